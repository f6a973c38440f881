"""The row records (csrc/layout.h) against the dense map over every form they replace it in: row lengths around the
16-node groups, folded y or z, unfolded periodic axes, open faces, tiles that split the rows' order, random and packed
walls (tests/native/row_records_check.cpp, built with the sanitizers)."""
import os
import shutil
import subprocess

import numpy as np
import pytest

REPO = os.path.abspath(os.path.join(os.path.dirname(__file__), ".."))


@pytest.fixture(scope="module")
def checker(tmp_path_factory):
    cxx = shutil.which("g++")
    if cxx is None:
        pytest.skip("g++ not available")
    exe = str(tmp_path_factory.mktemp("rows") / "row_records_check")
    r = subprocess.run([cxx, "-std=c++17", "-O1", "-g", "-fsanitize=address,undefined", "-fno-sanitize-recover=all", "-I",
                        os.path.join(REPO, "mf-lbm_amd", "csrc"), os.path.join(REPO, "tests", "native", "row_records_check.cpp"),
                        "-o", exe], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    return exe


# open_z, jper, kper, fold_y, fold_z
KINDS = [(1, 0, 0, 0, 0), (0, 0, 1, 0, 1), (0, 1, 0, 1, 0), (0, 1, 1, 0, 0), (0, 0, 0, 0, 0)]


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("shape,tile,solid", [((3, 3, 12), 32, 0.0), ((16, 5, 9), 4, 0.4), ((17, 33, 10), 8, 0.7),
                                              ((31, 12, 14), 1, 0.5), ((33, 40, 11), 64, 0.95), ((64, 7, 10), 32, 0.3)])
def test_row_records_equal_the_dense_map(checker, tmp_path, kind, shape, tile, solid):
    nx, ny, nz = shape
    rng = np.random.default_rng(nx * 100 + ny)
    w = np.ones((nz + 4, ny + 4, nx + 4), np.int8)
    w[2:-2, 2:-2, 2:-2] = rng.random((nz, ny, nx)) < solid
    open_z, jper, kper, fy, fz = kind
    if kper or open_z:   # the halo of a periodic or open face is not solid everywhere
        w[:2, 2:-2, 2:-2] = w[-4:-2, 2:-2, 2:-2]
        w[-2:, 2:-2, 2:-2] = w[2:4, 2:-2, 2:-2]
    if jper:
        w[:, :2] = w[:, -4:-2]
        w[:, -2:] = w[:, 2:4]
    path = str(tmp_path / "walls.bin")
    with open(path, "wb") as fh:
        fh.write(np.array([nx, ny, nz, *kind, tile], np.int32).tobytes())
        fh.write(w.tobytes())
    r = subprocess.run([checker, path], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout + r.stderr[-3000:]
    assert r.stdout.startswith("ok")
