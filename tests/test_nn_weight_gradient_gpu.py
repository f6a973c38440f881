"""The staged weight gradient at the edges of its tiles: rows shorter than, equal to and no multiple of a 32-position
tile, domains one node thin, channel counts that are no multiple of 16, several chunks, both channel groupings, and a
plane too large for a 2 GiB window (64-bit addressing)."""
import ctypes as C
import os
import sys

import numpy as np
import pytest

sys.path.insert(0, os.path.join(os.path.dirname(os.path.abspath(__file__)), "..", "oracle"))
import nn_oracle as O  # noqa: E402

pytestmark = pytest.mark.gpu


def _run(x, dy, cin, cout, shape):
    import torch
    from mflbm import native
    lib = native.load()
    P = lambda t: C.c_void_p(t.data_ptr())
    dw, db = torch.zeros((cout, 27 * cin), device="cuda"), torch.zeros(cout, device="cuda")
    need = int(lib.mflbm_nn_conv3d_dw_work(*shape, cin, cout))
    work = torch.empty(need, device="cuda")
    sp = C.c_void_p(torch.cuda.current_stream().cuda_stream)
    assert lib.mflbm_nn_conv3d_dw_ordered(P(x), P(dy), P(dw), P(db), P(work), need, *shape, cin, cout, sp) == 0
    torch.cuda.synchronize()
    return dw, db


@pytest.mark.parametrize("cin,cout,shape", [(8, 8, (3, 4, 3, 8)), (24, 40, (2, 1, 7, 24)), (16, 24, (1, 5, 1, 40)),
                                            (40, 16, (2, 3, 1, 8)), (8, 48, (1, 1, 1, 8)), (32, 32, (1, 9, 16, 32)),
                                            (64, 160, (1, 17, 32, 32))])
def test_weight_gradient_at_tile_edges(cin, cout, shape):
    """FP32 sums of BF16 products against the oracle's (another order): |error| <= 2e-3 of the largest gradient, as for
    the other shapes."""
    import torch
    rng = np.random.default_rng(cin + cout)
    x = O.to_bf16(rng.standard_normal(shape + (cin,)).astype(np.float32))
    g = O.to_bf16(rng.standard_normal(shape + (cout,)).astype(np.float32))
    bf = lambda a: torch.from_numpy(a).to("cuda", torch.bfloat16)
    dw, db = _run(bf(x), bf(g), cin, cout, shape)
    _, rgw, rgb = O.conv3d_grads(x, np.zeros((cout, 27, cin), np.float32), g)
    np.testing.assert_allclose(dw.cpu().numpy().reshape(cout, 27, cin), rgw, rtol=2e-3, atol=2e-3 * np.abs(rgw).max())
    np.testing.assert_allclose(db.cpu().numpy(), rgb, rtol=2e-3, atol=2e-3 * np.abs(rgb).max())


def test_weight_gradient_on_a_plane_beyond_the_window():
    """4096 x 4096 x 32 channels: 64-bit addressing.  128 tile sums and 4096 chunk sums in FP32: |error| <= 4300 * 2^-24
    of the sum of magnitudes."""
    import torch
    cin, cout, shape = 32, 8, (1, 1, 4096, 4096)
    gen = torch.Generator(device="cuda")
    gen.manual_seed(5)
    x = torch.randn(shape + (cin,), generator=gen, device="cuda", dtype=torch.bfloat16)
    g = torch.randn(shape + (cout,), generator=gen, device="cuda", dtype=torch.bfloat16)
    dw, _ = _run(x, g, cin, cout, shape)
    dw = dw.reshape(cout, 27, cin).double()
    assert torch.equal(dw[:, :9], torch.zeros_like(dw[:, :9])) and torch.equal(dw[:, 18:], torch.zeros_like(dw[:, 18:]))
    xd, gd = x[0, 0].double(), g[0, 0].double()
    for dyy, dx in ((-1, -1), (0, 0), (1, 1), (1, -1)):
        ys, yt = slice(max(0, dyy), 4096 + min(0, dyy)), slice(max(0, -dyy), 4096 + min(0, -dyy))
        xs, xt = slice(max(0, dx), 4096 + min(0, dx)), slice(max(0, -dx), 4096 + min(0, -dx))
        a, b = gd[yt, xt].reshape(-1, cout), xd[ys, xs].reshape(-1, cin)
        ref, mag = a.T @ b, a.abs().T @ b.abs()
        assert ((dw[:, 9 + 3 * (dyy + 1) + dx + 1] - ref).abs() <= 4300 * 2.0 ** -24 * mag).all()
