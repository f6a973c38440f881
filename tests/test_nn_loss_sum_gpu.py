"""The loss sum of the squared-error kernel where its grid passes over the tensor more than once, in both access widths,
with most of the sum in the last pass or in one work-group's share: no share may be missing."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

GROUPS, THREADS = 1024, 256   # work-groups the kernel has at most, threads of one


@pytest.mark.parametrize("npos,c,used", [(300000, 8, 4), (300000, 8, 8), (60000, 5, 5), (530000, 1, 1), (70000, 24, 20), (2000, 8, 8)])
@pytest.mark.parametrize("part", ["last pass", "one group", "even"])
def test_every_share_is_in_the_sum(npos, c, used, part):
    """A sum of non-negative FP32 values of depth k is within k * 2^-24 of it: the squares, a thread's values, 8 levels
    of the work-group's tree and one addition a work-group."""
    import torch
    from mflbm import native
    lib, P = native.load(), (lambda t: C.c_void_p(t.data_ptr()))
    gen = torch.Generator(device="cuda")
    gen.manual_seed(npos + c)
    y = torch.randn((npos, c), generator=gen, device="cuda")
    v = 8 if c % 8 == 0 else 1
    n, sweep = npos * c, v * THREADS * GROUPS
    heavy = torch.zeros(n, dtype=torch.bool, device="cuda")
    if part == "last pass":
        heavy[(n - 1) // sweep * sweep:] = True
    elif part == "one group":
        heavy[min(n // (v * THREADS), GROUPS) // 2 * v * THREADS:][:v * THREADS] = True
    scale = torch.where(heavy.view(npos, c), 64.0, 1.0 if part == "even" else 1.0 / 16)
    y = (y * scale).to(torch.bfloat16)
    t = torch.zeros_like(y)
    g, loss = torch.empty_like(y), torch.zeros(1, device="cuda")
    sp = C.c_void_p(torch.cuda.current_stream().cuda_stream)
    assert lib.mflbm_nn_mse(P(y), P(t), P(g), P(loss), npos, c, used, 1.0, sp) == 0
    sq = y.double().square()
    sq[:, used:] = 0.0
    want = float(sq.sum())
    if part != "even":
        assert float(sq.view(-1)[heavy].sum()) > 0.5 * want
    depth = 1 + v * -(-n // sweep) + 8 + min(GROUPS, -(-n // (v * THREADS)))
    print(f"[loss sum] {npos} x {c} {part}: {float(loss) / want - 1:.2e}, bound {depth * 2.0 ** -24:.2e}", flush=True)
    assert abs(float(loss) - want) <= depth * 2.0 ** -24 * want
