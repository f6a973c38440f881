"""Forward convolutions on domains that fill little of a spatial tile: the thin and the full domain take different
kernels with one order of sums, and a thin domain must not pay for the tile's missing planes."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _setup(cin, cout, seed):
    import torch
    from mflbm import native
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    wf = torch.zeros((cout, (27 * cin + 31) // 32 * 32), dtype=torch.bfloat16, device="cuda")
    wf[:, :27 * cin] = (torch.randn((cout, 27 * cin), generator=gen, device="cuda") * 0.05).to(torch.bfloat16)
    b = torch.randn(cout, generator=gen, device="cuda")
    return torch, native.load(), gen, wf, b, C.c_void_p(torch.cuda.current_stream().cuda_stream)


def _ptr(t):
    return C.c_void_p(t.data_ptr())


@pytest.mark.parametrize("cin,cout", [(8, 8), (16, 32), (32, 32), (32, 64), (64, 32), (64, 64), (128, 96), (256, 40)])
@pytest.mark.parametrize("axis", [0, 1, 2])
def test_thin_domain_equals_the_full_one_bit_for_bit(cin, cout, axis):
    """A domain one node thick is the middle plane of a 9-node one whose other planes hold zeros: equal bits."""
    torch, lib, gen, wf, b, sp = _setup(cin, cout, cin + cout)
    shape = [40, 40, 40]
    shape[axis] = 1
    x = torch.randn((2, *shape, cin), generator=gen, device="cuda").to(torch.bfloat16)
    full = list(shape)
    full[axis] = 9
    xf = torch.zeros((2, *full, cin), dtype=torch.bfloat16, device="cuda")
    xf.narrow(1 + axis, 4, 1).copy_(x)
    y = torch.empty((2, *shape, cout), dtype=torch.bfloat16, device="cuda")
    yf = torch.empty((2, *full, cout), dtype=torch.bfloat16, device="cuda")
    assert lib.mflbm_nn_conv3d_fwd(_ptr(x), _ptr(wf), _ptr(b), _ptr(y), 2, *shape, cin, cout, 0, sp) == 0
    assert lib.mflbm_nn_conv3d_fwd(_ptr(xf), _ptr(wf), _ptr(b), _ptr(yf), 2, *full, cin, cout, 0, sp) == 0
    torch.cuda.synchronize()
    assert torch.equal(y, yf.narrow(1 + axis, 4, 1))


def test_a_quarter_of_the_planes_takes_less_than_their_time():
    """4 x d x 64 x 64, 256 -> 256: d = 1 has a quarter of the work of d = 4 and must take less than 3/4 of its time."""
    torch, lib, gen, wf, b, sp = _setup(256, 256, 1)
    us = {}
    for d in (4, 1):
        x = torch.randn((4, d, 64, 64, 256), generator=gen, device="cuda").to(torch.bfloat16)
        y = torch.empty_like(x)
        best = 1e9
        for _ in range(5):
            t0, t1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            t0.record()
            for _ in range(5):
                assert lib.mflbm_nn_conv3d_fwd(_ptr(x), _ptr(wf), _ptr(b), _ptr(y), 4, d, 64, 64, 256, 256, 1, sp) == 0
            t1.record()
            t1.synchronize()
            best = min(best, t0.elapsed_time(t1))
        us[d] = best * 200
    print(us, flush=True)
    assert us[1] < 0.75 * us[4]
