"""Convolutions whose BF16 tensors start 2, 4, 6 and 8 bytes past a 16-byte boundary: the same values as on one."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _shifted(torch, t, off):
    """A copy of t whose storage starts ``off`` values past an aligned address."""
    a = torch.zeros(t.numel() + off + 8, dtype=t.dtype, device="cuda")
    assert a.data_ptr() % 16 == 0
    b = a[off:off + t.numel()].view(t.shape)
    b.copy_(t)
    return b


@pytest.mark.parametrize("off", [1, 2, 3, 4])
@pytest.mark.parametrize("cin,cout", [(8, 8), (24, 40), (64, 64)])
def test_shifted_inputs_give_the_same_values(cin, cout, off):
    import torch
    from mflbm import native
    lib, P = native.load(), (lambda t: C.c_void_p(t.data_ptr()))
    sp = C.c_void_p(torch.cuda.current_stream().cuda_stream)
    gen = torch.Generator(device="cuda")
    gen.manual_seed(cin)
    shape = (2, 5, 9, 16)
    x = torch.randn(shape + (cin,), generator=gen, device="cuda").to(torch.bfloat16)
    dy = torch.randn(shape + (cout,), generator=gen, device="cuda").to(torch.bfloat16)
    wf = torch.zeros((cout, (27 * cin + 31) // 32 * 32), dtype=torch.bfloat16, device="cuda")
    wf[:, :27 * cin] = (torch.randn((cout, 27 * cin), generator=gen, device="cuda") * 0.05).to(torch.bfloat16)
    need = int(lib.mflbm_nn_conv3d_dw_work(*shape, cin, cout))

    def both(x, dy, wf):
        y = torch.empty(shape + (cout,), dtype=torch.bfloat16, device="cuda")
        dw, db, work = torch.zeros((cout, 27 * cin), device="cuda"), torch.zeros(cout, device="cuda"), torch.empty(need, device="cuda")
        assert lib.mflbm_nn_conv3d_fwd(P(x), P(wf), None, P(y), *shape, cin, cout, 0, sp) == 0
        assert lib.mflbm_nn_conv3d_dw_ordered(P(x), P(dy), P(dw), P(db), P(work), need, *shape, cin, cout, sp) == 0
        torch.cuda.synchronize()
        return y, dw, db

    print(f"[alignment] {cin} -> {cout}, {2 * off} bytes", flush=True)
    want = both(x, dy, wf)
    for args in ((_shifted(torch, x, off), dy, wf), (x, _shifted(torch, dy, off), wf), (x, dy, _shifted(torch, wf, off))):
        for a, b in zip(both(*args), want):
            assert torch.equal(a, b)
