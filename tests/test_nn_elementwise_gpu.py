"""The elementwise kernels of the network in both access widths: lengths and channel counts that are and are not
multiples of 8, tensors that start off a 16-byte boundary, one value and more than one pass of the grid, against torch
on the same BF16 values (one rounding, the same operations: equal bits)."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _lib():
    import torch
    from mflbm import native
    return torch, native.load(), lambda t: C.c_void_p(t.data_ptr()), C.c_void_p(torch.cuda.current_stream().cuda_stream)


def _bf(torch, shape, seed, off=0):
    """A tensor of this shape whose storage starts `off` values past an aligned address."""
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    n = int(np.prod(shape))
    return torch.randn(n + off, generator=g, device="cuda").to(torch.bfloat16)[off:].view(shape)


@pytest.mark.parametrize("n,off", [(1, 0), (7, 0), (8, 0), (2048, 0), (2049, 0), (4096, 3), (800008, 0)])
def test_add_and_relu_gradient(n, off):
    torch, lib, P, sp = _lib()
    a, b = _bf(torch, (n,), 1, off), _bf(torch, (n,), 2, off)
    y = torch.empty(n + off, dtype=torch.bfloat16, device="cuda")[off:]
    assert lib.mflbm_nn_add(P(a), P(b), P(y), n, sp) == 0
    assert torch.equal(y, (a.float() + b.float()).to(torch.bfloat16))
    g = a.clone() if off == 0 else _bf(torch, (n,), 1, off)
    want = torch.where(b.float() > 0, g, torch.zeros_like(g))
    assert lib.mflbm_nn_relu_bwd(P(g), P(b), n, sp) == 0
    assert torch.equal(g, want)


@pytest.mark.parametrize("c,off", [(1, 0), (6, 0), (8, 0), (24, 0), (8, 1)])
def test_pooling_and_upsampling(c, off):
    torch, lib, P, sp = _lib()
    n, d, h, w = 2, 4, 6, 10
    x = _bf(torch, (n, d, h, w, c), 3, off)
    q = _bf(torch, (n, d // 2, h // 2, w // 2, c), 4, off)
    parts = x.float().view(n, d // 2, 2, h // 2, 2, w // 2, 2, c).permute(2, 4, 6, 0, 1, 3, 5, 7).reshape(8, *q.shape)
    s = torch.zeros_like(parts[0])
    for o in range(8):
        s = s + parts[o]
    rep = q.repeat_interleave(2, 1).repeat_interleave(2, 2).repeat_interleave(2, 3)
    coarse, fine = torch.empty_like(q), torch.empty_like(x)
    assert lib.mflbm_nn_pool2(P(x), P(coarse), n, d, h, w, c, 0, sp) == 0
    assert torch.equal(coarse, (0.125 * s).to(torch.bfloat16))
    assert lib.mflbm_nn_up2(P(x), P(coarse), n, d, h, w, c, 1, sp) == 0
    assert torch.equal(coarse, s.to(torch.bfloat16))
    assert lib.mflbm_nn_pool2(P(q), P(fine), n, d, h, w, c, 1, sp) == 0
    assert torch.equal(fine, (0.125 * rep.float()).to(torch.bfloat16))
    assert lib.mflbm_nn_up2(P(q), P(fine), n, d, h, w, c, 0, sp) == 0
    assert torch.equal(fine, rep)


@pytest.mark.parametrize("npos,c,used,off", [(1, 8, 4, 0), (100, 5, 3, 0), (300000, 8, 4, 0), (3000, 16, 16, 1)])
def test_squared_error(npos, c, used, off):
    """Gradient bits as torch's; the loss, a sum of npos * used squares in FP32 in any order: within npos * c * 2^-24."""
    torch, lib, P, sp = _lib()
    y, t = _bf(torch, (npos, c), 5, off), _bf(torch, (npos, c), 6, off)
    g, loss = torch.empty_like(y), torch.zeros(1, device="cuda")
    scale = float(np.float32(1.0 / npos))
    assert lib.mflbm_nn_mse(P(y), P(t), P(g), P(loss), npos, c, used, scale, sp) == 0
    d = y.float() - t.float()
    d[:, used:] = 0.0
    assert torch.equal(g, (torch.tensor(2.0 * scale, device="cuda") * d).to(torch.bfloat16))
    want = float(d.double().square().sum())
    assert abs(float(loss) - want) <= npos * c * 2.0 ** -24 * want
