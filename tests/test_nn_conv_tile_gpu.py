"""The tiled forward convolution at the edges of its tiles and of its dispatch: domains that are no multiple of a tile,
thinner than one, or one node wide; channel counts around every rule (8 .. 256 in, 1 .. 130 out), steps of 32 k that
span offsets; and the untiled kernel behind it (more than 256 input channels)."""
import ctypes as C
import os
import sys

import numpy as np
import pytest

sys.path.insert(0, os.path.join(os.path.dirname(os.path.abspath(__file__)), "..", "oracle"))
import nn_oracle as O  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cin,cout,shape,relu", [
    (8, 32, (2, 3, 9, 17), 1), (16, 20, (1, 5, 8, 7), 0), (24, 16, (1, 9, 1, 10), 1), (32, 1, (1, 4, 7, 9), 0),
    (32, 32, (2, 1, 1, 1), 1), (32, 70, (1, 5, 9, 8), 0), (40, 32, (1, 8, 9, 8), 1), (64, 30, (2, 64, 72, 65), 0),
    (56, 64, (1, 3, 8, 9), 1), (64, 66, (2, 33, 64, 72), 0), (72, 6, (1, 4, 4, 9), 0), (128, 64, (1, 5, 6, 8), 1),
    (136, 34, (1, 4, 5, 4), 0), (256, 130, (1, 5, 4, 3), 1), (264, 9, (1, 3, 2, 5), 0)])
def test_conv_forward_at_tile_edges(cin, cout, shape, relu):
    """FP32 sums of BF16 products rounded once: within one BF16 step (2^-7 of the largest value) of the oracle, as for
    the other shapes; large domains are compared on their last planes."""
    import torch
    from mflbm import native
    lib = native.load()
    P = lambda t: C.c_void_p(t.data_ptr())
    rng = np.random.default_rng(cin + cout)
    x = O.to_bf16(rng.standard_normal(shape + (cin,)).astype(np.float32))
    w = rng.standard_normal((cout, 27, cin)).astype(np.float32) * np.float32(np.sqrt(2.0 / (27 * cin)))
    b = (rng.standard_normal(cout) * 0.1).astype(np.float32)
    bf = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to("cuda", torch.bfloat16)
    gx, gb = bf(x), torch.from_numpy(b).cuda()
    wf = torch.zeros((cout, (27 * cin + 31) // 32 * 32), dtype=torch.bfloat16, device="cuda")
    wf[:, :27 * cin] = bf(w.reshape(cout, -1))
    y = torch.full(shape + (cout,), 7.0, dtype=torch.bfloat16, device="cuda")
    sp = C.c_void_p(torch.cuda.current_stream().cuda_stream)
    assert lib.mflbm_nn_conv3d_fwd(P(gx), P(wf), P(gb), P(y), *shape, cin, cout, relu, sp) == 0
    torch.cuda.synchronize()
    got = y.float().cpu().numpy()
    if shape[1] > 16:   # the oracle on the last planes, with the plane below them as halo
        ref = O.to_bf16(O.conv3d(x[:, -4:], O.to_bf16(w), b, bool(relu)))[:, 1:]
        got = got[:, -3:]
    else:
        ref = O.to_bf16(O.conv3d(x, O.to_bf16(w), b, bool(relu)))
    assert np.abs(got - ref).max() <= 2 ** -7 * np.abs(ref).max()


def test_conv_forward_into_an_unaligned_output():
    """An output that starts 2 bytes past an 8-byte boundary takes 2-byte stores: the same values, nothing around them."""
    import torch
    from mflbm import native
    lib = native.load()
    P = lambda t: C.c_void_p(t.data_ptr())
    gen = torch.Generator(device="cuda")
    gen.manual_seed(3)
    shape, cin, cout = (1, 5, 6, 9), 32, 8
    x = torch.randn(shape + (cin,), generator=gen, device="cuda").to(torch.bfloat16)
    wf = (torch.randn((cout, 27 * cin), generator=gen, device="cuda") * 0.05).to(torch.bfloat16)
    n = int(np.prod(shape)) * cout
    a, b = torch.zeros(n, dtype=torch.bfloat16, device="cuda"), torch.zeros(n + 8, dtype=torch.bfloat16, device="cuda")
    sp = C.c_void_p(torch.cuda.current_stream().cuda_stream)
    assert lib.mflbm_nn_conv3d_fwd(P(x), P(wf), None, P(a), *shape, cin, cout, 0, sp) == 0
    assert lib.mflbm_nn_conv3d_fwd(P(x), P(wf), None, P(b[1:]), *shape, cin, cout, 0, sp) == 0
    torch.cuda.synchronize()
    assert torch.equal(a, b[1:1 + n]) and float(b[0]) == 0.0 and float(b[1 + n:].abs().sum()) == 0.0
