"""Forward convolutions over so many small images that one work-group a tile would need 2^32 threads, more than a launch
has: the whole batch is computed, its last image as a batch of one."""
import ctypes as C

import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape,cout", [((8400000, 1, 1, 1), 8), ((8388607, 4, 8, 8), 1)])
def test_batch_beyond_a_launch_of_tiles(shape, cout):
    import torch
    from mflbm import native
    lib, P, cin = native.load(), (lambda t: C.c_void_p(t.data_ptr())), 8
    n, d, h, w = shape
    if torch.cuda.mem_get_info()[0] < 2 * n * d * h * w * (cin + cout) + (1 << 30):
        pytest.skip("not enough device memory")
    gen = torch.Generator(device="cuda")
    gen.manual_seed(2)
    wf = torch.zeros((cout, 224), dtype=torch.bfloat16, device="cuda")
    wf[:, :216] = torch.randn((cout, 216), generator=gen, device="cuda").to(torch.bfloat16)
    sp = C.c_void_p(torch.cuda.current_stream().cuda_stream)
    x = torch.zeros(shape + (cin,), dtype=torch.bfloat16, device="cuda")
    y = torch.full(shape + (cout,), 7.0, dtype=torch.bfloat16, device="cuda")
    one = torch.randn((1, d, h, w, cin), generator=gen, device="cuda").to(torch.bfloat16)
    want = torch.empty((1, d, h, w, cout), dtype=torch.bfloat16, device="cuda")
    for k in (0, n // 2, n - 1):
        x[k] = one[0]
    print(f"[many images] {shape} {cout}", flush=True)
    assert lib.mflbm_nn_conv3d_fwd(P(one), P(wf), None, P(want), 1, d, h, w, cin, cout, 0, sp) == 0
    assert lib.mflbm_nn_conv3d_fwd(P(x), P(wf), None, P(y), n, d, h, w, cin, cout, 0, sp) == 0
    torch.cuda.synchronize()
    assert float(want.abs().sum()) > 0
    for k in (0, n // 2, n - 1):
        assert torch.equal(y[k], want[0])
    assert float(y[1].abs().max()) == 0.0 and float(y[n - 2].abs().max()) == 0.0


def test_weight_gradient_beyond_one_launch():
    """8192 x 8192 channels over 128 chunks of positions: 2^24 work-groups.  One position in the first chunk and one in
    the last are not zero, so the centre offset's gradient is the sum of two exact products, rounded once."""
    import torch
    from mflbm import native
    lib, P, c, shape = native.load(), (lambda t: C.c_void_p(t.data_ptr())), 8192, (128, 1, 64, 64)
    if torch.cuda.mem_get_info()[0] < 40 << 30:
        pytest.skip("not enough device memory")
    gen = torch.Generator(device="cuda")
    gen.manual_seed(4)
    x, dy = (torch.zeros(shape + (c,), dtype=torch.bfloat16, device="cuda") for _ in range(2))
    want = torch.zeros((c, c), device="cuda")
    for at in ((0, 0, 3, 7), (127, 0, 63, 63)):
        a, b = (torch.randn(c, generator=gen, device="cuda").to(torch.bfloat16) for _ in range(2))
        x[at], dy[at] = a, b
        want += b.float()[:, None] * a.float()[None, :]
    dw = torch.zeros((c, 27, c), device="cuda")
    sp = C.c_void_p(torch.cuda.current_stream().cuda_stream)
    print("[weight gradient beyond one launch]", flush=True)
    assert lib.mflbm_nn_conv3d_dw(P(x), P(dy), P(dw), None, *shape, c, c, sp) == 0
    torch.cuda.synchronize()
    assert torch.equal(dw[:, 13], want)
    dw[:, 13] = 0
    assert float(dw.abs().max()) == 0.0
