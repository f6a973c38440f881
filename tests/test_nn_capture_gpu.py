"""The network's kernels under graph capture, each kernel's first launch of the process among them (the forward tiles ask
for more than 64 KB of LDS): every replay, with new inputs and other work between, equals the eager call."""
import ctypes as C
import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu

CHILD = """
import ctypes as C, sys
import torch
from mflbm import native
lib, P = native.load(), (lambda t: C.c_void_p(t.data_ptr()))
S = lambda: C.c_void_p(torch.cuda.current_stream().cuda_stream)
gen = torch.Generator(device="cuda"); gen.manual_seed(1)
R = lambda *s: torch.randn(s, generator=gen, device="cuda").to(torch.bfloat16)
calls = []
for cin, cout, shape in [(8, 32, (1, 8, 8, 16)), (32, 8, (1, 8, 8, 16)), (32, 32, (2, 8, 8, 16)), (32, 64, (2, 8, 8, 16)),
                         (64, 32, (1, 64, 64, 64)), (64, 64, (1, 32, 64, 64)), (64, 64, (1, 8, 8, 16)), (128, 64, (1, 8, 8, 8)),
                         (256, 64, (1, 4, 4, 8)), (264, 16, (1, 2, 3, 8)), (64, 64, (64, 1, 1, 8))]:
    wf = torch.zeros((cout, (27 * cin + 31) // 32 * 32), dtype=torch.bfloat16, device="cuda")
    wf[:, :27 * cin] = (torch.randn((cout, 27 * cin), generator=gen, device="cuda") * 0.05).to(torch.bfloat16)
    x, y = R(*shape, cin), torch.empty(shape + (cout,), dtype=torch.bfloat16, device="cuda")
    calls.append((x, y, lambda x=x, y=y, wf=wf, a=(*shape, cin, cout): lib.mflbm_nn_conv3d_fwd(P(x), P(wf), None, P(y), *a, 1, S())))
x, dy = R(1, 8, 16, 32, 32), R(1, 8, 16, 32, 32)
dw, db = torch.zeros((32, 27 * 32), device="cuda"), torch.zeros(32, device="cuda")
def grad():
    dw.zero_(); db.zero_()
    return lib.mflbm_nn_conv3d_dw_ordered_noalloc(P(x), P(dy), P(dw), P(db), 1, 8, 16, 32, 32, 32, S())
assert grad() == 0   # (its scratch array is looked up on the first call)
calls.append((x, dw, grad))
g = torch.cuda.CUDAGraph()
with torch.cuda.graph(g):
    rcs = [f() for _, _, f in calls]
assert rcs == [0] * len(calls), rcs
for k in range(4):
    for x, _, _ in calls:
        x.copy_(R(*x.shape))
    g.replay()
    torch.cuda.synchronize()
    got = [y.clone() for _, y, _ in calls]
    float(R(1000, 1000).float().sum())
    for (_, y, f), h in zip(calls, got):
        y.fill_(3.0)
        assert f() == 0
        torch.cuda.synchronize()
        assert torch.equal(y, h), k
print("replays equal", flush=True)
"""


def test_replays_equal_the_eager_calls():
    pkg = os.path.join(os.path.dirname(os.path.abspath(__file__)), "..", "mf-lbm_amd")
    r = subprocess.run([sys.executable, "-u", "-c", CHILD], capture_output=True, text=True, timeout=100,
                       env=dict(os.environ, PYTHONPATH=pkg + os.pathsep + os.environ.get("PYTHONPATH", "")))
    assert r.returncode == 0, r.stdout[-500:] + r.stderr[-2000:]
    assert "replays equal" in r.stdout
