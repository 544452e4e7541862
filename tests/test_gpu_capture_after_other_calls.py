"""Calls that can be captured once another call of the plan has run, because all
they need is there by then."""
import subprocess
import sys

import numpy as np
import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu

FUSED = """
import numpy as np, torch
import cunfft_adjoint_amd as cu
dt, cdt, prec = {dt}
rng = np.random.default_rng(2)
n, M = 200, {M}
x = torch.from_numpy(rng.uniform(-0.5, 0.5, n).astype(dt)).cuda()
y = torch.from_numpy(rng.standard_normal(n).astype(dt)).cuda()
plan = cu.NFFTPlan(x, M)
s = torch.cuda.Stream()
out = torch.empty((1, M), dtype=cdt, device="cuda")
plan.backward(y, torch.ones((1, M), dtype=cdt, device="cuda"))
torch.cuda.synchronize()
g = cu.capture(lambda: plan.adjoint(y, out=out, stream=s), s, prec)
for _ in range(3):
    out.zero_()
    torch.cuda.synchronize()
    g.launch(s)
    s.synchronize()
    got = out.cpu().numpy()
    assert np.array_equal(got, plan.adjoint(y).cpu().numpy())
print("done")
"""


@pytest.fixture(scope="module", autouse=True)
def _gpu():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")


@pytest.mark.parametrize("dt", ["np.float32, torch.complex64, 'f'", "np.float64, torch.complex128, 'd'"])
@pytest.mark.parametrize("M", [1 << 8, 1 << 12])
def test_fused_adjoint_after_a_backward(dt, M):
    """In a process of its own: twiddle tables are kept per process."""
    r = subprocess.run([sys.executable, "-c", FUSED.format(dt=dt, M=M)], capture_output=True,
                       text=True, timeout=100)
    assert r.returncode == 0 and "done" in r.stdout, r.stdout + r.stderr


@pytest.mark.parametrize("prec", ["f", "d"])
@pytest.mark.parametrize("lens", [[3000], [700, 0, 1900]])
def test_forward_after_a_backward(prec, lens):
    """Then there is one grid per curve, and the real and the imaginary part follow each
    other: the same sums as in one pass, so rel L2 1e-6 (libcunaf), 1e-13 (libcunad)
    of rounding."""
    import cunfft_adjoint_amd as cu
    M, offs = 1 << 11, np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    rt, ct = (torch.float32, torch.complex64) if prec == "f" else (torch.float64, torch.complex128)
    rng = np.random.default_rng(4)
    x = torch.from_numpy(rng.uniform(-0.5, 0.5, offs[-1])).to(rt).cuda()
    h = rng.standard_normal((len(lens), M)) + 1j * rng.standard_normal((len(lens), M))
    h = torch.from_numpy(h).to(ct).cuda()
    plan = cu.NFFTPlan(x, M, offsets=offs, tile_log2=8)
    s = torch.cuda.Stream()
    out = torch.empty(int(offs[-1]), dtype=ct, device="cuda")
    plan.backward(None, h)
    torch.cuda.synchronize()
    g = cu.capture(lambda: plan.forward(h, out=out, stream=s), s, prec)
    for _ in range(3):
        out.zero_()
        torch.cuda.synchronize()
        g.launch(s)
        s.synchronize()
        got = out.clone()
        want = plan.forward(h)
        assert torch.linalg.norm(got - want) <= (1e-6 if prec == "f" else 1e-13) * torch.linalg.norm(want)
