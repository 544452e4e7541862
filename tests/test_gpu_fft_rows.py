"""The largest transform that one workgroup holds (2^14 complex values in libcunaf,
2^13 in libcunad), where few rows go through two passes and many through one
workgroup each: row counts on both sides of the line, through the adjoint of several
value vectors, the forward transform of several curves and the compat bootstrap.
The same rows in a smaller call, on the other side of the line, and the direct sum;
tolerances are the library's parity bounds: rel L2 1e-5 (libcunaf), 1e-11 (libcunad,
the accurate filter's bound)."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

import cunfft_adjoint_amd as cu  # noqa: E402
import oracle  # noqa: E402
from tests._data import rel_l2, uniform_points  # noqa: E402

pytestmark = pytest.mark.gpu

NP = {"f": np.float32, "d": np.float64}
CP = {"f": torch.complex64, "d": torch.complex128}
TOL = {"f": 1e-5, "d": 1e-11}
LG = {"f": 14, "d": 13}
LINE = {"f": 100, "d": 32}


@pytest.fixture(scope="module", autouse=True)
def _gpu():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    torch.cuda.init()


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


@pytest.mark.parametrize("prec", ["f", "d"])
@pytest.mark.parametrize("extra", [0, 1])
def test_adjoint_rows(prec, extra):
    M, n, rows = 1 << LG[prec], 300, LINE[prec] + extra
    rng = np.random.default_rng(extra)
    x = rng.uniform(-0.5, 0.5, n).astype(NP[prec])
    y = rng.standard_normal((rows, n)).astype(NP[prec])
    plan = cu.NFFTPlan(dev(x), M, tile_log2=8)
    many = plan.adjoint_many(dev(y)).cpu().numpy()
    for r in (0, rows - 1):
        one = plan.adjoint(dev(y[r])).cpu().numpy()[0]
        assert rel_l2(many[r], one) < TOL[prec]
        assert rel_l2(one, oracle.ndft(x.astype(np.float64), y[r].astype(np.float64), M)) < TOL[prec]


@pytest.mark.parametrize("prec", ["f", "d"])
@pytest.mark.parametrize("curves", [1, 16, 17, 50, 51])
def test_forward_rows(prec, curves):
    """Two rows per curve."""
    M, n = 1 << LG[prec], 40
    rng = np.random.default_rng(curves)
    x = rng.uniform(-0.5, 0.5, curves * n).astype(NP[prec])
    g = dev(rng.standard_normal((curves, M)) + 1j * rng.standard_normal((curves, M))).to(CP[prec])
    f = cu.NFFTPlan(dev(x), M, offsets=np.arange(curves + 1, dtype=np.int32) * n).forward(g).cpu().numpy()
    for c in (0, curves - 1):
        ref = oracle.ndft_forward(x[c * n:(c + 1) * n].astype(np.float64),
                                  g[c].cpu().numpy().astype(np.complex128))
        assert rel_l2(f[c * n:(c + 1) * n], ref) < TOL[prec]


@pytest.mark.parametrize("prec", ["f", "d"])
def test_compat_bootstrap_rows(prec):
    ng, n, rows = 1 << (LG[prec] + 1), 700, LINE[prec] + 1
    x, y = uniform_points(n, ng, NP[prec])
    xd, yd = dev(x), dev(y)
    fp = cu.generate_filter_properties(xd, n, ng)
    many, few = (torch.empty((r, ng), dtype=CP[prec], device="cuda") for r in (rows, 5))
    cu.cunfft_adjoint_raw_async_bootstrap(xd, yd, many, n, ng, rows, fp, seed=9)
    cu.cunfft_adjoint_raw_async_bootstrap(xd, yd, few, n, ng, 5, fp, seed=9)
    assert rel_l2(few.cpu().numpy(), many[:5].cpu().numpy()) < TOL[prec]
    fp.free()
