"""The chirp transform at the largest length one workgroup holds (2^14 in libcunaf,
2^13 in libcunad), where few rows go through the three passes and many through one
workgroup each: row counts on both sides of the line, lengths at both ends of that
range.  The complex FFT against numpy in 64 bits and the compat bootstrap against
the same replicates on the other side of the line; tolerances are the library's
parity bounds: rel L2 1e-5 (libcunaf), 1e-12 (libcunad)."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

import cunfft_adjoint_amd as cu  # noqa: E402
from tests._data import rel_l2, uniform_points  # noqa: E402

pytestmark = pytest.mark.gpu

NP = {"f": np.float32, "d": np.float64}
CP = {"f": torch.complex64, "d": torch.complex128}
TOL = {"f": 1e-5, "d": 1e-12}


@pytest.fixture(scope="module", autouse=True)
def _gpu():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    torch.cuda.init()


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


@pytest.mark.parametrize("prec,n", [("f", 4099), ("f", 8191), ("d", 2050), ("d", 4095)])
@pytest.mark.parametrize("rows", [1, 31, 32, 33, 64, 65])
def test_complex_fft_rows(prec, n, rows):
    rng = np.random.default_rng(n + rows)
    z = rng.standard_normal((rows, n)) + 1j * rng.standard_normal((rows, n))
    d = dev(z).to(CP[prec])
    z = d.cpu().numpy().astype(np.complex128)
    assert rel_l2(cu.fft(d, 1).cpu().numpy(), np.fft.ifft(z, axis=1) * n) < TOL[prec]


@pytest.mark.parametrize("prec,ng", [("f", 5001), ("f", 13482), ("d", 2501), ("d", 8180)])
def test_compat_bootstrap_rows(prec, ng):
    n = 700
    x, y = uniform_points(n, ng, NP[prec])
    xd, yd = dev(x), dev(y)
    fp = cu.generate_filter_properties(xd, n, ng)
    many, few = (torch.empty((r, ng), dtype=CP[prec], device="cuda") for r in (70, 20))
    cu.cunfft_adjoint_raw_async_bootstrap(xd, yd, many, n, ng, 70, fp, seed=9)
    cu.cunfft_adjoint_raw_async_bootstrap(xd, yd, few, n, ng, 20, fp, seed=9)
    assert rel_l2(few.cpu().numpy(), many[:20].cpu().numpy()) < TOL[prec]
    fp.free()
