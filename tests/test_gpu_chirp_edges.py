"""The chirp transform where it changes form: lengths whose convolution is the
last to fit one workgroup (2^14 values in libcunaf, 2^13 in libcunad) and the
first of the three-launch form, even (paired) and odd grids, the smallest ones,
several batch rows.  The compat transform and its bootstrap against the CPU
oracle, the complex FFT against numpy in 64 bits; tolerances are the library's
parity bounds: rel L2 1e-5 (libcunaf), 1e-12 (libcunad)."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

import oracle  # noqa: E402
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


@pytest.mark.parametrize("prec", ["f", "d"])
@pytest.mark.parametrize("ng", [1, 2, 3, 6, 7, 4095, 4097, 8190, 8191, 8193, 8194, 16382, 16386, 65538, 65537])
def test_compat_vs_oracle(prec, ng):
    n = max(1, min(3000, ng // 2))
    x, y = uniform_points(n, ng, NP[prec])
    xd, yd = dev(x), dev(y)
    fp = cu.generate_filter_properties(xd, n, ng)
    out = torch.empty(ng, dtype=CP[prec], device="cuda")
    cu.cunfft_adjoint_raw_async(xd, yd, out, n, ng, fp)
    assert rel_l2(out.cpu().numpy(), oracle.compat_adjoint(x, y, ng, prec == "d")) < TOL[prec]
    boot = torch.empty((3, ng), dtype=CP[prec], device="cuda")
    cu.cunfft_adjoint_raw_async_bootstrap(xd, yd, boot, n, ng, 3, fp, seed=5)
    ref = oracle.compat_adjoint_bootstrap(x, y, ng, 3, 5, prec == "d").reshape(3, ng)
    assert rel_l2(boot.cpu().numpy(), ref) < TOL[prec]
    fp.free()


@pytest.mark.parametrize("prec", ["f", "d"])
@pytest.mark.parametrize("n", [1, 3, 12, 4095, 4097, 8191, 8193, 40001])
@pytest.mark.parametrize("sign", [1, -1])
def test_complex_fft_vs_numpy(prec, n, sign):
    rng = np.random.default_rng(n)
    z = rng.standard_normal((2, n)) + 1j * rng.standard_normal((2, n))
    d = dev(z).to(CP[prec])
    got = cu.fft(d, sign).cpu().numpy()
    z = dev(z).to(CP[prec]).cpu().numpy().astype(np.complex128)
    ref = np.fft.ifft(z, axis=1) * n if sign > 0 else np.fft.fft(z, axis=1)
    assert rel_l2(got, ref) < TOL[prec]
