"""Type-2 path (forward transform and gradients) at the sizes where it changes
form: the smallest grids, one-tile grids, the last single-workgroup inverse FFT
(2^13 complex values) and the first two-pass one, sigma = 4 (half of the
spectrum out of band), several tiles per gather workgroup (few points per tile)
and one (many), ragged curves with an empty one.  Against the FP64 direct sums;
tolerances are those of the library's accuracy contract: rel L2 1e-5 (libcunaf)
and 1e-11 (libcunad)."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

import oracle  # noqa: E402
import cunfft_adjoint_amd as cu  # noqa: E402
from tests._data import rel_l2  # noqa: E402

pytestmark = pytest.mark.gpu

NP = {"f": np.float32, "d": np.float64}
CP = {"f": np.complex64, "d": np.complex128}
TOL = {"f": 1e-5, "d": 1e-11}


@pytest.fixture(scope="module", autouse=True)
def _gpu():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    torch.cuda.init()


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


@pytest.mark.parametrize("prec", ["f", "d"])
@pytest.mark.parametrize("M,sigma,lens", [
    (2, 2, [1, 3]),
    (8, 2, [5, 0, 70]),
    (128, 2, [400]),
    (1 << 10, 4, [300, 0, 1, 2000]),
    (1 << 12, 4, [1500]),
    (1 << 13, 2, [700, 1300, 90]),
    (1 << 14, 2, [40, 900]),
    (1 << 15, 4, [130]),
])
def test_forward_and_backward_vs_direct_sums(prec, M, sigma, lens):
    rng = np.random.default_rng(M + sigma)
    offs = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    x = rng.uniform(-0.5, 0.5, offs[-1]).astype(NP[prec])
    y = rng.standard_normal(offs[-1]).astype(NP[prec])
    g = (rng.standard_normal((len(lens), M)) + 1j * rng.standard_normal((len(lens), M))).astype(CP[prec])
    plan = cu.NFFTPlan(dev(x), M, offsets=offs, sigma=sigma)
    f = plan.forward(dev(g)).cpu().numpy()
    dy, dx = (v.cpu().numpy() for v in plan.backward(dev(y), dev(g)))
    for c in range(len(lens)):
        sl = slice(offs[c], offs[c + 1])
        if sl.start == sl.stop:
            continue
        x64, g64 = x[sl].astype(np.float64), g[c].astype(np.complex128)
        assert rel_l2(f[sl], oracle.ndft_forward(x64, g64)) < TOL[prec]
        ady, adx = oracle.ndft_grad(x64, y[sl].astype(np.float64), M, g64)
        assert rel_l2(dy[sl], ady) < TOL[prec]
        assert rel_l2(dx[sl], adx) < TOL[prec]
