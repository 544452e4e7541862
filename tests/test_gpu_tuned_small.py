"""The autotuner on small grids: where the one-launch adjoint is the faster one (a
few hundred points, M = 2^11: one launch against two), the tuned plan takes it, and
its result meets the tolerance."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

import cunfft_adjoint_amd as cu  # noqa: E402
import oracle  # noqa: E402
from tests._data import rel_l2, uniform_points  # noqa: E402

pytestmark = pytest.mark.gpu


def test_tuned_plan_keeps_the_one_launch_adjoint():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    x, y = uniform_points(300, 5)
    xd, yd = (torch.from_numpy(np.ascontiguousarray(v)).cuda() for v in (x, y))
    M, tol = 1 << 11, 1e-5
    p = cu.autotune(xd, M, tol, cache_path="")
    got = cu.NFFTPlan(xd, M, **p).adjoint(yd).cpu().numpy()[0]
    assert rel_l2(got, oracle.ndft(x.astype(np.float64), y.astype(np.float64), M)) < tol
    assert (p["tile_log2"], p["fft_w"], p["fft_h"]) == (0, 0, 0)
