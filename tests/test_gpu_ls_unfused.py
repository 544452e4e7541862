"""Lomb-Scargle periodograms exist in the fused kernel only: a plan made without it
is refused on the host, before anything is launched, and stays usable."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

import cunfft_adjoint_amd as cu  # noqa: E402
from tests._data import uniform_points  # noqa: E402

pytestmark = pytest.mark.gpu


def test_unfused_plan_is_refused():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    x, y = (torch.from_numpy(np.ascontiguousarray(v)).cuda() for v in uniform_points(500, 3))
    plan = cu.NFFTPlan(x, 1 << 10, window2=True, unfused=True)
    with pytest.raises(cu.CunaError, match="CUNA_PLAN_UNFUSED"):
        plan.bootstrap_ls(y, 4, seed=1)
    fused = cu.NFFTPlan(x, 1 << 10, window2=True)
    got, want = (p.bootstrap(y, 2, seed=1, window=True) for p in (plan, fused))
    for a, b in zip(got, want):
        assert torch.linalg.norm(a - b) <= 1e-5 * torch.linalg.norm(b)
