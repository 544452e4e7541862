"""A batch whose curves have 2^26 spread tiles together, more than the work order's
launch takes at one thread group per tile: 8192 curves of one point on 2^19 cells in
tiles of 64.  A curve's spectrum is y exp(2 pi i k x); rel L2 1e-5."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

import cunfft_adjoint_amd as cu  # noqa: E402
from tests._data import rel_l2  # noqa: E402

pytestmark = pytest.mark.gpu


def test_more_tiles_than_one_launch():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    nc, M = 8192, 1 << 18
    rng = np.random.default_rng(6)
    x = rng.uniform(-0.5, 0.5, nc).astype(np.float32)
    y = rng.uniform(1.0, 2.0, nc).astype(np.float32)
    plan = cu.NFFTPlan(torch.from_numpy(x).cuda(), M, offsets=np.arange(nc + 1, dtype=np.int32),
                       tile_log2=6)
    assert nc * plan.info().ntiles == 1 << 26
    f = plan.adjoint(torch.from_numpy(y).cuda())
    k = np.arange(-M // 2, M // 2)
    for c in (0, nc // 2 - 1, nc // 2, nc - 1):  # (the launches meet at half the curves)
        want = y[c] * np.exp(2j * np.pi * ((k * np.float64(x[c])) % 1.0))
        assert rel_l2(f[c].cpu().numpy(), want) < 1e-5
    plan.close()
    del f
    cu.batch_cache_clear("f")
    torch.cuda.empty_cache()
