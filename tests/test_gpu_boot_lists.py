"""Merged draws of the fused bootstrap at the edges of its 16-bit lists: curves
one point below, at and above the longest merged one of a small grid (so that one
batch mixes merged and point-by-point replicates), one and two points, an empty
curve, odd lengths.  Spectra and windows against the unfused path (the same draws
through the plan's tiles), Lomb-Scargle power against the FP64 periodogram of the
same draws; replicates few and many (one or two transforms per queue item).
Tolerances: the library's rel L2 1e-5 / 1e-11, power 2e-5 / 1e-10 absolute."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

import oracle  # noqa: E402
import cunfft_adjoint_amd as cu  # noqa: E402
from tests._data import rel_l2  # noqa: E402

pytestmark = pytest.mark.gpu

NP = {"f": np.float32, "d": np.float64}
TOL = {"f": 1e-5, "d": 1e-11}
PTOL = {"f": 2e-5, "d": 1e-10}


@pytest.fixture(scope="module", autouse=True)
def _gpu():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    torch.cuda.init()


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def inputs(prec, M, seed):
    cap = 2 * M * (4 if prec == "f" else 8) // 2  # counters in the grid's space
    lens = [cap - 1, 1, cap, 0, cap + 1, 2, 101]
    rng = np.random.default_rng(seed)
    offs = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    x = rng.uniform(-0.5, 0.5, offs[-1]).astype(NP[prec])
    y = rng.standard_normal(offs[-1]).astype(NP[prec])
    return x, y, offs, lens


@pytest.mark.parametrize("prec", ["f", "d"])
@pytest.mark.parametrize("M,nbs", [(64, 3), (1 << 9, 2), (64, 1500)])
def test_spectra_equal_the_unfused_path(prec, M, nbs):
    x, y, offs, lens = inputs(prec, M, M + nbs)
    kw = dict(offsets=offs, window2=True)
    got = cu.NFFTPlan(dev(x), M, **kw).bootstrap(dev(y), nbs, seed=9, window=True)
    ref = cu.NFFTPlan(dev(x), M, unfused=True, **kw).bootstrap(dev(y), nbs, seed=9, window=True)
    for g, r in zip(got, ref):
        g = g.cpu().numpy().reshape(len(lens), nbs, M)
        r = r.cpu().numpy().reshape(len(lens), nbs, M)
        for c in range(len(lens)):
            if lens[c] == 0:
                assert not g[c].any()
            else:
                assert rel_l2(g[c], r[c]) < TOL[prec], (c, lens[c])


@pytest.mark.parametrize("prec", ["f", "d"])
def test_lomb_scargle_of_merged_and_single_draws(prec):
    M, nbs, seed = 64, 2, 21
    x, y, offs, lens = inputs(prec, M, 5)
    plan = cu.NFFTPlan(dev(x), M, offsets=offs, window2=True)
    power = plan.bootstrap_ls(dev(y), nbs, seed=seed)["power"].cpu().numpy().reshape(len(lens), nbs, M // 2)
    for c in (0, 2, 4, 6):
        sl = slice(offs[c], offs[c + 1])
        d = oracle.bootstrap_indices(seed, lens[c], nbs)
        for r in range(nbs):
            xr, yr = x[sl][d[r]].astype(np.float64), y[sl][d[r]].astype(np.float64)
            ref = oracle.lomb_scargle(xr, yr, 1.0, M // 2)
            # k = 0 has no power in either
            assert np.abs(power[c, r, 1:] - ref[1:]).max() < PTOL[prec], (c, r)
