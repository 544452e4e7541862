"""The one-workgroup adjoint of small grids against the exact sum and the tile
path: the smallest and largest grids of both libraries, every filter width it has,
empty and one-point curves, curves at the edges of its workgroup sizes, curves whose
densest window asks for a second round (all points in one cell), unit values,
several value vectors, and what it shares with the other directions of a plan.

Tolerances: the filter's own error at m = 8 (FP32) is below 1e-6 of a spectrum's
norm and rounding below 1e-6, so 1e-5 covers both; FP64 at m = 13 rounds near
1e-13 with a filter error near 1e-12, so 1e-11.  At a smaller m the two paths share
the filter's error, and their difference is rounding alone: 1e-6 and 1e-13 of the
norm times a margin of 10."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

import cunfft_adjoint_amd as cu  # noqa: E402
import oracle  # noqa: E402

pytestmark = pytest.mark.gpu

NP = {"f": np.float32, "d": np.float64}
TOL = {"f": 1e-5, "d": 1e-11}
PATHS = {"f": 1e-5, "d": 1e-12}


@pytest.fixture(scope="module", autouse=True)
def _gpu():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    torch.cuda.init()


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def exact(x, y, offs, M):
    return np.stack([oracle.ndft(x[b:e].astype(np.float64), y[b:e].astype(np.float64), M)
                     for b, e in zip(offs[:-1], offs[1:])])


def close(a, b, tol):
    for c in range(len(b)):  # per curve: a large one must not hide a small one
        assert np.linalg.norm(a[c] - b[c]) <= tol * np.linalg.norm(b[c]), c


def case(prec, lens, seed, one_cell=False):
    rng = np.random.default_rng(seed)
    offs = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    x = rng.uniform(-0.5, 0.5, offs[-1])
    if one_cell:
        x = 0.125 + 1e-7 * x
    y = rng.standard_normal(offs[-1]) + 0.5
    return x.astype(NP[prec]), y.astype(NP[prec]), offs


@pytest.mark.parametrize("prec", ["f", "d"])
@pytest.mark.parametrize("lens,M,one_cell", [
    ([1, 0, 63, 64, 65, 250], 1 << 6, False),
    ([250, 0, 1, 249], 1 << 6, True),
    ([255, 256, 257, 3] * 5, 1 << 9, False),
    ([0, 512, 511, 513] * 3, 1 << 11, True),
    ([1000, 7, 1023, 0], 1 << 13, False),
])
def test_against_the_exact_sum(prec, lens, M, one_cell):
    if prec == "d":
        lens = [min(v, 257) for v in lens]  # longer ones go through tiles
    x, y, offs = case(prec, lens, M, one_cell)
    kw = {"m": 8 if prec == "f" else 13}
    p = cu.NFFTPlan(dev(x), M, offsets=offs, **kw)
    want = exact(x, y, offs, M)
    close(p.adjoint(dev(y)).cpu().numpy(), want, TOL[prec])
    close(p.adjoint(None).cpu().numpy(), exact(x, np.ones_like(y), offs, M), TOL[prec])
    # several value vectors: bitwise the single ones
    ys = np.stack([y, -2 * y, y[::-1]])
    many = p.adjoint_many(dev(ys)).cpu().numpy().reshape(len(lens), 3, M)
    for r in range(3):
        assert np.array_equal(many[:, r], p.adjoint(dev(ys[r])).cpu().numpy())


@pytest.mark.parametrize("prec,M,m,long,short", [
    ("f", 1 << 14, 8, 8000, 900), ("f", 1 << 10, 6, 1050, 900), ("f", 1 << 12, 10, 1400, 900),
    ("d", 1 << 13, 13, 1700, 700), ("d", 1 << 10, 6, 430, 300), ("d", 1 << 12, 16, 1000, 700)])
@pytest.mark.parametrize("one_cell", [False, True])
def test_against_tiles(prec, M, m, long, short, one_cell):
    """Ragged batch with a curve about as long as the rule lets it be and one value
    that dominates its curve."""
    lens = [1, 100, 0, long] + [short] * 90
    x, y, offs = case(prec, lens, m, one_cell)
    y[offs[1]] = 1e6
    a, b = (cu.NFFTPlan(dev(x), M, offsets=offs, m=m, tile_log2=t) for t in (0, 8))
    pa, pb = (q.adjoint(dev(y)).cpu().numpy() for q in (a, b))
    close(pa, pb, PATHS[prec])
    # other directions after a fused call build what they need themselves
    g = np.random.default_rng(1).standard_normal((len(lens), M)) + 0j
    g = dev(g.astype(pa.dtype))
    assert torch.equal(a.forward(g), b.forward(g))


@pytest.mark.parametrize("prec", ["f", "d"])
def test_values_that_are_not_finite_stay_in_their_curve(prec):
    lens = [200, 200, 200]
    x, y, offs = case(prec, lens, 5)
    p = cu.NFFTPlan(dev(x), 1 << 9, offsets=offs)
    want = p.adjoint(dev(y)).cpu().numpy()
    for bad in (np.nan, np.inf):
        v = y.copy()
        v[250] = bad
        got = p.adjoint(dev(v)).cpu().numpy()
        assert not np.isfinite(got[1]).all()
        assert np.array_equal(got[[0, 2]], want[[0, 2]])
