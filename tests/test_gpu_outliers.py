"""Values of very different size (log-normal, or one that dominates its curve) keep
the accuracy of ordinary ones: the spread's fixed-point unit follows what a cell can
receive, not the largest value times the densest window.  FP32 against the FP64
library at m = 16 (1e-14, checked against direct sums elsewhere).

Bounds.  The two-pass FFT's own rounding is near 2.2e-7 of the spectrum's norm.  A
batch in large spread tiles may be 1.1 times as far off as in tiles of 256 cells,
which leaves the spread's rounding 0.45 of the FFT's."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

import cunfft_adjoint_amd as cu  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _gpu():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    torch.cuda.init()


def values(kind, n, rng):
    y = rng.standard_normal(n)
    if kind == "lognormal":
        return np.exp(2.0 * y)
    if kind != "even":
        y[n // 3] = float(kind)
    return y


def points(kind, n, rng):
    x = rng.uniform(-0.5, 0.5, n)
    if kind == "clustered":
        k = int(0.8 * n)
        x[:k] = rng.uniform(-0.5, 0.5, 50)[rng.integers(0, 50, k)] + 0.005 * rng.standard_normal(k)
        x = (rng.permutation(x) + 0.5) % 1.0 - 0.5
    return x


def batch(pts, kind, n, curves, rows):
    """`curves` curves of n points, the first `rows` of them of the kind asked for."""
    rng = np.random.default_rng(11)
    x = np.concatenate([points(pts, n, rng) for _ in range(curves)]).astype(np.float32)
    y = np.concatenate([values(kind if c < rows else "even", n, rng) for c in range(curves)])
    return (torch.from_numpy(v).cuda() for v in (x, y.astype(np.float32)))


def reference(x, y, n, rows, M):
    x, y = x[:rows * n].double(), y[:rows * n].double()
    return cu.NFFTPlan(x, M, offsets=np.arange(rows + 1, dtype=np.int32) * n, m=16).adjoint(y)


def error(f, ref):
    return (torch.linalg.norm(f.to(torch.complex128) - ref) / torch.linalg.norm(ref)).item()


@pytest.mark.parametrize("pts", ["uniform", "clustered"])
@pytest.mark.parametrize("kind", ["even", "lognormal", "1000", "1e6"])
def test_large_spread_tiles(pts, kind):
    n, M, curves, rows = 20_000, 1 << 16, 64, 2
    x, y = batch(pts, kind, n, curves, rows)
    offs = np.arange(curves + 1, dtype=np.int32) * n
    ref = reference(x, y, n, rows, M)
    large, small = (cu.NFFTPlan(x, M, offsets=offs, tile_log2=t) for t in (0, 8))
    assert large.info().tile_log2 > 8
    e = [error(p.adjoint(y)[:rows], ref) for p in (large, small)]
    assert e[0] <= 1.1 * e[1], e


@pytest.mark.parametrize("n,M,curves,pts", [
    (1000, 1 << 11, 1, "uniform"), (1000, 1 << 11, 1, "clustered"), (200, 1 << 9, 4, "uniform"),
    (4700, 1 << 14, 256, "uniform"), (4700, 1 << 14, 256, "clustered"),
    (12_000, 1 << 14, 256, "uniform"), (12_000, 1 << 14, 256, "clustered")])
@pytest.mark.parametrize("kind", ["even", "lognormal", "30", "100", "1000", "1e6"])
def test_fused_adjoint(n, M, curves, pts, kind):
    """One workgroup's FFT rounds near 2.1e-7 (2.6e-7 for dense clumps), and the rule
    keeps the grid's rounding below 0.75e-7: together 2.7e-7, times a margin of 1.2.
    One curve of the kind asked for, the rest short, so that the batch is fused."""
    x, y = batch(pts, kind, n, 1, 1)
    if curves > 1:
        rng = np.random.default_rng(12)
        fill = 100 * (curves - 1)
        x = torch.cat([x, torch.from_numpy(rng.uniform(-0.5, 0.5, fill).astype(np.float32)).cuda()])
        y = torch.cat([y, torch.from_numpy(rng.standard_normal(fill).astype(np.float32)).cuda()])
    offs = np.concatenate([[0, n], n + 100 * np.arange(1, curves)]).astype(np.int32)
    ref = reference(x, y, n, 1, M)
    fused, tiles = (cu.NFFTPlan(x, M, offsets=offs, unfused=u) for u in (False, True))
    got = fused.adjoint(y)
    assert error(got[:1], ref) <= 3.2e-7
    assert error(tiles.adjoint(y)[:1], ref) <= 3.2e-7  # and so have the tiles
    # the same bits each time, whatever the order in which the rounds' atomics land
    assert torch.equal(got, fused.adjoint(y))
