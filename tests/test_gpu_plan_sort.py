"""The one-launch sort of short curves against the multi-launch one: the same
curves planned alone (or together) and next to one curve that is too long for
the one-launch sort give bitwise the same spectra, since the sorted order, the
buckets and the tiles' covers are the same.  Lengths at the edges of its
workgroup sizes (2048, 8192, 23552 points), one point, empty curves, all points
in one cell; grids of one to three sort digits."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

import cunfft_adjoint_amd as cu  # noqa: E402

pytestmark = pytest.mark.gpu

NP = {"f": np.float32, "d": np.float64}
LONG = 23 * 1024 + 1  # one point more than the one-launch sort takes


@pytest.fixture(scope="module", autouse=True)
def _gpu():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    torch.cuda.init()


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def spectra(x, y, lens, M):
    offs = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    # an explicit tile size asks for the tile path, also on small grids
    return cu.NFFTPlan(dev(x), M, offsets=offs, tile_log2=8).adjoint(dev(y)).cpu().numpy()


@pytest.mark.parametrize("prec", ["f", "d"])
@pytest.mark.parametrize("lens,M,one_cell", [
    ([1, 0, 63, 64, 65, 2048], 1 << 5, False),
    ([2049, 5, 0, 1025], 1 << 9, False),
    ([8192, 300], 1 << 12, False),
    ([8193, 23 * 1024], 1 << 16, False),
    ([1000, 2047], 1 << 19, False),
    ([3000], 1 << 12, True),
])
def test_same_spectra_as_the_multi_launch_sort(prec, lens, M, one_cell):
    rng = np.random.default_rng(sum(lens) + M)
    n = sum(lens)
    x = rng.uniform(-0.5, 0.5, n + LONG).astype(NP[prec])
    if one_cell:
        x[:n] = (0.2 + rng.uniform(0, 0.2, n) / (2 * M)).astype(NP[prec])
    y = rng.standard_normal(n + LONG).astype(NP[prec])
    short = spectra(x[:n], y[:n], lens, M)
    mixed = spectra(x, y, lens + [LONG], M)
    assert np.isfinite(short).all() and np.abs(short).max() > 0
    assert np.array_equal(short, mixed[:len(lens)])
