"""Calls that are promised to agree bit for bit: a curve of a compat batch and the
call on that curve alone, a value vector of adjoint_many and the adjoint of that
vector.  Batches on both sides of where the library changes tile or FFT form, at
grids whose transform one workgroup holds (compat: powers of two up to 2^15 in
libcunaf and 2^14 in libcunad, other lengths up to 2^13 and 2^12; accurate: M up to
2^14 and 2^13)."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

import cunfft_adjoint_amd as cu  # noqa: E402

pytestmark = pytest.mark.gpu

RT = {"f": torch.float32, "d": torch.float64}
CT = {"f": torch.complex64, "d": torch.complex128}


@pytest.fixture(scope="module", autouse=True)
def _gpu():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    torch.cuda.init()


def compat_batch_equals_single_calls(prec, ng, curves, n):
    rng = np.random.default_rng(ng + curves)
    lens = [n + i % 7 for i in range(curves)]
    off = np.concatenate([[0], np.cumsum(lens)])
    x = torch.from_numpy(rng.uniform(-0.5, 0.5, off[-1])).to(RT[prec]).cuda()
    y = torch.from_numpy(rng.standard_normal(off[-1])).to(RT[prec]).cuda()
    out = torch.zeros(curves * ng, dtype=CT[prec], device="cuda")
    cu.cunfft_adjoint_raw_batched_async(x, y, out, lens, [ng] * curves, None)
    for i in (0, curves // 2, curves - 1):
        one = torch.zeros(ng, dtype=CT[prec], device="cuda")
        sl = slice(int(off[i]), int(off[i + 1]))
        cu.cunfft_adjoint_raw_async(x[sl].clone(), y[sl].clone(), one, lens[i], ng, None)
        assert torch.equal(out[i * ng:(i + 1) * ng], one), i


@pytest.mark.parametrize("prec", ["f", "d"])
def test_compat_batch_of_sparse_curves(prec):
    compat_batch_equals_single_calls(prec, 1 << 13, 520, 100)


@pytest.mark.parametrize("prec,ng", [("f", 1 << 15), ("f", 3001), ("f", 4097), ("f", 5001), ("f", 8191),
                                     ("d", 1 << 14), ("d", 2049), ("d", 2501), ("d", 4095)])
@pytest.mark.parametrize("curves", [2, 70, 130])
def test_compat_batch(prec, ng, curves):
    compat_batch_equals_single_calls(prec, ng, curves, 900)


@pytest.mark.parametrize("prec,M", [("f", 1 << 13), ("f", 1 << 14), ("d", 1 << 12), ("d", 1 << 13)])
@pytest.mark.parametrize("curves,nrhs", [(1, 2), (1, 60), (1, 130), (40, 3), (60, 2), (110, 2)])
def test_adjoint_many(prec, M, curves, nrhs):
    rng = np.random.default_rng(M + nrhs)
    n = 1500 * curves
    x = torch.from_numpy(rng.uniform(-0.5, 0.5, n)).to(RT[prec]).cuda()
    y = torch.from_numpy(rng.standard_normal((nrhs, n))).to(RT[prec]).cuda()
    plan = cu.NFFTPlan(x, M, offsets=np.arange(curves + 1, dtype=np.int32) * 1500, tile_log2=8)
    many = plan.adjoint_many(y).reshape(curves, nrhs, M)
    for r in (0, nrhs - 1):
        assert torch.equal(many[:, r], plan.adjoint(y[r]))


@pytest.mark.parametrize("prec,ng,rows", [("f", 1 << 15, 97), ("f", 1 << 15, 96), ("d", 1 << 14, 49),
                                          ("d", 1 << 14, 48)])
def test_compat_bootstrap_within_rounding(prec, ng, rows):
    """Replicates choose the form by their number: the same ones in a call on the other
    side of the line (3/8 and 3/16 of the CUs) within rounding, 1e-6 and 1e-14."""
    rng = np.random.default_rng(rows)
    n = 700
    x = torch.from_numpy(rng.uniform(-0.5, 0.5, n)).to(RT[prec]).cuda()
    y = torch.from_numpy(rng.standard_normal(n)).to(RT[prec]).cuda()
    fp = cu.generate_filter_properties(x, n, ng)
    many, few = (torch.empty((r, ng), dtype=CT[prec], device="cuda") for r in (rows, 5))
    cu.cunfft_adjoint_raw_async_bootstrap(x, y, many, n, ng, rows, fp, seed=9)
    cu.cunfft_adjoint_raw_async_bootstrap(x, y, few, n, ng, 5, fp, seed=9)
    assert torch.linalg.norm(many[:5] - few) <= (1e-6 if prec == "f" else 1e-14) * torch.linalg.norm(few)
    fp.free()
