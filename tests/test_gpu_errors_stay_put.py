"""A HIP error that one call has reported, or that a release has met, is not reported
again by the next call: a captured stream refuses the memory of a first call, and a
plan is destroyed while its thread captures.  The capture is lost either way; work on
another stream goes on.  The runtime leaves the captured stream unusable, so it is
one of the test's own, not of torch's pool."""
import ctypes

import numpy as np
import pytest

torch = pytest.importorskip("torch")

import cunfft_adjoint_amd as cu  # noqa: E402
from tests._data import uniform_points  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,n", [(1 << 11, 3000), (1 << 16, 50_000)])  # blocks not kept, and kept
@pytest.mark.parametrize("what", ["first call", "destroy"])
def test_next_call_on_another_stream(what, M, n):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    torch.cuda.init()
    cu.batch_cache_clear("f")
    x, y = (torch.from_numpy(np.ascontiguousarray(v)).cuda() for v in uniform_points(n, 3))
    plan, other = (cu.NFFTPlan(x, M, tile_log2=8) for _ in range(2))
    out = torch.empty((1, M), dtype=torch.complex64, device="cuda")
    want = plan.adjoint(y).cpu().numpy()
    if what == "destroy":
        other.adjoint(y)
    raw = ctypes.c_void_p()
    assert ctypes.CDLL("libamdhip64.so").hipStreamCreate(ctypes.byref(raw)) == 0
    captured, after = torch.cuda.ExternalStream(raw.value), torch.cuda.Stream()
    torch.cuda.synchronize()

    def run():
        if what == "destroy":
            other.close()
            plan.adjoint(y, out=out, stream=captured)
        else:
            other.adjoint(y, out=out, stream=captured)

    try:
        cu.capture(run, captured).close()
    except cu.CunaError:
        pass
    plan.adjoint(y, out=out, stream=after)
    after.synchronize()
    assert np.array_equal(out.cpu().numpy(), want)
