"""Device blocks kept from destroyed plans: new plans on other streams and with
other sizes get the right results from reused blocks, while the old plan's work
may still be queued when it is destroyed; a captured stream is refused a kept
block as it is refused hipMalloc; cuna_batch_cache_clear gives the memory back."""
import ctypes

import numpy as np
import pytest

torch = pytest.importorskip("torch")

import cunfft_adjoint_amd as cu  # noqa: E402
from tests._data import uniform_points  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _gpu():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    torch.cuda.init()


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def test_reused_blocks_across_streams():
    sizes = [(100_000, 1 << 17), (90_000, 1 << 17), (30_000, 1 << 15), (100_000, 1 << 17)]
    data = [tuple(dev(v) for v in uniform_points(n, 50 + i)) for i, (n, _) in enumerate(sizes)]
    want = []
    for (x, y), (_, M) in zip(data, sizes):
        plan = cu.NFFTPlan(x, M)
        want.append(plan.adjoint(y).cpu().numpy())
        plan.close()
    streams = [torch.cuda.Stream() for _ in range(3)]
    torch.cuda.synchronize()
    for rep in range(3):
        got = []
        for i, ((x, y), (_, M)) in enumerate(zip(data, sizes)):
            s = streams[(i + rep) % 3]
            with torch.cuda.stream(s):
                plan = cu.NFFTPlan(x, M)
                got.append(plan.adjoint(y))
                plan.close()  # its transform may still be queued
        torch.cuda.synchronize()
        for g, w in zip(got, want):
            assert np.array_equal(g.cpu().numpy(), w)


def test_capture_refuses_a_kept_block_and_clear_gives_back():
    x, y = (dev(v) for v in uniform_points(50_000, 7))
    M = 1 << 16
    plan = cu.NFFTPlan(x, M)
    plan.adjoint(y)
    plan.close()  # its grid is kept
    plan = cu.NFFTPlan(x, M)
    out = torch.empty((1, M), dtype=torch.complex64, device="cuda")
    s = torch.cuda.Stream()
    with pytest.raises(cu.CunaError):
        cu.capture(lambda: plan.adjoint(y, out=out, stream=s), s)
    plan.adjoint(y, out=out, stream=s)
    s.synchronize()
    ref = out.cpu().numpy().copy()
    g = cu.capture(lambda: plan.adjoint(y, out=out, stream=s), s)
    for _ in range(3):
        out.zero_()
        torch.cuda.synchronize()
        g.launch(s)
        s.synchronize()
        assert np.array_equal(out.cpu().numpy(), ref)
    g.close()
    plan.close()
    hip = ctypes.CDLL("libamdhip64.so")
    free, total = ctypes.c_size_t(), ctypes.c_size_t()

    def free_bytes():
        assert hip.hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
        return free.value

    big = cu.NFFTPlan(x, 1 << 22)  # a grid of 32 MiB
    big.adjoint(y)
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    held = free_bytes()
    big.close()
    cu.batch_cache_clear("f")
    assert free_bytes() >= held + (32 << 20)
