"""A graph keeps working while its plan goes on: an eager call that needs larger
workspaces than the captured one leaves the memory whose address the graph holds
with the plan, so a replay gives the captured call's result and writes into no
other plan.  Sizes: the blocks that the plan would give up (its grid of 2^17 cells)
are of the size class of the second plan's chirp table (65,251 values)."""
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


def spectrum(M, rows=1):
    g = np.random.default_rng(3).standard_normal((rows, M, 2)).astype(np.float32)
    return torch.view_as_complex(dev(g))


def other_plan():
    """A plan whose tables take a block of 512 KiB, and its result."""
    x, y = (dev(v) for v in uniform_points(20_000, 8))
    p = cu.NFFTPlan(x, 87_000, mode="compat")
    return p, y, p.adjoint(y).cpu().numpy()


def replays_equal(g, s, out, want):
    for _ in range(3):
        out.zero_()
        torch.cuda.synchronize()
        g.launch(s)
        s.synchronize()
        assert np.array_equal(out.cpu().numpy(), want)


@pytest.mark.parametrize("later", ["forward", "adjoint_many", "both"])
def test_adjoint_graph_after_larger_calls(later):
    M = 1 << 16
    cu.batch_cache_clear("f")
    x, y = (dev(v) for v in uniform_points(50_000, 7))
    plan = cu.NFFTPlan(x, M)
    s = torch.cuda.Stream()
    out = torch.empty((1, M), dtype=torch.complex64, device="cuda")
    torch.cuda.synchronize()
    plan.adjoint(y, out=out, stream=s)
    s.synchronize()
    want = out.cpu().numpy().copy()
    g = cu.capture(lambda: plan.adjoint(y, out=out, stream=s), s)
    if later != "adjoint_many":
        plan.forward(spectrum(M))
    if later != "forward":
        plan.adjoint_many(torch.stack([y, 2 * y, 3 * y]).contiguous())
    torch.cuda.synchronize()
    p2, y2, want2 = other_plan()
    replays_equal(g, s, out, want)
    assert np.array_equal(p2.adjoint(y2).cpu().numpy(), want2)
    g.close()
    plan.close()
    p2.close()


def test_fused_adjoint_graph_after_a_backward():
    """More curves than resident workgroups: the fused adjoint's rows are fewer than
    the grids of the other directions."""
    M, nc, n = 1 << 13, 700, 20
    cu.batch_cache_clear("f")
    rng = np.random.default_rng(5)
    x = dev(rng.uniform(-0.5, 0.5, nc * n).astype(np.float32))
    y = dev(rng.standard_normal(nc * n).astype(np.float32))
    plan = cu.NFFTPlan(x, M, offsets=np.arange(nc + 1, dtype=np.int32) * n)
    s = torch.cuda.Stream()
    out = torch.empty((nc, M), dtype=torch.complex64, device="cuda")
    torch.cuda.synchronize()
    plan.adjoint(y, out=out, stream=s)
    s.synchronize()
    want = out.cpu().numpy().copy()
    g = cu.capture(lambda: plan.adjoint(y, out=out, stream=s), s)
    plan.backward(y, spectrum(M, nc))
    torch.cuda.synchronize()
    p2, y2, want2 = other_plan()
    replays_equal(g, s, out, want)
    assert np.array_equal(p2.adjoint(y2).cpu().numpy(), want2)
    g.close()
    plan.close()
    p2.close()


def test_compat_graph_after_a_bootstrap():
    """The chirp transform's workspace grows with the replicates."""
    n, ng = 20_000, 65_538
    cu.batch_cache_clear("f")
    x, y = (dev(v) for v in uniform_points(n, 9))
    fp = cu.generate_filter_properties(x, n, ng)
    s = torch.cuda.Stream()
    out = torch.empty(ng, dtype=torch.complex64, device="cuda")
    torch.cuda.synchronize()

    def run():
        cu.cunfft_adjoint_raw_async_noalloc(x, y, out, n, ng, fp, stream=s)

    run()
    s.synchronize()
    want = out.cpu().numpy().copy()
    g = cu.capture(run, s)
    boot = torch.empty((4, ng), dtype=torch.complex64, device="cuda")
    cu.cunfft_adjoint_raw_async_bootstrap(x, y, boot, n, ng, 4, fp, seed=1)
    torch.cuda.synchronize()
    p2, y2, want2 = other_plan()
    replays_equal(g, s, out, want)
    assert np.array_equal(p2.adjoint(y2).cpu().numpy(), want2)
    g.close()
    fp.free()
    p2.close()
