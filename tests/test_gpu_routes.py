"""Which kernels a call runs, where a flag or the sizes decide it: names from
the in-process profiler's trace of the call.  (What the kernels compute is
compared elsewhere; forms that give the same bits cannot be told apart by
their results.)"""
import pytest

from genericschur import gen

pytestmark = pytest.mark.gpu


def _trace(f):
    import torch
    from torch.profiler import ProfilerActivity, profile
    with profile(activities=[ProfilerActivity.CUDA]) as p:
        f()
        torch.cuda.synchronize()
    return {e.name for e in p.events() if "kernel" in e.name}


@pytest.fixture(scope="module")
def kernels():
    """names of the library's kernels that f() runs"""
    import torch
    x = torch.ones(64, device="cuda")
    if not _trace(lambda: x.mul_(2.0)):
        pytest.skip("no kernel trace on this system")

    def names(f):
        f()  # allocations
        return sorted(n.split("(")[0] for n in _trace(f) if "gs::" in n)
    return names


@pytest.mark.parametrize("cplx", [False, True])
def test_single_zlog_flags(gs, kernels, cplx):
    """A single matrix of a resident order: Z through the log, or, with
    zdirect, in place (no replay)."""
    n = 30
    A = gen.ginibre_complex(n, gen.stream(51, 1, n)) if cplx else gen.ginibre_real(n, gen.stream(51, 1, n))
    replay = "zlog_kernel" if cplx else "dlog_kernel"
    for kw, logs in (({}, True), ({"zlog_tiny": True}, True), ({"zdirect": True}, False), ({"wantZ": False}, False)):
        assert any(replay in k for k in kernels(lambda: gs.gschur(A, **kw))) == logs, kw


@pytest.mark.parametrize("cplx", [False, True])
@pytest.mark.parametrize("left", [False, True])
def test_small_vectors_one_launch(gs, kernels, cplx, left):
    """Eigenvectors of orders up to 32: one kernel; of 33, those over the columns."""
    for n in (2, 16, 17, 32, 33):
        A = gen.ginibre_complex(n, gen.stream(52, 1, n)) if cplx else gen.ginibre_real(n, gen.stream(52, 1, n))
        S = gs.gschur(A)
        k = kernels(lambda: gs.geigvecs(S, left=left))
        assert len(k) >= 3 if n > 32 else (len(k) == 1 and "trevc_small" in k[0]), k
