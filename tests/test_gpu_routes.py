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
        return " ".join(sorted(n for n in _trace(f) if "gs::" in n))
    return names


@pytest.mark.parametrize("cplx", [False, True])
def test_single_zlog_flags(gs, kernels, cplx):
    """A single matrix of a resident order: Z through the log, or, with
    zdirect, in place (no replay)."""
    n = 30
    A = gen.ginibre_complex(n, gen.stream(51, 1, n)) if cplx else gen.ginibre_real(n, gen.stream(51, 1, n))
    replay = "zlog_kernel" if cplx else "dlog_kernel"
    assert replay in kernels(lambda: gs.gschur(A))
    assert replay in kernels(lambda: gs.gschur(A, zlog_tiny=True))
    assert replay not in kernels(lambda: gs.gschur(A, zdirect=True))
    assert replay not in kernels(lambda: gs.gschur(A, wantZ=False))
