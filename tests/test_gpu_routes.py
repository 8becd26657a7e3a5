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


def _device_batch(ns, cplx):
    import numpy as np
    import torch
    ns = np.ascontiguousarray(ns, dtype=np.int32)
    off = np.zeros(len(ns), dtype=np.int64)
    off[1:] = np.cumsum(ns[:-1].astype(np.int64) ** 2)
    g = torch.Generator(device="cuda").manual_seed(5)
    A = torch.randn((2 if cplx else 1) * int((ns.astype(np.int64) ** 2).sum()), generator=g, device="cuda",
                    dtype=torch.float64)
    T, Z = torch.zeros_like(A), torch.zeros_like(A)
    W = torch.zeros(2 * int(ns.sum()), device="cuda", dtype=torch.float64)
    return ns, off, A, T, Z, W, torch.zeros(len(ns), device="cuda", dtype=torch.int32)


@pytest.mark.parametrize("count", [85, 86])
def test_noalloc_cooperative_form_by_call(gs, kernels, count):
    """The 512-thread windowed form where the call (not one of its launches,
    which run side by side) has at most a matrix above order 48 per CU."""
    import ctypes
    from genericschur import _lib
    ns, off, A, T, Z, W, info = _device_batch([20] * 300 + [96] * count + [80] * count + [64] * (256 - 2 * 85), True)
    p = lambda t: ctypes.c_void_p(t.data_ptr())
    h = _lib.handle()

    def call():
        rc = _lib.lib().gs_schur_batched_z_noalloc(h, len(ns), ctypes.c_void_p(ns.ctypes.data),
                                                   ctypes.c_void_p(off.ctypes.data), p(A), p(T), p(Z), p(W), p(info),
                                                   _lib.GS_SCALE)
        _lib.check(rc, h, "gs_schur_batched_z_noalloc")
    k = kernels(call)
    assert any("zqrw2_kernel<true, 512>" in x for x in k) == (count == 85), k
    assert any("zqrw2_kernel<true, 128>" in x for x in k) == (count == 86), k


@pytest.mark.parametrize("n,wantZ,zdirect,nt", [(550, True, False, 512), (551, True, False, 1024), (551, False, False, 512),
                                                (768, True, False, 512), (768, True, True, 1024)])
def test_single_complex_threads(gs, kernels, n, wantZ, zdirect, nt):
    """Threads of one complex matrix's QR kernel: 1024 already above order 550
    where Z is updated in place (without the log, which starts at 768)."""
    A = gen.ginibre_complex(n, gen.stream(53, 1, n))
    k = kernels(lambda: gs.gschur(A, wantZ=wantZ, zdirect=zdirect))
    assert any(f"zqrw2_kernel<true, {nt}>" in x for x in k), k


@pytest.mark.parametrize("n,name", [(96, "dlog_kernel<96>"), (97, "dlog_lds_kernel"), (128, "dlog_lds_kernel")])
def test_real_replay_form(gs, kernels, n, name):
    """The real Z log's replay: Z's rows in registers up to order 96, Z in LDS above."""
    A = [gen.ginibre_real(n, gen.stream(54, 1, n))] * 2
    assert any(name in x for x in kernels(lambda: gs.gschur_batched(A)))
