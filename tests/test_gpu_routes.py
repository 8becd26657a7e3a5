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


@pytest.mark.parametrize("cplx", [False, True])
@pytest.mark.parametrize("small,large,own", [(256, [33, 64], False), (257, [33, 64], True), (256, [65], True)])
def test_small_vectors_joined(gs, kernels, cplx, small, large, own):
    """Up to 256 matrices of orders up to 32 go with the list's orders 33 to 64,
    if there are any; either way with the single calls' bits."""
    import ctypes
    import numpy as np
    from genericschur import _lib
    ns = [int(n) for n in gen.stream(56, small, len(large)).integers(1, 33, size=small)] + large + [0]
    r = gen.stream(56, 1, small)
    Ss, _ = gs.gschur_batched([gen.ginibre_complex(n, r) if cplx else gen.ginibre_real(n, r) for n in ns])
    n_, off, T = gs.pack([S.T for S in Ss], np.complex128 if cplx else np.float64)
    _, _, Z = gs.pack([S.Z for S in Ss], T.dtype)
    V = np.zeros(T.shape, dtype=np.complex128)
    h = _lib.handle()
    p = lambda a: ctypes.c_void_p(a.ctypes.data)
    f = _lib.lib().gs_trevc_batched_z if cplx else _lib.lib().gs_trevc_batched_d
    k = kernels(lambda: _lib.check(f(h, len(n_), p(n_), p(off), p(T), p(Z), p(V), 0, 1, 0), h, "gs_trevc_batched"))
    assert any("trevc_small" in x for x in k) == own, k
    for S, X in list(zip(Ss, gs.unpack(n_, off, V)))[:-1:16]:
        assert np.array_equal(X, gs.geigvecs(S))


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
    """The 512-thread windowed form where the call (not one of its launches)
    has at most a matrix above order 48 to a CU (three to four CUs beside
    smaller ones)."""
    import ctypes
    from genericschur import _lib
    ns, off, A, T, Z, W, info = _device_batch([20] * 300 + [96] * count + [80] * count + [64] * (192 - 2 * 85), True)
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


# (orders, whether the work queue, the 512-thread form, the resident form, and a replay of orders above 48 run)
ROUTES = [([64] * 256, False, True, False, False),
          ([64] * 257, True, False, False, False),
          ([64] * 192 + [20] * 10, False, True, True, False),
          ([64] * 193 + [20] * 10, True, False, False, False),
          ([81] * 257, True, False, False, True),
          ([64] * 560, True, False, False, False),
          ([64] * 561, True, False, False, True),
          ([49] + [20] * 1000, False, True, True, False),
          ([48] * 300, False, False, True, False)]


@pytest.mark.parametrize("case", range(len(ROUTES)))
def test_complex_batch_routes(gs, kernels, case):
    """Complex batches at the lines between the forms."""
    orders, queue, coop, resident, replay = ROUTES[case]
    ns, off, A, T, Z, W, info = _device_batch(orders, True)
    k = kernels(lambda: gs.gschur_batched_device(ns, off, A, T, Z, W, info, True))
    assert int(info.abs().sum()) == 0
    got = [any(x in y for y in k) for x in ("zqrw2_queue_kernel", "zqrw2_kernel<true, 512>", "zqrr_kernel")]
    assert got == [queue, coop, resident], k
    assert any("zlog_kernel<" + c in y for y in k for c in ("64", "80", "96")) == replay, k
    assert any("zlog_kernel<32" in y or "zlog_kernel<48" in y for y in k) == resident, k


def test_complex_batch_one_windowed_launch(gs, kernels):
    """Bins above the resident orders in one 512-thread launch, with the results
    of one launch per bin (as when timed) and of the queue (the same matrices
    among more), bit for bit."""
    import torch
    from genericschur import _lib
    orders = [99, 97, 80, 60, 49, 48, 30, 5, 1] * 20
    ns, off, A, T, Z, W, info = _device_batch(orders, True)
    gs.gschur_batched_device(ns, off, A, T, Z, W, info, True)
    T1, Z1, W1 = torch.zeros_like(T), torch.zeros_like(Z), torch.zeros_like(W)
    gs.gschur_batched_device(ns, off, A, T1, Z1, W1, info, True, timing=True)
    qr = [r for r in _lib.last_launches() if r["kind"] == "qr"]
    assert sum(r["nmax"] > 48 for r in qr) >= 2 and sum(r["count"] for r in qr) == len(orders)
    assert torch.equal(T, T1) and torch.equal(Z, Z1) and torch.equal(W, W1)
    ns2, off2, A2, T2, Z2, W2, info2 = _device_batch(orders + [60] * 300, True)
    A2[:A.numel()] = A
    assert any("queue" in x for x in kernels(lambda: gs.gschur_batched_device(ns2, off2, A2, T2, Z2, W2, info2, True)))
    m = A.numel()
    assert torch.equal(T, T2[:m]) and torch.equal(Z, Z2[:m]) and torch.equal(W, W2[:W.numel()])
