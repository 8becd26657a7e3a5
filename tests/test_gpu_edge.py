"""GPU parity on the reference's own test families, error paths and the
oracle's T, Z and slot order.

The families (tests/families.py) re-create those of the reference's tests:
Jordan blocks, random unitary / orthogonal (normal) matrices, general
matrices with specified eigenvalues in modes 4/3/1/5 with eigenvector
condition 1 and 1/sqrt(ulp) at magnitudes 1, ovfl*ulp and unfl/ulp,
diagonal, Hermitian, general and triangular random-entry matrices,
triangular matrices with a repeated eigenvalue, 100 floatmin and
floatmax / 100 scalings (which run _scale!), zero and identity, and the
cyclic shift that only the exceptional shifts move; plus the short QR sweep
regression (test/complex.jl:156-166) and Godunov's matrix
(test/testfuncs.jl:127-142; in Float64 only its backward error is
meaningful, econd = 7e16).

Each case runs through the single-matrix kernels (LDS-resident, plain, and
the large real path), and the family set as one batch, through the C ABI.
Every result is held to the reference's schurtest at tolerance 20, the
acceptance bounds 50 n eps, and the oracle's eigenvalues within
10 n eps ||A||_2 cond(lambda).  T, Z and the diagonal slot order are compared
with the oracle's up to the Schur form's own freedom; the share that match is
printed, and where the eigenvalues are well separated it must be high.
"""
import ctypes

import numpy as np
import pytest

import checks
from families import families, oracle_result
from genericschur import gen

pytestmark = pytest.mark.gpu

TOL = 20.0
EPS = np.finfo(np.float64).eps
TINY = np.finfo(np.float64).tiny


def check_case(oracle, name, A, S, normal, tally):
    n = A.shape[0]
    print(f"case {name} n={n} dtype={A.dtype}", flush=True)
    checks.schur_invariants(A, S.T, S.Z, S.values, TOL, normal=normal)
    assert checks.rel_backward(A, S.T, S.Z) <= 50 * n * EPS
    assert checks.rel_orth(S.Z) <= 50 * n * EPS
    To, Zo, wo, cond, _ = oracle_result(oracle, A)
    checks.eigen_parity(A, S.values, wo, cond)
    m = checks.schur_form_match(A, S.T, S.Z, S.values, To, Zo, wo, cond)
    wc = checks.well_conditioned(A, wo, cond)
    tally.setdefault(m, []).append((f"{name}/{n}", wc))
    return m


def report(tag, tally, min_share=0.8):
    """Prints how the results compare with the oracle's T, Z and slot order.
    Where every eigenvalue is simple and well separated (checks.
    well_conditioned) the Schur form is determined up to phases, so the
    results must match the oracle's there, apart from the rare matrix whose
    eigenvalues converge in another order after a rounding-level difference
    (FMA contraction, summation order) moved a deflation."""
    tot = sum(len(v) for v in tally.values())
    parts = ", ".join(f"{k} {len(v)}" for k, v in sorted(tally.items()))
    print(f"{tag}: T/Z vs oracle over {tot} cases: {parts}", flush=True)
    g = [c for v in tally.values() for c, wc in v if wc]
    good = [c for k in ("bitwise", "phases") for c, wc in tally.get(k, []) if wc]
    if g:
        share = len(good) / len(g)
        print(f"{tag}: well-conditioned cases matching up to phases: {len(good)}/{len(g)} = {share:.2f}",
              flush=True)
        assert share >= min_share, [c for c in g if c not in good]
    return tally


@pytest.mark.parametrize("cplx,sizes", [(True, (4, 32, 96)), (False, (4, 32, 128))])
def test_families_single(gs, oracle, cplx, sizes):
    """Single-matrix LDS-resident kernels (complex n <= 99, real n <= 141)."""
    tally = {}
    for n in sizes:
        for name, A, normal in families(n, cplx):
            S = gs.gschur(A)
            check_case(oracle, name, A, S, normal, tally)
    report(f"single {'complex' if cplx else 'real'}", tally)


@pytest.mark.parametrize("n", [100, 130, 200, 260])
def test_families_single_complex_windowed(gs, oracle, n):
    """Complex orders above the LDS-resident range: Hessenberg + Q in global
    memory (one workgroup below order 192, grid-wide launches per column
    from 192 up), then the windowed QR kernel with H and Z in HBM."""
    assert n > gs.batched_max_n(True)
    tally = {}
    for name, A, normal in families(n, True, seed=4):
        S = gs.gschur(A)
        check_case(oracle, name, A, S, normal, tally)
    report(f"windowed complex n={n}", tally)


@pytest.mark.parametrize("cplx", [True, False])
def test_families_batched(gs, oracle, cplx):
    """All families and orders as one batch (size bins, graph, Z log)."""
    sizes = (4, 5, 17, 32, 64, 96) if cplx else (4, 5, 17, 32, 64, 128)
    cases = [(name, A, normal) for n in sizes for name, A, normal in families(n, cplx, seed=1)]
    Ss, info = gs.gschur_batched([A for _, A, _ in cases])
    assert np.all(info == 0)
    tally = {}
    for (name, A, normal), S in zip(cases, Ss):
        check_case(oracle, name, A, S, normal, tally)
    report(f"batched {'complex' if cplx else 'real'}", tally)


def test_families_multishift(gs, oracle):
    """Real orders with multishift sweeps (from 256), whose diagonal order is
    their own: the invariants, the acceptance bounds and the eigenvalues."""
    for name, A, normal in families(300, False, seed=5):
        print(f"case {name} n=300", flush=True)
        S = gs.gschur(A)
        checks.schur_invariants(A, S.T, S.Z, S.values, TOL, normal=normal)
        assert checks.rel_backward(A, S.T, S.Z) <= 50 * 300 * EPS and checks.rel_orth(S.Z) <= 50 * 300 * EPS
        To, Zo, wo, cond, _ = oracle_result(oracle, A)
        checks.eigen_parity(A, S.values, wo, cond)


@pytest.mark.parametrize("cplx,n", [(True, 40), (True, 130), (False, 40), (False, 160)])
def test_families_plain(gs, oracle, cplx, n):
    """The plain unblocked global-memory kernel (GS_PLAIN)."""
    tally = {}
    for name, A, normal in families(n, cplx, seed=2):
        S = gs.gschur(A, plain=True)
        check_case(oracle, name, A, S, normal, tally)
    report(f"plain {'complex' if cplx else 'real'} n={n}", tally)


def test_families_large_real(gs, oracle):
    """The large real path (blocked Hessenberg, chunked QR) above n = 141."""
    n = 160
    assert n > gs.batched_max_n(False)
    tally = {}
    for name, A, normal in families(n, False, seed=3):
        S = gs.gschur(A)
        check_case(oracle, name, A, S, normal, tally)
    report("large real n=160", tally)


def test_short_qr_sweep(gs, oracle):
    """The 5 x 5 mode-4 matrix with cond 1/ulp that broke v0.4.0
    (test/complex.jl:156-166), complex and real, single and batched."""
    tally = {}
    for cplx in (True, False):
        mats = [gen.latme_like(5, 4, 1.0 / EPS, 1.0, 1.0, gen.stream(s, 78, int(cplx)), cplx) for s in range(8)]
        Ss, info = gs.gschur_batched(mats)
        assert np.all(info == 0)
        for A, S in zip(mats, Ss):
            check_case(oracle, "short-sweep-batched", A, S, False, tally)
            check_case(oracle, "short-sweep-single", A, gs.gschur(A), False, tally)
    report("short QR sweep", tally, 0.0)


def test_godunov(gs, oracle):
    """Godunov (test/testfuncs.jl:127-142): backward error below
    100 eps ||A|| as the reference demands; eigenvalues against the oracle
    within the cond-weighted bound."""
    A, exact, econd = gen.godunov()
    tally = {}
    for M in (A, A.astype(np.complex128)):
        for S in (gs.gschur(M), gs.gschur(M, plain=True), gs.gschur_batched([M])[0][0]):
            assert np.linalg.norm(S.Z @ S.T @ S.Z.conj().T - M) < 100 * EPS * np.linalg.norm(M)
            check_case(oracle, "godunov", M, S, False, tally)
    report("godunov", tally, 0.0)


def test_exceptional_shifts(gs, oracle):
    """The cyclic shift: the oracle needs the exceptional shifts (more than
    10 iterations on its first eigenvalue); the GPU runs the same number of
    QR sweeps as the oracle, kernel by kernel."""
    for cplx in (True, False):
        for n in (6, 24, 64):
            A = gen.cyclic_shift(n, cplx)
            _, _, _, _, stats = oracle_result(oracle, A)
            iters, sweeps = stats[0], stats[1]
            print(f"case cyclic n={n} cplx={cplx}: oracle iterations {iters}, sweeps {sweeps}", flush=True)
            assert iters > 10
            for plain in (False, True):
                S = gs.gschur(A, plain=plain)
                st = gs._lib.last_stats()
                check_case(oracle, "cyclic", A, S, True, {})
                assert st[0] == sweeps, (plain, st, stats)


def test_sweep_counts_match_oracle(gs, oracle):
    """The control flow (deflation tests, shifts, start rows) against the
    oracle's: the number of QR sweeps per matrix, single-matrix kernels.
    Rounding differences may move a deflation by a sweep in rare cases, so
    the share of exact matches is printed and must be high."""
    same = tot = 0
    for cplx in (True, False):
        for n in (8, 33, 64):
            for s in range(4):
                rng = gen.stream(s, 79, n)
                A = gen.ginibre_complex(n, rng) if cplx else gen.ginibre_real(n, rng)
                gs.gschur(A)
                st = gs._lib.last_stats()
                _, _, _, _, stats = oracle_result(oracle, A)
                tot += 1
                same += int(st[0] == stats[1])
    print(f"QR sweep counts equal to the oracle's: {same}/{tot}", flush=True)
    assert same >= 0.8 * tot


# ---------------------------------------------------------------- API paths
@pytest.mark.parametrize("cplx,n", [(True, 5), (True, 60), (True, 120), (False, 5), (False, 60), (False, 150)])
def test_hessenberg_input(gs, oracle, cplx, n):
    """gschur!(H::Hessenberg, Z) (GenericSchur.jl:194-335, :513-699) with Z
    (GS_HESSENBERG | GS_WANTZ: Z updated from the caller's transformation)
    and without Z; against the oracle's schur_hess on the same H, Z."""
    rng = gen.stream(5, 80, n)
    A = gen.ginibre_complex(n, rng) if cplx else gen.ginibre_real(n, rng)
    _, _, Q, H = oracle.hessenberg(A)
    S = gs.gschur_hessenberg_(H, Z=Q)
    checks.schur_invariants(A, S.T, S.Z, S.values, TOL)
    assert checks.rel_backward(A, S.T, S.Z) <= 50 * n * EPS
    To, Zo, wo, info = oracle.schur_hess(H, Q)
    assert info == 0
    To = np.triu(To) if cplx else np.triu(To, -1)
    VR = oracle.eigvecs(To, Zo, left=False)
    VL = oracle.eigvecs(To, Zo, left=True)
    cond = checks.eig_conditions(VR, VL)
    checks.eigen_parity(A, S.values, wo, cond)
    m = checks.schur_form_match(A, S.T, S.Z, S.values, To, Zo, wo, cond)
    print(f"case hessenberg n={n} cplx={cplx}: T/Z vs oracle {m}", flush=True)
    assert m in ("bitwise", "phases")
    S2 = gs.gschur_hessenberg_(H)
    assert S2.Z.shape == (0, 0)
    assert np.array_equal(S2.values, S.values) and np.array_equal(S2.T, S.T)


@pytest.mark.parametrize("n", [5, 120])
def test_checksd_argument_error(gs, oracle, n):
    """A complex Hessenberg matrix with a non-real subdiagonal is rejected
    (test/errors.jl:1-5), on the LDS-resident (n = 5) and plain (n = 120)
    kernels, as the oracle rejects it."""
    H = np.diag(np.full(n - 1, -1.0 + 1.0j), -1) + np.triu(gen.stream(6, 80, n).random((n, n)))
    assert oracle.schur_hess(H, checksd=True)[3] == oracle.NONREAL_SUB
    with pytest.raises(gs.ArgumentError):
        gs.gschur_hessenberg_(H)
    with pytest.raises(gs.ArgumentError):
        gs.gschur_hessenberg_(H, Z=np.eye(n, dtype=complex))


@pytest.mark.parametrize("cplx,n,plain", [(True, 32, False), (False, 32, False), (True, 120, True),
                                          (True, 120, False), (False, 160, True), (False, 200, False)])
def test_maxiter_unconverged(gs, oracle, cplx, n, plain):
    """maxiter = 1 raises UnconvergedException (GenericSchur.jl:234-236,
    :554-556) on every kernel, as in the oracle."""
    rng = gen.stream(7, 80, n)
    A = gen.ginibre_complex(n, rng) if cplx else gen.ginibre_real(n, rng)
    assert oracle.gschur(A, maxiter=1)[3] == oracle.UNCONVERGED
    with pytest.raises(gs.UnconvergedException):
        gs.gschur(A, maxiter=1, plain=plain)
    S = gs.gschur(A, plain=plain)  # and the handle still works
    assert checks.rel_backward(A, S.T, S.Z) <= 50 * n * EPS


@pytest.mark.parametrize("cplx", [True, False])
def test_eigvals_sorted(gs, oracle, cplx):
    """eigvals!(A) (pirates.jl:17-27): gschur!(A; wantZ=false), sorted by
    (Re, Im), equal to the oracle's sorted values; wantZ=false leaves T
    bitwise as with Z (the LDS kernels and the large path)."""
    for n in (7, 48, 150):
        rng = gen.stream(8, 80, n)
        A = gen.ginibre_complex(n, rng) if cplx else gen.ginibre_real(n, rng)
        v = gs.eigvals_(A)
        key = np.lexsort((v.imag, v.real))
        assert np.array_equal(key, np.arange(n))
        _, _, wo, cond, _ = oracle_result(oracle, A)
        checks.eigen_parity(A, v, wo, cond)
        if not cplx or n <= gs.batched_max_n(True):
            S = gs.gschur(A)
            S0 = gs.gschur(A, wantZ=False)
            assert np.array_equal(S.T, S0.T)


def test_quad_double_statement(gs, oracle):
    """Eigenvalue error of the batched kernels against the oracle run in
    quad-double (about 212 bits), on a sample of the batched complex and real
    workloads; printed (the accuracy statement) and held to the bound."""
    for cplx in (True, False):
        mats = gen.workload2(seed=11, count=8) if cplx else gen.workload3(seed=11, count=8)[0]
        Ss, info = gs.gschur_batched(mats)
        assert np.all(info == 0)
        worst = rmax = 0.0
        rels = []
        for A, S in zip(mats, Ss):
            n = A.shape[0]
            w_hp, _, inf = oracle.eig_hp(A, prec=2)
            assert inf == 0
            _, _, wo, cond, _ = oracle_result(oracle, A)
            perm, _ = checks.match_eigenvalues(w_hp, wo)
            ref = w_hp[perm]
            _, err = checks.match_eigenvalues(S.values, ref)
            bound = 10 * n * EPS * np.linalg.norm(A, 2) * cond
            worst = max(worst, float((err / bound).max()))
            rel = err / np.maximum(np.abs(ref), TINY)
            rmax = max(rmax, float(rel.max()))
            rels.append(rel)
            checks.eigen_parity(A, S.values, ref, cond)
        print(f"{'complex' if cplx else 'real'} batch sample vs quad-double: max err/bound {worst:.3e}, "
              f"max rel {rmax:.3e}, median rel {np.median(np.concatenate(rels)):.3e}", flush=True)


# --------------------------------------------------------- bad batch layouts
def test_batched_bad_offsets_rejected(gs):
    """A negative offset or overlapping matrix spans return GS_E_ARG before
    any launch: the outputs keep their contents (batched Schur, batched
    eigenvectors, VJP)."""
    from genericschur import _lib
    L = _lib.lib()
    h = _lib.handle()
    p = lambda a: ctypes.c_void_p(a.ctypes.data)
    ns = np.array([4, 4], dtype=np.int32)
    for off in (np.array([0, 8], dtype=np.int64), np.array([-16, 16], dtype=np.int64),
                np.array([16, 0 - 1], dtype=np.int64)):
        A = np.ones(64, dtype=np.complex128)
        T = np.full(64, 7.0 + 0j)
        Z = np.full(64, 7.0 + 0j)
        W = np.full(8, 7.0 + 0j)
        info = np.full(2, 9, dtype=np.int32)
        rc = L.gs_schur_batched_z(h, 2, p(ns), p(off), p(A), p(T), p(Z), p(W), p(info), _lib.GS_WANTZ)
        assert rc == _lib.GS_E_ARG, rc
        assert np.all(T == 7.0) and np.all(Z == 7.0) and np.all(W == 7.0) and np.all(info == 9)
        Ar = np.ones(64)
        Tr = np.full(64, 7.0)
        Zr = np.full(64, 7.0)
        rc = L.gs_schur_batched_d(h, 2, p(ns), p(off), p(Ar), p(Tr), p(Zr), p(W), p(info), 0)
        assert rc == _lib.GS_E_ARG and np.all(Tr == 7.0)
        V = np.full(64, 7.0 + 0j)
        rc = L.gs_trevc_batched_z(h, 2, p(ns), p(off), p(T), p(Z), p(V), 0, 1, 0)
        assert rc == _lib.GS_E_ARG and np.all(V == 7.0)
        g = np.zeros(8, dtype=np.complex128)
        Ab = np.full(64, 7.0)
        rc = L.gs_eig_vjp_batched_d(h, 2, p(ns), p(off), p(Tr), p(Tr), p(g), p(Ab), p(info), 0)
        assert rc == _lib.GS_E_ARG and np.all(Ab == 7.0)
    msg = L.gs_last_error(h).decode()
    assert "offset" in msg or "overlap" in msg


@pytest.mark.parametrize("n", [200, 800])
def test_single_complex_zlog_matches_direct(gs, oracle, n):
    """Complex orders from 768 up log Z's updates during the sweeps and
    replay the log onto Z's rows over the whole GPU afterwards; Z updated
    during the sweeps (the default below 768, zdirect above) and a log of
    one sweep (zlog_tiny: the QR kernel applies the log itself before almost
    every sweep, and the rest is replayed over the GPU) give the same T and Z
    bit for bit, and the logged form passes the invariants."""
    A = gen.ginibre_complex(n, gen.stream(31, 1, n))
    S = gs.gschur(A)
    Sd = gs.gschur(A, zdirect=True)
    St = gs.gschur(A, zlog_tiny=True)
    assert np.array_equal(S.T, Sd.T) and np.array_equal(S.T, St.T)
    assert np.array_equal(S.Z, Sd.Z) and np.array_equal(S.Z, St.Z)
    if n <= 200:
        check_case(oracle, "ginibre", A, S, False, {})
    else:
        eps = np.finfo(np.float64).eps
        assert checks.rel_backward(A, S.T, S.Z) <= 50 * n * eps
        assert checks.rel_orth(S.Z) <= 50 * n * eps
