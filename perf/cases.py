"""Performance cases: the work a program has this library do, over the range of its real use.

Each case goes through the public entry points (the Python API, or the C ABI
where only that takes device pointers).  Sizes and distributions are those
of gen.py, the tests and bench.py: complex and real Ginibre matrices, the
mixed-size batches, Hermitian matrices, and quasi-triangular Schur factors.

kind     entry points                                   outputs
batch    gschur_batched_device, gs_trevc_batched_z      values (diagonal order) and right eigenvectors, packed
vjp      SchurEigvals forward + backward                eigenvalue loss and the gradient of every matrix, packed
eigvals  eigvals_ (one matrix, host arrays)             values sorted by (re, im)
eigen    eigen_ (one matrix, host arrays)               sorted values, normalized eigenvectors
vectors  geigvecs (a Schur factorization, host arrays)  eigenvectors
heev     gs_heev_z / gs_heev_d (device batch)           values, vectors
herm     geigen_hermitian (one matrix, host arrays)     values, vectors

T and Z of a Schur form are determined up to a phase per column, and those phases follow the rounding: two correct
implementations differ in them by as much as the entries themselves.  So the cases end where a program's use of T and
Z ends, in eigenvalues, eigenvectors and gradients, each of which depends on all of T and Z.  Hermitian eigenvectors
have the same freedom, which run takes out as a program that compares them does: a real, positive first entry.
"""
import ctypes
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "genericschur.jl_amd"))
import genericschur as gs  # noqa: E402
from genericschur import _lib  # noqa: E402
from genericschur.autodiff import make_schur_eigvals  # noqa: E402

SchurEigvals = make_schur_eigvals(torch)


def listed():
    return [
        # the eigenvalues of one small matrix (a stability test inside a loop): a drop-in call, where launches,
        # copies and the latency of a few short sweeps count
        {"name": "eigvals-complex-13", "kind": "eigvals", "complex": True, "n": 13},
        # eigen of one small real matrix (balancing, Schur, triangularization, vectors): many short launches
        {"name": "eigen-real-24", "kind": "eigen", "complex": False, "n": 24},
        # many small systems at once, ragged orders (one block each of a larger model)
        {"name": "batch-complex-4-24", "kind": "batch", "count": 1000, "nmin": 4, "nmax": 24, "layout": 1},
        # bench.py's headline batch, with the eigenvectors that its T and Z are computed for
        {"name": "batch-complex-8-96", "kind": "batch", "count": 8192, "nmin": 8, "nmax": 96, "layout": 0},
        # bench.py's real batch (its Ginibre kind), forward and backward through the eigenvalues
        {"name": "vjp-16-128", "kind": "vjp", "count": 4096, "nmin": 16, "nmax": 128, "layout": 0},
        # a training step through the eigenvalues (bench.py's differentiation batch)
        {"name": "vjp-32-64", "kind": "vjp", "count": 2048, "nmin": 32, "nmax": 64, "layout": 0},
        # the reference's own single-matrix case, complex, above the LDS-resident orders
        {"name": "eigvals-complex-256", "kind": "eigvals", "complex": True, "n": 256},
        # one large real matrix, values only (blocked Hessenberg and chunked sweeps)
        {"name": "eigvals-real-1500", "kind": "eigvals", "complex": False, "n": 1500},
        # one medium real matrix with vectors: the large path with Z, then every step of eigen!
        {"name": "eigen-real-501", "kind": "eigen", "complex": False, "n": 501},
        # left eigenvectors of a large real Schur factorization
        {"name": "vectors-left-real-2048", "kind": "vectors", "complex": False, "n": 2048, "left": True},
        # batched Hermitian eigensystems (bench.py's Hermitian batch)
        {"name": "heev-complex-4096x64", "kind": "heev", "complex": True, "count": 4096, "n": 64},
        # one large Hermitian eigensystem
        {"name": "herm-complex-1000", "kind": "herm", "complex": True, "n": 1000},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["batch", "batch", "vjp", "eigvals", "eigen", "vectors", "heev", "herm"])
    cplx = rng.random() < 0.5
    if kind == "batch":
        nmin = rng.randint(1, 32)
        return {"kind": kind, "count": _log_int(rng, 16, 4096), "nmin": nmin, "nmax": rng.randint(nmin, 96),
                "layout": rng.randint(0, 1 << 20)}
    if kind == "vjp":
        nmin = rng.randint(1, 48)
        return {"kind": kind, "count": _log_int(rng, 16, 2048), "nmin": nmin, "nmax": rng.randint(nmin, 128),
                "layout": rng.randint(0, 1 << 20)}
    if kind == "eigvals":
        return {"kind": kind, "complex": cplx, "n": _log_int(rng, 2, 400 if cplx else 1500)}
    if kind == "eigen":
        return {"kind": kind, "complex": cplx, "n": _log_int(rng, 2, 300 if cplx else 600)}
    if kind == "vectors":
        return {"kind": kind, "complex": cplx, "n": _log_int(rng, 16, 1024 if cplx else 2048), "left": rng.random() < 0.5}
    if kind == "heev":
        return {"kind": kind, "complex": cplx, "count": _log_int(rng, 1, 4096), "n": rng.randint(2, 96 if cplx else 128)}
    return {"kind": kind, "complex": cplx, "n": _log_int(rng, 100, 1000)}


def _orders(case):
    """The orders of a ragged batch: the same for every seed (a program's layout), U{nmin..nmax}."""
    r = np.random.Generator(np.random.Philox(key=[case["layout"], case["count"]]))
    ns = r.integers(case["nmin"], case["nmax"] + 1, size=case["count"]).astype(np.int32)
    off = np.zeros(case["count"], dtype=np.int64)
    off[1:] = np.cumsum(ns[:-1].astype(np.int64) ** 2)
    return ns, off


def _ginibre(case, n, seed):
    r = np.random.Generator(np.random.Philox(key=[seed, 7]))
    a = r.standard_normal((n, n))
    if case["complex"]:
        a = (a + 1j * r.standard_normal((n, n))) * math.sqrt(0.5)
    return a


def _randn(shape, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return torch.randn(shape, generator=g, device="cuda", dtype=torch.float64)


def _hermitian(case, shape, seed):
    a = _randn(shape + ((2,) if case["complex"] else ()), seed)
    if case["complex"]:
        a = torch.view_as_complex(a)
    return (a + a.mH) * 0.5


def _schur_factor(case, seed):
    """A Schur factorization as gschur gives one: T (quasi-)triangular with half its real eigenvalues in standard-form
    pairs, a strictly upper part of the size that a Ginibre matrix's has, and an orthogonal / unitary Z."""
    n = case["n"]
    r = np.random.Generator(np.random.Philox(key=[seed, 11]))
    T = np.triu(r.standard_normal((n, n)), 1)
    z = _randn((n, n), seed)
    s = math.sqrt(n)
    if case["complex"]:
        T = (T + 1j * np.triu(r.standard_normal((n, n)), 1)) * math.sqrt(0.5)
        w = s * np.sqrt(r.random(n)) * np.exp(2j * np.pi * r.random(n))
        T[np.diag_indices(n)] = w
        z = torch.complex(z, _randn((n, n), seed + 1))
    else:
        w = s * r.uniform(-1.0, 1.0, n) + 0j
        for j in range(0, n - 1, 4):
            re, im = s * r.uniform(-1.0, 1.0), s * r.uniform(0.05, 1.0)
            T[j, j] = T[j + 1, j + 1] = re
            b = im * r.uniform(0.5, 2.0)
            T[j, j + 1], T[j + 1, j] = b, -im * im / b
            w[j] = complex(re, math.sqrt(abs(T[j, j + 1])) * math.sqrt(abs(T[j + 1, j])))
            w[j + 1] = w[j].conjugate()
        single = np.ones(n, dtype=bool)
        for j in range(0, n - 1, 4):
            single[j] = single[j + 1] = False
        T[np.diag_indices(n)] = np.where(single, w.real, np.diag(T))
    # columns orthonormal: Cholesky QR, twice
    for _ in range(2):
        L = torch.linalg.cholesky((z.mH.contiguous() @ z).cpu()).to(z.device)
        z = torch.linalg.solve_triangular(L, z.mH.contiguous(), upper=False).mH.contiguous()
    return gs.Schur(np.asfortranarray(T), np.asfortranarray(z.cpu().numpy()), w)


def prepare(case, seed):
    k = case["kind"]
    s = {"case": case}
    if k in ("eigvals", "eigen"):
        s["A"] = _ginibre(case, case["n"], seed)
    elif k in ("batch", "vjp"):
        ns, off = _orders(case)
        s["ns"], s["off"] = ns, off
        m = int((ns.astype(np.int64) ** 2).sum())
        if k == "batch":
            s["A"] = torch.view_as_complex(_randn((m, 2), seed) * math.sqrt(0.5))
            for name in ("T", "Z", "V"):
                s[name] = torch.zeros_like(s["A"])
            s["W"] = torch.zeros(int(ns.sum()), dtype=torch.complex128, device="cuda")
            s["info"] = torch.zeros(len(ns), dtype=torch.int32, device="cuda")
        else:
            s["A"] = _randn(m, seed).requires_grad_(True)
    elif k == "vectors":
        s["S"] = _schur_factor(case, seed)
    elif k == "heev":
        c, n = case["count"], case["n"]
        s["A"] = _hermitian(case, (c, n, n), seed).contiguous()
        s["W"] = torch.zeros((c, n), dtype=torch.float64, device="cuda")
        s["V"] = torch.zeros_like(s["A"])
        s["info"] = torch.zeros(c, dtype=torch.int32, device="cuda")
    else:
        s["A"] = _hermitian(case, (case["n"], case["n"]), seed).cpu().numpy()
    torch.cuda.synchronize()
    return s


def _ptr(t):
    return ctypes.c_void_p(t.data_ptr())


def _unit_first(V, axis):
    """Columns scaled to a real, positive first entry (axis: the columns' index along the last two)."""
    f = V[..., :1, :] if axis == -1 else V[..., :, :1]
    return V * (f.conj() / abs(f))


def run(s):
    case = s["case"]
    k = case["kind"]
    if k == "batch":
        ns, off = s["ns"], s["off"]
        gs.gschur_batched_device(ns, off, s["A"], s["T"], s["Z"], s["W"], s["info"], True)
        h = _lib.handle()
        rc = _lib.lib().gs_trevc_batched_z(h, len(ns), ctypes.c_void_p(ns.ctypes.data), ctypes.c_void_p(off.ctypes.data),
                                           _ptr(s["T"]), _ptr(s["Z"]), _ptr(s["V"]), 0, 1, _lib.GS_DEVICE_PTRS)
        _lib.check(rc, h, "gs_trevc_batched_z")
        return [s["W"], s["V"], s["info"]]
    if k == "vjp":
        s["A"].grad = None
        w = SchurEigvals.apply(s["A"], s["ns"], s["off"])
        # the same function of every eigenvalue, so the gradient does not depend on their order
        loss = (w.real.square() + w.imag.square()).mean()
        loss.backward()
        return [loss.detach(), s["A"].grad]
    if k == "eigvals":
        return [gs.eigvals_(s["A"])]
    if k == "eigen":
        E = gs.eigen_(s["A"])
        return [E.values, E.vectors]
    if k == "vectors":
        return [gs.geigvecs(s["S"], left=case["left"])]
    if k == "heev":
        c, n = case["count"], case["n"]
        h = _lib.handle()
        f = _lib.lib().gs_heev_z if case["complex"] else _lib.lib().gs_heev_d
        rc = f(h, c, n, _ptr(s["A"]), n, n * n, 0, _ptr(s["W"]), _ptr(s["V"]), n, n * n, _ptr(s["info"]),
               _lib.GS_WANTZ | _lib.GS_SORT | _lib.GS_DEVICE_PTRS)
        _lib.check(rc, h, "gs_heev")
        return [s["W"], _unit_first(s["V"], -2), s["info"]]
    E = gs.geigen_hermitian(s["A"])
    return [E.values, _unit_first(E.vectors, -1)]


def work(case):
    """Inputs read once and outputs written once, and the method's operations (Golub & Van Loan, 4th ed., 7.5.6 and
    8.3.3: real Schur form with Z 25 n^3, values only 10 n^3, vectors of a triangular matrix n^3 and the
    back-transform 2 n^3; symmetric with vectors 9 n^3; complex four times as many)."""
    k = case["kind"]
    if k in ("batch", "vjp"):
        ns = _orders(case)[0].astype(np.float64)
        n1, n2, n3 = float(ns.sum()), float((ns ** 2).sum()), float((ns ** 3).sum())
        if k == "batch":
            return {"bytes": 2 * 16 * n2 + 16 * n1, "flops": 112 * n3}
        # backward: both sets of (complex) vectors, and the sum of the outer products
        return {"bytes": 2 * 8 * n2, "flops": (25 + 6 + 4) * n3}
    n = float(case["n"])
    c, e = (4.0, 16.0) if case["complex"] else (1.0, 8.0)
    if k == "eigvals":
        return {"bytes": n * n * e + 16 * n, "flops": 10 * c * n ** 3}
    if k == "eigen":
        return {"bytes": n * n * (e + 16) + 16 * n, "flops": 28 * c * n ** 3}
    if k == "vectors":
        return {"bytes": n * n * (1.5 * e + 16), "flops": 3 * c * n ** 3}
    m = float(case.get("count", 1))
    return {"bytes": m * (2 * n * n * e + 8 * n), "flops": m * 9 * c * n ** 3}


def tolerance(case):
    # Measured: the path on inputs perturbed by 2e-16 relative (the effect of another order of its sums) against itself,
    # over the listed cases and 40 drawn ones: values up to 1.6e-14; vectors and gradients 1e-14 to 1e-13 as a rule,
    # with the nearly defective pairs of single matrices up to 1.7e-12 (their share falls off slowly, hence the margin)
    return {"rel": 1e-13 if case["kind"] == "eigvals" else 1e-11}


def _eig(A, left):
    """Values and unit eigenvectors (columns, the first largest entry real and positive) of A, or of A^H for left."""
    w, X = np.linalg.eig(A.conj().T if left else A)
    return (w.conj() if left else w), _unit_largest(X)


def _unit_largest(X):
    X = X / np.linalg.norm(X, axis=0)
    f = X[np.argmax(abs(X), axis=0), np.arange(X.shape[1])]
    return X * (f.conj() / abs(f))


def exact(case, seed):
    k = case["kind"]
    if k == "batch":
        return None  # the order of the diagonal is the iteration's own
    if k == "vectors" and case["n"] > 700:
        return None
    s = prepare(case, seed)
    if k == "vjp":
        ns, off = s["ns"], s["off"]
        A = s["A"].detach().cpu().numpy()
        G = np.zeros_like(A)
        loss, tot = 0.0, int(ns.sum())
        for n, o in zip(ns, off):
            w, X = np.linalg.eig(A[o:o + n * n].reshape((n, n), order="F"))
            loss += float((w.real ** 2 + w.imag ** 2).sum()) / tot
            # sum_k gbar_k y_k x_k^H / conj(y_k^H x_k) = X^-H diag(gbar) X^H
            G[o:o + n * n] = np.linalg.solve(X.conj().T, (2.0 / tot * w)[:, None] * X.conj().T).real.reshape(-1, order="F")
        return [np.array(loss), G]
    if k == "vectors":
        S = s["S"]
        w, X = _eig(S.T, case["left"])
        order = [int(np.argmin(abs(w - v))) for v in S.values]
        return [_unit_largest(S.Z @ X[:, order])]
    if k == "heev":
        # the buffer is read column by column: the transpose of the tensor's matrices
        w, V = np.linalg.eigh(s["A"].cpu().numpy().transpose(0, 2, 1))
        return [w, _unit_first(V, -1).transpose(0, 2, 1), None]
    if k == "herm":
        w, V = np.linalg.eigh(s["A"])
        return [w, _unit_first(V, -1)]
    if k == "eigvals":
        w = np.linalg.eigvals(s["A"])
        return [w[np.lexsort((w.imag, w.real))]]
    w, X = _eig(s["A"], False)
    p = np.lexsort((w.imag, w.real))
    return [w[p], X[:, p]]
