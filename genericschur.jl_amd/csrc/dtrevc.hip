// Eigenvectors of a real standard-form Schur factorization (T
// quasi-triangular, Z) on gfx950, following GenericSchur.jl:
//   right   vectors.jl:133-362 (dtrevc-style)
//   left    vectors.jl:462-698
//   1x1 / 2x2 solves  _xsolve util.jl:698-751, _safe_lu_solve! :603-687
//   unit 2-norm, largest entry real: _enormalize! util.jl:572-592
//
// Same organisation as the complex kernels (trevc_grid.h): one wavefront per
// eigenvector (or conjugate pair) with the complex solution in its lanes.
// The conjugate partner of a complex pair is written last as the conjugate
// of the finished column, which equals the reference's copy-then-normalise.
#include <algorithm>

#include "dev_common.h"
#include "internal.h"
#include "trevc_grid.h"
#include "wavevec.h"

namespace gs {

// One step of a substitution, (a A - lam I) x = s B for the 1 x 1 or 2 x 2
// diagonal block A at the step (_xsolve, util.jl:698-751, _safe_lu_solve!
// :603-687, complete pivoting), split in two: what does not depend on B is
// factored for the 64 rows of a chunk at once, one row per lane (DFac in
// LDS); a step then reads its factors as broadcasts and applies them to B.
// The operations on B are those of the unsplit form, in its order.  The
// factorization's moduli and divisions are most of a step's instructions,
// and every lane used to repeat them at every step.
struct DFac {
  zd l;       // 2 x 2: A21 / A11 after pivoting; 1 x 1: Smith's (ratio, denominator)
  zd u;       // 2 x 2: A12 / A11
  zd t0, t1;  // 2 x 2: 1 / A11, 1 / A22
  double a0, a3;  // 2 x 2: |A11|, |A22|; 1 x 1: a0 = abs1 of the pivot
  double beta;    // the column norm(s) of the overflow guard
  double flags;   // bits below
};
enum { DF_TWO = 1, DF_IP = 2, DF_JP = 4, DF_SMALL = 8, DF_SWAP = 16 };

GS_DEV void dfac1(DFac& f, double diag, zd lam, double smin, double beta) {
  smin = fmax(smin, 2.0 * GS_FMIN);
  double csr = diag - lam.x, csi = -lam.y;
  double cnorm = fabs(csr) + fabs(csi);
  if (cnorm < smin) {
    csr = smin;
    csi = 0.0;
    cnorm = smin;
  }
  // Smith's division by (csr, csi): the part without the numerator
  const bool sw = fabs(csi) > fabs(csr);
  const double r = sw ? csr / csi : csi / csr;
  const double d = sw ? csr * r + csi : csr + csi * r;
  f.l = zmk(r, d);
  f.a0 = cnorm;
  f.beta = beta;
  f.flags = sw ? (double)DF_SWAP : 0.0;
}

// A column-major: a11, a21, a12, a22
GS_DEV void dfac2(DFac& f, double a11, double a21, double a12, double a22, zd lam, double smin, double beta) {
  smin = fmax(smin, 2.0 * GS_FMIN);
  zd A[4] = {zr(a11) - lam, zr(a21), zr(a12), zr(a22) - lam};
  int fl = DF_TWO;
  const double cmax = fmax(fmax(zabs1(A[0]), zabs1(A[1])), fmax(zabs1(A[2]), zabs1(A[3])));
  f.beta = beta;
  if (cmax < smin) {
    f.flags = (double)(fl | DF_SMALL);
    return;
  }
  const double m0 = zabs(A[0]), m1 = zabs(A[1]), m2 = zabs(A[2]), m3 = zabs(A[3]);
  const double sm = fmax(GS_EPS * fmax(fmax(m0, m1), fmax(m2, m3)), GS_FMIN / GS_EPS);
  // complete pivoting: the last maximal entry in (row, column) order
  int ip = 0, jp = 0;
  double xm = 0.0;
  if (m0 >= xm) { xm = m0; ip = 0; jp = 0; }
  if (m2 >= xm) { xm = m2; ip = 0; jp = 1; }
  if (m1 >= xm) { xm = m1; ip = 1; jp = 0; }
  if (m3 >= xm) { xm = m3; ip = 1; jp = 1; }
  if (ip) {
    const zd t = A[0], u = A[2];
    A[0] = A[1];
    A[1] = t;
    A[2] = A[3];
    A[3] = u;
    fl |= DF_IP;
  }
  if (jp) {
    const zd t = A[0], u = A[1];
    A[0] = A[2];
    A[2] = t;
    A[1] = A[3];
    A[3] = u;
    fl |= DF_JP;
  }
  if (zabs(A[0]) < sm) A[0] = zr(sm);
  A[1] = A[1] / A[0];
  A[3] = A[3] - A[1] * A[2];
  if (zabs(A[3]) < sm) A[3] = zr(sm);
  f.l = A[1];
  f.t1 = zdiv(zr(1.0), A[3]);
  f.t0 = zdiv(zr(1.0), A[0]);
  f.u = f.t0 * A[2];
  f.a0 = zabs(A[0]);
  f.a3 = zabs(A[3]);
  f.flags = (double)fl;
}

GS_DEV double dapply1(const DFac& f, int fl, zd& B, double& xnorm) {
  const double bignum = 1.0 / (2.0 * GS_FMIN);
  double s = 1.0;
  const double bnorm = zabs1(B);
  if (f.a0 < 1.0 && bnorm > 1.0 && bnorm > bignum * f.a0) s = 1.0 / bnorm;
  const zd a = B * s;
  const bool sw = (fl & DF_SWAP) != 0;
  const double p = sw ? a.y : a.x, q = sw ? a.x : a.y;
  const double x = (p + q * f.l.x) / f.l.y, y = (q - p * f.l.x) / f.l.y;
  B = zmk(x, sw ? -y : y);
  xnorm = zabs1(B);
  return s;
}

GS_DEV double dapply2(const DFac& f, int fl, zd* B, double smin, double& xnorm) {
  double s = 1.0;
  if (fl & DF_SMALL) {
    const double bignum = 1.0 / (2.0 * GS_FMIN);
    smin = fmax(smin, 2.0 * GS_FMIN);
    const double bnorm = fmax(zabs1(B[0]), zabs1(B[1]));
    if (smin < 1.0 && bnorm > 1.0 && bnorm > bignum * smin) s = 1.0 / bnorm;
    const double t = s / smin;
    B[0] = B[0] * t;
    B[1] = B[1] * t;
  } else {
    if (fl & DF_IP) {
      const zd t = B[0];
      B[0] = B[1];
      B[1] = t;
    }
    B[1] = B[1] - f.l * B[0];
    const double a8 = 8.0 * (GS_FMIN / GS_EPS);
    // |b| <= abs1(b): the moduli only where the cheap bound cannot decide
    if (!(a8 * zabs1(B[0]) <= f.a0 && a8 * zabs1(B[1]) <= f.a3) &&
        ((a8 * zabs(B[0]) > f.a0) || (a8 * zabs(B[1]) > f.a3))) {
      s = (1.0 / 8.0) / fmax(zabs(B[0]), zabs(B[1]));
      B[0] = B[0] * s;
      B[1] = B[1] * s;
    }
    B[1] = B[1] * f.t1;
    B[0] = B[0] * f.t0;
    B[0] = B[0] - f.u * B[1];
    if (fl & DF_JP) {
      const zd t = B[0];
      B[0] = B[1];
      B[1] = t;
    }
  }
  xnorm = sqrt(zabs2(B[0]) + zabs2(B[1]));
  return s;
}

// The columns of T a substitution reads.  Up to R = 8 entries per lane the two
// that the next step needs are loaded a step ahead; above, each entry is read
// where it is used.
template <int R, class TA, bool LEFT> struct DCols {
  static constexpr bool PF = R <= 8;
  static constexpr int NR = PF ? R : 1;
  const TA& Tc;
  int n;  // rows and columns that may be read
  double ca[NR], cb[NR], na[NR], nb[NR];
  // line j: column j (right) or row j (left) of T, lanes along it
  GS_DEV double at(int i, int j) const { return LEFT ? Tc(j, i) : Tc(i, j); }
  GS_DEV void load(double (&c)[NR], int j) const {
    if constexpr (PF) {
#pragma unroll
      for (int q = 0; q < R; ++q) c[q] = at(min((int)(threadIdx.x & 63) + 64 * q, n - 1), min(max(j, 0), n - 1));
    }
  }
  static constexpr int D = LEFT ? 1 : -1;
  // lines j and j + D in ca, cb; the two after them on the way
  GS_DEV void start(int j) {
    load(ca, j);
    load(cb, j + D);
  }
  GS_DEV void ahead(int j) {
    load(na, j + 2 * D);
    load(nb, j + 3 * D);
  }
  GS_DEV void advance(bool two) {
    if constexpr (PF) {
#pragma unroll
      for (int q = 0; q < R; ++q) {
        ca[q] = two ? na[q] : cb[q];
        cb[q] = two ? nb[q] : na[q];
      }
    }
  }
  GS_DEV double first(int q, int i, int j) const {
    if constexpr (PF) return ca[q];
    else return at(i, j);
  }
  GS_DEV double second(int q, int i, int j) const {
    if constexpr (PF) return cb[q];
    else return at(i, j);
  }
};

// ------------------------------------------------------------- right
// Solution for column ki (0-based) with ip = 0 (real wr) or -1 (pair,
// lambda = wr + i wi, ki the second row of the block).  Entries 0..ki hold
// the vector on exit.
template <int R, class TA, class VEC> GS_DEV void dsolve_right(const TA& Tc, const double* sub, const double* tnorms, int ki,
                                                     int ip, double smallnum, double bignum, VEC& v, DFac* fac) {
  const int lane = threadIdx.x & 63;
  const double ulp = GS_EPS;
  const double wr = Tc(ki, ki);
  const double wi = (ip == 0) ? 0.0 : sqrt(fabs(sub[ki - 1])) * sqrt(fabs(Tc(ki - 1, ki)));
  const double smin = fmax(ulp * (fabs(wr) + fabs(wi)), smallnum);
  const zd lam = zmk(wr, wi);
  int jtop;
  if (ip == 0) {
#pragma unroll
    for (int q = 0; q < R; ++q) {
      const int i = lane + 64 * q;
      v.v[q] = (i < ki) ? zr(-Tc(i, ki)) : (i == ki ? zr(1.0) : zr(0.0));
    }
    jtop = ki - 1;
  } else {
    zd a, c;
    if (fabs(Tc(ki - 1, ki)) >= fabs(sub[ki - 1])) {
      a = zr(1.0);
      c = zmk(0.0, wi / Tc(ki - 1, ki));
    } else {
      a = zr(-wi / sub[ki - 1]);
      c = zmk(0.0, 1.0);
    }
#pragma unroll
    for (int q = 0; q < R; ++q) {
      const int i = lane + 64 * q;
      zd val = zr(0.0);
      if (i < ki - 1) val = zmk(-a.x * Tc(i, ki - 1), -(c.y * Tc(i, ki)));
      else if (i == ki - 1) val = a;
      else if (i == ki) val = c;
      v.v[q] = val;
    }
    jtop = ki - 2;
  }
  int j = jtop;
  DCols<R, TA, false> dc{Tc, ki + 1};
  if (j >= 0) dc.start(j);
  int chunk = -1;  // the 64 rows whose factors are in fac
  while (j >= 0) {
    dc.ahead(j);
    if ((j >> 6) != chunk) {
      chunk = j >> 6;
      const int i = 64 * chunk + lane;
      wsync();
      if (i <= j) {
        DFac f;
        if (i > 0 && sub[i - 1] != 0.0)
          dfac2(f, Tc(i - 1, i - 1), sub[i - 1], Tc(i - 1, i), Tc(i, i), lam, smin, fmax(tnorms[i - 1], tnorms[i]));
        else
          dfac1(f, Tc(i, i), lam, smin, tnorms[i]);
        fac[lane] = f;
      }
      wsync();
    }
    const DFac f = fac[j & 63];
    const int fl = __builtin_amdgcn_readfirstlane((int)f.flags);
    const bool two = (fl & DF_TWO) != 0;
    zd B[2] = {v.get(j), zr(0.0)};
    double t1, vscale;
    if (!two) {
      vscale = dapply1(f, fl, B[0], t1);
    } else {
      B[1] = B[0];
      B[0] = v.get(j - 1);
      vscale = dapply2(f, fl, B, smin, t1);
    }
    // t1 > 1 && beta > bignum / t1, the quotient only near the limit
    if (t1 > 1.0 && !(f.beta * t1 <= 0.5 * bignum) && f.beta > bignum / t1) {
      B[0] = B[0] / t1;
      if (two) B[1] = B[1] / t1;
      vscale /= t1;
    }
    if (vscale != 1.0) {
#pragma unroll
      for (int q = 0; q < R; ++q)
        if (lane + 64 * q <= ki) v.v[q] = v.v[q] * vscale;
    }
    if (!two) {
      v.set(j, B[0]);
#pragma unroll
      for (int q = 0; q < R; ++q) {
        const int i = lane + 64 * q;
        if (i < j) v.v[q] = v.v[q] - B[0] * dc.first(q, i, j);
      }
    } else {
      v.set(j - 1, B[0]);
      v.set(j, B[1]);
#pragma unroll
      for (int q = 0; q < R; ++q) {
        const int i = lane + 64 * q;
        if (i < j - 1) v.v[q] = (v.v[q] - B[0] * dc.second(q, i, j - 1) - B[1] * dc.first(q, i, j));
      }
    }
    j -= two ? 2 : 1;
    dc.advance(two);
  }
}

// -------------------------------------------------------------- left
// Solution for column ki with ip = 0 or 1 (pair, ki the first row of the
// block, lambda = wr - i wi in the solves).  Entries ki..n-1 hold it.
// Forward substitution in axpy form; the reference's overflow guards
// (vmax, vcrit) and the j1 = j + 1 quirk of vectors.jl:627 are kept.
template <int R, class TA, class VEC> GS_DEV void dsolve_left(const TA& Tc, const double* sub, const double* tnorms, int n,
                                                    int ki, int ip, double smallnum, double bignum, VEC& v,
                                                    DFac* fac) {
  const int lane = threadIdx.x & 63;
  const double ulp = GS_EPS;
  const double wr = Tc(ki, ki);
  const double wi = (ip == 0) ? 0.0 : sqrt(fabs(Tc(ki, ki + 1))) * sqrt(fabs(sub[ki]));
  const double smin = fmax(ulp * (fabs(wr) + fabs(wi)), smallnum);
  int jstart;
  zd lam;
  if (ip == 0) {
#pragma unroll
    for (int q = 0; q < R; ++q) {
      const int i = lane + 64 * q;
      v.v[q] = (i > ki && i < n) ? zr(-Tc(ki, i)) : (i == ki ? zr(1.0) : zr(0.0));
    }
    jstart = ki + 1;
    lam = zr(wr);
  } else {
    zd a, c;
    if (fabs(Tc(ki, ki + 1)) >= fabs(sub[ki])) {
      a = zr(wi / Tc(ki, ki + 1));
      c = zmk(0.0, 1.0);
    } else {
      a = zr(1.0);
      c = zmk(0.0, -wi / sub[ki]);
    }
#pragma unroll
    for (int q = 0; q < R; ++q) {
      const int i = lane + 64 * q;
      zd val = zr(0.0);
      if (i > ki + 1 && i < n) val = zmk(-a.x * Tc(ki, i), -(c.y * Tc(ki + 1, i)));
      else if (i == ki) val = a;
      else if (i == ki + 1) val = c;
      v.v[q] = val;
    }
    jstart = ki + 2;
    lam = zmk(wr, -wi);
  }
  const bool pair = (ip != 0);
  double vmax = 1.0;  // the reference's vcrit is bignum / vmax
  int j = jstart;
  DCols<R, TA, true> dc{Tc, n};
  if (j < n) dc.start(j);
  int chunk = -1;
  while (j < n) {
    dc.ahead(j);
    if ((j >> 6) != chunk) {
      chunk = j >> 6;
      const int i = 64 * chunk + lane;
      wsync();
      if (i >= j && i < n) {
        DFac f;
        // with a pair the 2 x 2 guard reads tnorms[i-1]
        if (i < n - 1 && sub[i] != 0.0)
          dfac2(f, Tc(i, i), Tc(i, i + 1), sub[i], Tc(i + 1, i + 1), lam, smin,
                fmax(tnorms[pair ? i - 1 : i + 1], tnorms[i]));
        else
          dfac1(f, Tc(i, i), lam, smin, tnorms[i]);
        fac[lane] = f;
      }
      wsync();
    }
    const DFac f = fac[j & 63];
    const int fl = __builtin_amdgcn_readfirstlane((int)f.flags);
    const bool two = (fl & DF_TWO) != 0;
    // beta > bignum / vmax, the quotient only near the limit
    if (!(f.beta * vmax <= 0.5 * bignum) && f.beta > bignum / vmax) {
      const double t1 = 1.0 / vmax;
#pragma unroll
      for (int q = 0; q < R; ++q)
        if (lane + 64 * q >= ki) v.v[q] = v.v[q] * t1;
      vmax = 1.0;
    }
    zd B[2] = {v.get(j), zr(0.0)};
    double xn;
    double vscale;
    if (!two) {
      vscale = dapply1(f, fl, B[0], xn);
    } else {
      B[1] = v.get(j + 1);
      vscale = dapply2(f, fl, B, smin, xn);
    }
    if (vscale != 1.0) {
#pragma unroll
      for (int q = 0; q < R; ++q)
        if (lane + 64 * q >= ki) v.v[q] = v.v[q] * vscale;
    }
    // abs1 bounds the modulus
    const double b1 = two ? fmax(zabs1(B[0]), zabs1(B[1])) : zabs1(B[0]);
    if (pair) vmax = fmax(b1, vmax);
    else if (!(b1 <= vmax)) vmax = fmax(two ? fmax(zabs(B[0]), zabs(B[1])) : zabs(B[0]), vmax);
    // remove x from the later right-hand sides
    v.set(j, B[0]);
    if (!two) {
#pragma unroll
      for (int q = 0; q < R; ++q) {
        const int i = lane + 64 * q;
        if (i > j && i < n) v.v[q] = v.v[q] - B[0] * dc.first(q, i, j);
      }
    } else {
      v.set(j + 1, B[1]);
#pragma unroll
      for (int q = 0; q < R; ++q) {
        const int i = lane + 64 * q;
        if (i > j + 1 && i < n) v.v[q] = v.v[q] - B[0] * dc.first(q, i, j) - B[1] * dc.second(q, i, j + 1);
      }
    }
    j += two ? 2 : 1;
    dc.advance(two);
  }
}

template <int R, class VEC> GS_DEV void enormalize_w(VEC& v, int n);

// max-|.| normalisation of a finished column (maximum(abs, ...) or abs1)
template <int R, class VEC> GS_DEV void scale_by_max(VEC& y, int lo, int hi, bool use_abs1) {
  const int lane = threadIdx.x & 63;
  double m = 0.0;
#pragma unroll
  for (int q = 0; q < R; ++q) {
    const int i = lane + 64 * q;
    if (i >= lo && i < hi) m = fmax(m, use_abs1 ? zabs1(y.v[q]) : zabs(y.v[q]));
  }
  m = wave_max(m);
  const double s = 1.0 / m;
#pragma unroll
  for (int q = 0; q < R; ++q) y.v[q] = y.v[q] * s;
}

template <int R, class VEC> GS_DEV void enormalize_w(VEC& v, int n) {
  const int lane = threadIdx.x & 63;
  double am = 0.0;
#pragma unroll
  for (int q = 0; q < R; ++q)
    if (lane + 64 * q < n) am = fmax(am, fmax(fabs(v.v[q].x), fabs(v.v[q].y)));
  am = wave_max(am);
  double ss = 0.0, best = -1.0;
  int bi = 0x7fffffff;
#pragma unroll
  for (int q = 0; q < R; ++q) {
    const int i = lane + 64 * q;
    if (i < n) {
      const double a = v.v[q].x / am, b = v.v[q].y / am;
      ss += a * a + b * b;
      const double u = zabs2(v.v[q]);
      if (u > best) {
        best = u;
        bi = i;
      }
    }
  }
  ss = wave_sum(ss);
  const double nrm = am * sqrt(ss);
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    const double ob = __shfl_xor(best, o, 64);
    const int oi = __shfl_xor(bi, o, 64);
    if (ob > best || (ob == best && oi < bi)) {
      best = ob;
      bi = oi;
    }
  }
  bi = min(bi, n - 1);  // no entry compared (NaN throughout): any of them, within the vector
  const zd vi0 = v.get(bi);
  const zd tt = ((1.0 / nrm) * zconj(vi0)) / sqrt(zabs2(vi0));
#pragma unroll
  for (int q = 0; q < R; ++q) v.v[q] = v.v[q] * tt;
  const zd r0 = v.get(bi);
  v.set(bi, zr(r0.x));
}

// Column norms, subdiagonal and block kinds, one wavefront per column.
// kind: 0 a real eigenvalue; the row of a 2 x 2 block that solves its pair
// (right: the second, -1; left: the first, 1); 2 its partner.  The reference
// walks ki = n..1 (right) or 1..n (left) and skips the partner of each pair,
// so within a run of nonzero subdiagonal entries (one entry, for a
// quasi-triangular T) the distance from the end where the walk enters it
// decides.
template <class SUB> GS_DEV int dtrevc_kind(const SUB& sub, int j, bool left) {
  int d = 0;
  if (left) {
    while (sub(j - 1 - d) != 0.0) ++d;
    return (d & 1) ? 2 : (sub(j) != 0.0 ? 1 : 0);
  }
  while (sub(j + d) != 0.0) ++d;
  return (d & 1) ? 2 : (sub(j - 1) != 0.0 ? -1 : 0);
}
__global__ void __launch_bounds__(256) dtrevc_norms_kernel(TrevcArgs a) {
  const TrevcMat<double> t = trevc_mat<double>(a, blockIdx.y);
  const int n = t.n;
  const int j = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (j >= n) return;
  double s = 0.0;
  for (int i = lane; i < j; i += 64) s += fabs(t.T[i + (int64_t)j * t.ldt]);
  s = wave_sum(s);
  if (lane != 0) return;
  auto sub = [&](int i) { return (i >= 0 && i + 1 < n) ? t.T[(i + 1) + (int64_t)i * t.ldt] : 0.0; };
  t.cn[j] = s;
  t.sub[j] = sub(j);
  t.kind[j] = dtrevc_kind(sub, j, a.left != 0);
}

// workgroup (t, matrix) solves column n-1-t (right) or t (left): the longest
// solves are dispatched first
template <int R, bool LEFT> __global__ void __launch_bounds__(64) dtrevc_solve_kernel(TrevcArgs a) {
  extern __shared__ double smem[];
  const TrevcMat<double> t = trevc_mat<double>(a, blockIdx.y);
  const int n = t.n, lane = threadIdx.x & 63, b = blockIdx.x;
  if (b >= n) return;
  const int ki = LEFT ? b : n - 1 - b;
  const int kd = t.kind[ki];
  zd* xo = t.X + (int64_t)ki * n;
  if (kd == 2) {
    for (int i = lane; i < n; i += 64) xo[i] = zr(0.0);
    return;
  }
  const double ulp = GS_EPS;
  const double smallnum = GS_FMIN * ((double)n / ulp);  // vectors.jl:146,475
  const double bignum = (1.0 - ulp) / smallnum;
  WaveVec<R> v;
  wavevec_bind(v.v, smem);
  typedef typename std::conditional<LEFT, TransG<double>, ColG<double>>::type TA;
  const TA Tc = LEFT ? TA{t.Tt, n} : TA{t.T, t.ldt};
  __shared__ DFac fac[64];
  if (!LEFT) dsolve_right<R>(Tc, t.sub, t.cn, ki, kd, smallnum, bignum, v, fac);
  else dsolve_left<R>(Tc, t.sub, t.cn, n, ki, kd, smallnum, bignum, v, fac);
#pragma unroll
  for (int q = 0; q < R; ++q) {
    const int i = lane + 64 * q;
    if (i < n) xo[i] = v.v[q];
  }
}

// Scaling and normalization of column ki, and its store with a pair's partner.
// y: the column of Z X (whole), or without Z of X (entries lo .. hi - 1).  edge:
// a column of Z itself, which the reference only normalizes.
template <int R, class VEC> GS_DEV void dtrevc_store(const TrevcMat<double>& t, VEC& y, int ki, int kd, bool left,
                                                     bool normalize, bool edge) {
  const int n = t.n, lane = threadIdx.x & 63;
  const bool conj = !left && kd == -1;
  auto flip = [&] {
#pragma unroll
    for (int q = 0; q < R; ++q) y.v[q] = zconj(y.v[q]);
  };
  if (t.Z) {
    if (!edge) {
      scale_by_max<R>(y, 0, n, false);
      if (conj) flip();
    }
  } else {
    if (conj) flip();
    scale_by_max<R>(y, left ? ki : 0, left ? n : ki + 1, kd != 0);
  }
  if (normalize) enormalize_w<R>(y, n);
  zd* vo = t.V + (int64_t)ki * t.ldv;
  zd* po = t.V + (int64_t)(left ? ki + 1 : ki - 1) * t.ldv;
#pragma unroll
  for (int q = 0; q < R; ++q) {
    const int r = lane + 64 * q;
    if (r < n) {
      const zd z = y.v[q];
      vo[r] = z;
      // the conjugate partner of a pair
      if (kd != 0) po[r] = zconj(z);
    }
  }
}

GS_DEV bool dtrevc_edge(int n, int ki, int kd, bool left) { return kd == 0 && ki == (left ? n - 1 : 0); }

template <int R> __global__ void __launch_bounds__(64) dtrevc_finish_kernel(TrevcArgs a) {
  extern __shared__ double smem[];
  const TrevcMat<double> t = trevc_mat<double>(a, blockIdx.y);
  const int n = t.n, lane = threadIdx.x & 63, ki = blockIdx.x;
  if (ki >= n) return;
  const bool left = a.left != 0;
  const int kd = t.kind[ki];
  if (kd == 2) return;
  WaveVec<R> y;
  wavevec_bind(y.v, smem);
  const int lo = left ? ki : 0, hi = left ? n : ki + 1;
  const bool edge = dtrevc_edge(n, ki, kd, left);
  const zd* vo = t.V + (int64_t)ki * t.ldv;
  const zd* xo = t.X + (int64_t)ki * n;
#pragma unroll
  for (int q = 0; q < R; ++q) {
    const int r = lane + 64 * q;
    zd v = zr(0.0);
    if (t.Z) {
      if (r < n) v = edge ? zr(t.Z[r + (int64_t)ki * t.ldz]) : vo[r];
    } else {
      if (r >= lo && r < hi) v = xo[r];
    }
    y.v[q] = v;
  }
  dtrevc_store<R>(t, y, ki, kd, left, a.normalize != 0, edge);
}

// Orders up to kTrevcSmallN: the columns of a matrix by the wavefronts of one
// workgroup, T in LDS (pitch NM + 1), the back-transform and the scaling in the
// solving wavefront's registers.
template <int NM, bool LEFT> __global__ void __launch_bounds__(1024) dtrevc_small_kernel(TrevcArgs a) {
  extern __shared__ double smem[];  // DFac[NM] per wavefront
  constexpr int P = NM + 1;
  __shared__ double Ts[P * NM], cn[NM], sub[NM];
  __shared__ int kind[NM];
  const TrevcMat<double> t = trevc_mat<double, false>(a, blockIdx.x);
  const int n = t.n, lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  trevc_stage<P>(t, false, Ts, cn);
  if ((int)threadIdx.x < n) {
    auto sb = [&](int i) { return (i >= 0 && i + 1 < n) ? Ts[(i + 1) + i * P] : 0.0; };
    sub[threadIdx.x] = sb(threadIdx.x);
    kind[threadIdx.x] = dtrevc_kind(sb, threadIdx.x, LEFT);
  }
  __syncthreads();
  const double ulp = GS_EPS;
  const double smallnum = GS_FMIN * ((double)n / ulp);  // vectors.jl:146,475
  const double bignum = (1.0 - ulp) / smallnum;
  const ColG<double> Tc{Ts, P};
  DFac* const fac = reinterpret_cast<DFac*>(smem) + NM * wave;
  for (int b = wave; b < n; b += blockDim.x >> 6) {
    const int ki = LEFT ? b : n - 1 - b;
    const int kd = __builtin_amdgcn_readfirstlane(kind[ki]);
    if (kd == 2) continue;
    WaveVec<1> y;
    if (!LEFT) dsolve_right<1>(Tc, sub, cn, ki, kd, smallnum, bignum, y, fac);
    else dsolve_left<1>(Tc, sub, cn, n, ki, kd, smallnum, bignum, y, fac);
    const int lo = LEFT ? ki : 0, hi = LEFT ? n : ki + 1;
    if (!(lane >= lo && lane < hi)) y.v[0] = zr(0.0);
    const bool edge = dtrevc_edge(n, ki, kd, LEFT);
    if (t.Z) {
      if (edge) y.v[0] = lane < n ? zr(t.Z[lane + (int64_t)ki * t.ldz]) : zr(0.0);
      else y.v[0] = trevc_back_small(t, y, lo, hi - 1);
    }
    dtrevc_store<1>(t, y, ki, kd, LEFT, a.normalize != 0, edge);
  }
}

static hipError_t launch_dtrevc_small(const TrevcArgs& a, int nmax, hipStream_t s) {
  const int nw = trevc_small_waves(a.count);
  if (nmax <= 16) {
    const size_t lds = 16 * sizeof(DFac) * nw;
    if (a.left) hipLaunchKernelGGL((dtrevc_small_kernel<16, true>), dim3(a.count), dim3(64 * nw), lds, s, a);
    else hipLaunchKernelGGL((dtrevc_small_kernel<16, false>), dim3(a.count), dim3(64 * nw), lds, s, a);
  } else {
    const size_t lds = 32 * sizeof(DFac) * nw;
    if (a.left) hipLaunchKernelGGL((dtrevc_small_kernel<32, true>), dim3(a.count), dim3(64 * nw), lds, s, a);
    else hipLaunchKernelGGL((dtrevc_small_kernel<32, false>), dim3(a.count), dim3(64 * nw), lds, s, a);
  }
  return hipGetLastError();
}

template <int R> static hipError_t launch_dtrevc_r(const TrevcArgs& a, int nmax, hipStream_t s) {
  const size_t lds = wavevec_lds_bytes<R>();
  const int nt = (nmax + 63) / 64;
  hipLaunchKernelGGL(dtrevc_norms_kernel, dim3((nmax + 3) / 4, a.count), dim3(256), 0, s, a);
  if (a.left) {
    hipLaunchKernelGGL(trevc_transpose_kernel<double>, dim3((nmax + 31) / 32, (nmax + 31) / 32, a.count), dim3(256),
                       0, s, a);
    hipLaunchKernelGGL((dtrevc_solve_kernel<R, true>), dim3(nmax, a.count), dim3(64), lds, s, a);
  } else {
    hipLaunchKernelGGL((dtrevc_solve_kernel<R, false>), dim3(nmax, a.count), dim3(64), lds, s, a);
  }
  if (a.Z) hipLaunchKernelGGL(trevc_back_kernel<double>, dim3(nt, nt, a.count), dim3(256), 0, s, a);
  hipLaunchKernelGGL(dtrevc_finish_kernel<R>, dim3(nmax, a.count), dim3(64), lds, s, a);
  return hipGetLastError();
}

hipError_t launch_dtrevc(const TrevcArgs& a, int nmax, hipStream_t s) {
  if (nmax <= kTrevcSmallN) return launch_dtrevc_small(a, nmax, s);
  switch (trevc_class(nmax)) {
    case 1: return launch_dtrevc_r<1>(a, nmax, s);
    case 2: return launch_dtrevc_r<2>(a, nmax, s);
    case 4: return launch_dtrevc_r<4>(a, nmax, s);
    case 8: return launch_dtrevc_r<8>(a, nmax, s);
    case 16: return launch_dtrevc_r<16>(a, nmax, s);
    case 32: return launch_dtrevc_r<32>(a, nmax, s);
    case 64: return launch_dtrevc_r<64>(a, nmax, s);
    default: return hipErrorInvalidValue;
  }
}

int trevc_max_n() { return 4096; }

// Workspace of one launch group, per matrix: X (16 n^2), the transpose
// (left), and 8 n + 8 n + 4 n for norms, subdiagonal and kinds; each array
// 256-byte aligned.  A group ends where the next matrix needs another class,
// would take the workspace above kGroupBytes, or fills the grid's z
// dimension; the small orders, without workspace, are one group, or, up to
// kTrevcJoin of them, part of the group of orders 33 to 64 if there is one.
constexpr size_t kGroupBytes = size_t(1) << 30;
constexpr int kGroupCount = 32768;
static size_t seg(size_t bytes) { return (bytes + 255) & ~size_t(255); }

void trevc_groups(const int32_t* n, const int32_t* order, int64_t count, bool cplx, TrevcPlan& p) {
  const size_t es = cplx ? 16 : 8;
  p.groups.clear();
  p.wsn.clear();
  p.wsnn.clear();
  p.bytes = 0;
  int64_t nsmall = 0;
  for (int64_t q = 0; q < count; ++q) nsmall += n[q] > 0 && n[q] <= kTrevcSmallN;
  const bool join = nsmall <= kTrevcJoin;
  for (int64_t q = 0; q < count;) {
    if (n[order[q]] <= 0) break;  // descending: only empty matrices remain
    TrevcGroup g;
    g.first = q;
    g.nmax = n[order[q]];
    const int cls = trevc_class(g.nmax);
    int64_t sn = 0, snn = 0;
    int64_t k = q;
    const bool small = g.nmax <= kTrevcSmallN;
    while (small && k < count && n[order[k]] > 0) ++k;
    for (; !small && k < count && k - q < kGroupCount; ++k) {
      const int64_t m = n[order[k]];
      if (m <= (join ? 0 : kTrevcSmallN) || trevc_class((int)m) != cls) break;
      if (k > q && (16 + es) * (size_t)(snn + m * m) > kGroupBytes) break;
      p.wsn.push_back(sn);
      p.wsnn.push_back(snn);
      sn += m;
      snn += m * m;
    }
    g.count = k - q;
    g.sn = sn;
    g.snn = snn;
    p.groups.push_back(g);
    if (small) break;  // the last: without workspace
    p.bytes = std::max(p.bytes, seg(16 * (size_t)snn) + seg(es * (size_t)snn) + 2 * seg(8 * (size_t)sn) +
                                    seg(4 * (size_t)sn));
    q = k;
  }
}

hipError_t launch_trevc(bool cplx, TrevcArgs a, const TrevcPlan& p, void* ws, hipStream_t s) {
  const int32_t* order = a.order;
  const int64_t *wsn = a.wsn, *wsnn = a.wsnn;
  const size_t es = cplx ? 16 : 8;
  for (const TrevcGroup& g : p.groups) {
    char* w = static_cast<char*>(ws);
    a.wX = w;
    w += seg(16 * (size_t)g.snn);
    a.wT = w;
    w += seg(es * (size_t)g.snn);
    a.wcn = reinterpret_cast<double*>(w);
    w += seg(8 * (size_t)g.sn);
    a.wsub = reinterpret_cast<double*>(w);
    w += seg(8 * (size_t)g.sn);
    a.wkind = reinterpret_cast<int*>(w);
    a.order = order + g.first;
    if (g.nmax > kTrevcSmallN) {
      a.wsn = wsn + g.first;
      a.wsnn = wsnn + g.first;
    }
    a.count = (int)g.count;
    const hipError_t e = cplx ? launch_ztrevc(a, g.nmax, s) : launch_dtrevc(a, g.nmax, s);
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

}  // namespace gs
