// Eigenvectors of a complex Schur factorization (T upper triangular, Z) on
// gfx950, following GenericSchur.jl:
//   right   vectors.jl:45-131   with _usolve!  util.jl:128-293 (zlatrs)
//   left    vectors.jl:372-460  with _cusolve! util.jl:301-461
//   unit 2-norm, largest entry real: _enormalize! util.jl:572-592
//
// The launches over a list of matrices are described in trevc_grid.h; here
// one wavefront per eigenvector, the scalar control of the scaled solver
// running uniformly in every lane.
#include "dev_common.h"
#include "internal.h"
#include "trevc_grid.h"
#include "wavevec.h"

namespace gs {

// ------------------------------------------------------------------------
// Shifted, clamped diagonal of the solve: T(j,j) - lam, replaced by smin
// when its abs1 is below smin (vectors.jl:87-90 / :412-415).
template <class TA> GS_DEV zd shifted_diag(const TA& Tc, int j, zd lam, double smin) {
  zd d = Tc(j, j) - lam;
  if (zabs1(d) < smin) d = zr(smin);
  return d;
}

// The substitutions without scaling divide by the shifted diagonal with
// Smith's algorithm, whose ratio and denominator depend on the diagonal only:
// ZFac holds them for the 64 rows of a chunk, one row per lane (LDS), and a
// step reads its row's as a broadcast.
struct ZFac {
  double r, d, sw, pad;
};
GS_DEV ZFac zfac(zd b) {
  const bool sw = fabs(b.y) > fabs(b.x);
  const double r = sw ? b.x / b.y : b.y / b.x;
  return ZFac{r, sw ? b.x * r + b.y : b.x + b.y * r, sw ? 1.0 : 0.0, 0.0};
}
GS_DEV zd zfac_div(zd a, ZFac f) {
  const bool sw = __builtin_amdgcn_readfirstlane((int)f.sw) != 0;
  const double p = sw ? a.y : a.x, q = sw ? a.x : a.y;
  const double x = (p + q * f.r) / f.d, y = (q - p * f.r) / f.d;
  return zmk(x, sw ? -y : y);
}

// Whether the growth estimate of zlatrs is certain to allow the substitution
// without scaling: with every |t_jj| >= smallnum the estimate is at least
// grow0 times the product of min(1, t_jj) / 1 at its smallest and of
// t_jj / (t_jj + cnorm_j) (left: min(1, t_jj / (1 + cnorm_j)) and 1 / (1 +
// cnorm_j)), here bounded from below by powers of two summed over the lanes.
// The estimate itself is a chain of n divisions; it runs where this bound
// does not decide.
template <bool LEFT, class TA> GS_DEV bool grow_certain(const TA& Tc, const double* cnorm, int o, int m, zd lam,
                                                        double smin, double grow0) {
  const int lane = threadIdx.x & 63;
  const double smallnum = GS_FMIN / GS_EPS;
  int e = 0, emin = 0;
  bool ok = true;
  for (int j = lane; j < m; j += 64) {
    zd d = Tc(o + j, o + j) - lam;
    if (zabs1(d) < smin) d = zr(smin);
    const double t = zabs1(d);
    ok = ok && t >= smallnum && t < 0x1p1000 && cnorm[j] < 0x1p1000;
    const int et = ilogb(t);
    if (LEFT) {
      const int ec = ilogb(1.0 + cnorm[j]) + 1;  // 1 + cnorm < 2^ec
      e += min(0, et - ec);
      emin = min(emin, -ec);
    } else {
      e += et - (ilogb(t + cnorm[j]) + 1);  // t / (t + c) > 2^(et - ec)
      emin = min(emin, et);
    }
  }
  // 64 lanes: sums of exponents by lane exchange
  for (int s = 32; s > 0; s >>= 1) {
    e += __shfl_xor(e, s, 64);
    emin = min(emin, __shfl_xor(emin, s, 64));
  }
  if (__builtin_amdgcn_ballot_w64(!ok) != 0) return false;
  return grow0 >= 0x1p-1000 && ilogb(grow0) + e + emin > ilogb(smallnum) + 2;
}

// _usolve! on entries 0..m-1 of x (A = T shifted by lam, leading m x m).
template <int R, class TA, class VEC> GS_DEV double usolve_w(const TA& Tc, const double* cnorm, int m, zd lam,
                                                             double smin, VEC& x, ZFac* fac) {
  const int lane = threadIdx.x & 63;
  const double half = 0.5;
  const double smallnum = GS_FMIN / GS_EPS;
  const double bignum = 1.0 / smallnum;
  double xscale = 1.0;
  auto inrange = [&](int q) { return lane + 64 * q < m; };
  auto cabs1half = [](zd z) { return fabs(z.x / 2) + fabs(z.y / 2); };
  double tmax = 0.0;
  for (int j = lane; j < m; j += 64) tmax = fmax(tmax, fabs(cnorm[j]));
  tmax = wave_max(tmax);
  double tscale;
  if (tmax <= bignum * half) tscale = 1.0;
  else tscale = half / (smallnum * tmax);
  double xmax = 0.0;
#pragma unroll
  for (int q = 0; q < R; ++q)
    if (inrange(q)) xmax = fmax(xmax, cabs1half(x.v[q]));
  xmax = wave_max(xmax);
  double xbound = xmax;
  double grow;
  if (tscale != 1.0) {
    grow = 0.0;
  } else {
    grow = half / fmax(xbound, smallnum);
    xbound = grow;
    bool toosmall = false;
    if (!grow_certain<false>(Tc, cnorm, 0, m, lam, smin, grow))
    for (int j = m - 1; j >= 0; --j) {
      toosmall = (grow <= smallnum);
      if (toosmall) break;
      const double tjj = zabs1(shifted_diag(Tc, j, lam, smin));
      if (tjj >= smallnum) xbound = fmin(xbound, fmin(1.0, tjj) * grow);
      else xbound = 0.0;
      const double cn = cnorm[j] * tscale;
      if (tjj + cn >= smallnum) grow *= (tjj / (tjj + cn));
      else grow = 0.0;
    }
    if (!toosmall) grow = xbound;
  }
  if (grow * tscale > smallnum) {
    // columns of T one step ahead up to R = 4 entries per lane
    constexpr bool PF = R <= 4;
    zd c[PF ? R : 1];
    auto load = [&](int j) {
      if constexpr (PF) {
#pragma unroll
        for (int q = 0; q < R; ++q) c[q] = Tc(min(lane + 64 * q, m - 1), max(j, 0));
      }
    };
    load(m - 1);
    int chunk = -1;
    for (int j = m - 1; j >= 0; --j) {
      if ((j >> 6) != chunk) {
        chunk = j >> 6;
        wsync();
        fac[lane] = zfac(shifted_diag(Tc, min(64 * chunk + lane, m - 1), lam, smin));
        wsync();
      }
      zd k[PF ? R : 1];
      if constexpr (PF) {
#pragma unroll
        for (int q = 0; q < R; ++q) k[q] = c[q];
      }
      load(j - 1);
      const zd xj = zfac_div(x.get(j), fac[j & 63]);
      x.set(j, xj);
#pragma unroll
      for (int q = 0; q < R; ++q) {
        const int i = lane + 64 * q;
        if constexpr (PF) {
          if (i < j) x.v[q] = x.v[q] - k[q] * xj;
        } else {
          if (i < j) x.v[q] = x.v[q] - Tc(i, j) * xj;
        }
      }
    }
    return xscale;
  }
  // careful scaled solve
  if (xmax > bignum * half) {
    xscale = (bignum * half) / xmax;
    x.scale(xscale);
    xmax = bignum;
  } else {
    xmax *= 2.0;
  }
  for (int j = m - 1; j >= 0; --j) {
    zd xjv = x.get(j);
    double xj = zabs1(xjv);
    const zd tjjs = shifted_diag(Tc, j, lam, smin) * tscale;
    const double tjj = zabs1(tjjs);
    const double cnj = cnorm[j] * tscale;
    if (tjj > smallnum) {
      if (tjj < 1.0 && xj > tjj * bignum) {
        const double rec = 1.0 / xj;
        x.scale(rec);
        xscale *= rec;
        xmax *= rec;
        xjv = x.get(j);
      }
      xjv = xjv / tjjs;
      x.set(j, xjv);
      xj = zabs1(xjv);
    } else if (tjj > 0.0) {
      if (xj > tjj * bignum) {
        double rec = (tjj * bignum) / xj;
        if (cnj > 1.0) rec /= cnj;
        x.scale(rec);
        xscale *= rec;
        xmax *= rec;
        xjv = x.get(j);
      }
      xjv = xjv / tjjs;
      x.set(j, xjv);
      xj = zabs1(xjv);
    } else {
#pragma unroll
      for (int q = 0; q < R; ++q) x.v[q] = zr(0.0);
      x.set(j, zr(1.0));
      xjv = zr(1.0);
      xscale = 0.0;
      xmax = 0.0;
    }
    if (xj > 1.0) {
      double rec = 1.0 / xj;
      if (cnj > (bignum - xmax) * rec) {
        rec *= half;
        x.scale(rec);
        xscale *= rec;
      }
    } else if (xj * cnj > bignum - xmax) {
      x.scale(half);
      xscale *= half;
    }
    if (j > 0) {
      const zd xjt = x.get(j) * tscale;
      double xm = 0.0;
#pragma unroll
      for (int q = 0; q < R; ++q) {
        const int i = lane + 64 * q;
        if (i < j) {
          x.v[q] = x.v[q] - xjt * Tc(i, j);
          xm = fmax(xm, zabs1(x.v[q]));
        }
      }
      xmax = wave_max(xm);
    }
  }
  xscale /= tscale;
  return xscale;
}

// _cusolve! on entries o..o+m-1 of x: (A)^H y = s b with
// A(i, j) = T(o+i, o+j) for i < j and the shifted, clamped diagonal; cnorm
// is indexed from 0 (the reference passes the full tnorms, vectors.jl:417-420).
template <int R, class TA, class VEC> GS_DEV double cusolve_w(const TA& Tc, const double* cnorm, int o, int m, zd lam,
                                                              double smin, VEC& x, ZFac* fac) {
  const int lane = threadIdx.x & 63;
  const double half = 0.5;
  const double smallnum = GS_FMIN / GS_EPS;
  const double bignum = 1.0 / smallnum;
  double xscale = 1.0;
  auto inrange = [&](int q) {
    const int i = lane + 64 * q;
    return i >= o && i < o + m;
  };
  auto cabs1half = [](zd z) { return fabs(z.x / 2) + fabs(z.y / 2); };
  double tmax = 0.0;
  for (int j = lane; j < m; j += 64) tmax = fmax(tmax, fabs(cnorm[j]));
  tmax = wave_max(tmax);
  double tscale;
  if (tmax <= bignum * half) tscale = 1.0;
  else tscale = half / (smallnum * tmax);
  double xmax = 0.0;
#pragma unroll
  for (int q = 0; q < R; ++q)
    if (inrange(q)) xmax = fmax(xmax, cabs1half(x.v[q]));
  xmax = wave_max(xmax);
  double xbound = xmax;
  double grow;
  if (tscale != 1.0) {
    grow = 0.0;
  } else {
    grow = half / fmax(xbound, smallnum);
    xbound = grow;
    bool toosmall = false;
    if (!grow_certain<true>(Tc, cnorm, o, m, lam, smin, grow))
    for (int j = 0; j < m; ++j) {
      toosmall = (grow <= smallnum);
      if (toosmall) break;
      const double xj = 1.0 + cnorm[j] * tscale;
      grow = fmin(grow, xbound / xj);
      const double tjj = zabs1(shifted_diag(Tc, o + j, lam, smin));
      if (tjj >= smallnum) {
        if (xj > tjj) xbound *= (tjj / xj);
      } else {
        xbound = 0.0;
      }
    }
    if (!toosmall) grow = fmin(grow, xbound);
  }
  if (grow * tscale > smallnum) {
    // forward substitution in axpy form: after x[j] is final, remove its
    // contribution from the later right-hand sides
    constexpr bool PF = R <= 4;
    zd c[PF ? R : 1];
    auto load = [&](int j) {
      if constexpr (PF) {
#pragma unroll
        for (int q = 0; q < R; ++q) c[q] = Tc(o + min(j, m - 1), min(lane + 64 * q, o + m - 1));
      }
    };
    load(0);
    int chunk = -1;
    for (int j = 0; j < m; ++j) {
      if (((o + j) >> 6) != chunk) {
        chunk = (o + j) >> 6;
        wsync();
        fac[lane] = zfac(zconj(shifted_diag(Tc, min(max(64 * chunk + lane, o), o + m - 1), lam, smin)));
        wsync();
      }
      zd k[PF ? R : 1];
      if constexpr (PF) {
#pragma unroll
        for (int q = 0; q < R; ++q) k[q] = c[q];
      }
      load(j + 1);
      const zd xj = zfac_div(x.get(o + j), fac[(o + j) & 63]);
      x.set(o + j, xj);
#pragma unroll
      for (int q = 0; q < R; ++q) {
        const int i = lane + 64 * q;  // absolute entry index
        if constexpr (PF) {
          if (i > o + j && i < o + m) x.v[q] = x.v[q] - zconj(k[q]) * xj;
        } else {
          if (i > o + j && i < o + m) x.v[q] = x.v[q] - zconj(Tc(o + j, i)) * xj;
        }
      }
    }
    return xscale;
  }
  if (xmax > bignum * half) {
    xscale = (bignum * half) / xmax;
    x.scale(xscale);
    xmax = bignum;
  } else {
    xmax *= 2.0;
  }
  for (int j = 0; j < m; ++j) {
    double xj = zabs1(x.get(o + j));
    zd uscale = zr(tscale);
    double rec = 1.0 / fmax(xmax, 1.0);
    zd tjjs = zconj(shifted_diag(Tc, o + j, lam, smin)) * tscale;
    const double cnj = cnorm[j] * tscale;
    if (cnj > (bignum - xj) * rec) {
      rec *= half;
      const double tjj = zabs1(tjjs);
      if (tjj > 1.0) {
        rec = fmin(1.0, rec * tjj);
        uscale = uscale / tjjs;
      }
      if (rec < 1.0) {
        x.scale(rec);
        xscale *= rec;
        xmax *= rec;
      }
    }
    // csumj = sum_{i<j} (conj(A(i,j)) * uscale) * x[i]
    zd part = zr(0.0);
#pragma unroll
    for (int q = 0; q < R; ++q) {
      const int i = lane + 64 * q;
      if (i >= o && i < o + j) part = part + (zconj(Tc(i, o + j)) * uscale) * x.v[q];
    }
    const zd csumj = wave_zsum(part);
    const bool unscaled = (uscale.x == tscale && uscale.y == 0.0) || isnan(uscale.x) || isnan(uscale.y);
    if (unscaled) {
      zd xjv = x.get(o + j) - csumj;
      xj = zabs1(xjv);
      tjjs = zconj(shifted_diag(Tc, o + j, lam, smin)) * tscale;
      const double tjj = zabs1(tjjs);
      if (tjj > smallnum) {
        if (tjj < 1.0 && xj > tjj * bignum) {
          const double rec2 = 1.0 / xj;
          x.scale(rec2);
          xscale *= rec2;
          xmax *= rec2;
          xjv = xjv * rec2;
        }
        xjv = xjv / tjjs;
        x.set(o + j, xjv);
      } else if (tjj > 0.0) {
        if (xj > tjj * bignum) {
          const double rec2 = (tjj * bignum) / xj;
          x.scale(rec2);
          xscale *= rec2;
          xmax *= rec2;
          xjv = xjv * rec2;
        }
        xjv = xjv / tjjs;
        x.set(o + j, xjv);
      } else {
#pragma unroll
        for (int q = 0; q < R; ++q)
          if (inrange(q)) x.v[q] = zr(0.0);
        x.set(o + j, zr(1.0));
        xscale = 0.0;
        xmax = 0.0;
      }
    } else {
      x.set(o + j, x.get(o + j) / tjjs - csumj);
    }
    xmax = fmax(xmax, zabs1(x.get(o + j)));
  }
  xscale /= tscale;
  return xscale;
}

// max abs1 scaling then _enormalize! of one column held in a WaveVecZ
// (entries 0..n-1); normalize = 0 stops after the max-abs1 scaling.
template <int R, class VEC> GS_DEV void normalize_col(VEC& v, int n, bool enorm) {
  const int lane = threadIdx.x & 63;
  double t0 = 0.0;
#pragma unroll
  for (int q = 0; q < R; ++q)
    if (lane + 64 * q < n) t0 = fmax(t0, zabs1(v.v[q]));
  t0 = wave_max(t0);
  const double remax = 1.0 / t0;
#pragma unroll
  for (int q = 0; q < R; ++q) v.v[q] = v.v[q] * remax;
  if (!enorm) return;
  // 2-norm without over/underflow, and the first index of the largest |v|^2
  double am = 0.0;
#pragma unroll
  for (int q = 0; q < R; ++q)
    if (lane + 64 * q < n) am = fmax(am, fmax(fabs(v.v[q].x), fabs(v.v[q].y)));
  am = wave_max(am);
  double ss = 0.0;
  double best = -1.0;
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
  // largest |v|^2, first index among ties (util.jl:578-584 uses strict >)
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
  const double s = 1.0 / nrm;
  const zd tt = (s * zconj(vi0)) / sqrt(zabs2(vi0));
#pragma unroll
  for (int q = 0; q < R; ++q) v.v[q] = v.v[q] * tt;
  const zd r0 = v.get(bi);
  v.set(bi, zr(r0.x));
}

// strictly-upper column norms: abs for right (vectors.jl:70-75), abs1 for
// left (vectors.jl:395-400); one wavefront per column
__global__ void __launch_bounds__(256) ztrevc_norms_kernel(TrevcArgs a) {
  const TrevcMat<zd> t = trevc_mat<zd>(a, blockIdx.y);
  const int j = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (j >= t.n) return;
  double s = 0.0;
  for (int i = lane; i < j; i += 64) s += tmag(t.T[i + (int64_t)j * t.ldt], a.left != 0);
  s = wave_sum(s);
  if (lane == 0) t.cn[j] = s;
}

// workgroup (t, matrix) solves column n-1-t (right) or t (left), the longest
// first; the scale goes to the diagonal slot
template <int R, bool LEFT> __global__ void __launch_bounds__(64) ztrevc_solve_kernel(TrevcArgs a) {
  extern __shared__ double smem[];
  const TrevcMat<zd> t = trevc_mat<zd>(a, blockIdx.y);
  const int n = t.n, lane = threadIdx.x & 63, b = blockIdx.x;
  if (b >= n) return;
  const int kk = LEFT ? b : n - 1 - b;
  typedef typename std::conditional<LEFT, TransG<zd>, ColG<zd>>::type TA;
  const TA Tc = LEFT ? TA{t.Tt, n} : TA{t.T, t.ldt};
  const zd lam = Tc(kk, kk);
  const double smin = fmax(GS_EPS * zabs1(lam), GS_FMIN * (double)n);  // vectors.jl:61,386
  WaveVec<R> x;
  wavevec_bind(x.v, smem);
#pragma unroll
  for (int q = 0; q < R; ++q) {
    const int i = lane + 64 * q;
    zd v = zr(0.0);
    if (!LEFT) {
      if (i < kk) v = -Tc(i, kk);
    } else {
      if (i > kk && i < n) v = -zconj(Tc(kk, i));
    }
    x.v[q] = v;
  }
  __shared__ ZFac fac[64];
  double vscale;
  if (!LEFT) vscale = (kk > 0) ? usolve_w<R>(Tc, t.cn, kk, lam, smin, x, fac) : 1.0;
  else vscale = (kk < n - 1) ? cusolve_w<R>(Tc, t.cn, kk + 1, n - 1 - kk, lam, smin, x, fac) : 1.0;
  x.set(kk, zr(vscale));
  zd* xo = t.X + (int64_t)kk * n;
#pragma unroll
  for (int q = 0; q < R; ++q) {
    const int i = lane + 64 * q;
    if (i < n) xo[i] = (LEFT ? (i >= kk) : (i <= kk)) ? x.v[q] : zr(0.0);
  }
}

template <int R> __global__ void __launch_bounds__(64) ztrevc_finish_kernel(TrevcArgs a) {
  extern __shared__ double smem[];
  const TrevcMat<zd> t = trevc_mat<zd>(a, blockIdx.y);
  const int n = t.n, lane = threadIdx.x & 63, kk = blockIdx.x;
  if (kk >= n) return;
  WaveVec<R> y;
  wavevec_bind(y.v, smem);
  zd* vo = t.V + (int64_t)kk * t.ldv;
  const zd* src = t.Z ? vo : t.X + (int64_t)kk * n;
#pragma unroll
  for (int q = 0; q < R; ++q) {
    const int r = lane + 64 * q;
    y.v[q] = (r < n) ? src[r] : zr(0.0);
  }
  normalize_col<R>(y, n, a.normalize != 0);
#pragma unroll
  for (int q = 0; q < R; ++q) {
    const int r = lane + 64 * q;
    if (r < n) vo[r] = y.v[q];
  }
}

// Orders up to kTrevcSmallN: the columns of a matrix by the wavefronts of one
// workgroup, T in LDS (pitch NM + 1), the back-transform and the scaling in the
// solving wavefront's registers.
template <int NM, bool LEFT> __global__ void __launch_bounds__(1024) ztrevc_small_kernel(TrevcArgs a) {
  extern __shared__ double smem[];  // ZFac[64] per wavefront
  constexpr int P = NM + 1;
  __shared__ zd Ts[P * NM];
  __shared__ double cn[NM];
  const TrevcMat<zd> t = trevc_mat<zd, false>(a, blockIdx.x);
  const int n = t.n, lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  trevc_stage<P>(t, LEFT, Ts, cn);
  __syncthreads();
  const ColG<zd> Tc{Ts, P};
  ZFac* const fac = reinterpret_cast<ZFac*>(smem) + 64 * wave;
  for (int b = wave; b < n; b += blockDim.x >> 6) {
    const int kk = LEFT ? b : n - 1 - b;
    const zd lam = Tc(kk, kk);
    const double smin = fmax(GS_EPS * zabs1(lam), GS_FMIN * (double)n);  // vectors.jl:61,386
    WaveVec<1> x;
    x.v[0] = zr(0.0);
    if (!LEFT) {
      if (lane < kk) x.v[0] = -Tc(lane, kk);
    } else {
      if (lane > kk && lane < n) x.v[0] = -zconj(Tc(kk, lane));
    }
    double vscale;
    if (!LEFT) vscale = (kk > 0) ? usolve_w<1>(Tc, cn, kk, lam, smin, x, fac) : 1.0;
    else vscale = (kk < n - 1) ? cusolve_w<1>(Tc, cn, kk + 1, n - 1 - kk, lam, smin, x, fac) : 1.0;
    x.set(kk, zr(vscale));
    if (!(LEFT ? (lane >= kk && lane < n) : (lane <= kk))) x.v[0] = zr(0.0);
    if (t.Z) x.v[0] = trevc_back_small(t, x, LEFT ? kk : 0, LEFT ? n - 1 : kk);
    normalize_col<1>(x, n, a.normalize != 0);
    if (lane < n) t.V[lane + (int64_t)kk * t.ldv] = x.v[0];
  }
}

static hipError_t launch_ztrevc_small(const TrevcArgs& a, int nmax, hipStream_t s) {
  const int nw = trevc_small_waves(a.count);
  const size_t lds = 64 * sizeof(ZFac) * nw;
  if (nmax <= 16) {
    if (a.left) hipLaunchKernelGGL((ztrevc_small_kernel<16, true>), dim3(a.count), dim3(64 * nw), lds, s, a);
    else hipLaunchKernelGGL((ztrevc_small_kernel<16, false>), dim3(a.count), dim3(64 * nw), lds, s, a);
  } else {
    if (a.left) hipLaunchKernelGGL((ztrevc_small_kernel<32, true>), dim3(a.count), dim3(64 * nw), lds, s, a);
    else hipLaunchKernelGGL((ztrevc_small_kernel<32, false>), dim3(a.count), dim3(64 * nw), lds, s, a);
  }
  return hipGetLastError();
}

template <int R> static hipError_t launch_ztrevc_r(const TrevcArgs& a, int nmax, hipStream_t s) {
  const size_t lds = wavevec_lds_bytes<R>();
  const int nt = (nmax + 63) / 64;
  hipLaunchKernelGGL(ztrevc_norms_kernel, dim3((nmax + 3) / 4, a.count), dim3(256), 0, s, a);
  if (a.left) {
    hipLaunchKernelGGL(trevc_transpose_kernel<zd>, dim3((nmax + 31) / 32, (nmax + 31) / 32, a.count), dim3(256), 0, s,
                       a);
    hipLaunchKernelGGL((ztrevc_solve_kernel<R, true>), dim3(nmax, a.count), dim3(64), lds, s, a);
  } else {
    hipLaunchKernelGGL((ztrevc_solve_kernel<R, false>), dim3(nmax, a.count), dim3(64), lds, s, a);
  }
  if (a.Z) hipLaunchKernelGGL(trevc_back_kernel<zd>, dim3(nt, nt, a.count), dim3(256), 0, s, a);
  hipLaunchKernelGGL(ztrevc_finish_kernel<R>, dim3(nmax, a.count), dim3(64), lds, s, a);
  return hipGetLastError();
}

hipError_t launch_ztrevc(const TrevcArgs& a, int nmax, hipStream_t s) {
  if (nmax <= kTrevcSmallN) return launch_ztrevc_small(a, nmax, s);
  switch (trevc_class(nmax)) {
    case 1: return launch_ztrevc_r<1>(a, nmax, s);
    case 2: return launch_ztrevc_r<2>(a, nmax, s);
    case 4: return launch_ztrevc_r<4>(a, nmax, s);
    case 8: return launch_ztrevc_r<8>(a, nmax, s);
    case 16: return launch_ztrevc_r<16>(a, nmax, s);
    case 32: return launch_ztrevc_r<32>(a, nmax, s);
    case 64: return launch_ztrevc_r<64>(a, nmax, s);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace gs
