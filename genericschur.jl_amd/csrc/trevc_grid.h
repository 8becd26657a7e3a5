// Shared pieces of the eigenvector path (vectors.jl:12-20): every matrix of a
// list over the whole GPU, one wavefront per eigenvector.
//
//   1. column norms of T's strict upper triangle (one wavefront per column;
//      real: also the subdiagonal and the block kinds);
//   2. left only: T's transpose, which turns the row walks of the left
//      solves into coalesced column reads;
//   3. solves: workgroup (column, matrix) of one wavefront, the solution in
//      registers (orders up to 256) or LDS, T from global memory through L2;
//      the solution goes to a workspace X;
//   4. back-transform Z X as FP64 MFMA tiles (trevc_back_kernel);
//   5. one wavefront per column scales and normalises in V.
//
// The orders up to kTrevcSmallN go through one launch of their own, unless they
// are few beside orders 33 to 64 (kTrevcJoin).  The rest of the list is processed in classes of orders that need the same number R of
// entries per lane.  Bound by the latency of the substitutions, of which one
// matrix has n in flight and a batch n per matrix.  Before, one workgroup of
// 4 wavefronts per matrix solved its n columns in turn with T's triangle in
// LDS (one or two workgroups per CU; T from L2 above order 192), each lane
// repeating the diagonal blocks' factorization at every step: one real matrix
// of order 64 / 128 / 512 / 1024 took 538 / 2452 / 47154 / 776375 us, now 66 /
// 114 / 523 / 1643 us (complex 128 / 1024: 1932 / 926396 -> 100 / 3162 us);
// right and left vectors of 4096 real matrices n ~ U{16..128} 15.4 -> 6.5 ms,
// right vectors of 8192 complex matrices n ~ U{8..96} 8.1 -> 4.7 ms.
#pragma once
#include "dev_common.h"
#include "internal.h"
#include "wavevec.h"

namespace gs {

// One matrix of a class, as the kernels see it.  X, Tt, cn, sub, kind: its
// workspace segments.
template <class E> struct TrevcMat {
  int n;
  const E* T;
  const E* Z;  // may be null
  zd* V;
  int64_t ldt, ldz, ldv;
  zd* X;       // n x n, ld n
  E* Tt;       // n x n, ld n (left)
  double* cn;  // n
  double* sub; // n (real)
  int* kind;   // n (real)
};
// WS: with the workspace segments.
template <class E, bool WS = true> GS_DEV TrevcMat<E> trevc_mat(const TrevcArgs& a, int q) {
  const int m = a.order[q];
  const int n = a.n[m];
  const int64_t o = a.off[m];
  TrevcMat<E> t;
  t.n = n;
  t.T = reinterpret_cast<const E*>(a.T) + o;
  t.Z = a.Z ? reinterpret_cast<const E*>(a.Z) + o : nullptr;
  t.V = reinterpret_cast<zd*>(a.V) + o;
  t.ldt = a.ldt > 0 ? a.ldt : n;
  t.ldz = a.ldz > 0 ? a.ldz : n;
  t.ldv = a.ldv > 0 ? a.ldv : n;
  if constexpr (WS) {
    const int64_t w = a.wsn[q], ww = a.wsnn[q];
    t.X = reinterpret_cast<zd*>(a.wX) + ww;
    t.Tt = reinterpret_cast<E*>(a.wT) + ww;
    t.cn = a.wcn + w;
    t.sub = a.wsub + w;
    t.kind = a.wkind + w;
  }
  return t;
}

// Tt(j, i) = T(i, j); 32 x 32 tiles through LDS, grid (tiles, tiles, count),
// 256 threads.
template <class E> __global__ void __launch_bounds__(256) trevc_transpose_kernel(TrevcArgs a) {
  __shared__ E tile[32][33];
  const TrevcMat<E> t = trevc_mat<E>(a, blockIdx.z);
  const int n = t.n;
  const int bx = blockIdx.x * 32, by = blockIdx.y * 32;
  if (bx >= n || by >= n) return;
  const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
  for (int k = ty; k < 32; k += 8) {
    const int r = bx + tx, c = by + k;
    if (r < n && c < n) tile[k][tx] = t.T[r + (int64_t)c * t.ldt];
  }
  __syncthreads();
  for (int k = ty; k < 32; k += 8) {
    const int r = by + tx, c = bx + k;  // Tt(r, c) = T(c, r) = tile[tx][k]
    if (r < n && c < n) t.Tt[r + (int64_t)c * n] = tile[tx][k];
  }
}

GS_DEV double tmag(double x, bool) { return fabs(x); }
GS_DEV double tmag(zd z, bool abs1) { return abs1 ? zabs1(z) : zabs(z); }

// Entry (i, j) of T: T itself, or through the transpose (the left solves'
// row walks T(j, i), i along the lanes, become column reads).
template <class E> struct ColG {
  const E* p;
  int64_t ld;
  GS_DEV E operator()(int i, int j) const { return p[i + (int64_t)j * ld]; }
};
template <class E> struct TransG {
  const E* p;
  int64_t ld;
  GS_DEV E operator()(int i, int j) const { return p[j + (int64_t)i * ld]; }
};

// V = Z X for the matrices of a class on v_mfma_f64_16x16x4_f64 (operand
// layout in dgemm.hip): grid (row tiles, column tiles, matrices), four
// wavefronts per 64 x 64 complex tile, each 32 x 32 (the real and imaginary
// parts as separate accumulators, so that a lane stores whole entries; complex,
// the two products of each part in accumulators of their own: added in turn to
// one, twice as many sums are rounded as in a product of complex entries, and
// the vectors were 10 to 18 % further from the exact ones, n = 260 8.2 against
// 6.9e-16; two wavefronts to a SIMD, since with one, by the registers that the
// compiler takes unasked, 4000 n = 65 take 3.1 instead of 2.7 ms).
// Slabs of 16 rows of X through LDS as planes.  X is upper (right) or lower
// (left) triangular: the contraction runs over the tile's own support only.
template <class E> __global__ void __launch_bounds__(256, 2) trevc_back_kernel(TrevcArgs a) {
  constexpr bool CPLX = sizeof(E) == sizeof(zd);
  constexpr int BT = 64, KB = 16, LD = BT + 16;
  typedef double v4d __attribute__((ext_vector_type(4)));
  __shared__ double Az[CPLX ? 2 : 1][KB * LD], Bx[2][KB * LD];
  const TrevcMat<E> t = trevc_mat<E>(a, blockIdx.z);
  const int n = t.n;
  const int r0 = blockIdx.x * BT, c0 = blockIdx.y * BT;
  if (r0 >= n || c0 >= n) return;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wr = (wave & 1) * 32, wc = (wave >> 1) * 32;
  const int kb = a.left ? c0 : 0, ke = a.left ? n : min(n, c0 + BT);
  // Z tile: lane = row, X tile: lane % 16 = k, so both walk memory in order
  const int ar = min(r0 + lane, n - 1);
  E ra[KB / 4];
  zd rx[KB / 4];
  auto fetch = [&](int k0) {
#pragma unroll
    for (int q = 0; q < KB / 4; ++q) {
      ra[q] = t.Z[ar + (int64_t)min(k0 + wave + 4 * q, n - 1) * t.ldz];
      rx[q] = t.X[min(k0 + (tid & 15), n - 1) + (int64_t)min(c0 + (tid >> 4) + 16 * q, n - 1) * n];
    }
  };
  v4d re[2][2], im[2][2], re2[2][2], im2[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) re[i][j] = im[i][j] = re2[i][j] = im2[i][j] = v4d{0.0, 0.0, 0.0, 0.0};
  fetch(kb);
  for (int k0 = kb; k0 < ke; k0 += KB) {
    __syncthreads();
#pragma unroll
    for (int q = 0; q < KB / 4; ++q) {
      const int kz = wave + 4 * q, kx = tid & 15, cx = (tid >> 4) + 16 * q;
      // entries past the support meet zeros on both sides
      const bool vz = k0 + kz < ke, vx = k0 + kx < ke;
      if constexpr (CPLX) {
        Az[0][kz * LD + lane] = vz ? ra[q].x : 0.0;
        Az[1][kz * LD + lane] = vz ? ra[q].y : 0.0;
      } else {
        Az[0][kz * LD + lane] = vz ? ra[q] : 0.0;
      }
      Bx[0][kx * LD + cx] = vx ? rx[q].x : 0.0;
      Bx[1][kx * LD + cx] = vx ? rx[q].y : 0.0;
    }
    __syncthreads();
    fetch(k0 + KB);
#pragma unroll
    for (int k4 = 0; k4 < KB / 4; ++k4) {
      const int kk = (4 * k4 + (lane >> 4)) * LD;
      double zr_[2], zi_[2], xr[2], xi[2];
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        zr_[i] = Az[0][kk + wr + 16 * i + (lane & 15)];
        if constexpr (CPLX) zi_[i] = Az[1][kk + wr + 16 * i + (lane & 15)];
        xr[i] = Bx[0][kk + wc + 16 * i + (lane & 15)];
        xi[i] = Bx[1][kk + wc + 16 * i + (lane & 15)];
      }
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          re[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(xr[j], zr_[i], re[i][j], 0, 0, 0);
          im[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(xi[j], zr_[i], im[i][j], 0, 0, 0);
          if constexpr (CPLX) {
            re2[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(xi[j], zi_[i], re2[i][j], 0, 0, 0);
            im2[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(xr[j], zi_[i], im2[i][j], 0, 0, 0);
          }
        }
    }
  }
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int gr = r0 + wr + 16 * i + (lane & 15), gc = c0 + wc + 16 * j + (lane >> 4) + 4 * r;
        if (gr < n && gc < n)
          t.V[gr + (int64_t)gc * t.ldv] =
              CPLX ? zmk(re[i][j][r] - re2[i][j][r], im[i][j][r] + im2[i][j][r]) : zmk(re[i][j][r], im[i][j][r]);
      }
}

// Orders up to this take one launch of a workgroup per matrix (the small
// kernels of ztrevc.hip and dtrevc.hip) instead of the four or five over the
// columns, whose launches cost a small matrix more than its solves, and a large
// batch the solutions' way through memory.  Measured, complex, five launches /
// one: one matrix n = 2 35 / 26 us, n = 16 39 / 33, n = 24 45 / 42, n = 32 47 / 55;
// 16384 of n = 16 1.41 / 0.94 ms, of n = 32 3.16 / 2.08 (real 1.64 / 1.02 and
// 3.77 / 2.06).
constexpr int kTrevcSmallN = 32;

// Small matrices of a list that go through the grid launches of its orders 33
// to 64 all the same, if it has any: up to this many cost those less than a
// launch of their own.  Measured, own launch / joined, right vectors, beside 8
// matrices: 16 complex of n = 17..32 93 / 61 us, 256 105 / 102, 512 130 / 141
// (real 96 / 64, 111 / 84, 137 / 112; n = 2..16 75 / 62, 82 / 76, 94 / 95);
// beside 300: 200 / 168, 210 / 202, 237 / 249.
constexpr int64_t kTrevcJoin = 256;

// Wavefronts of a small matrix's workgroup: one per column or two where the
// matrices are fewer than the CUs, down to four where they fill the GPU.
// Measured, 16 / 8 / 4: one complex matrix n = 32 55 / 62 / 89 us, 1000 of n =
// 4..24 99 / 97 / 105, 16384 of n = 16 1.05 / 0.97 / 0.94 ms (real 1.35 / 1.15 /
// 1.02).
inline int trevc_small_waves(int count) { return count <= 256 ? 16 : (count <= 1024 ? 8 : 4); }

// A small matrix in LDS with pitch P: T, and its strictly upper column norms
// by one lane per column.  Every thread of the workgroup calls it.
template <int P, class E> GS_DEV void trevc_stage(const TrevcMat<E>& t, bool abs1, E* Ts, double* cn) {
  constexpr int NM = P - 1;
  const int n = t.n, r = threadIdx.x % NM;
  for (int c = threadIdx.x / NM; c < n; c += blockDim.x / NM)
    if (r < n) Ts[r + c * P] = t.T[r + (int64_t)c * t.ldt];
  __syncthreads();
  if ((int)threadIdx.x < n) {
    double s = 0.0;
    for (int i = 0; i < (int)threadIdx.x; ++i) s += tmag(Ts[i + threadIdx.x * P], abs1);
    cn[threadIdx.x] = s;
  }
}

// y = Z x over the support lo .. hi of x, row lane of the product in lane, each
// sum an fma chain of its own in the columns' order: the MFMA tiles' bits.
template <class E, class VEC> GS_DEV zd trevc_back_small(const TrevcMat<E>& t, const VEC& x, int lo, int hi) {
  constexpr bool CPLX = sizeof(E) == sizeof(zd);
  const E* z = t.Z + min((int)(threadIdx.x & 63), t.n - 1);
  zd y = zr(0.0), y2 = zr(0.0);
#pragma unroll 8
  for (int k = lo; k <= hi; ++k) {
    const E a = z[(int64_t)k * t.ldz];
    const zd b = x.get(k);
    if constexpr (CPLX) {
      y = zmk(fma(a.x, b.x, y.x), fma(a.x, b.y, y.y));
      y2 = zmk(fma(a.y, b.y, y2.x), fma(a.y, b.x, y2.y));
    } else {
      y = y + a * b;
    }
  }
  if constexpr (CPLX) y = zmk(y.x - y2.x, y.y + y2.y);
  return y;
}

// entries per lane of the class an order belongs to
inline int trevc_class(int n) {
  int r = 1;
  while (64 * r < n) r *= 2;
  return r;
}

}  // namespace gs
