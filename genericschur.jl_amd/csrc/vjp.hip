// Eigenvalue vector-Jacobian product on gfx950 (no counterpart in the
// reference; the backward of the eigenvalue rrule).
//
// For A = X Lambda X^{-1} with right eigenvectors x_k and left eigenvectors
// y_k (A^H y_k = conj(lambda_k) y_k), a real loss L(lambda) with cotangent
// gbar_k = dL/dRe(lambda_k) + i dL/dIm(lambda_k) per eigenvalue slot has
//     dL = Re sum_k conj(gbar_k) y_k^H dA x_k / (y_k^H x_k),
// so the gradient with respect to a real A is
//     Abar = Re( sum_k c_k y_k x_k^H ),   c_k = gbar_k / conj(y_k^H x_k),
// i.e. Re(X^{-H} diag(gbar) X^H).  The eigenvectors are recomputed from the
// Schur factors by the eigenvector kernels (normalised, any scaling cancels
// in c_k y_k x_k^H); the kernels here form c_k and the rank-n sum: one
// workgroup per matrix with the two n x n complex factors staged in LDS, or,
// above the LDS-resident orders, as FP64 MFMA tiles.
#include <algorithm>

#include "dev_common.h"
#include "internal.h"

namespace gs {

template <int NT> __global__ void __launch_bounds__(NT) vjp_assemble_kernel(VjpArgs a) {
  extern __shared__ double smem[];
  const int b = blockIdx.x;
  if (b >= a.count) return;
  const int m = a.order ? a.order[b] : b;
  const int n = a.n[m];
  if (n <= 0) {
    if (threadIdx.x == 0) a.info[m] = 0;
    return;
  }
  const int64_t o = a.off[m];
  const zd* VR = reinterpret_cast<const zd*>(a.VR) + o;
  const zd* VL = reinterpret_cast<const zd*>(a.VL) + o;
  const zd* g = reinterpret_cast<const zd*>(a.gbar) + a.woff[m];
  double* Ab = a.Abar + o;
  zd* sR = reinterpret_cast<zd*>(smem);  // n x n, ld = n + 1
  const int ld = n + 1;
  zd* sL = sR + (size_t)ld * n;
  zd* c = sL + (size_t)ld * n;
  int* bad = reinterpret_cast<int*>(c + n);
  const int tid = threadIdx.x;
  for (int e = tid; e < n * n; e += NT) {
    const int col = e / n, row = e - col * n;
    sR[row + col * ld] = VR[e];
    sL[row + col * ld] = VL[e];
  }
  if (tid == 0) *bad = 0;
  __syncthreads();
  // c_k = gbar_k / conj(y_k^H x_k), one wavefront per column k
  const int lane = tid & 63, w = tid >> 6;
  for (int k = w; k < n; k += NT / 64) {
    zd s = zr(0.0);
    for (int i = lane; i < n; i += 64) s = s + zconj(sL[i + k * ld]) * sR[i + k * ld];
    s = wave_zsum(s);
    if (lane == 0) {
      const zd d = zconj(s);
      if (d.x == 0.0 && d.y == 0.0) {
        *bad = 1;
        c[k] = zr(0.0);
      } else {
        c[k] = g[k] / d;
      }
    }
  }
  __syncthreads();
  // Abar[r, s] = Re sum_k c_k yL[r, k] conj(xR[s, k])
  for (int e = tid; e < n * n; e += NT) {
    const int s = e / n, r = e - s * n;
    double acc = 0.0;
    for (int k = 0; k < n; ++k) {
      const zd t = c[k] * sL[r + k * ld];
      const zd x = sR[s + k * ld];
      acc += t.x * x.x + t.y * x.y;  // Re(t * conj(x))
    }
    Ab[e] = acc;
  }
  if (tid == 0) a.info[m] = *bad;
}

// Orders whose two factors do not fit LDS, every matrix of a size class in
// two launches.  First, in place in the left vectors' buffer, y_k := c_k y_k
// (one wavefront per column); info = 1 when some y_k^H x_k vanished.
__global__ void __launch_bounds__(256) vjp_scale_kernel(VjpArgs a, zd* VL) {
  const int m = a.order[blockIdx.y];
  const int n = a.n[m];
  const int lane = threadIdx.x & 63;
  const int k = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (k >= n) return;
  const zd* x = reinterpret_cast<const zd*>(a.VR) + a.off[m] + (int64_t)k * n;
  zd* y = VL + a.off[m] + (int64_t)k * n;
  zd s = zr(0.0);
  for (int i = lane; i < n; i += 64) s = s + zconj(y[i]) * x[i];
  s = wave_zsum(s);
  const zd d = zconj(s);
  const bool zero = d.x == 0.0 && d.y == 0.0;
  const zd c = zero ? zr(0.0) : (reinterpret_cast<const zd*>(a.gbar) + a.woff[m])[k] / d;
  if (zero && lane == 0) a.info[m] = 1;
  for (int i = lane; i < n; i += 64) y[i] = c * y[i];
}

// Then Abar(r, s) = sum_k Re(y_k[r] conj(x_k[s])), an n x n x 2n real
// product of the interleaved factors (k and the real / imaginary part are
// the contraction index) on v_mfma_f64_16x16x4_f64 (operand layout in
// dgemm.hip).  One workgroup of four wavefronts owns a 64 x 64 tile of one
// matrix, each wavefront 32 x 32; slabs of 8 vectors (16 contraction
// entries) through two LDS buffers, the next slab's loads in flight during
// the current slab's MFMAs.  Bound by the reads of the two factors (16
// bytes per 2 flops and tile side).  One launch covers every matrix of the
// class instead of a GEMM per matrix, whose single 128 x 128 tile left 255
// CUs idle: 4096 real matrices n ~ U{16..128}, the 2119 of order above 70
// took
// 105 ms more in 6357 launches (forward and backward 146.9 -> 42.3 ms).
constexpr int VT = 64, VKB = 8, VLD = VT + 16;
__global__ void __launch_bounds__(256) vjp_gemm_kernel(VjpArgs a) {
  __shared__ double As[2][2 * VKB * VLD], Bs[2][2 * VKB * VLD];
  typedef double v4d __attribute__((ext_vector_type(4)));
  const int m = a.order[blockIdx.z];
  const int n = a.n[m];
  const int r0 = blockIdx.x * VT, s0 = blockIdx.y * VT;
  if (r0 >= n || s0 >= n) return;
  const zd* Y = reinterpret_cast<const zd*>(a.VL) + a.off[m];
  const zd* X = reinterpret_cast<const zd*>(a.VR) + a.off[m];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wr = (wave & 1) * 32, wc = (wave >> 1) * 32;
  const int ty = min(r0 + lane, n - 1), tx = min(s0 + lane, n - 1);
  const bool vy = r0 + lane < n, vx = s0 + lane < n;
  zd ry[2], rx[2];
  // unconditional loads from clamped addresses; entries outside the factors
  // are zeroed when staged
  auto fetch = [&](int k0) {
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      const int64_t k = min(k0 + wave + 4 * q, n - 1);
      ry[q] = Y[ty + k * n];
      rx[q] = X[tx + k * n];
    }
  };
  auto stage = [&](int k0, int buf) {
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      const int kk = wave + 4 * q;
      const bool vk = k0 + kk < n;
      As[buf][(2 * kk) * VLD + lane] = (vk && vy) ? ry[q].x : 0.0;
      As[buf][(2 * kk + 1) * VLD + lane] = (vk && vy) ? ry[q].y : 0.0;
      Bs[buf][(2 * kk) * VLD + lane] = (vk && vx) ? rx[q].x : 0.0;
      Bs[buf][(2 * kk + 1) * VLD + lane] = (vk && vx) ? rx[q].y : 0.0;
    }
  };
  v4d acc[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) acc[i][j] = v4d{0.0, 0.0, 0.0, 0.0};
  const int ns = (n + VKB - 1) / VKB;
  fetch(0);
  stage(0, 0);
  for (int sl = 0; sl < ns; ++sl) {
    const int buf = sl & 1;
    __syncthreads();
    fetch((sl + 1) * VKB);
#pragma unroll
    for (int k4 = 0; k4 < 2 * VKB / 4; ++k4) {
      const int kk = 4 * k4 + (lane >> 4);
      double af[2], bf[2];
#pragma unroll
      for (int i = 0; i < 2; ++i) af[i] = As[buf][kk * VLD + wr + 16 * i + (lane & 15)];
#pragma unroll
      for (int j = 0; j < 2; ++j) bf[j] = Bs[buf][kk * VLD + wc + 16 * j + (lane & 15)];
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(bf[j], af[i], acc[i][j], 0, 0, 0);
    }
    if (sl + 1 < ns) stage((sl + 1) * VKB, buf ^ 1);
  }
  double* Ab = a.Abar + a.off[m];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int gr = r0 + wr + 16 * i + (lane & 15), gc = s0 + wc + 16 * j + (lane >> 4) + 4 * r;
        if (gr < n && gc < n) Ab[gr + (int64_t)gc * n] = acc[i][j][r];
      }
}

// a.order lists matrices whose orders need the same number of tiles; VL is
// a.VL, writable (scaled in place)
hipError_t launch_vjp_class(const VjpArgs& a, double* VL, int nmax, hipStream_t s) {
  if (a.count <= 0 || nmax <= 0) return hipSuccess;
  const int nt = (nmax + VT - 1) / VT;
  // grid dimensions y and z hold at most 65535
  for (int first = 0; first < a.count; first += 65535) {
    VjpArgs b = a;
    b.order = a.order + first;
    b.count = std::min(a.count - first, 65535);
    hipLaunchKernelGGL(vjp_scale_kernel, dim3((nmax + 3) / 4, b.count), dim3(256), 0, s, b,
                       reinterpret_cast<zd*>(VL));
    hipLaunchKernelGGL(vjp_gemm_kernel, dim3(nt, nt, b.count), dim3(256), 0, s, b);
  }
  return hipGetLastError();
}

int vjp_tiles(int n) { return (n + VT - 1) / VT; }

__global__ void vjp_info_clear_kernel(int32_t* info, int count) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i < count) info[i] = 0;
}

hipError_t launch_vjp_info_clear(int32_t* info, int count, hipStream_t s) {
  if (count <= 0) return hipSuccess;
  hipLaunchKernelGGL(vjp_info_clear_kernel, dim3((count + 255) / 256), dim3(256), 0, s, info, count);
  return hipGetLastError();
}

size_t vjp_lds_bytes(int n) { return 16 * (2 * (size_t)(n + 1) * n + (size_t)n) + 16; }

hipError_t launch_vjp_assemble(const VjpArgs& a, int nmax, hipStream_t s) {
  if (a.count <= 0) return hipSuccess;
  const size_t lds = vjp_lds_bytes(nmax);
  if (lds > 160 * 1024) return hipErrorInvalidValue;
  (void)hipFuncSetAttribute((const void*)vjp_assemble_kernel<256>, hipFuncAttributeMaxDynamicSharedMemorySize,
                            (int)lds);
  hipLaunchKernelGGL(vjp_assemble_kernel<256>, dim3(a.count), dim3(256), lds, s, a);
  return hipGetLastError();
}

}  // namespace gs
