// Multishift sweeps of the large real QR iteration (dlarge.hip): MNB double
// shifts, the eigenvalues of the trailing 2 MNB x 2 MNB block of the active
// block, chased as a train of small bulges MSP rows apart (Braman, Byers and
// Mathias, "The multishift QR algorithm, part I", SIAM J. Matrix Anal. Appl.
// 23(4), 2002).  At time t bulge j performs the step k = istart + t - MSP j of
// a double-shift sweep (GenericSchur.jl:877-949); the bulges of one time lie
// MSP rows apart, so their left updates touch disjoint rows and their right
// updates disjoint columns, and one wavefront takes each.
//
// A sweep runs in chunks of MST times.  Workgroup 0 chases the chunk's train
// in an MNW x MNW window of H in LDS and logs the reflectors; the other
// workgroups of the launch apply the previous chunk's log outside its window:
// columns right of the current window, rows above the previous one, and Z.
#pragma once
#include "dchase.h"
#include "dev_common.h"

namespace gs {

// Smallest order with multishift sweeps.  They deflate the eigenvalues in an
// order of their own, so T's diagonal is another one of the matrix's valid
// ones than the double-shift iteration's.  They are faster from the LDS-resident
// range on, so the line is not the measurements': it keeps the double-shift
// iteration's order, which is the oracle's slot by slot and is held by the
// tests up to n = 160, for the orders below 256.  Measured, QR phase with Z,
// multishift against double-shift sweeps: n = 160 16.2 / 22.4 ms, n = 200 21.5 /
// 30.9, n = 256 29.1 / 48.4, n = 501 71.5 / 155, n = 1500 405 / 1191.
constexpr int MSMINN = 256;
// Smallest active block with multishift sweeps.  Measured, QR phase: n = 300
// 36.0 ms from 64 rows, 35.7 from 48, 36.2 from 80; n = 200 21.4, 23.9, 23.8.
constexpr int MSMIN = 64;
constexpr int MNB = 8;                                // bulges (wavefronts of the chase)
constexpr int MSP = 3;                                // rows between bulges
constexpr int MNW = 89;                               // window rows and columns
constexpr int MST = MNW - MSP * (MNB - 1) - 4;        // times per chunk
constexpr int MWP = MNW | 1;                          // odd LDS pitch of a window column
constexpr int MLP = 65;                               // pitch of the line buffer: 64 lines, odd
constexpr int MLB = 8;                                // times per block of ms_lines
constexpr int MLG = 3 * MNB * MST;                    // doubles of a chunk's log
static_assert(MST <= 64, "a chunk's new columns are the lines of one wavefront");
static_assert(MSP >= 3, "bulges of one time, and of neighbouring blocks of ms_lines, touch disjoint elements");
constexpr int MS_LDS = 8 * (MWP * MNW + MLP * (MNW + 2) + MLG);
static_assert(MS_LDS <= 160 * 1024, "LDS of a gfx950 CU");
static_assert(8 * MWP * (MNW + 64) <= MS_LDS && MWP >= 64, "the chase's unmasked loads stay in the LDS of the workgroup");

// State of the iteration between sweeps, on the device.
struct LState {
  int64_t iter, nsweep, nstep;
  int iend, istart, iterqr, iwcur, phase, status, mx, nb;  // nb > 0: a multishift sweep is due
  double v0, v1, v2;
  double sh[4 * MNB];  // (r1r, r1i, r2r, r2i) per bulge
};

// Chunk c (0-based) of a multishift sweep: times t0 .. t1 (t0 > t1: no chase,
// flush only), the previous chunk's pt0 .. pt1 (pt0 > pt1: none).
struct MChunk {
  int t0, t1, pt0, pt1;
};
__host__ GS_DEV int ms_times(int I, int E) { return E - I + MSP * (MNB - 1); }
__host__ GS_DEV int ms_chunks(int I, int E) { return (ms_times(I, E) + MST - 1) / MST; }
GS_DEV bool ms_chunk_of(int I, int E, int c, MChunk& ck) {
  const int nt = ms_times(I, E), nch = ms_chunks(I, E);
  if (c > nch) return false;
  ck.t0 = c < nch ? c * MST : 1;
  ck.t1 = c < nch ? min(c * MST + MST, nt) - 1 : 0;
  ck.pt0 = c > 0 ? (c - 1) * MST : 1;
  ck.pt1 = c > 0 ? min(c * MST, nt) - 1 : 0;
  return true;
}
// rows and columns that the times t0 .. t1 touch
GS_DEV int ms_wb(int I, int t0) { return max(I, I + t0 - MSP * (MNB - 1) - 1); }
GS_DEV int ms_we(int I, int E, int t1) { return min(E, I + t1 + 3); }

// tau fitted to the vector (1, v2, v3) as rounded: a Newton step towards
// 2 / (1 + v2^2 + v3^2).  What the reflector formulas leave of it is most of
// what Z loses.  n = 400, |Z^T Z - I| 1.63e-13 with the step, 2.25 without, 2.16
// by double-shift sweeps (7 % fewer reflectors); |A Z - Z T| / |A| 0.98, 1.28 and
// 1.23e-14.  Fitting the log's tau only, so that Z takes another reflector than
// T, gives 1.66e-13 and 1.12e-14, and eigenvector residuals 10 % above the
// double-shift ones instead of 15 % below.  Two more dependent operations of a
// step; n = 1500 462 ms with it, 465 without.
GS_DEV double ms_fit(double tau, double v2, double v3) {
  const double vv = fma(v3, v3, fma(v2, v2, 1.0));
  return fma(tau, fma(-0.5 * tau, vv, 1.0), tau);
}

// One 3-element reflector on a line.
GS_DEV void ms_apply(double& x0, double& x1, double& x2, double tau, double v2, double v3) {
  const double ss = x0 + v2 * x1 + v3 * x2;
  x0 = x0 - ss * tau;
  x1 = x1 - ss * (tau * v2);
  x2 = x2 - ss * (tau * v3);
}

// The log of times t0 .. t1 applied to 64 lines in LDS, element of row (or
// column) b + e of line l at buf[e MLP + l], two rows beyond the last one zero.
// Wavefront j applies bulge j, MLB times in registers, one block of times
// behind wavefront j - 1: the two then touch disjoint elements, and every
// element receives the reflectors in the order of the sweep.  MNB wavefronts.
GS_DEV void ms_lines(double* buf, const double* lg, int t0, int t1, int I, int E, int b) {
  const int lane = threadIdx.x & 63;
  const int j = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int nblk = (t1 - t0 + MLB) / MLB;
  for (int u = 0; u < nblk + MNB - 1; ++u) {
    const int q = u - j;
    if (q >= 0 && q < nblk) {
      const int lo = max(t0 + MLB * q, MSP * j);
      const int hi = min(min(t0 + MLB * q + MLB - 1, t1), E - 1 - I + MSP * j);
      if (lo <= hi) {
        double* p = buf + (I + lo - MSP * j - b) * MLP + lane;
        const double* l3 = lg + 3 * ((lo - t0) * MNB + j);
        const int cnt = hi - lo + 1;
        if (cnt == MLB) {
          double x[MLB + 2];
#pragma unroll
          for (int i = 0; i < MLB + 2; ++i) x[i] = p[i * MLP];
#pragma unroll
          for (int i = 0; i < MLB; ++i)
            ms_apply(x[i], x[i + 1], x[i + 2], l3[3 * MNB * i], l3[3 * MNB * i + 1], l3[3 * MNB * i + 2]);
#pragma unroll
          for (int i = 0; i < MLB + 2; ++i) p[i * MLP] = x[i];
        } else {
          double x0 = p[0], x1 = p[MLP];
          for (int i = 0; i < cnt; ++i) {
            double x2 = p[(i + 2) * MLP];
            ms_apply(x0, x1, x2, l3[3 * MNB * i], l3[3 * MNB * i + 1], l3[3 * MNB * i + 2]);
            p[i * MLP] = x0;
            x0 = x1;
            x1 = x2;
          }
          p[cnt * MLP] = x0;
          p[(cnt + 1) * MLP] = x1;
        }
      }
    }
    __syncthreads();
  }
}

// First column of (H - s1)(H - s2) (GenericSchur.jl:851-876) from H's leading
// entries and the shifts sh (r1r, r1i, r2r, r2i), scaled to unit 1-norm.  The
// block is unreduced when the sweep begins, but the bulges after the first
// meet the entries that those before them have left: a column that has
// vanished gives zeros (an identity reflector: that bulge moves nothing), not
// a quotient by zero.
__host__ GS_DEV void ms_first(double h11, double h12, double h21, double h22, double h32, const double* sh, double& v0,
                              double& v1, double& v2) {
  v0 = v1 = v2 = 0.0;
  double sx = fabs(h11 - sh[2]) + fabs(sh[3]) + fabs(h21);
  if (sx == 0.0) return;
  h21 = h21 / sx;
  const double w0 = h21 * h12 + (h11 - sh[0]) * ((h11 - sh[2]) / sx) - sh[1] * (sh[3] / sx);
  const double w1 = h21 * (h11 + h22 - sh[0] - sh[2]);
  const double w2 = h21 * h32;
  sx = fabs(w0) + fabs(w1) + fabs(w2);
  if (sx == 0.0) return;
  v0 = w0 / sx;
  v1 = w1 / sx;
  v2 = w2 / sx;
}

// Times t0 .. t1 of the train in the window win (rows and columns wb .. we,
// entry (r, c) at win[(r - wb) + (c - wb) MWP]), wavefront j with bulge j;
// the reflectors (tau, v2, v3) to lg[3 ((t - t0) MNB + j)].  Per time: the
// left updates of all bulges, a barrier, the right updates, a barrier.  The
// next reflector's input comes from the right update's lanes, so no LDS round
// trip lies between it and the reflector, and its operands are loaded before
// the reflector.  Bulges inside the block (I < k <= E - 3) take the short form:
// the annihilated column rides in lane 0 of the left update, addresses advance
// by a constant, idle lanes load whatever lies there and store nothing.
GS_DEV void ms_chase(double* win, double* lg, const double* sh, int t0, int t1, int I, int E, int wb, int we) {
  const int lane = threadIdx.x & 63;
  const int j = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  auto W = [&](int r, int c) -> double& { return win[(r - wb) + (c - wb) * MWP]; };
  double nv0 = 0.0, nv1 = 0.0, nv2 = 0.0;
  int k = I + t0 - MSP * j;
  if (k > I && k <= E - 1) {
    nv0 = W(k, k - 1);
    nv1 = W(k + 1, k - 1);
    nv2 = k + 2 <= E ? W(k + 2, k - 1) : 0.0;
  }
  nv0 = rdfirst(nv0);
  nv1 = rdfirst(nv1);
  nv2 = rdfirst(nv2);
  int oL = (k - wb) + (k - 1 - wb + lane) * MWP;       // (k, k - 1 + lane)
  int oR = (k + 3 - lane - wb) + (k - wb) * MWP;       // (k + 3 - lane, k)
  double lt = 0.0, l2 = 0.0, l3 = 0.0;                 // lane s: the reflector of time t0 + s
  for (int t = t0; t <= t1; ++t, ++k, oL += MWP + 1, oR += MWP + 1) {
    const bool act = k >= I && k <= E - 1;
    const bool inner = k > I && k <= E - 3;
    const bool three = k <= E - 2;
    double tau = 0.0, v2 = 0.0, v3 = 0.0, tau2 = 0.0, tau3 = 0.0;
    if (inner) {
      double* const p = win + oL;
      const bool two = k + 63 <= we;  // uniform
      double a0 = p[0], a1 = p[1], a2 = p[2];
      double b0 = 0.0, b1 = 0.0, b2 = 0.0;
      double* const q = &W(k, k + 63) + min(lane, we - k - 63) * MWP;
      if (two) {
        b0 = q[0];
        b1 = q[1];
        b2 = q[2];
      }
      double beta = nv0;
      v2 = nv1;
      v3 = nv2;
      tau = ms_fit(dreflector3_wave(beta, v2, v3), v2, v3);
      tau2 = tau * v2;
      tau3 = tau * v3;
      const bool l0 = lane == 0;
      const double sa = a0 + v2 * a1 + v3 * a2;
      a0 = l0 ? beta : a0 - sa * tau;
      a1 = l0 ? 0.0 : a1 - sa * tau2;
      a2 = l0 ? 0.0 : a2 - sa * tau3;
      if (lane <= we - k + 1) {
        p[0] = a0;
        p[1] = a1;
        p[2] = a2;
      }
      if (two) {
        const double sb = b0 + v2 * b1 + v3 * b2;
        if (lane <= we - k - 63) {
          q[0] = b0 - sb * tau;
          q[1] = b1 - sb * tau2;
          q[2] = b2 - sb * tau3;
        }
      }
    } else if (act) {
      if (k == I) {
        ms_first(W(I, I), W(I, I + 1), W(I + 1, I), W(I + 1, I + 1), W(I + 2, I + 1), sh + 4 * j, nv0, nv1, nv2);
      }
      double beta = nv0;
      v2 = nv1;
      v3 = nv2;
      if (three) {
        tau = dreflector3_wave(beta, v2, v3);
      } else {
        tau = dreflector_fast(2, beta, v2, v3);
        v3 = 0.0;
      }
      tau = ms_fit(tau, v2, v3);
      tau2 = tau * v2;
      tau3 = tau * v3;
      for (int c = k + lane; c <= we; c += 64) {
        double* const p = &W(k, c);
        const double a0 = p[0], a1 = p[1], a2 = three ? p[2] : 0.0;
        const double sa = a0 + v2 * a1 + v3 * a2;
        p[0] = a0 - sa * tau;
        p[1] = a1 - sa * tau2;
        if (three) p[2] = a2 - sa * tau3;
      }
      if (lane == 0 && k > I) {
        double* const z = &W(k, k - 1);
        z[0] = beta;
        z[1] = 0.0;
        if (three) z[2] = 0.0;
      }
    }
    {
      const bool me = lane == t - t0;
      lt = me ? tau : lt;
      l2 = me ? v2 : l2;
      l3 = me ? v3 : l3;
    }
    __syncthreads();
    if (inner) {
      double* const p = win + oR;
      const bool two = k - 61 >= wb;  // uniform
      double a0 = p[0], a1 = p[MWP], a2 = p[2 * MWP];
      double b0 = 0.0, b1 = 0.0, b2 = 0.0;
      if (two) {
        b0 = p[-64];
        b1 = p[MWP - 64];
        b2 = p[2 * MWP - 64];
      }
      const double sa = a0 + v2 * a1 + v3 * a2;
      a0 = a0 - sa * tau;
      // rows k + 1 .. k + 3 of column k: the next step's input
      nv0 = rdlane(a0, 2);
      nv1 = rdlane(a0, 1);
      nv2 = rdlane(a0, 0);
      if (lane <= k + 3 - wb) {
        p[0] = a0;
        p[MWP] = a1 - sa * tau2;
        p[2 * MWP] = a2 - sa * tau3;
      }
      if (two) {
        const double sb = b0 + v2 * b1 + v3 * b2;
        if (lane <= k - 61 - wb) {
          p[-64] = b0 - sb * tau;
          p[MWP - 64] = b1 - sb * tau2;
          p[2 * MWP - 64] = b2 - sb * tau3;
        }
      }
    } else if (act) {
      const int jm = min(k + 3, E);
      for (int r = jm - lane; r >= wb; r -= 64) {
        double* const p = &W(r, k);
        const double a0 = p[0], a1 = p[MWP], a2 = three ? p[2 * MWP] : 0.0;
        const double sa = a0 + v2 * a1 + v3 * a2;
        p[0] = a0 - sa * tau;
        p[MWP] = a1 - sa * tau2;
        if (three) p[2 * MWP] = a2 - sa * tau3;
      }
      wsync();
      if (k <= E - 2) {
        nv0 = rdfirst(W(k + 1, k));
        nv1 = rdfirst(W(k + 2, k));
        nv2 = k + 3 <= E ? rdfirst(W(k + 3, k)) : 0.0;
      }
    }
    __syncthreads();
  }
  if (lane <= t1 - t0) {
    double* const g = lg + 3 * (lane * MNB + j);
    g[0] = lt;
    g[1] = l2;
    g[2] = l3;
  }
}

hipError_t launch_dshift(const double* H, int64_t ld, LState* st, int64_t maxiter, hipStream_t s);

}  // namespace gs
