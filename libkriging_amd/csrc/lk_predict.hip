// Prediction kernels on gfx950, FP64 (KrigingImpl.cpp:145-291): mean and
// variance at m new points, their covariance and derivatives, from the
// model's L^-1, M = L^-1 F, z and R*.
//
// R_on and C = L^-1 R_on keep the points contiguous, (1 + d) groups of mpad
// columns beside each other when derivatives are wanted: one launch takes
// L^-1 through all of them, every operand is read in whole 128-byte lines,
// and the sums over the design run with a point per lane.
#include <hip/hip_runtime.h>

#include <type_traits>

#include <math.h>

#include "lk_device.hpp"
#include "lk_kernels.h"

namespace lk {

// d ln k / d dx_k (Covariance.cpp:52-63, 90-101, 132-146, 181-198), dx =
// x_new - x_obs, it = 1 / theta_k
__device__ inline double dlncov_dx(int kern, double dx, double it) {
  const double sg = dx > 0.0 ? 1.0 : (dx < 0.0 ? -1.0 : 0.0);
  if (kern == K_GAUSS) return -dx * it * it;
  if (kern == K_EXP) return -sg * it;
  if (kern == K_MATERN32) {
    const double u = SQRT3 * fabs(dx * it);
    return -SQRT3 * sg * (u / (1.0 + u)) * it;
  }
  const double u = SQRT5 * fabs(dx * it);
  const double aa = 1.0 + u, bb = u * (1.0 / 3.0);
  return -SQRT5 * sg * ((aa * bb) / (aa + u * bb)) * it;
}

// R_on(i, j) = factor * k(x_i - xn_j), 1 where the points coincide
// (|dx_k| <= eps for all k, KrigingImpl.cpp:202-205), and in the groups 1 + k
// its derivative R_on d ln k / d dx_k; zero padding.  64 points by ROWS
// design rows per workgroup.  Bound by the covariances (one exp per pair):
// 16 rows when 64-row tiles would not fill the chip (n = 200, 1000 points:
// 13.2 -> 6.9 us), else 64.  grid (mpad / 64, npad / ROWS)
template <int DT, int ROWS, bool DERIV>
__global__ __launch_bounds__(TPB) void k_pred_cross(PredictArgs a) {
  const int j0 = blockIdx.x * NB, i0 = blockIdx.y * ROWS, tid = threadIdx.x;
  const int n = a.n, m = a.m, d = a.d;
  const size_t ld = (size_t)a.groups * a.mpad;
  __shared__ double sXo[DT * ROWS];
  __shared__ double sXn[DT * NB];
  for (int q = tid; q < d * ROWS; q += TPB) {
    const int k = q / ROWS, r = q % ROWS;
    sXo[q] = (i0 + r < n) ? a.X[(size_t)k * n + i0 + r] : 0.0;
  }
  for (int q = tid; q < d * NB; q += TPB) {
    const int k = q / NB, r = q % NB;
    sXn[q] = (j0 + r < m) ? a.Xn[(size_t)k * m + j0 + r] : 0.0;
  }
  __syncthreads();
  const int jj = tid & 63, gj = j0 + jj;
  double dx[DT];
  for (int r = 0; r < ROWS / 4; ++r) {
    const int ii = (tid >> 6) + 4 * r, gi = i0 + ii;
    double v = 0.0;
    const bool in = gi < n && gj < m;
    if (in) {
      bool same = true;
#pragma unroll
      for (int k = 0; k < DT; ++k) {
        dx[k] = (k < d) ? sXo[k * ROWS + ii] - sXn[k * NB + jj] : 0.0;
        same = same && fabs(dx[k]) <= 2.220446049250313e-16;
      }
      v = same ? 1.0 : kern_rho<DT>(a.kernel, dx, a.itheta) * a.factor;
    }
    double* R = a.Ron + (size_t)gi * ld + gj;
    R[0] = v;
    if constexpr (DERIV)
      for (int k = 0; k < d; ++k) {
        const double g = in ? dlncov_dx(a.kernel, sXn[k * NB + jj] - sXo[k * ROWS + ii], a.itheta[k]) : 0.0;
        R[(size_t)(k + 1) * a.mpad] = v * g;
      }
  }
}

// ---------------------------------------------------------------------------
// A 64 x 64 tile: sum_k P(i0 + row, k) Q(j0 + col, k) over [0, 4 nst), P and Q
// with rows contiguous (P[k * ldp + row]).  Each wave runs the whole tile (16
// blocks of 16 x 16 for 8 operand loads a step) over a quarter of the K range,
// its operands straight from memory into registers four steps ahead, with no
// LDS and no barrier in the loop; the four sums s_w meet in LDS as (s_0 + s_2)
// + (s_1 + s_3), the order of tile32_sum too: an element has the same bits in
// either.  v[r]: element (w + 4 r, lane).  sS: 2 NB LDSS doubles.
// ---------------------------------------------------------------------------
template <bool NEG>
__device__ inline void tile64(const double* __restrict__ P, int ldp, int i0, const double* __restrict__ Q, int ldq,
                              int j0, int nst, double* __restrict__ sS, double (&v)[16], int tid) {
  const int lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6), r16 = lane & 15, kq = lane >> 4;
  const int s0 = nst * w / 4, s1 = nst * (w + 1) / 4;
  const double* Pl = P + (size_t)kq * ldp + i0 + r16;
  const double* Ql = Q + (size_t)kq * ldq + j0 + r16;
  d4 acc[4][4];
#pragma unroll
  for (int x = 0; x < 4; ++x)
#pragma unroll
    for (int y = 0; y < 4; ++y) acc[x][y] = d4{0.0, 0.0, 0.0, 0.0};
  constexpr int D = 4;
  double p[D][4], q[D][4];
  auto load = [&](int u, int s) __attribute__((always_inline)) {
    const size_t k = 4 * (size_t)min(s, s1 - 1);
#pragma unroll
    for (int x = 0; x < 4; ++x) {
      p[u][x] = gload(Pl + k * ldp + 16 * x);
      q[u][x] = gload(Ql + k * ldq + 16 * x);
    }
  };
#pragma unroll
  for (int u = 0; u < D; ++u) {
    __builtin_amdgcn_sched_barrier(0);
    load(u, s0 + u);
  }
  for (int s = s0; s < s1; s += D) {
#pragma unroll
    for (int u = 0; u < D; ++u) {
      __builtin_amdgcn_sched_barrier(0);
      if (s + u < s1) {
#pragma unroll
        for (int x = 0; x < 4; ++x)
#pragma unroll
          for (int y = 0; y < 4; ++y)
            acc[x][y] = __builtin_amdgcn_mfma_f64_16x16x4f64(NEG ? -p[u][x] : p[u][x], q[u][y], acc[x][y], 0, 0, 0);
      }
      load(u, s + u + D);
    }
  }
  auto put = [&](double* d) __attribute__((always_inline)) {
#pragma unroll
    for (int x = 0; x < 4; ++x)
#pragma unroll
      for (int y = 0; y < 4; ++y)
#pragma unroll
        for (int e = 0; e < 4; ++e) d[(16 * x + kq + 4 * e) * LDSS + 16 * y + r16] = acc[x][y][e];
  };
  if (w >= 2) put(sS + (w - 2) * NB * LDSS);
  __syncthreads();
  if (w < 2) {
    const double* d = sS + w * NB * LDSS;
#pragma unroll
    for (int x = 0; x < 4; ++x)
#pragma unroll
      for (int y = 0; y < 4; ++y) {
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[x][y][e] += d[(16 * x + kq + 4 * e) * LDSS + 16 * y + r16];
        __builtin_amdgcn_sched_barrier(0);
      }
  }
  __syncthreads();
  if (w < 2) put(sS + w * NB * LDSS);
  __syncthreads();
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    const int o = (w + 4 * r) * LDSS + lane;
    v[r] = sS[o] + sS[o + NB * LDSS];
  }
}

// C = L^-1 R_on on 64 x 64 tiles, the longest rows first.  Bound by the MFMA:
// n = 3001, 5003 points: 810 us, 58 TFLOP/s, the MFMA busy 84 % of the time
// (staged through LDS, a quadrant per wave: 850 .. 890 us and 76 %; 128 x 64
// tiles that way: 837 us).
// grid (columns / 64, npad / 64)
__global__ __launch_bounds__(TPB, 2) void k_pred_trmm(PredictArgs a) {
  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int t0 = blockIdx.x * NB, i0 = ((int)gridDim.y - 1 - (int)blockIdx.y) * NB;
  const int ld = a.groups * a.mpad;
  __shared__ double sS[2 * NB * LDSS];
  double v[16];
  tile64<false>(a.Linv, a.npad, i0, a.Ron, ld, t0, (i0 + NB) / 4, sS, v, tid);
#pragma unroll
  for (int r = 0; r < 16; ++r) a.C[(size_t)(i0 + w + 4 * r) * ld + t0 + lane] = v[r];
}

// ---------------------------------------------------------------------------
// 32 x 32 tiles for products too small to fill the chip with 64 x 64 ones:
// the four waves take a quarter of the K range each, operands straight from
// memory into the MFMA's registers (T32_D steps of 4 in flight), and add up
// through LDS: a sixteenth of the chain per wave, for twice the reads.
// ---------------------------------------------------------------------------
constexpr int T32 = 32;
constexpr int T32_D = 8;
constexpr int T32_S = T32 + 1;  // row pitch of the partial sums

// part (this wave's) = sum_k P(i0 + row, k) Q(j0 + col, k) for its quarter of
// [0, kend), P and Q with rows contiguous (P[k * ldp + row]); the sums of the
// four waves to sS: row-major, col fastest
template <bool NEG>
__device__ inline void tile32(const double* __restrict__ P, int ldp, int i0, const double* __restrict__ Q, int ldq,
                              int j0, int kend, double* __restrict__ sS, int tid) {
  const int lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6), r16 = lane & 15, kq = lane >> 4;
  const int nst = kend / 4, s0 = nst * w / 4, s1 = nst * (w + 1) / 4;
  const double* Pl = P + (size_t)kq * ldp + i0 + r16;
  const double* Ql = Q + (size_t)kq * ldq + j0 + r16;
  d4 acc[2][2];
  acc_zero(acc);
  double p[T32_D][2], q[T32_D][2];
  auto load = [&](int u, int s) __attribute__((always_inline)) {
    const size_t k = 4 * (size_t)min(s, s1 - 1);
    p[u][0] = gload(Pl + k * ldp);
    p[u][1] = gload(Pl + k * ldp + 16);
    q[u][0] = gload(Ql + k * ldq);
    q[u][1] = gload(Ql + k * ldq + 16);
  };
  if (s0 < s1) {
#pragma unroll
    for (int u = 0; u < T32_D; ++u) {
      __builtin_amdgcn_sched_barrier(0);
      load(u, s0 + u);
    }
    for (int s = s0; s < s1; s += T32_D) {
#pragma unroll
      for (int u = 0; u < T32_D; ++u) {
        __builtin_amdgcn_sched_barrier(0);
        if (s + u < s1) {
#pragma unroll
          for (int bi = 0; bi < 2; ++bi)
#pragma unroll
            for (int bj = 0; bj < 2; ++bj)
              acc[bi][bj] = __builtin_amdgcn_mfma_f64_16x16x4f64(NEG ? -p[u][bi] : p[u][bi], q[u][bj], acc[bi][bj], 0, 0, 0);
        }
        load(u, s + u + T32_D);
      }
    }
  }
  double* part = sS + w * T32 * T32_S;
#pragma unroll
  for (int bi = 0; bi < 2; ++bi)
#pragma unroll
    for (int bj = 0; bj < 2; ++bj)
#pragma unroll
      for (int e = 0; e < 4; ++e) part[(16 * bi + kq + 4 * e) * T32_S + 16 * bj + r16] = acc[bi][bj][e];
  __syncthreads();
}
__device__ inline double tile32_sum(const double* sS, int row, int col) {
  const double* s = sS + row * T32_S + col;
  return (s[0] + s[2 * T32 * T32_S]) + (s[T32 * T32_S] + s[3 * T32 * T32_S]);
}

// K ends with the 64-row block, as in k_pred_trmm: the quarters are the same,
// and L^-1 is zero beyond the diagonal.  grid (columns / 32, npad / 32)
__global__ __launch_bounds__(TPB) void k_pred_trmm32(PredictArgs a) {
  const int tid = threadIdx.x, t0 = blockIdx.x * T32, i0 = ((int)gridDim.y - 1 - (int)blockIdx.y) * T32;
  const int ld = a.groups * a.mpad;
  __shared__ double sS[4 * T32 * T32_S];
  tile32<false>(a.Linv, a.npad, i0, a.Ron, ld, t0, (i0 / NB + 1) * NB, sS, tid);
  const int col = tid & 31;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int row = (tid >> 5) + 8 * r;
    a.C[(size_t)(i0 + row) * ld + t0 + col] = tile32_sum(sS, row, col);
  }
}

// ---------------------------------------------------------------------------
// The sums over the design: with x a column of C, sum_i x_i z_i and x_i
// M_iq (q < p), and sum_i x_i c_i with c the point's column of group 0.
// Group 0 gives the mean and variance factor,
//   mean = f_j beta + C' z,  1 - |C|^2 + |E circ_j|^2 with
//   E circ_j = (f_j - C' M) R*^-1  (KrigingImpl.cpp:227-242), clipped at 0;
// group 1 + k, with W = L^-1 dR_on / dx_k, the derivatives
//   dmean_k = (dF_j beta)_k + W' z
//   dvar_k  = -2 C' W + 2 Ecirc_j DEcirc_k, DEcirc_k = solve_lower(R*',
//             dF_j(k, :)' - M' W)  (KrigingImpl.cpp:276-288).
// PS_P points per workgroup, lane = (point, one of PS_R rows); 16 waves share
// the rows, PS_U loads of PS_R rows in flight each, and their sums are added
// in order.  Bound by the chain of its loads where there are few points (n =
// 1000, 500 points, 6 columns: 17 us; one wave per point and a pass per
// column: 31), by reading C and the coefficients beside it where there are
// many (n = 3001, 5003 points: 42 us, 50; 64 points per workgroup: 43).
// grid (mpad / PS_P) or (mpad / PS_P, d)
// ---------------------------------------------------------------------------
constexpr int PS_W = 16;
constexpr int PS_P = 16;
constexpr int PS_R = 64 / PS_P;
constexpr int PS_U = 4;

// PS_Q: columns of [M | z] per pass
template <bool DERIV, int PS_Q>
__global__ __launch_bounds__(64 * PS_W) void k_pred_sums(PredictArgs a) {
  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r16 = lane % PS_P, kq = lane / PS_P;
  const int k = blockIdx.y, n = a.n, p = a.p, m = a.m;
  const size_t ld = (size_t)a.groups * a.mpad;
  const double* c = a.C + (size_t)kq * ld + blockIdx.x * PS_P + r16;
  const double* x = c + (DERIV ? (size_t)(k + 1) * a.mpad : 0);
  __shared__ double red[PS_W][PS_Q + 1][PS_P];
  __shared__ double sS[PMAX + 2][PS_P];         // sums over M_q (q < p), z, c; then e
  __shared__ double sK[PMAX + PMAX * PMAX];     // beta, R*
  for (int q = tid; q < p + p * p; q += 64 * PS_W) sK[q] = a.coef[q];
  const int nst = (n + PS_R - 1) / PS_R;
  for (int q0 = 0; q0 <= p; q0 += PS_Q) {
    const int nq = min(PS_Q, p + 1 - q0);
    const double* mz = a.MZ + (size_t)q0 * a.npad + kq;
    double s[PS_Q] = {}, sc = 0.0;
    for (int s0 = PS_U * w; s0 < nst; s0 += PS_U * PS_W) {
      double xv[PS_U], cv[PS_U], mv[PS_U][PS_Q];
      bool on[PS_U];
#pragma unroll
      for (int u = 0; u < PS_U; ++u) {
        const int st = s0 + u, row = PS_R * min(st, nst - 1);
        const bool in = st < nst && row + kq < n;
        xv[u] = gload(x + (size_t)row * ld);
        cv[u] = (DERIV && q0 == 0) ? gload(c + (size_t)row * ld) : xv[u];
        // columns past nq re-read the last one and are dropped
#pragma unroll
        for (int q = 0; q < PS_Q; ++q) mv[u][q] = gload(mz + (size_t)min(q, nq - 1) * a.npad + row);
        on[u] = in;
      }
#pragma unroll
      for (int u = 0; u < PS_U; ++u) {
        const double xu = on[u] ? xv[u] : 0.0;
#pragma unroll
        for (int q = 0; q < PS_Q; ++q) s[q] = fma(xu, on[u] ? mv[u][q] : 0.0, s[q]);
        sc = fma(xu, cv[u], sc);
      }
    }
#pragma unroll
    for (int q = 0; q <= PS_Q; ++q) {
      double v = q < PS_Q ? s[q] : sc;
      v += __shfl_xor(v, 16, 64);
      v += __shfl_xor(v, 32, 64);
      if (kq == 0) red[w][q][r16] = v;
    }
    __syncthreads();
    const int q = tid / PS_P, t = tid % PS_P;
    if (q < nq || (q0 == 0 && q == PS_Q)) {
      double v = red[0][q][t];
#pragma unroll
      for (int u = 1; u < PS_W; ++u) v += red[u][q][t];
      sS[q == PS_Q ? PMAX + 1 : q0 + q][t] = v;
    }
    __syncthreads();
  }
  const int j = blockIdx.x * PS_P + tid;
  if (tid >= PS_P || j >= m) return;
  const double* beta = sK;
  const double* Rs = sK + p;
  // the point's own column of sS: e, then the forward substitution R*' c = e
  auto solve = [&](auto use) __attribute__((always_inline)) {
    for (int q = 0; q < p; ++q) {
      double t = sS[q][tid];
      for (int r = 0; r < q; ++r) t -= Rs[r + q * p] * sS[r][tid];
      t /= Rs[q + q * p];
      sS[q][tid] = t;
      use(q, t);
    }
  };
  if constexpr (!DERIV) {
    double mean = sS[p][tid], ee = 0.0;
    for (int q = 0; q < p; ++q) {
      const double f = (q == 0) ? 1.0 : a.Xn[(size_t)(q - 1) * m + j];
      mean = fma(f, beta[q], mean);
      sS[q][tid] = f - sS[q][tid];
    }
    solve([&](int q, double t) {
      ee = fma(t, t, ee);
      if (a.ecirc != nullptr) a.ecirc[(size_t)q * m + j] = t;
    });
    double v = 1.0 - sS[PMAX + 1][tid] + ee;
    if (isnan(v) || v < 0.0) v = 0.0;
    a.out[j] = mean;
    a.out[m + j] = v;
  } else {
    double dm = sS[p][tid];
    if (a.linear_trend) dm += beta[k + 1];  // dF(k, q) = 1 for q = k + 1
    a.dmean[(size_t)k * m + j] = dm;
    if (!a.want_var) return;
    for (int q = 0; q < p; ++q) sS[q][tid] = ((a.linear_trend && q == k + 1) ? 1.0 : 0.0) - sS[q][tid];
    double ed = 0.0;
    solve([&](int q, double t) { ed = fma(a.ecirc[(size_t)q * m + j], t, ed); });
    a.dvar[(size_t)k * m + j] = -2.0 * sS[PMAX + 1][tid] + 2.0 * ed;
  }
}

// ---------------------------------------------------------------------------
// predictive covariance: Sigma = R_nn - C' C + Ecirc Ecirc' (before
// var_scale).  R_nn as LinearAlgebra::covMat_sym_X (LinearAlgebra.cpp:531-596):
// factor * k(xn_i - xn_j) off the diagonal, 1 on it.  Sigma is symmetric:
// grid T (T + 1) / 2 over the lower tiles, T = mpad / S, each off-diagonal
// tile stored at both of its places.  S = 64 or, with few tiles, 32.
// ---------------------------------------------------------------------------
template <int DT>
__device__ inline double pred_sigma(const PredictArgs& a, double cc, const double* sXi, const double* sXj, int S,
                                    int r, int c, int gi, int gj) {
  double rnn = 1.0;
  if (gi != gj) {
    double dx[DT];
#pragma unroll
    for (int k = 0; k < DT; ++k) dx[k] = sXi[k * S + r] - sXj[k * S + c];
    rnn = kern_rho<DT>(a.kernel, dx, a.itheta) * a.nn_factor;
  }
  double ec = 0.0;
  for (int q = 0; q < a.p; ++q) ec = fma(a.ecirc[(size_t)q * a.m + gi], a.ecirc[(size_t)q * a.m + gj], ec);
  return cc + rnn + ec;
}

template <int DT>
__device__ inline void pred_stage_points(const PredictArgs& a, double* sXi, double* sXj, int S, int i0, int j0,
                                         int tid) {
  for (int q = tid; q < DT * S; q += TPB) {
    const int k = q / S, r = q % S;
    sXi[q] = (k < a.d && i0 + r < a.m) ? a.Xn[(size_t)k * a.m + i0 + r] : 0.0;
    sXj[q] = (k < a.d && j0 + r < a.m) ? a.Xn[(size_t)k * a.m + j0 + r] : 0.0;
  }
}

template <int DT>
__global__ __launch_bounds__(TPB, 2) void k_pred_cov(PredictArgs a) {
  int ti, tj;
  tri_decode(blockIdx.x, ti, tj);
  const int i0 = ti * NB, j0 = tj * NB;
  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int m = a.m, ld = a.groups * a.mpad;
  __shared__ double sS[2 * NB * LDSS];
  double v[16];
  tile64<true>(a.C, ld, j0, a.C, ld, i0, a.npad / 4, sS, v, tid);  // rows j, columns i
  static_assert(2 * DMAX * NB <= 2 * NB * LDSS && NB * (NB + 1) <= 2 * NB * LDSS, "what follows in sS");
  double* sXi = sS;
  double* sXj = sS + DT * NB;
  __syncthreads();  // every wave has read its sums
  pred_stage_points<DT>(a, sXi, sXj, NB, i0, j0, tid);
  __syncthreads();
  const int gi = i0 + lane;
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    const int c = w + 4 * r, gj = j0 + c;
    if (gi >= m || gj >= m) continue;
    v[r] = pred_sigma<DT>(a, v[r], sXi, sXj, NB, lane, c, gi, gj);
    a.cov[(size_t)gj * m + gi] = v[r];
  }
  if (ti == tj) return;
  // the transpose of an off-diagonal tile, through LDS: stored in rows too
  __syncthreads();  // every wave is done with sXi / sXj
#pragma unroll
  for (int r = 0; r < 16; ++r) sS[lane * (NB + 1) + w + 4 * r] = v[r];
  __syncthreads();
  for (int r = 0; r < 16; ++r) {
    const int row = w + 4 * r;
    if (i0 + row < m && j0 + lane < m) a.cov[(size_t)(i0 + row) * m + j0 + lane] = sS[row * (NB + 1) + lane];
  }
}

template <int DT>
__global__ __launch_bounds__(TPB) void k_pred_cov32(PredictArgs a) {
  int ti, tj;
  tri_decode(blockIdx.x, ti, tj);
  const int i0 = ti * T32, j0 = tj * T32, tid = threadIdx.x;
  const int m = a.m, ld = a.groups * a.mpad;
  __shared__ double sS[4 * T32 * T32_S];
  __shared__ double sXi[DT * T32];
  __shared__ double sXj[DT * T32];
  pred_stage_points<DT>(a, sXi, sXj, T32, i0, j0, tid);
  tile32<true>(a.C, ld, j0, a.C, ld, i0, a.npad, sS, tid);  // rows j, columns i
  const int x = tid & 31, y = tid >> 5;
  double v[4];
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int c = y + 8 * r, gi = i0 + x, gj = j0 + c;
    v[r] = 0.0;
    if (gi < m && gj < m) {
      v[r] = pred_sigma<DT>(a, tile32_sum(sS, c, x), sXi, sXj, T32, x, c, gi, gj);
      a.cov[(size_t)gj * m + gi] = v[r];
    }
  }
  if (ti == tj) return;
  __syncthreads();
#pragma unroll
  for (int r = 0; r < 4; ++r) sS[x * T32_S + y + 8 * r] = v[r];
  __syncthreads();
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int gi = i0 + y + 8 * r, gj = j0 + x;
    if (gi < m && gj < m) a.cov[(size_t)gi * m + gj] = sS[(y + 8 * r) * T32_S + x];
  }
}

// ---------------------------------------------------------------------------
// launchers
// ---------------------------------------------------------------------------
// up to here (in 64 x 64 tiles) a product runs on 32 x 32 tiles: n = 200,
// 1000 points (64 tiles) 6.5 us, 14 with 64 x 64 ones staged through LDS; the
// covariance of 500 points at n = 1000 (36 tiles) 18 us, 65; 640 tiles at n =
// 1000 66 us, 65
constexpr int PRED_SMALL_TILES = 512;

template <class F>
static void with_dims(int d, F f) {
  if (d <= 4)
    f(std::integral_constant<int, 4>{});
  else if (d <= 8)
    f(std::integral_constant<int, 8>{});
  else if (d <= 16)
    f(std::integral_constant<int, 16>{});
  else
    f(std::integral_constant<int, 32>{});
}

template <bool DERIV>
static void launch_sums(const PredictArgs& a, hipStream_t stream) {
  const dim3 grid(a.mpad / PS_P, DERIV ? a.d : 1), block(64 * PS_W);
  // one pass up to a constant trend, else six columns a pass
  if (a.p + 1 <= 2)
    hipLaunchKernelGGL((k_pred_sums<DERIV, 2>), grid, block, 0, stream, a);
  else
    hipLaunchKernelGGL((k_pred_sums<DERIV, 6>), grid, block, 0, stream, a);
}

hipError_t launch_predict(const PredictArgs& a, hipStream_t stream) {
  const int cols = a.groups * a.mpad, tiles = (a.mpad / NB) * (a.npad / NB);
  with_dims(a.d, [&](auto tag) {
    constexpr int DT = decltype(tag)::value;
    const dim3 g64(a.mpad / NB, a.npad / NB), g16(a.mpad / NB, a.npad / 16);
    if (tiles <= PRED_SMALL_TILES) {
      if (a.groups > 1)
        hipLaunchKernelGGL((k_pred_cross<DT, 16, true>), g16, dim3(TPB), 0, stream, a);
      else
        hipLaunchKernelGGL((k_pred_cross<DT, 16, false>), g16, dim3(TPB), 0, stream, a);
    } else {
      if (a.groups > 1)
        hipLaunchKernelGGL((k_pred_cross<DT, 64, true>), g64, dim3(TPB), 0, stream, a);
      else
        hipLaunchKernelGGL((k_pred_cross<DT, 64, false>), g64, dim3(TPB), 0, stream, a);
    }
  });
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  if (a.groups * tiles <= PRED_SMALL_TILES)
    hipLaunchKernelGGL(k_pred_trmm32, dim3(cols / T32, a.npad / T32), dim3(TPB), 0, stream, a);
  else
    hipLaunchKernelGGL(k_pred_trmm, dim3(cols / NB, a.npad / NB), dim3(TPB), 0, stream, a);
  if ((e = hipGetLastError()) != hipSuccess) return e;
  launch_sums<false>(a, stream);
  return hipGetLastError();
}

hipError_t launch_predict_deriv(const PredictArgs& a, hipStream_t stream) {
  if (a.groups != 1 + a.d) return hipErrorInvalidValue;
  launch_sums<true>(a, stream);
  return hipGetLastError();
}

hipError_t launch_predict_cov(const PredictArgs& a, hipStream_t stream) {
  const int T = a.mpad / NB, tiles = T * (T + 1) / 2;
  with_dims(a.d, [&](auto tag) {
    constexpr int DT = decltype(tag)::value;
    if (tiles <= PRED_SMALL_TILES)
      hipLaunchKernelGGL(k_pred_cov32<DT>, dim3(T * (2 * T + 1)), dim3(TPB), 0, stream, a);
    else
      hipLaunchKernelGGL(k_pred_cov<DT>, dim3(tiles), dim3(TPB), 0, stream, a);
  });
  return hipGetLastError();
}

}  // namespace lk
