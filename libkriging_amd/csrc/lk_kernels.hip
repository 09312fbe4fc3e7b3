// Kriging concentrated log-likelihood + adjoint gradient, FP64, gfx950.
//
// One "slot" is one LL(+grad) evaluation of one design at one parameter
// vector.  Every kernel below works on a batch of slots (grid.y or grid.x =
// slot) so that 64 multistart evaluations, or 256 uneven NestedKriging
// submodels, run in the same launches.  Matrices live in HBM as FP64
// column-major npad x npad (npad = n rounded up to 64, the padded part set to
// the identity so that every kernel works on whole 64 x 64 tiles).
//
// Pipeline of one evaluation (reference: Kriging::_logLikelihood,
// src/lib/Kriging.cpp:214-338, and KrigingImpl::populate_Model,
// src/lib/KrigingImpl.cpp:73-125):
//   build           R = factor * k(x_i - x_j; theta), unit (+jitter) diagonal
//   potrf chain/rows/update   blocked right-looking Cholesky, FP64 MFMA
//                   (chain and rows in lk_potrf.hip)
//   trtri           L^-1 by recursive doubling, FP64 MFMA
//   solve_fy, gls, solve_e, solve_x   F* = L^-1 F, y* = L^-1 y, GLS beta,
//                   E* = L^-1 (y - F beta), x = L^-T E*, |L|_1, |L^-1|_1
//   finalize_ll     log-det, SSE, LL, rcond check (and its 1-norm estimate)
//   lauum_adjoint   R^-1 = L^-T L^-1 tile by tile on MFMA; each tile is
//                   contracted at once with dR/dtheta_k recomputed from X
//                   (all k, plus the nugget direction), never stored
//   finalize_grad   deterministic reduction of the per-tile partial sums
#include <hip/hip_runtime.h>

#include <math.h>

#include <type_traits>

#include "lk_device.hpp"
#include "lk_kernels.h"

namespace lk {

// ---------------------------------------------------------------------------
// (0) Parameters in, results out: one wave per slot reads its parameters from
// (writes its results to) pinned host memory.  As launches of the captured
// pipeline these replace a copy before it and one after it, each its own
// submission with 8 - 12 us between it and the kernels (n = 200: 20 us of a
// 225 us evaluation).  grid (nslots), 64 threads
// ---------------------------------------------------------------------------
static_assert(sizeof(SlotParams) % 4 == 0 && sizeof(SlotOut) % 8 == 0, "copied by words");
__global__ __launch_bounds__(64) void k_params_in(const SlotParams* __restrict__ host, SlotParams* __restrict__ params) {
  const int* src = reinterpret_cast<const int*>(host + blockIdx.x);
  int* dst = reinterpret_cast<int*>(params + blockIdx.x);
  for (int i = threadIdx.x; i < (int)(sizeof(SlotParams) / 4); i += 64) dst[i] = src[i];
}
__device__ inline void result_out(const SlotOut* out, SlotOut* host, int tid, int nthreads) {
  const double* src = reinterpret_cast<const double*>(out);
  double* dst = reinterpret_cast<double*>(host);
  for (int i = tid; i < (int)(sizeof(SlotOut) / 8); i += nthreads) dst[i] = src[i];
}
__global__ __launch_bounds__(64) void k_results_out(const SlotOut* __restrict__ out, SlotOut* __restrict__ host) {
  result_out(out + blockIdx.x, host + blockIdx.x, threadIdx.x, 64);
}
hipError_t launch_params_in(const Batch& B) {
  if (B.host_params == nullptr) return hipSuccess;
  hipLaunchKernelGGL(k_params_in, dim3(B.nslots), dim3(64), 0, B.stream, B.host_params,
                     const_cast<SlotParams*>(B.params));
  return hipGetLastError();
}
hipError_t launch_results_out(const Batch& B) {
  if (B.host_out == nullptr) return hipSuccess;
  hipLaunchKernelGGL(k_results_out, dim3(B.nslots), dim3(64), 0, B.stream, B.out, B.host_out);
  return hipGetLastError();
}

// ---------------------------------------------------------------------------
// (1) covariance build: lower 64 x 64 tiles (diagonal tiles in full)
// grid (ntiles(nblk_max), nslots), 256 threads
// ---------------------------------------------------------------------------
template <int DT>
__global__ __launch_bounds__(TPB) void k_build(const Slot* __restrict__ slots, const SlotParams* __restrict__ params,
                                               SlotOut* __restrict__ out) {
  const TileSlot ts = tile_slot();
  const int b = ts.slot;
  const Slot S = slots[b];
  const SlotParams& P = params[b];
  if (!P.active) {
    if (ts.tile == 0 && threadIdx.x == 0) out[b].status = ST_INACTIVE;
    return;
  }
  if (ts.tile == 0 && threadIdx.x == 0) out[b].status = ST_OK;
  const int ntiles = S.nblk * (S.nblk + 1) / 2;
  if (ts.tile >= ntiles) return;
  int ti, tj;
  tri_decode(ts.tile, ti, tj);
  const int i0 = ti * NB, j0 = tj * NB;
  const int n = S.n, d = S.d, tid = threadIdx.x;
  if (P.mode != MODE_KERNEL) {
    // the input matrix's lower triangle (diagonal tiles: zero above), the
    // padded part the identity; the matrix mode adds the retry ladder's
    // cumulative jitter to the diagonal in the reference's order
    // (LinearAlgebra.cpp:88: X.diag() += num_nugget * 10^inc, per retry)
    const int ii = tid & 63, gi = i0 + ii;
    for (int r = 0; r < NB / 4; ++r) {
      const int jj = (tid >> 6) + 4 * r, gj = j0 + jj;
      double v;
      if (gi >= n || gj >= n) {
        v = (gi == gj) ? 1.0 : 0.0;
      } else if (gi < gj) {
        v = 0.0;
      } else {
        v = S.M[(size_t)gj * n + gi];
        // a given factor's columns are taken with a positive diagonal: the
        // 1-norm condition number does not change with column signs
        if (P.mode == MODE_FACTOR && S.M[(size_t)gj * n + gj] < 0.0) v = -v;
        if (gi == gj && P.mode == MODE_MATRIX) {
          double p10 = 1.0;
          for (int q = 0; q < P.inc; ++q) {
            v += P.num_nugget * p10;
            p10 *= 10.0;
          }
        }
      }
      S.A[(size_t)gj * S.npad + gi] = v;
    }
    return;
  }

  __shared__ double sXi[DT * NB];
  __shared__ double sXj[DT * NB];
  for (int q = tid; q < d * NB; q += TPB) {
    const int k = q / NB, r = q % NB;
    sXi[q] = (i0 + r < n) ? S.X[(size_t)k * n + i0 + r] : 0.0;
    sXj[q] = (j0 + r < n) ? S.X[(size_t)k * n + j0 + r] : 0.0;
  }
  double it[DT];
#pragma unroll
  for (int k = 0; k < DT; ++k) it[k] = (k < d) ? 1.0 / P.theta[k] : 1.0;
  const double factor = (S.noise == NOISE_NUGGET) ? P.alpha : 1.0;
  // diagonal: 1 plus the cumulative jitter of the retry ladder, added in the
  // same order as LinearAlgebra.cpp:88 (X.diag() += num_nugget * 10^inc)
  double dval = 1.0;
  {
    double p10 = 1.0;
    for (int q = 0; q < P.inc; ++q) {
      dval += P.num_nugget * p10;
      p10 *= 10.0;
    }
  }
  __syncthreads();

  const int ii = tid & 63;
  const int gi = i0 + ii;
  // specialised per covariance kernel (one kernel's code runs)
  auto fill = [&](auto ktag) __attribute__((always_inline)) {
    constexpr int KT = decltype(ktag)::value;
    double dx[DT];
    // up to 8 dimensions two elements per iteration: all sixteen unrolled are
    // 58 KB of code over the four kernels, each run once per workgroup (n =
    // 200: 12.7 -> 10.3 us; no slower at n = 1024 .. 4096); beyond, unrolled (n
    // = 8192, d = 10: 135 against 164 us)
#pragma unroll(DT <= 8 ? 2 : NB / 4)
    for (int r = 0; r < NB / 4; ++r) {
      const int jj = (tid >> 6) + 4 * r;
      const int gj = j0 + jj;
      double v;
      if (gi >= n || gj >= n) {
        v = (gi == gj) ? 1.0 : 0.0;
      } else if (gi == gj) {
        v = dval;
      } else {
#pragma unroll
        for (int k = 0; k < DT; ++k) dx[k] = (k < d) ? sXj[k * NB + jj] - sXi[k * NB + ii] : 0.0;
        v = kern_rho<DT>(KT, dx, it, DT <= 8 ? d : DT) * factor;  // padded coordinates skipped up to 8 dimensions (beyond, the branches cost more than they save: n = 8192, d = 10 build 0.216 vs 0.143 ms)
      }
      S.A[(size_t)gj * S.npad + gi] = v;
    }
  };
  switch (S.kernel) {
    case K_GAUSS: fill(std::integral_constant<int, K_GAUSS>{}); break;
    case K_EXP: fill(std::integral_constant<int, K_EXP>{}); break;
    case K_MATERN32: fill(std::integral_constant<int, K_MATERN32>{}); break;
    default: fill(std::integral_constant<int, K_MATERN52>{}); break;
  }
}

// ---------------------------------------------------------------------------
// (2c) deferred update: A(r, c) -= sum_{k in [kb, ke)} L(r, k) L(c, k)^T
// over tile columns c in [c0, c1] (c1 < 0: every column from c0 on) and
// rows r >= c.  Two-level blocking: inside a panel of P block columns the
// update reaches only the panel's own columns (K = 64); the rest of the
// matrix is updated once per panel with K = 64 P, so the trailing matrix is
// read and written 1 / P as often.
// grid (tiles of the widest slot, nslots), 256 threads, four waves per SIMD
// (128 registers, no spill: the 64 x n = 1024 batch's Cholesky 1.035 ->
// 1.021 ms against three)
// ---------------------------------------------------------------------------
// tile number `tile` of the update's tile set -> (r, c); false when out of range
__device__ inline bool update_tile_rc(int tile, int nb, int c0, int c1, int& r, int& c) {
  if (c1 < 0) {
    const int T = nb - c0;
    if (tile >= T * (T + 1) / 2) return false;
    int ti, tj;
    tri_decode(tile, ti, tj);
    r = c0 + ti;
    c = c0 + tj;
    return true;
  }
  int t = tile;
  c = c0;
  const int cl = min(c1, nb - 1);
  while (c <= cl && t >= nb - c) {
    t -= nb - c;
    ++c;
  }
  if (c > cl) return false;
  r = c + t;
  return true;
}

__device__ inline void update_tile(const Slot& S, int r, int c, int kb, int ke, double* sbuf) {
  const int i0 = r * NB, j0 = c * NB, ld = S.npad;
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, wr = w >> 1, wc = w & 1;
  d4 acc[2][2];
  double* C = S.A + (size_t)j0 * ld + i0;
  acc_load(acc, C, ld, lane, wr, wc);
  tile_mainloop<false, false, true>(S.A, ld, i0, S.A, ld, j0, kb * NB, ke * NB, sbuf, acc, tid, lane, wr, wc);
  acc_store(acc, C, ld, lane, wr, wc);
}

__global__ __launch_bounds__(TPB, 4) void k_potrf_update(const Slot* __restrict__ slots,
                                                      const SlotParams* __restrict__ params,
                                                      SlotOut* __restrict__ out, int kb, int ke, int c0, int c1) {
  const TileSlot ts = tile_slot();
  const int b = ts.slot;
  const Slot S = slots[b];
  if (!slot_live(params[b], out[b]) || params[b].mode == MODE_FACTOR) return;
  const int nb = S.nblk;
  if (c0 >= nb || ke > nb) return;
  int r, c;
  if (!update_tile_rc(ts.tile, nb, c0, c1, r, c)) return;
  __shared__ double sbuf[4 * KC * LDSS];
  update_tile(S, r, c, kb, ke, sbuf);
}

// The same, a quarter of a tile (32 x 32) per workgroup and 16 x 16 of it per
// wave: bound by one load, K / 4 MFMAs and one store in a row.  grid (4
// tiles, nslots)
__global__ __launch_bounds__(TPB) void k_potrf_update_s(const Slot* __restrict__ slots,
                                                        const SlotParams* __restrict__ params,
                                                        SlotOut* __restrict__ out, int kb, int ke, int c0, int c1) {
  const TileSlot ts = tile_slot();
  const int b = ts.slot;
  const Slot S = slots[b];
  if (!slot_live(params[b], out[b]) || params[b].mode == MODE_FACTOR) return;
  const int nb = S.nblk;
  if (c0 >= nb || ke > nb) return;
  int r, c;
  if (!update_tile_rc(ts.tile >> 2, nb, c0, c1, r, c)) return;
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, ld = S.npad;
  const int i0 = r * NB + 32 * (ts.tile & 1) + 16 * (w & 1), j0 = c * NB + 16 * (ts.tile & 2) + 16 * (w >> 1);
  double* C = S.A + (size_t)(j0 + (lane >> 4)) * ld + i0 + (lane & 15);
  d4 acc;
#pragma unroll
  for (int e = 0; e < 4; ++e) acc[e] = gload(C + (size_t)(4 * e) * ld);
  block16_direct<true>(S.A, ld, i0, S.A, ld, j0, kb * NB, ke * NB, acc, lane);
#pragma unroll
  for (int e = 0; e < 4; ++e) C[(size_t)(4 * e) * ld] = acc[e];
}

// The trailing update (every column from c0 on) on 128 x 64 tiles: column c's
// row blocks c, c+1, ... taken in pairs (the last one alone when their count
// is odd).  Tile t -> (c, first row block).  grid (tiles, nslots)
__device__ inline bool update_tile_w(int tile, int nb, int c0, int& r, int& c) {
  int t = tile;
  for (c = c0; c < nb; ++c) {
    const int pairs = (nb - c + 1) / 2;
    if (t < pairs) {
      r = c + 2 * t;
      return true;
    }
    t -= pairs;
  }
  return false;
}

__global__ __launch_bounds__(TPB, 2) void k_potrf_update_w(const Slot* __restrict__ slots,
                                                        const SlotParams* __restrict__ params,
                                                        SlotOut* __restrict__ out, int kb, int ke, int c0) {
  const TileSlot ts = tile_slot();
  const int b = ts.slot;
  const Slot S = slots[b];
  if (!slot_live(params[b], out[b]) || params[b].mode == MODE_FACTOR) return;
  const int nb = S.nblk;
  if (c0 >= nb || ke > nb) return;
  int r, c;
  if (!update_tile_w(ts.tile, nb, c0, r, c)) return;
  const int i0 = r * NB, j0 = c * NB, ld = S.npad;
  const int rows_valid = (r + 1 < nb) ? WROWS : NB;
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, wr = w >> 1, wc = w & 1;
  __shared__ double sbuf[2 * KC * (LDSW + LDSS)];
  d4 acc[4][2];
  double* C = S.A + (size_t)j0 * ld + i0;
  accw_load(acc, C, ld, lane, wr, wc, rows_valid);
  tile_mainloop_w<true>(S.A, ld, i0, S.A, ld, j0, kb * NB, ke * NB, sbuf, acc, tid, lane, wr, wc, rows_valid);
  accw_store(acc, C, ld, lane, wr, wc, rows_valid);
}

// The same update for one slot by a persistent grid: workgroup g takes tiles
// g, g + G, g + 2G, ... (G = gridDim.x).  Launched with about two
// workgroups per CU, it leaves room on every CU (LDS and registers) for the
// diagonal-block, panel and look-ahead launches of the next panel, which
// run beside it on another stream.  Each tile gets the same arithmetic as in
// k_potrf_update.
__global__ __launch_bounds__(TPB) void k_potrf_update_persistent(const Slot* __restrict__ slots,
                                                                 const SlotParams* __restrict__ params,
                                                                 SlotOut* __restrict__ out, int kb, int ke, int c0,
                                                                 int c1, int tiles) {
  const Slot S = slots[0];
  if (!slot_live(params[0], out[0]) || params[0].mode == MODE_FACTOR) return;
  const int nb = S.nblk;
  if (c0 >= nb || ke > nb) return;
  __shared__ double sbuf[4 * KC * LDSS];
  for (int t = blockIdx.x; t < tiles; t += gridDim.x) {
    int r, c;
    if (!update_tile_rc(t, nb, c0, c1, r, c)) return;  // tiles are in increasing order: the rest are out too
    update_tile(S, r, c, kb, ke, sbuf);
  }
}

// ---------------------------------------------------------------------------
// (3) L^-1 by recursive doubling.  At level s (block size s tiles), for each
// aligned pair (top = 2ps, bot = top + s):
//   step 0:  T = L(bot, top) * Linv(top, top)          -> W upper (transposed)
//   step 1:  Linv(bot, top) = -Linv(bot, bot) * T      -> W lower
// grid (npairs_max * s * s, nslots), 256 threads, four waves per SIMD (124
// registers, no spill: 64 x n = 1024 L^-1 0.664 -> 0.651 ms against three)
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(TPB, 4) void k_trtri(const Slot* __restrict__ slots, const SlotParams* __restrict__ params,
                                               SlotOut* __restrict__ out, int s, int step) {
  const TileSlot ts = tile_slot();
  const int b = ts.slot;
  const Slot S = slots[b];
  if (!slot_live(params[b], out[b])) return;
  const int per_pair = s * s;
  const int pr = ts.tile / per_pair;
  const int rem = ts.tile % per_pair;
  // tiles in order of falling K length (longest first, the short ones fill
  // the tail), and consecutive workgroups, which the dispatcher deals to the
  // 8 XCDs in turn, with equal K: step 0's K falls with tj, step 1's grows
  // with ti
  const int ti = (step == 0) ? rem % s : s - 1 - rem / s;
  const int tj = (step == 0) ? rem / s : rem % s;
  const int top = 2 * pr * s, bot = top + s;
  const int it = bot + ti, jt = top + tj;  // tile row / col of the output
  if (bot >= S.nblk || it >= S.nblk) return;
  const int ld = S.npad;
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, wr = w >> 1, wc = w & 1;
  const int i0 = it * NB, j0 = jt * NB;
  __shared__ double sbuf[4 * KC * LDSS];
  d4 acc[2][2];
  acc_zero(acc);
  if (step == 0) {
    // T(i, j) = sum_{k = jt*NB}^{(top + s)*NB - 1} L(i, k) Linv(k, j)
    tile_mainloop<false, true, false>(S.A, ld, i0, S.W, ld, j0, jt * NB, (top + s) * NB, sbuf, acc, tid, lane, wr,
                                      wc);
    // T(i, j) stored at W[(i0 + row) * ld + j0 + col] (strict upper triangle of W)
    acc_store_t(acc, S.W + (size_t)i0 * ld + j0, ld, lane, wr, wc);
  } else {
    // Linv(i, j) = -sum_{k = bot*NB}^{(it + 1)*NB - 1} Linv(i, k) T(k, j)
    tile_mainloop<false, false, true>(S.W, ld, i0, S.W, ld, j0, bot * NB, (it + 1) * NB, sbuf, acc, tid, lane, wr,
                                      wc);
    acc_store(acc, S.W + (size_t)j0 * ld + i0, ld, lane, wr, wc);
  }
}

// The same, a quarter of a tile (32 x 32) per workgroup and 16 x 16 of it per
// wave.  Step 0's Linv is transposed and goes through LDS (read straight from
// memory a level of n = 1500 took 41 us, so 18).  grid (4 npairs_max * s * s,
// nslots)
__global__ __launch_bounds__(TPB) void k_trtri_s(const Slot* __restrict__ slots, const SlotParams* __restrict__ params,
                                                 SlotOut* __restrict__ out, int s, int step) {
  const TileSlot ts = tile_slot();
  const int b = ts.slot;
  const Slot S = slots[b];
  if (!slot_live(params[b], out[b])) return;
  const int per_pair = s * s, tile = ts.tile >> 2;
  const int pr = tile / per_pair, rem = tile % per_pair;
  const int ti = (step == 0) ? rem % s : s - 1 - rem / s;
  const int tj = (step == 0) ? rem / s : rem % s;
  const int top = 2 * pr * s, bot = top + s;
  const int it = bot + ti, jt = top + tj;
  if (bot >= S.nblk || it >= S.nblk) return;
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, ld = S.npad;
  const int i0 = it * NB + 32 * (ts.tile & 1) + 16 * (w & 1), j0 = jt * NB + 16 * (ts.tile & 2) + 16 * (w >> 1);
  const int i = i0 + (lane & 15), j = j0 + (lane >> 4);
  d4 acc = d4{0.0, 0.0, 0.0, 0.0};
  if (step == 0) {
    __shared__ double sB[2 * B16_BUF];
    block16_bt(S.A, ld, i0, S.W, ld, jt * NB + 16 * (ts.tile & 2), 16 * (w >> 1), jt * NB, (top + s) * NB, sB, acc,
               (int)threadIdx.x);
#pragma unroll
    for (int e = 0; e < 4; ++e) S.W[(size_t)i * ld + j + 4 * e] = acc[e];
  } else {
    block16_direct<true>(S.W, ld, i0, S.W, ld, j0, bot * NB, (it + 1) * NB, acc, lane);
#pragma unroll
    for (int e = 0; e < 4; ++e) S.W[(size_t)(j + 4 * e) * ld + i] = acc[e];
  }
}

// ---------------------------------------------------------------------------
// (4) triangular products with the explicit inverse.
// V columns: [0, p) F*, p y*, p+1 r, p+2 E*, p+3 x, p+4.. p+6 estimator scratch
// ---------------------------------------------------------------------------
// [F* | y*] = Linv [F | y]
__global__ __launch_bounds__(MV_TPB) void k_solve_fy(const Slot* __restrict__ slots,
                                                  const SlotParams* __restrict__ params,
                                                  SlotOut* __restrict__ out) {
  const TileSlot ts = tile_slot();
  const int b = ts.slot;
  const Slot S = slots[b];
  if (!slot_live(params[b], out[b]) || ts.tile >= S.nblk) return;
  const int rb = ts.tile;
  // [F | y] -> V columns 0 .. p in one pass over this row block of Linv
  lower_matvec_block<false>(S, rb, S.F, S.n, S.n, S.p + 1, S.V, S.npad, nullptr, S.y);
  // this row block's part of F*'F* and F*'y* (upper triangle and last column
  // of [F* | y*]'[F* | y*], a-major), for k_gls: its columns were just
  // written by this workgroup
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, p = S.p;
  const double* v = S.V + rb * NB + lane;
  double* part = S.V + (size_t)v_gram(p) * S.npad + (size_t)rb * gram_entries(p);
  int e = 0;
  for (int a = 0; a < p; ++a)
    for (int c = a; c <= p; ++c, ++e)
      if (e % MV_W == w) {
        const double t = wave_sum(v[(size_t)a * S.npad] * v[(size_t)c * S.npad]);
        if (lane == 0) part[e] = t;
      }
}

// GLS: R* = chol_upper(F*'F*), beta = R*^-1 R*^-T F*'y*, r = y - F beta
// (KrigingImpl.cpp:105-121).  Every workgroup adds the row blocks' Gram sums
// and factors the p x p system for itself (one wave, lane = column), then
// takes 256 rows of r: one pass over F instead of one per entry of F*'F* by a
// single workgroup (n = 4096, p = 9: 194 us; n = 8192, p = 1: 40 us).
// grid (ceil(nblk_max / 4), nslots), 256 threads
__global__ __launch_bounds__(TPB) void k_gls(const Slot* __restrict__ slots, const SlotParams* __restrict__ params,
                                             SlotOut* __restrict__ out) {
  const int b = blockIdx.y;
  const Slot S = slots[b];
  if (!slot_live(params[b], out[b]) || (int)blockIdx.x * TPB >= S.npad) return;
  const int tid = threadIdx.x, p = S.p, n = S.n, ld = S.npad;
  __shared__ double G[PMAX * (PMAX + 1)];  // p x (p + 1): [F*'F* | F*'y*], then [R* | R*^-T F*'y*]
  __shared__ double part[TPB];
  __shared__ double beta[PMAX];
  const int ne = gram_entries(p);
  const double* gram = S.V + (size_t)v_gram(p) * ld;
  // entry e of the sums at G(a, c); consecutive threads take consecutive
  // entries, and with fewer entries than threads the row blocks are dealt to
  // np groups of threads whose sums are added in order
  const int np = (ne >= TPB || ne == 0) ? 1 : TPB / ne;
  for (int e0 = 0; e0 < ne; e0 += TPB) {
    const int e = e0 + tid % (np > 1 ? ne : TPB), g = np > 1 ? tid / ne : 0;
    double s = 0.0;
    if (e < ne && g < np)
      for (int q = g; q < S.nblk; q += np) s += gload(gram + (size_t)q * ne + e);
    part[tid] = s;
    __syncthreads();
    if (e < ne && g == 0) {
      for (int q = 1; q < np; ++q) s += part[tid + q * ne];
      int a = 0, r = e;
      while (r > p - a) r -= p - a + 1, ++a;
      G[a + (a + r) * PMAX] = s;
    }
    __syncthreads();
  }
  if (tid < 64) {
    // upper Cholesky in place, row by row: lane c has column c; column p
    // becomes R*^-T F*'y* on the way
    bool ok = true;
    const int c = tid;
    for (int j = 0; j < p; ++j) {
      const double d = G[j + j * PMAX];
      ok = ok && (d > 0.0);
      const double ujj = sqrt(d);
      double u = 0.0;
      if (c >= j && c <= p) u = (c == j) ? ujj : G[j + c * PMAX] / ujj;
      wave_lds_fence();
      if (c >= j && c <= p) G[j + c * PMAX] = u;
      wave_lds_fence();
      if (c > j && c <= p)
        for (int i = j + 1; i < p && i <= c; ++i) G[i + c * PMAX] = fma(-G[j + i * PMAX], u, G[i + c * PMAX]);
      wave_lds_fence();
    }
    // R* beta = z, lane c holds z_c
    double z = (c < p) ? G[c + p * PMAX] : 0.0;
    for (int a = p - 1; a >= 0; --a) {
      const double ba = __shfl(z, a, 64) / G[a + a * PMAX];
      if (c == a) z = ba;
      if (c < a) z = fma(-G[c + a * PMAX], ba, z);
    }
    if (c < p) beta[c] = z;
    if (blockIdx.x == 0) {
      if (c < p) out[b].beta[c] = z;
      double* rs = S.red + red_rstar_off(S.nblk);
      for (int q = 0; q < p; ++q)
        if (c < p) rs[c + q * p] = (c <= q) ? G[c + q * PMAX] : 0.0;
      const double ldr = wave_sum(c < p ? log(G[c + c * PMAX]) : 0.0);
      if (c == 0) {
        out[b].logdet_rstar = ldr;
        if (!ok) out[b].status = ST_CHOL_FAILED;
      }
    }
  }
  __syncthreads();
  // residual r = y - F beta into V column p + 1 (zero in padded rows)
  const int i = blockIdx.x * TPB + tid;
  if (i >= ld) return;
  double v = 0.0;
  if (i < n) {
    double s = 0.0;
    for (int a = 0; a < p; ++a) s = fma(S.F[(size_t)a * n + i], beta[a], s);
    v = S.y[i] - s;
  }
  S.V[(size_t)(p + 1) * ld + i] = v;
}

// E* = Linv r, SSE partials
__global__ __launch_bounds__(MV_TPB) void k_solve_e(const Slot* __restrict__ slots,
                                                 const SlotParams* __restrict__ params,
                                                 SlotOut* __restrict__ out) {
  const TileSlot ts = tile_slot();
  const int b = ts.slot;
  const Slot S = slots[b];
  if (!slot_live(params[b], out[b]) || ts.tile >= S.nblk) return;
  const double* r = S.V + (size_t)(S.p + 1) * S.npad;
  double* e = S.V + (size_t)(S.p + 2) * S.npad;
  lower_matvec_block<true>(S, ts.tile, r, S.npad, S.n, 1, e, S.npad, S.red + red_sse_off(S.nblk));
}

// x = Linv^T E*, and the 1-norms (max column abs sums) of L and Linv
__global__ __launch_bounds__(MV_TPB) void k_solve_x(const Slot* __restrict__ slots,
                                                 const SlotParams* __restrict__ params,
                                                 SlotOut* __restrict__ out) {
  const TileSlot ts = tile_slot();
  const int b = ts.slot;
  const Slot S = slots[b];
  if (!slot_live(params[b], out[b]) || ts.tile >= S.nblk) return;
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, ld = S.npad, n = S.n;
  const double* e = S.V + (size_t)(S.p + 2) * ld;
  double* x = S.V + (size_t)(S.p + 3) * ld;
  double mW = 0.0, mL = 0.0;
  // ||L||_1: L's columns are read only inside the diagonal block; below it
  // the sums of 16 rows each that the Cholesky left stand in for them (a factor
  // given as input had no panel step: then all of L is read)
  const int lend = (params[b].mode == MODE_FACTOR) ? ld : (ts.tile + 1) * NB;
  // wave w takes the block's columns c0 .. c0 + CW - 1 together: one pass
  // down the rows (the reductions run once per column at the end)
  constexpr int CW = NB / MV_W;  // columns per wave
  const int c0 = ts.tile * NB + CW * w;
  double s[CW], aw[CW];
#pragma unroll
  for (int q = 0; q < CW; ++q) {
    s[q] = 0.0;
    aw[q] = 0.0;
  }
  // the diagonal block's rows, then XU groups of 64 whole rows at a time: XU
  // (CW + 1) loads in flight per lane, no test per element (n = 4096: 50 ->
  // 45 us, n = 8192: 128 -> 116)
  {
    const int i = ts.tile * NB + lane;
    const double ev = gload(e + i);
#pragma unroll
    for (int q = 0; q < CW; ++q) {
      const double wv = gload(S.W + (size_t)(c0 + q) * ld + i);
      if (i >= c0 + q) {  // the lower triangle only
        s[q] = fma(wv, ev, s[q]);
        aw[q] += fabs(wv);
      }
    }
  }
  constexpr int XU = 4;
  auto rows = [&](int i0, auto utag) __attribute__((always_inline)) {
    constexpr int U = decltype(utag)::value;
    double ev[U], wv[U][CW];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      ev[u] = gload(e + i0 + 64 * u + lane);
#pragma unroll
      for (int q = 0; q < CW; ++q) wv[u][q] = gload(S.W + (size_t)(c0 + q) * ld + i0 + 64 * u + lane);
    }
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int q = 0; q < CW; ++q) {
        s[q] = fma(wv[u][q], ev[u], s[q]);
        aw[q] += fabs(wv[u][q]);
      }
  };
  int i0 = (ts.tile + 1) * NB;
  for (; i0 + 64 * XU <= ld; i0 += 64 * XU) rows(i0, std::integral_constant<int, XU>{});
  for (; i0 < ld; i0 += 64) rows(i0, std::integral_constant<int, 1>{});
  // |L|'s column sums: the four columns' loads together
  double al4[CW];
#pragma unroll
  for (int q = 0; q < CW; ++q) al4[q] = 0.0;
  for (int i = ts.tile * NB + lane; i < lend; i += 64)
#pragma unroll
    for (int q = 0; q < CW; ++q) {
      const double v = fabs(gload(S.A + (size_t)(c0 + q) * ld + i));
      if (i >= c0 + q) al4[q] += v;
    }
  if (lend < ld)
    // four partial sums per row block (lcol_part in lk_potrf.hip)
    for (int r = 4 * (ts.tile + 1) + lane; r < 4 * S.nblk; r += 64) {
      const double* Lp = S.A + (size_t)((r >> 2) * NB + (r & 3)) * ld + c0;
#pragma unroll
      for (int q = 0; q < CW; ++q) al4[q] += gload(Lp + q);
    }
#pragma unroll
  for (int q = 0; q < CW; ++q) {
    const int c = c0 + q;
    double al = al4[q];
    const double sx = wave_sum(s[q]);
    const double awx = wave_sum(aw[q]);
    al = wave_sum(al);
    if (lane == 0) x[c] = sx;
    if (c < n) {
      mW = fmax(mW, awx);
      mL = fmax(mL, al);
    }
  }
  __shared__ double sm[2][MV_W];
  if (lane == 0) {
    sm[0][w] = mW;
    sm[1][w] = mL;
  }
  __syncthreads();
  // the block's share of the log-determinant, sum log L_cc
  if (w == MV_W - 1) {
    const int c = ts.tile * NB + lane;
    const double t = wave_sum(log(gload(S.A + (size_t)c * ld + c)));
    if (lane == 0) S.red[RED_LOGDET + ts.tile] = t;
  }
  if (tid == 0) {
    double a = sm[0][0], l = sm[1][0];
    for (int q = 1; q < MV_W; ++q) {
      a = fmax(a, sm[0][q]);
      l = fmax(l, sm[1][q]);
    }
    S.red[red_colW_off(S.nblk) + ts.tile] = a;
    S.red[red_colL_off(S.nblk) + ts.tile] = l;
  }
}

// ---------------------------------------------------------------------------
// (6) fused R^-1 tile + adjoint contraction.  Tile (i >= j) of
// R^-1 = Linv^T Linv is accumulated on MFMA; then every strictly-lower
// element (gi > gj) contributes, with dR_ij/dtheta_k = R_ij g_k(x_j - x_i)
// recomputed from X (KrigingImpl.cpp:871-884, Kriging.cpp:303-316):
//   s1_k += (x_i x_j - sigma2 Rinv_ij) R_ij g_k   (the finaliser's
//           s1 / sigma2 - s2 in one sum; the s2 partials are zero)
//   a1   += x_i x_j rho_ij        a2   += Rinv_ij rho_ij   (nugget models
//           whose parameter vector has alpha only)
// and diagonal elements add x_i^2 and Rinv_ii.  Partials per tile go to
// red[grad_off + tile * GRAD_STRIDE]: [s1 (DT) | s2 (DT) | a1 a2 dg1 dg2].
// LMP: the log-marginal-posterior gradient (KrigingImpl.cpp:887-921) has the
// same contraction with B = R^-1 - R^-1 F (F'R^-1 F)^-1 F'R^-1 = R^-1 - G'G in
// place of R^-1 (G = R*^-T F*' L^-1, columns of V from the leave-one-out
// pass k_loo_g), subtracted from each tile before the contraction.
// grid (nblk_max (nblk_max + 1) / 2, nslots), 256 threads.  Waves per SIMD:
// 4 up to 8 dimensions (128 registers: 0.717 -> 0.680 ms per 64 x n = 1024
// launch against 3 waves; the diagonal elements' sums are taken before the
// element loop; the 8-dimension instance spills a few values), 2
// for 9..16 dimensions (1 before: 9.5 -> 8 ms at n = 8192, d = 10).  Beyond
// 8 dimensions the epilogue runs its four 16 x 16 blocks as a loop (the
// sixteen elements are not unrolled there): with the block picked by
// selects instead of an index into the accumulators, which had moved them
// to scratch memory, n = 8192, d = 10 went from 7.61 to 3.69 ms per launch
// (24 -> 50 TFLOP/s) and 64 x n = 1024, d = 10 from 1.55 to 1.06 ms.  9..12
// dimensions use their own instance, which skips the padded coordinates
// (166 registers, three waves: d = 10 at 3.53 / 0.96 ms); up to 6
// dimensions the 6-dimension instance (64 x n = 1024, d = 6: 0.667 -> 0.630
// ms against the 8-dimension one, which computes two padded coordinates)
// ---------------------------------------------------------------------------
template <int DT, bool LMP>
__global__ __launch_bounds__(TPB, (DT == 16 || DT == 12 ? 2 : (DT <= 8 ? 4 : 1))) void k_lauum_adjoint(const Slot* __restrict__ slots,
                                                       const SlotParams* __restrict__ params,
                                                       SlotOut* __restrict__ out) {
  const TileSlot ts = tile_slot();
  const int b = ts.slot;
  const Slot S = slots[b];
  const SlotParams& P = params[b];
  if (!slot_live(P, out[b]) || !P.want_grad) return;
  const int ntiles = S.nblk * (S.nblk + 1) / 2;
  if (ts.tile >= ntiles) return;
  int it, jt;
  tri_decode(ts.tile, it, jt);
  const int ld = S.npad, n = S.n, d = S.d;
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, wr = w >> 1, wc = w & 1;
  const int i0 = it * NB, j0 = jt * NB;
  __shared__ double sbuf[4 * KC * LDSS];
  d4 acc[2][2];
  acc_zero(acc);
  // Linv(k, i0 + ii) Linv(k, j0 + jj) over k >= it * NB
  // (the epilogue reads only elements on or below the diagonal)
  tile_mainloop<true, true, false, true>(S.W, ld, i0, S.W, ld, j0, it * NB, S.nblk * NB, sbuf, acc, tid, lane, wr,
                                         wc, !upper_quadrant(it == jt, wr, wc));

  // epilogue: X rows of both blocks and the x vector in LDS (reuse sbuf)
  // the X rows need 2 DT NB doubles: in the staging buffer when it is large
  // enough (it is idle now), else in an array of their own
  constexpr bool kReuse = 4 * KC * LDSS >= 2 * DT * NB;
  __shared__ double sXown[kReuse ? 1 : 2 * DT * NB];
  double* sXi = kReuse ? sbuf : sXown;  // d x NB
  double* sXj = sXi + DT * NB;
  __shared__ double sxi[NB], sxj[NB];
  const double* xv = S.V + (size_t)(S.p + 3) * ld;
  // all DT coordinate rows, zero from d on: the padded coordinate
  // differences are then zero without a select per element
  for (int q = tid; q < DT * NB; q += TPB) {
    const int k = q / NB, r = q % NB;
    sXi[q] = (k < d && i0 + r < n) ? S.X[(size_t)k * n + i0 + r] : 0.0;
    sXj[q] = (k < d && j0 + r < n) ? S.X[(size_t)k * n + j0 + r] : 0.0;
  }
  if (tid < NB) {
    sxi[tid] = xv[i0 + tid];
    sxj[tid] = xv[j0 + tid];
  }
  __shared__ double sG[LMP ? 2 * PMAX * NB : 1];
  if (LMP) {
    const double* Gt = S.V + (size_t)v_loo_g(S.p) * ld;
    for (int q = tid; q < S.p * NB; q += TPB) {
      const int a = q / NB, r = q % NB;
      sG[q] = Gt[(size_t)a * ld + i0 + r];
      sG[PMAX * NB + q] = Gt[(size_t)a * ld + j0 + r];
    }
  }
  // 1 / theta_k: in registers up to 8 dimensions; beyond, read from LDS
  // (broadcast) so that the epilogue's registers leave room for more waves
  constexpr bool kItLds = DT > 8;
  __shared__ double sIt[kItLds ? DT : 1];
  double itr[kItLds ? 1 : DT];
  if (kItLds) {
    if (tid < DT) sIt[tid] = 1.0 / ((tid < d) ? P.theta[tid] : 1.0);
  } else {
#pragma unroll
    for (int k = 0; k < (kItLds ? 1 : DT); ++k) itr[k] = 1.0 / ((k < d) ? P.theta[k] : 1.0);
  }
  __syncthreads();
  const double* it_ = kItLds ? sIt : itr;
  const double factor = (S.noise == NOISE_NUGGET) ? P.alpha : 1.0;
  const int kern = S.kernel;
  // one sum per theta_k: sum (x_i x_j - sigma2 Rinv_ij) dR_ij/dtheta_k, the
  // finaliser's s1 / sigma2 - s2 with sigma2 (k_finalize_ll, earlier in the
  // pipeline) folded in per element; the s2 partials are written as zero
  const double s2g = out[b].sigma2;
  double sg[DT];
#pragma unroll
  for (int k = 0; k < DT; ++k) sg[k] = 0.0;
  double a1 = 0.0, a2 = 0.0;
  // the diagonal elements' sums first (diagonal tiles only), reduced at once
  // so that their accumulators are not live across the element loop
  __shared__ double sred[4][2 * DT + 4];
  if (it == jt) {
    double dg1 = 0.0, dg2 = 0.0;
#pragma unroll
    for (int bi = 0; bi < 2; ++bi)
#pragma unroll
      for (int bj = 0; bj < 2; ++bj)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int r = acc_row(lane, wr, bi), c = acc_col(lane, wc, bj, e);
          const int gi = i0 + r, gj = j0 + c;
          if (gi >= n || gi != gj) continue;
          double rinv = acc[bi][bj][e];
          if (LMP)
            for (int a = 0; a < S.p; ++a) rinv = fma(-sG[a * NB + r], sG[PMAX * NB + a * NB + c], rinv);
          dg1 += sxi[r] * sxj[c];
          dg2 += rinv;
        }
    const double v2 = wave_sum(dg1), v3 = wave_sum(dg2);
    if (lane == 0) {
      sred[w][2 * DT + 2] = v2;
      sred[w][2 * DT + 3] = v3;
    }
  } else if (lane == 0) {
    sred[w][2 * DT + 2] = 0.0;
    sred[w][2 * DT + 3] = 0.0;
  }

  // the alpha direction's sums only for a nugget model whose gamma has alpha
  const bool need_alpha = S.noise == NOISE_NUGGET && P.gamma_has_alpha;
  // unit inverse length-scales for kern_rho on scaled differences (folded)
  [[maybe_unused]] double kOnes[DT];
#pragma unroll
  for (int k = 0; k < DT; ++k) kOnes[k] = 1.0;
  // one element (r, c) of the tile, R^-1 value rinv
  auto element = [&](auto ktag, int r, int c, double rinv) __attribute__((always_inline)) {
    constexpr int KT = decltype(ktag)::value;
    const int gi = i0 + r, gj = j0 + c;
    if (gi >= n || gj > gi) return;
    if (LMP)
      for (int a = 0; a < S.p; ++a) rinv = fma(-sG[a * NB + r], sG[PMAX * NB + a * NB + c], rinv);
    const double xx = sxi[r] * sxj[c];
    if (gi == gj) return;
    // in the 12-dimension instance the coordinates from d on are skipped
    // (uniform branches): fewer registers, three waves per SIMD
    constexpr bool kSkip = DT == 12;
    double dx[DT];
#pragma unroll
    for (int k = 0; k < DT; ++k) dx[k] = sXj[k * NB + c] - sXi[k * NB + r];
    // rho first, then each g_k recomputed from dx_k while accumulating:
    // no g[] held across the exp (fewer live registers, more waves)
    const double rho = kern_rho<DT>(KT, dx, it_, kSkip ? d : DT);
    const double Rij = rho * factor;
    const double wf = fma(-s2g, rinv, xx) * Rij;  // one product per element, not per k
#pragma unroll
    for (int k = 0; k < DT; ++k) {
      if (kSkip && k >= d) break;
      sg[k] = fma(wf, kern_g(KT, dx[k], it_[k]), sg[k]);
    }
    a1 = fma(xx, rho, a1);
    a2 = fma(rinv, rho, a2);
  };
  if constexpr (DT <= 8) {
    // the element loop specialised per covariance kernel: the executed code
    // is one kernel's, contiguous, instead of all four's interleaved per
    // element (0.611 -> 0.563 ms per 64 x n = 1024, d = 6 launch)
    auto elements = [&](auto ktag) __attribute__((always_inline)) {
      constexpr int KT = decltype(ktag)::value;
#pragma unroll
      for (int bi = 0; bi < 2; ++bi)
#pragma unroll
        for (int bj = 0; bj < 2; ++bj)
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const int r = acc_row(lane, wr, bi), c = acc_col(lane, wc, bj, e);
            const int gi = i0 + r, gj = j0 + c;
            double rinv = acc[bi][bj][e];
            if (gi >= n || gj > gi) continue;
            if (LMP)
              for (int a = 0; a < S.p; ++a) rinv = fma(-sG[a * NB + r], sG[PMAX * NB + a * NB + c], rinv);
            const double xx = sxi[r] * sxj[c];
            if (gi == gj) continue;
            // scaled coordinate differences dx_k / theta_k (the products
            // kern_rho forms): rho from them, and g_k = d ln rho / d theta_k
            // as g(dx_k / theta_k; 1) / theta_k, the 1 / theta_k applied once
            // per tile (one product per coordinate fewer)
            double dx[DT];
#pragma unroll
            for (int k = 0; k < DT; ++k) dx[k] = (sXj[k * NB + c] - sXi[k * NB + r]) * it_[k];
            // rho first, then each g_k recomputed from dx_k while accumulating:
            // no g[] held across the exp (fewer live registers, more waves);
            // the padded coordinates are computed (zeros): skipping them by
            // branches here makes the unrolled elements spill
            const double rho = kern_rho<DT>(KT, dx, kOnes);
            const double Rij = rho * factor;
            const double wf = fma(-s2g, rinv, xx) * Rij;  // one product per element, not per k
#pragma unroll
            for (int k = 0; k < DT; ++k) sg[k] = fma(wf, kern_g(KT, dx[k], 1.0), sg[k]);
            if (need_alpha) {
              a1 = fma(xx, rho, a1);
              a2 = fma(rinv, rho, a2);
            }
          }
    };
    switch (kern) {
      case K_GAUSS: elements(std::integral_constant<int, K_GAUSS>{}); break;
      case K_EXP: elements(std::integral_constant<int, K_EXP>{}); break;
      case K_MATERN32: elements(std::integral_constant<int, K_MATERN32>{}); break;
      default: elements(std::integral_constant<int, K_MATERN52>{}); break;
    }
  } else {
    // beyond 8 dimensions the sixteen elements do not unroll: the four
    // 16 x 16 blocks in a loop, each picked from the accumulators by
    // selects (a loop index into acc would move it to scratch memory)
    // (specialised per covariance kernel, as above)
    auto blocks = [&](auto ktag) __attribute__((always_inline)) {
#pragma unroll 1
      for (int q = 0; q < 4; ++q) {
        const d4 blk = (q == 0) ? acc[0][0] : ((q == 1) ? acc[0][1] : ((q == 2) ? acc[1][0] : acc[1][1]));
#pragma unroll
        for (int e = 0; e < 4; ++e) element(ktag, acc_row(lane, wr, q >> 1), acc_col(lane, wc, q & 1, e), blk[e]);
      }
    };
    switch (kern) {
      case K_GAUSS: blocks(std::integral_constant<int, K_GAUSS>{}); break;
      case K_EXP: blocks(std::integral_constant<int, K_EXP>{}); break;
      case K_MATERN32: blocks(std::integral_constant<int, K_MATERN32>{}); break;
      default: blocks(std::integral_constant<int, K_MATERN52>{}); break;
    }
  }

  // up to 8 dimensions g_k carried 1 / theta_k as a common factor
  if constexpr (DT <= 8) {
#pragma unroll
    for (int k = 0; k < DT; ++k) sg[k] *= it_[k];
  }
  // workgroup reduction of the 2 * DT + 4 partials
  double* dst = S.red + red_grad_off(S.nblk) + (size_t)ts.tile * GRAD_STRIDE;
#pragma unroll
  for (int k = 0; k < DT; ++k) {
    const double v1 = wave_sum(sg[k]);
    if (lane == 0) {
      sred[w][k] = v1;
      sred[w][DT + k] = 0.0;
    }
  }
  {
    const double v0 = wave_sum(a1), v1 = wave_sum(a2);
    if (lane == 0) {
      sred[w][2 * DT + 0] = v0;
      sred[w][2 * DT + 1] = v1;
    }
  }
  __syncthreads();
  if (tid < 2 * DT + 4) {
    const double v = sred[0][tid] + sred[1][tid] + sred[2][tid] + sred[3][tid];
    int q;
    if (tid < DT) q = tid;                       // s1 (sigma2 folded in, see above)
    else if (tid < 2 * DT) q = DMAX + tid - DT;  // s2 (zero)
    else q = 2 * DMAX + (tid - 2 * DT);          // a1 a2 dg1 dg2
    dst[q] = v;
  }
}

// ---------------------------------------------------------------------------
// (7) gradient (Kriging.cpp:303-326): sums of the tile partials in tile order
// ---------------------------------------------------------------------------
constexpr int FG_TPB = 1024;  // 16 waves
// a slot of at least FG_SPLIT_MIN tiles (n >= 4096) is summed in two levels:
// FG_GROUPS workgroups each add a contiguous run of its tiles in tile order
// and leave the sum in the run's first tile row, then k_finalize_grad adds
// those FG_GROUPS rows in order (one workgroup alone reads the 4.5 MB of an
// n = 8192 slot's partials at a fraction of the chip's bandwidth)
constexpr int FG_SPLIT_MIN = 2048;
constexpr int FG_GROUPS = 128;
constexpr int FG1_TPB = 256;
__device__ inline int fg_group_start(int ntiles, int g) { return (int)(((long long)ntiles * g) / FG_GROUPS); }

__global__ __launch_bounds__(FG1_TPB) void k_grad_groups(const Slot* __restrict__ slots,
                                                         const SlotParams* __restrict__ params,
                                                         SlotOut* __restrict__ out) {
  const int g = blockIdx.x, b = blockIdx.y;
  const Slot S = slots[b];
  const SlotParams& P = params[b];
  if (!slot_live(P, out[b]) || !P.want_grad) return;
  const int ntiles = S.nblk * (S.nblk + 1) / 2;
  if (ntiles < FG_SPLIT_MIN) return;
  constexpr int NW = FG1_TPB / 64;
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  double* src = S.red + red_grad_off(S.nblk);
  const int g0 = fg_group_start(ntiles, g), g1 = fg_group_start(ntiles, g + 1);
  const int t0 = g0 + (g1 - g0) * w / NW, t1 = g0 + (g1 - g0) * (w + 1) / NW;
  __shared__ double part[NW][GRAD_STRIDE];
  for (int q = lane; q < GRAD_STRIDE; q += 64) {
    double sm[4] = {0.0, 0.0, 0.0, 0.0};
    int t = t0;
    for (; t + 3 < t1; t += 4) {
#pragma unroll
      for (int u = 0; u < 4; ++u) sm[u] += src[(size_t)(t + u) * GRAD_STRIDE + q];
    }
    for (; t < t1; ++t) sm[0] += src[(size_t)t * GRAD_STRIDE + q];
    part[w][q] = (sm[0] + sm[1]) + (sm[2] + sm[3]);
  }
  // every read of this run is done before its first row is overwritten;
  // the runs of the other workgroups are disjoint
  __syncthreads();
  for (int q = threadIdx.x; q < GRAD_STRIDE; q += FG1_TPB) {
    double s = part[0][q];
#pragma unroll
    for (int v = 1; v < NW; ++v) s += part[v][q];
    src[(size_t)g0 * GRAD_STRIDE + q] = s;
  }
}

__device__ inline void finalize_grad(const Slot& S, const SlotParams& P, SlotOut& O) {
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int ntiles = S.nblk * (S.nblk + 1) / 2;
  constexpr int NW = FG_TPB / 64;
  __shared__ double tot[GRAD_STRIDE];
  __shared__ double part[NW][GRAD_STRIDE];
  // wave w sums the tiles of its sixteenth, lane = component (a tile's
  // partials are contiguous: coalesced rows), eight running sums in tile
  // order (eight loads in flight); the sixteenths are added in order:
  // deterministic for a given tile count
  if (ntiles >= FG_SPLIT_MIN) {
    // the FG_GROUPS run sums of k_grad_groups, in run order
    const double* src = S.red + red_grad_off(S.nblk);
    constexpr int RW = FG_GROUPS / NW;  // runs per wave
    static_assert(FG_GROUPS % NW == 0 && FG_SPLIT_MIN >= 16 * FG_GROUPS, "whole runs per wave, >= 16 tiles a run");
    for (int q = lane; q < GRAD_STRIDE; q += 64) {
      double sm = 0.0;
#pragma unroll
      for (int u = 0; u < RW; ++u) sm += src[(size_t)fg_group_start(ntiles, w * RW + u) * GRAD_STRIDE + q];
      part[w][q] = sm;
    }
  } else {
    const double* src = S.red + red_grad_off(S.nblk);
    const int t0 = (int)(((long long)ntiles * w) / NW);
    const int t1 = (int)(((long long)ntiles * (w + 1)) / NW);
    for (int q = lane; q < GRAD_STRIDE; q += 64) {
      double sm[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) sm[u] = 0.0;
      int t = t0;
      for (; t + 7 < t1; t += 8) {
#pragma unroll
        for (int u = 0; u < 8; ++u) sm[u] += src[(size_t)(t + u) * GRAD_STRIDE + q];
      }
      for (; t < t1; ++t) sm[0] += src[(size_t)t * GRAD_STRIDE + q];
      part[w][q] = ((sm[0] + sm[1]) + (sm[2] + sm[3])) + ((sm[4] + sm[5]) + (sm[6] + sm[7]));
    }
  }
  __syncthreads();
  for (int q = threadIdx.x; q < GRAD_STRIDE; q += FG_TPB) {
    double s = part[0][q];
    for (int v = 1; v < NW; ++v) s += part[v][q];
    tot[q] = s;
  }
  __syncthreads();
  const int q = threadIdx.x;
  if (q != 0) return;
  const int d = S.d;
  const double s2g = O.sigma2;
  for (int k = 0; k < d; ++k) {
    // term1 = 2 s1, term2 = -2 s2, grad = (term1 / sigma2 + term2) / 2
    O.grad[k] = tot[k] / s2g - tot[DMAX + k];
  }
  if (P.gamma_has_alpha && S.noise == NOISE_NUGGET) {
    const double a1 = tot[2 * DMAX], a2 = tot[2 * DMAX + 1], dg1 = tot[2 * DMAX + 2], dg2 = tot[2 * DMAX + 3];
    const double a = P.alpha;
    double ga;
    if (P.objective == OBJ_LMP) {
      // -tr(Wb)/2 + y'Wb'Q_output/(2 sigma2), Wb = D B, D = R / alpha with
      // zero diagonal (Kriging.cpp:612-618); the prior term is the host's
      ga = a1 / s2g - a2;
    } else if (P.est_sigma2 && P.est_nugget) {
      // -0.5 * (-(x' D x) / var + <Rinv, D>), D = R / alpha with zero diagonal
      ga = -0.5 * (-(2.0 * a1) / s2g + 2.0 * a2);
    } else if (P.est_sigma2 && !P.est_nugget) {
      const double tv = s2g;
      const double q1 = 2.0 * a1 + dg1;
      const double tr = (2.0 * a2 + dg2) / tv;
      ga = -0.5 * (-q1 / (tv * tv) + tr) * P.nugget / (1.0 - a) / (1.0 - a);
    } else {
      ga = 0.0;
    }
    O.grad[d] = ga;
  }
}

// with `host`, also the last launch of the pipeline: every slot's results
// (failed and inactive ones' status too) to the pinned table
__global__ __launch_bounds__(FG_TPB) void k_finalize_grad(const Slot* __restrict__ slots,
                                                          const SlotParams* __restrict__ params,
                                                          SlotOut* __restrict__ out, SlotOut* __restrict__ host) {
  const int b = blockIdx.x;
  if (slot_live(params[b], out[b]) && params[b].want_grad) {
    const Slot S = slots[b];
    finalize_grad(S, params[b], out[b]);
  }
  if (host == nullptr) return;
  __syncthreads();
  result_out(out + b, host + b, threadIdx.x, FG_TPB);
}

// ---------------------------------------------------------------------------
// (8) LL value, and the 1-norm estimate of Linv (Higham, ACM TOMS 14 (1988) 381-396, Alg. 4.1
// with the alternating-sign extra estimate), run only for slots whose exact
// rcond fell below the threshold.  The estimate never exceeds the exact norm,
// so an exact rcond above the threshold implies the estimate-based one is
// too.  One workgroup per slot; uses V columns p+4 .. p+6 as scratch.
// ---------------------------------------------------------------------------
__device__ void est_lower_mv(const Slot& S, const double* __restrict__ in, double* __restrict__ o) {
  // o = Linv * in  (row i: sum_{k <= i} W[k*ld + i] in[k]) ; thread per row
  const int ld = S.npad, n = S.n;
  for (int i = threadIdx.x; i < n; i += TPB) {
    double s = 0.0;
    for (int k = 0; k <= i; ++k) s = fma(S.W[(size_t)k * ld + i], in[k], s);
    o[i] = s;
  }
}
__device__ void est_upper_mv(const Slot& S, const double* __restrict__ in, double* __restrict__ o) {
  // o = Linv^T * in  (column c: sum_{i >= c} W[c*ld + i] in[i]) ; wave per column
  const int ld = S.npad, n = S.n, lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  for (int c = w; c < n; c += TPB / 64) {
    double s = 0.0;
    for (int i = c + lane; i < n; i += 64) s = fma(S.W[(size_t)c * ld + i], in[i], s);
    s = wave_sum(s);
    if (lane == 0) o[c] = s;
  }
}

// ---------------------------------------------------------------------------
// (5) LL value and condition check (Kriging.cpp:247-289,
// LinearAlgebra.cpp:68-115), by one thread, from the row blocks' sums and
// maxima.
// ---------------------------------------------------------------------------
__device__ inline void finalize_ll(const Slot& S, const SlotParams& P, SlotOut& O, double logdet, double sse,
                                   double nL, double nW) {
  const double n = (double)S.n;
  const double two_pi = 2.0 * 3.14159265358979323846;
  O.logdet = logdet;
  O.sse = sse;
  O.norm1_L = nL;
  O.norm1_Linv = nW;
  const double rc = (1.0 / nL) / nW;
  O.rcond2 = rc * rc;
  if (P.rcond_check && !(O.rcond2 >= P.min_rcond) && O.status == ST_OK)
    O.status = ST_RCOND_SUSPECT;
  // a given factor: rcond from the 1-norm estimator, as arma::rcond
  if (P.mode == MODE_FACTOR && O.status == ST_OK) O.status = ST_RCOND_SUSPECT;
  double ll, s2g;
  if (P.objective == OBJ_LMP) {
    // log marginal likelihood of Kriging::_logMargPost (Kriging.cpp:560-583),
    // S_2 = y'R^-1 y - y'P y = SSE; the prior term is added by the host
    const double nmp = n - S.p;
    if (S.noise == NOISE_NUGGET) {
      if (P.est_sigma2 && P.est_nugget) s2g = sse / nmp;
      else if (P.est_sigma2 || P.est_nugget) s2g = P.sigma2 / P.alpha;
      else s2g = P.sigma2 + P.nugget;
    } else {
      s2g = P.est_sigma2 ? sse / nmp : P.sigma2;
    }
    O.ll = -logdet - O.logdet_rstar - 0.5 * nmp * log(s2g * nmp);
    O.sigma2 = s2g;
    return;
  }
  if (S.noise == NOISE_NUGGET) {
    const double a = P.alpha;
    double s2 = P.sigma2, nug = P.nugget;
    if (P.est_sigma2) {
      if (P.est_nugget) {
        const double var = sse / n;
        s2 = a * var;
        nug = (1.0 - a) * var;
      } else {
        s2 = P.nugget * a / (1.0 - a);
      }
    } else if (P.est_nugget) {
      nug = P.sigma2 * (1.0 - a) / a;
    }
    const double tv = s2 + nug;
    ll = -0.5 * (n * log(two_pi * tv) + 2.0 * logdet + sse / tv);
    s2g = tv;
  } else if (P.est_sigma2) {
    s2g = sse / n;
    ll = -0.5 * (n * log(two_pi * s2g) + 2.0 * logdet + n);
  } else {
    s2g = P.sigma2;
    ll = -0.5 * (n * log(two_pi * s2g) + 2.0 * logdet + sse / s2g);
  }
  O.ll = ll;
  O.sigma2 = s2g;
}

// One workgroup per slot: the sums above, finalize_ll, and the estimate where
// it is needed.
__global__ __launch_bounds__(TPB) void k_finalize_ll(const Slot* __restrict__ slots,
                                                        const SlotParams* __restrict__ params,
                                                        SlotOut* __restrict__ out) {
  const int b = blockIdx.x;
  const Slot S = slots[b];
  const SlotParams& P = params[b];
  SlotOut& O = out[b];
  if (!slot_live(P, O)) return;
  const int n = S.n, ld = S.npad, tid = threadIdx.x;
  __shared__ double sred[4][TPB / 64];
  __shared__ int suspect;
  {
    const int nb = S.nblk, lane = tid & 63, w = tid >> 6;
    double logdet = 0.0, sse = 0.0, nL = 0.0, nW = 0.0;
    for (int q = tid; q < nb; q += TPB) {
      logdet += S.red[RED_LOGDET + q];
      sse += S.red[red_sse_off(nb) + q];
      nL = fmax(nL, S.red[red_colL_off(nb) + q]);
      nW = fmax(nW, S.red[red_colW_off(nb) + q]);
    }
    logdet = wave_sum(logdet);
    sse = wave_sum(sse);
    nL = wave_max(nL);
    nW = wave_max(nW);
    if (lane == 0) {
      sred[0][w] = logdet;
      sred[1][w] = sse;
      sred[2][w] = nL;
      sred[3][w] = nW;
    }
    __syncthreads();
    if (tid == 0) {
      for (int q = 1; q < TPB / 64; ++q) {
        logdet += sred[0][q];
        sse += sred[1][q];
        nL = fmax(nL, sred[2][q]);
        nW = fmax(nW, sred[3][q]);
      }
      finalize_ll(S, P, O, logdet, sse, nL, nW);
      suspect = O.status == ST_RCOND_SUSPECT;
    }
    __syncthreads();
  }
  if (!suspect) return;
  double* x = S.V + (size_t)(S.p + 4) * ld;
  double* xi = S.V + (size_t)(S.p + 5) * ld;
  double* y = S.V + (size_t)(S.p + 6) * ld;
  __shared__ double sh[TPB];
  __shared__ int shi[TPB];
  __shared__ double sest, sestold;
  __shared__ int sj, sflag;

  auto block_sum_abs = [&](const double* v) -> double {
    double s = 0.0;
    for (int i = tid; i < n; i += TPB) s += fabs(v[i]);
    sh[tid] = s;
    __syncthreads();
    for (int h = TPB / 2; h > 0; h >>= 1) {
      if (tid < h) sh[tid] += sh[tid + h];
      __syncthreads();
    }
    const double r = sh[0];
    __syncthreads();
    return r;
  };
  auto block_argmax_abs = [&](const double* v) -> int {
    double best = -1.0;
    int bi = 0;
    for (int i = tid; i < n; i += TPB)
      if (fabs(v[i]) > best) {
        best = fabs(v[i]);
        bi = i;
      }
    sh[tid] = best;
    shi[tid] = bi;
    __syncthreads();
    for (int h = TPB / 2; h > 0; h >>= 1) {
      if (tid < h) {
        const double o = sh[tid + h];
        const int oi = shi[tid + h];
        if (o > sh[tid] || (o == sh[tid] && oi < shi[tid])) {
          sh[tid] = o;
          shi[tid] = oi;
        }
      }
      __syncthreads();
    }
    const int r = shi[0];
    __syncthreads();
    return r;
  };

  double est;
  for (int i = tid; i < n; i += TPB) x[i] = 1.0 / n;
  __syncthreads();
  est_lower_mv(S, x, y);
  __syncthreads();
  if (n == 1) {
    est = fabs(y[0]);
  } else {
    est = block_sum_abs(y);
    for (int i = tid; i < n; i += TPB) xi[i] = (y[i] >= 0.0) ? 1.0 : -1.0;
    __syncthreads();
    est_upper_mv(S, xi, x);
    __syncthreads();
    int j = block_argmax_abs(x);
    int iter = 2;
    for (;;) {
      for (int i = tid; i < n; i += TPB) x[i] = (i == j) ? 1.0 : 0.0;
      __syncthreads();
      est_lower_mv(S, x, y);
      __syncthreads();
      const double estold = est;
      est = block_sum_abs(y);
      if (tid == 0) sflag = 0;
      __syncthreads();
      for (int i = tid; i < n; i += TPB)
        if (((y[i] >= 0.0) ? 1.0 : -1.0) != xi[i]) sflag = 1;
      __syncthreads();
      const int changed = sflag;
      __syncthreads();
      if (!changed || est <= estold) break;
      for (int i = tid; i < n; i += TPB) xi[i] = (y[i] >= 0.0) ? 1.0 : -1.0;
      __syncthreads();
      est_upper_mv(S, xi, x);
      __syncthreads();
      const int jlast = j;
      j = block_argmax_abs(x);
      if (x[jlast] != fabs(x[j]) && iter < 5) {
        ++iter;
        continue;
      }
      break;
    }
    for (int i = tid; i < n; i += TPB) x[i] = ((i & 1) ? -1.0 : 1.0) * (1.0 + (double)i / (double)(n - 1));
    __syncthreads();
    est_lower_mv(S, x, y);
    __syncthreads();
    double temp = block_sum_abs(y);
    temp = 2.0 * (temp / (double)(3 * n));
    if (temp > est) est = temp;
  }
  (void)sest;
  (void)sestold;
  (void)sj;
  if (tid == 0) {
    const double rc = (1.0 / O.norm1_L) / est;
    O.rcond2 = rc * rc;
    O.status = (P.mode != MODE_FACTOR && O.rcond2 < P.min_rcond) ? ST_RCOND_LOW : ST_OK;
  }
}

// ---------------------------------------------------------------------------
// launchers
// ---------------------------------------------------------------------------
static inline int tri(int t) { return t * (t + 1) / 2; }

// Covariance between two point sets, LinearAlgebra::covMat_rect
// (LinearAlgebra.cpp:600-660) as used by KrigingImpl::covMat:
// out(i, j) = scale k(x1_i - x2_j; theta), n1 x n2 column-major.
// grid (ceil(n2 / 64), ceil(n1 / 64)), 256 threads
template <int DT>
__global__ __launch_bounds__(TPB) void k_cov_mat(CovMatArgs a) {
  const int j0 = blockIdx.x * NB, i0 = blockIdx.y * NB, tid = threadIdx.x;
  const int n1 = a.n1, n2 = a.n2, d = a.d;
  __shared__ double s1[DT * NB];
  __shared__ double s2[DT * NB];
  for (int q = tid; q < d * NB; q += TPB) {
    const int k = q / NB, r = q % NB;
    s1[q] = (i0 + r < n1) ? a.X1[(size_t)k * n1 + i0 + r] : 0.0;
    s2[q] = (j0 + r < n2) ? a.X2[(size_t)k * n2 + j0 + r] : 0.0;
  }
  double it[DT];
#pragma unroll
  for (int k = 0; k < DT; ++k) it[k] = (k < d) ? 1.0 / a.theta[k] : 1.0;
  __syncthreads();
  const int ii = tid & 63, gi = i0 + ii;
  double dx[DT];
  for (int r = 0; r < NB / 4; ++r) {
    const int jj = (tid >> 6) + 4 * r, gj = j0 + jj;
    if (gi >= n1 || gj >= n2) continue;
#pragma unroll
    for (int k = 0; k < DT; ++k) dx[k] = (k < d) ? s1[k * NB + ii] - s2[k * NB + jj] : 0.0;
    a.out[(size_t)gj * n1 + gi] = (a.unit_diag && gi == gj) ? 1.0 : kern_rho<DT>(a.kernel, dx, it) * a.scale;
  }
}

hipError_t launch_cov_mat(const CovMatArgs& a, hipStream_t stream) {
  if (a.n1 <= 0 || a.n2 <= 0) return hipSuccess;
  const dim3 grid((a.n2 + NB - 1) / NB, (a.n1 + NB - 1) / NB);
  if (a.d <= 4)
    hipLaunchKernelGGL(k_cov_mat<4>, grid, dim3(TPB), 0, stream, a);
  else if (a.d <= 8)
    hipLaunchKernelGGL(k_cov_mat<8>, grid, dim3(TPB), 0, stream, a);
  else if (a.d <= 16)
    hipLaunchKernelGGL(k_cov_mat<16>, grid, dim3(TPB), 0, stream, a);
  else
    hipLaunchKernelGGL(k_cov_mat<32>, grid, dim3(TPB), 0, stream, a);
  return hipGetLastError();
}

// C(it, jt) = sum_{kt <= it} Linv(it, kt) B(kt, jt); grid (cpad / 64, npad / 64)
__global__ __launch_bounds__(TPB) void k_trmm_lower(const double* __restrict__ Linv, const double* __restrict__ B,
                                                    double* __restrict__ C, int ld) {
  const int jt = blockIdx.x, it = blockIdx.y;
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, wr = w >> 1, wc = w & 1;
  const int i0 = it * NB, j0 = jt * NB;
  __shared__ double sbuf[4 * KC * LDSS];
  d4 acc[2][2];
  acc_zero(acc);
  // Linv(i0 + ii, k) B(k, j0 + jj) over k < (it + 1) * NB
  tile_mainloop<false, true, false>(Linv, ld, i0, B, ld, j0, 0, (it + 1) * NB, sbuf, acc, tid, lane, wr, wc);
  acc_store(acc, C + (size_t)j0 * ld + i0, ld, lane, wr, wc);
}

hipError_t launch_trmm_lower(const double* Linv, const double* B, double* C, int npad, int cpad, hipStream_t stream) {
  if (cpad <= 0 || npad <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_trmm_lower, dim3(cpad / NB, npad / NB), dim3(TPB), 0, stream, Linv, B, C, npad);
  return hipGetLastError();
}

// S = Cuu - U' U over the lower tiles of S (grid T (T + 1) / 2, T = mpad /
// 64); an off-diagonal tile also writes its transpose
__global__ __launch_bounds__(TPB) void k_schur(SchurArgs a) {
  int ti, tj;
  tri_decode(blockIdx.x, ti, tj);
  const int i0 = ti * NB, j0 = tj * NB;
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, wr = w >> 1, wc = w & 1;
  __shared__ double sbuf[4 * KC * LDSS];
  d4 acc[2][2];
  acc_zero(acc);
  tile_mainloop<true, true, true>(a.U, a.kdim, i0, a.U, a.kdim, j0, 0, a.kdim, sbuf, acc, tid, lane, wr, wc);
  const int m = a.m;
#pragma unroll
  for (int bi = 0; bi < 2; ++bi)
#pragma unroll
    for (int bj = 0; bj < 2; ++bj)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int gi = i0 + acc_row(lane, wr, bi), gj = j0 + acc_col(lane, wc, bj, e);
        if (gi >= m || gj >= m || (ti == tj && gi < gj)) continue;
        const double v = a.Cuu[(size_t)gj * m + gi] + acc[bi][bj][e];
        a.S[(size_t)gj * m + gi] = v;
        if (gi != gj) a.S[(size_t)gi * m + gj] = v;
      }
}

hipError_t launch_schur(const SchurArgs& a, hipStream_t stream) {
  if (a.m <= 0) return hipSuccess;
  const int T = a.mpad / NB;
  hipLaunchKernelGGL(k_schur, dim3(tri(T)), dim3(TPB), 0, stream, a);
  return hipGetLastError();
}

// grid (ceil(n / 64), ceil(n / 64)), 256 threads; lane = row (coalesced
// stores, the transposed reads of U are strided)
__global__ __launch_bounds__(TPB) void k_block_assemble(BlockAssembleArgs a) {
  const int i = blockIdx.x * NB + (threadIdx.x & 63);
  if (i >= a.n) return;
  for (int r = 0; r < NB / 4; ++r) {
    const int j = blockIdx.y * NB + (threadIdx.x >> 6) + 4 * r;
    if (j >= a.n) break;
    double v = 0.0;
    if (i >= j) {
      if (j < a.no)
        v = (i < a.no) ? a.Loo[(size_t)j * a.ldo + i] : a.U[(size_t)(i - a.no) * a.ldu + j];
      else
        v = a.Luu[(size_t)(j - a.no) * a.ldl + (i - a.no)];
    }
    a.L[(size_t)j * a.n + i] = v;
  }
}

hipError_t launch_block_assemble(const BlockAssembleArgs& a, hipStream_t stream) {
  if (a.n <= 0) return hipSuccess;
  const int T = (a.n + NB - 1) / NB;
  hipLaunchKernelGGL(k_block_assemble, dim3(T, T), dim3(TPB), 0, stream, a);
  return hipGetLastError();
}

hipError_t launch_build(const Batch& B) {
  dim3 grid(tri(B.nblk_max), B.nslots);
  if (B.dmax <= 4)
    hipLaunchKernelGGL(k_build<4>, grid, dim3(TPB), 0, B.stream, B.slots, B.params, B.out);
  else if (B.dmax <= 8)
    hipLaunchKernelGGL(k_build<8>, grid, dim3(TPB), 0, B.stream, B.slots, B.params, B.out);
  else if (B.dmax <= 16)
    hipLaunchKernelGGL(k_build<16>, grid, dim3(TPB), 0, B.stream, B.slots, B.params, B.out);
  else
    hipLaunchKernelGGL(k_build<32>, grid, dim3(TPB), 0, B.stream, B.slots, B.params, B.out);
  return hipGetLastError();
}
// Up to here (64 x 64 tiles in the launch) the quarter-tile kernels: below,
// the launch is one tile's chain, above it is the MFMA and LDS staging reads
// the operands once for four waves.  Updates of one n = 4096 Cholesky: 697 us
// without the line, 621 at 256 tiles, 631 at 512, 681 at 1024; its L^-1
// levels: 581, 584 at 256, 563 at 512.  n = 1000: an update 11.9 -> 6.3 us, a
// level 20.3 -> 8.8; n = 1500: 12.5 -> 8.1 and 26 -> 13.4.
constexpr int kUpdateSmall = 256;
constexpr int kTrtriSmall = 512;
hipError_t launch_potrf_update(const Batch& B, int kb, int ke, int c0, int c1) {
  const int nb = B.nblk_max;
  if (c0 >= nb) return hipSuccess;
  int tiles = 0;
  if (c1 < 0) {
    tiles = tri(nb - c0);
  } else {
    for (int c = c0; c <= c1 && c < nb; ++c) tiles += nb - c;
  }
  if (tiles <= 0) return hipSuccess;
  if (tiles * B.nslots <= kUpdateSmall) {
    hipLaunchKernelGGL(k_potrf_update_s, dim3(4 * tiles, B.nslots), dim3(TPB), 0, B.stream, B.slots, B.params, B.out, kb,
                       ke, c0, c1);
    return hipGetLastError();
  }
  hipLaunchKernelGGL(k_potrf_update, dim3(tiles, B.nslots), dim3(TPB), 0, B.stream, B.slots, B.params, B.out, kb, ke,
                     c0, c1);
  return hipGetLastError();
}
hipError_t launch_potrf_update_trailing(const Batch& B, int kb, int ke, int c0) {
  const int nb = B.nblk_max;
  if (c0 >= nb) return hipSuccess;
  int tiles = 0;
  for (int c = c0; c < nb; ++c) tiles += (nb - c + 1) / 2;
  hipLaunchKernelGGL(k_potrf_update_w, dim3(tiles, B.nslots), dim3(TPB), 0, B.stream, B.slots, B.params, B.out, kb, ke,
                     c0);
  return hipGetLastError();
}
hipError_t launch_potrf_update_persistent(const Batch& B, int kb, int ke, int c0, int c1, int workgroups) {
  if (B.nslots != 1) return hipErrorInvalidValue;
  const int nb = B.nblk_max;
  if (c0 >= nb) return hipSuccess;
  int tiles = 0;
  if (c1 < 0) {
    tiles = tri(nb - c0);
  } else {
    for (int c = c0; c <= c1 && c < nb; ++c) tiles += nb - c;
  }
  if (tiles <= 0) return hipSuccess;
  const int g = workgroups < 1 ? 1 : (workgroups < tiles ? workgroups : tiles);
  hipLaunchKernelGGL(k_potrf_update_persistent, dim3(g), dim3(TPB), 0, B.stream, B.slots, B.params, B.out, kb, ke,
                     c0, c1, tiles);
  return hipGetLastError();
}
int trtri_levels(int nblk) {
  int lv = 0;
  while ((1 << lv) < nblk) ++lv;
  return lv;
}
hipError_t launch_trtri_level(const Batch& B, int s, int step) {
  const int npairs = (B.nblk_max + 2 * s - 1) / (2 * s);
  if (npairs <= 0) return hipSuccess;
  if (npairs * s * s * B.nslots <= kTrtriSmall) {
    hipLaunchKernelGGL(k_trtri_s, dim3(4 * npairs * s * s, B.nslots), dim3(TPB), 0, B.stream, B.slots, B.params, B.out,
                       s, step);
    return hipGetLastError();
  }
  hipLaunchKernelGGL(k_trtri, dim3(npairs * s * s, B.nslots), dim3(TPB), 0, B.stream, B.slots, B.params, B.out, s,
                     step);
  return hipGetLastError();
}
hipError_t launch_solve_fy(const Batch& B) {
  hipLaunchKernelGGL(k_solve_fy, dim3(B.nblk_max, B.nslots), dim3(MV_TPB), 0, B.stream, B.slots, B.params, B.out);
  return hipGetLastError();
}
hipError_t launch_gls(const Batch& B) {
  hipLaunchKernelGGL(k_gls, dim3((B.nblk_max + 3) / 4, B.nslots), dim3(TPB), 0, B.stream, B.slots, B.params, B.out);
  return hipGetLastError();
}
hipError_t launch_solve_e(const Batch& B) {
  hipLaunchKernelGGL(k_solve_e, dim3(B.nblk_max, B.nslots), dim3(MV_TPB), 0, B.stream, B.slots, B.params, B.out);
  return hipGetLastError();
}
hipError_t launch_solve_x(const Batch& B) {
  hipLaunchKernelGGL(k_solve_x, dim3(B.nblk_max, B.nslots), dim3(MV_TPB), 0, B.stream, B.slots, B.params, B.out);
  return hipGetLastError();
}
hipError_t launch_finalize_ll(const Batch& B) {
  hipLaunchKernelGGL(k_finalize_ll, dim3(B.nslots), dim3(TPB), 0, B.stream, B.slots, B.params, B.out);
  return hipGetLastError();
}
template <bool LMP>
static hipError_t launch_lauum_adjoint_t(const Batch& B) {
  dim3 grid(tri(B.nblk_max), B.nslots);
  const int dmax_batch = B.dmax;
  if (dmax_batch <= 4)
    hipLaunchKernelGGL((k_lauum_adjoint<4, LMP>), grid, dim3(TPB), 0, B.stream, B.slots, B.params, B.out);
  else if (dmax_batch <= 6)
    hipLaunchKernelGGL((k_lauum_adjoint<6, LMP>), grid, dim3(TPB), 0, B.stream, B.slots, B.params, B.out);
  else if (dmax_batch <= 8)
    hipLaunchKernelGGL((k_lauum_adjoint<8, LMP>), grid, dim3(TPB), 0, B.stream, B.slots, B.params, B.out);
  else if (dmax_batch <= 12)
    hipLaunchKernelGGL((k_lauum_adjoint<12, LMP>), grid, dim3(TPB), 0, B.stream, B.slots, B.params, B.out);
  else if (dmax_batch <= 16)
    hipLaunchKernelGGL((k_lauum_adjoint<16, LMP>), grid, dim3(TPB), 0, B.stream, B.slots, B.params, B.out);
  else
    hipLaunchKernelGGL((k_lauum_adjoint<32, LMP>), grid, dim3(TPB), 0, B.stream, B.slots, B.params, B.out);
  return hipGetLastError();
}
hipError_t launch_lauum_adjoint(const Batch& B) { return launch_lauum_adjoint_t<false>(B); }
hipError_t launch_lmp_adjoint(const Batch& B) { return launch_lauum_adjoint_t<true>(B); }
hipError_t launch_finalize_grad(const Batch& B) {
  if (tri(B.nblk_max) >= FG_SPLIT_MIN) {
    hipLaunchKernelGGL(k_grad_groups, dim3(FG_GROUPS, B.nslots), dim3(FG1_TPB), 0, B.stream, B.slots, B.params,
                       B.out);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
  }
  hipLaunchKernelGGL(k_finalize_grad, dim3(B.nslots), dim3(FG_TPB), 0, B.stream, B.slots, B.params, B.out, B.host_out);
  return hipGetLastError();
}
}  // namespace lk
