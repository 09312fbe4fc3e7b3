// Blocked Cholesky of a batch of slots, FP64, gfx950 (LinearAlgebra.cpp:71),
// and the inverses of the factor's 256 x 256 diagonal blocks.
//
// Per 128 columns (two 64-column blocks, fewer at the end of a panel):
//   k_potrf_chain   the 128 x 128 diagonal square: both 64 x 64 diagonal
//                   factors, their inverses and the tile between them, one
//                   workgroup per slot
//   k_potrf_rows    those columns of every row below the square
// and then k_potrf_update (lk_kernels.hip) for the columns to the right.
#include <hip/hip_runtime.h>

#include <math.h>

#include "lk_device.hpp"
#include "lk_kernels.h"

namespace lk {

// The value, opaque to the compiler: what is computed from it inside a loop
// is not hoisted out (the LDS and memory addresses of the chain kernel's
// phases, all kept live across each other, spilled 300 registers)
__device__ inline int opaque(int v) {
  asm volatile("" : "+v"(v));
  return v;
}
__device__ inline int opaque_s(int v) {
  asm volatile("" : "+s"(v));
  return v;
}

// a^-1/2: y = v_rsq_f64(a) (relative error below 2^-22), then one third-order
// step: with e = 1 - a y^2, a^-1/2 = y (1 - e)^-1/2 = y (1 + e/2 + 3e^2/8 +
// O(e^3)); two dependent operations fewer than two Newton steps
__device__ inline double pivot_rsqrt(double a) {
  const double y = __builtin_amdgcn_rsq(a);
  const double t = a * y;
  const double e = fma(-t, y, 1.0);
  const double p = fma(e, 0.375, 0.5);
  return fma(y * e, p, y);
}

// ---------------------------------------------------------------------------
// (2a) the diagonal square.  512 threads: 8 waves.
//
// One 64 x 64 block (diag_block) is factored in four panels of 16 columns.
// Wave 0 holds a panel in registers, lane = row: the 16 diagonal rows, 16
// identity rows, which the same column operations turn into L_pp^-T, and the
// rows of the next two 16-row blocks; a column's pivot and multipliers are
// broadcast with v_readlane, so a panel has no LDS round trip and no barrier
// (wave 1 repeats panel 0 for the fourth block's rows).  The other waves apply
// a finished panel on MFMA, the next panel's tiles at once, the rest beside
// wave 0's next panel; there they also store what is final and form the
// inverse: wave 5 + q owns 16-column block q of X = L^-1 in registers, X_iq =
// -X_ii sum_k L_ik X_kq, whose operands are the MFMA results themselves (a
// result's register s is the operand of K-step s).  FP64 MFMA and FP64 VALU
// do not run side by side on a SIMD, so wave 4, on wave 0's, only stores.
// What bounds it: the 128 dependent pivots, each the chain of a reciprocal
// square root and the issue of the panel's own updates (about 185 cycles), then
// the panels' two barriers, and the 64 x 64 products between the blocks at one
// CU's MFMA rate.  One launch takes 24 us (n = 200 .. 1000) in place of the
// 45 us of the two diagonal-block launches, the panel and the update launch it
// replaces (a diagonal block took 14.6 us, four columns per step, exchanged
// through LDS at 18 barriers).  On the way: a panel's multipliers through LDS
// instead of v_readlane, 188 against 156 cycles per column; conditions and
// addresses of all eight roles in one loop, 2 300 cycles of scalar work and
// spills in front of wave 0's panel.
// ---------------------------------------------------------------------------
constexpr int CH_TPB = 512;
constexpr int CS = NB + 2;  // column stride of the LDS blocks (doubles)

struct ChainLds {
  double L[NB * CS];  // the diagonal block, then its factor (above the diagonal: not meaningful)
  double X[NB * CS];  // its inverse's lower 16 x 16 blocks, by rows: X(i, k) at [i * CS + k]
  double T[NB * CS];  // the tile below it: A, then L
  double U[NB * CS];  // refinement: the unrefined tile; then diag_panel's copy of block (0, 0)
  double eye[16 * CS];  // identity, 16 x 16
  double piv[NB];     // pivots; given factor: reciprocals of its diagonal
  double mx[5];
  int bad;
};

__device__ inline d4 tile_load(const ChainLds& sh, int rb, int cb, int l) {
  const double* C = sh.L + (16 * cb + (l >> 4)) * CS + 16 * rb + (l & 15);
  return d4{C[0], C[4 * CS], C[8 * CS], C[12 * CS]};
}
__device__ inline void tile_put(ChainLds& sh, int rb, int cb, const d4& t, int l) {
  double* C = sh.L + (16 * cb + (l >> 4)) * CS + 16 * rb + (l & 15);
#pragma unroll
  for (int e = 0; e < 4; ++e) C[4 * e * CS] = t[e];
}
// t -= M(rb, cols) M(cb, cols)^T over 4 S columns of the block M from column
// c0.  All operands are read first: with each read next to its MFMA the
// compiler waits for LDS once per MFMA.
template <int S>
__device__ inline void tile_syrk(d4& t, const double* M, int c0, int rb, int cb, int l) {
  const double* col = M + (c0 + (l >> 4)) * CS + (l & 15);
  double a[S], b[S];
#pragma unroll
  for (int s = 0; s < S; ++s) {
    a[s] = col[4 * s * CS + 16 * cb];
    b[s] = col[4 * s * CS + 16 * rb];
  }
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int s = 0; s < S; ++s) t = __builtin_amdgcn_mfma_f64_16x16x4f64(-a[s], b[s], t, 0, 0, 0);
}
// tile (rb, cb) of the block -= L(rb, panel p) L(cb, panel p)^T
__device__ inline void diag_tile_update(ChainLds& sh, int rb, int cb, int p, int l) {
  d4 t = tile_load(sh, rb, cb, l);
  tile_syrk<4>(t, sh.L, 16 * p, rb, cb, l);
  tile_put(sh, rb, cb, t, l);
}

// Panel p by one wave.  Lanes 0-15: rows of the diagonal 16 x 16 block; 16-31:
// identity rows, becoming L_pp^-T; 32-63: rows of 16-row blocks p + 1 and
// p + 2 (lanes past the block's end compute values that are dropped).  With
// `last`, a repetition of panel 0 for block 3's rows alone (lanes 16-31); its
// diagonal rows are read from sh.U, for the first wave overwrites them in
// sh.L with no barrier between.
__device__ inline void diag_panel(ChainLds& sh, int p, bool last, int l) {
  const int j0 = 16 * p, gi = l >> 4, r = l & 15;
  int row = j0 + r;
  if (gi >= 2) row += 16 * (gi - 1);
  if (last && gi == 1) row = 48 + r;
  const bool ident = gi == 1 && !last;
  const bool keep = last ? gi == 1 : (ident || row < NB);
  const double* src = ident ? sh.eye + r : (last && gi != 1) ? sh.U + r : sh.L + j0 * CS + min(row, NB - 1);
  double v[16];
#pragma unroll
  for (int c = 0; c < 16; ++c) v[c] = src[c * CS];
  double piv = 1.0;  // lane c: pivot c
#pragma unroll
  for (int c = 0; c < 16; ++c) {
    const double d = readlane_d(v[c], c);
    piv = (l == c) ? d : piv;
    v[c] *= pivot_rsqrt(d);
#pragma unroll
    for (int q = c + 1; q < 16; ++q) v[q] = fma(-v[c], readlane_d(v[c], q), v[q]);
  }
  // L's columns (rows above the diagonal carry values that nothing reads; the
  // diagonal itself is written from the pivots, diag_roots) and the inverse's
  // block
  double* dst = (ident ? sh.X + j0 * CS + j0 + r : sh.L + j0 * CS + row);
  if (keep) {
#pragma unroll
    for (int c = 0; c < 16; ++c) dst[c * CS] = v[c];
  }
  if (!last && l < 16) sh.piv[j0 + l] = piv;
}

// The diagonal of panel p (lanes 0-15): the pivots' roots, corrected by one
// Newton step; sh.bad on a non-positive or NaN pivot.  The wave's other lanes
// read them afterwards.
__device__ inline void diag_roots(ChainLds& sh, int p, int l) {
  if (l < 16) {
    const int c = 16 * p + l;
    const double a = sh.piv[c], iv = pivot_rsqrt(a), t = a * iv;
    sh.L[c * CS + c] = fma(fma(-t, t, a), 0.5 * iv, t);
    if (!(a > 0.0)) sh.bad = 1;
  }
  wave_lds_fence();
}

// Given factor: X_qq = L_qq^-1 (16 x 16) into sh.X, lane = column
__device__ inline void given_inverse16(ChainLds& sh, int q, int l) {
  const int j = l & 15, o = 16 * q;
  const double* Lq = sh.L + o * CS + o;
  double x[16];
#pragma unroll
  for (int i = 0; i < 16; ++i) x[i] = (i == j) ? 1.0 : 0.0;
#pragma unroll
  for (int k = 0; k < 16; ++k) {
    x[k] *= sh.piv[o + k];
    int at = k * CS;
    // two columns' reads at a time: all 120 at once would spill
    if ((k & 1) == 0) asm volatile("" : "+v"(at), "+v"(x[k]));
#pragma unroll
    for (int i = k + 1; i < 16; ++i) x[i] = fma(-Lq[at + i], x[k], x[i]);
  }
  if (l < 16)
#pragma unroll
    for (int i = 0; i < 16; ++i) sh.X[(o + i) * CS + o + j] = x[i];
}

__device__ inline double max_abs(const d4& t, double m) {
#pragma unroll
  for (int e = 0; e < 4; ++e) m = fmax(m, fabs(t[e]));
  return m;
}

// X_iq = -X_ii S, into sh.X
__device__ inline d4 inverse_block(ChainLds& sh, int i, int q, const d4& S, int l) {
  const int r = l & 15, g = l >> 4;
  d4 x = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
  for (int s = 0; s < 4; ++s)
    x = __builtin_amdgcn_mfma_f64_16x16x4f64(-sh.X[(16 * i + r) * CS + 16 * i + 4 * s + g], S[s], x, 0, 0, 0);
#pragma unroll
  for (int e = 0; e < 4; ++e) sh.X[(16 * i + g + 4 * e) * CS + 16 * q + r] = x[e];
  return x;
}

// Wave q's share of the inverse after panel t - 1 (t = 1 .. 3): its block of
// row t - 1 (the diagonal one from the panel, the others from the sum of the
// step before), then the sum of row t.  X[j] holds block (q + j, q).
// Returns the running maximum of their magnitude.
__device__ inline double inverse_step(ChainLds& sh, int t, int q, d4 (&X)[3], d4& S, double m, int l) {
  const int r = l & 15, g = l >> 4;
  if (q > t - 1) return m;
  if (q == t - 1) {
    const double* x = sh.X + (16 * q + g) * CS + 16 * q + r;
    X[0] = d4{x[0], x[4 * CS], x[8 * CS], x[12 * CS]};
    m = max_abs(X[0], m);
  } else {
    const d4 x = inverse_block(sh, t - 1, q, S, l);
    m = max_abs(x, m);
#pragma unroll
    for (int j = 1; j < 3; ++j)
      if (q + j == t - 1) X[j] = x;
  }
  S = d4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
  for (int j = 0; j < 3; ++j)
    if (q + j <= t - 1) {
#pragma unroll
      for (int s = 0; s < 4; ++s)
        S = __builtin_amdgcn_mfma_f64_16x16x4f64(sh.L[(16 * (q + j) + 4 * s + g) * CS + 16 * t + r], X[j][s], S, 0, 0,
                                                 0);
    }
  return m;
}

// |L| column sums over 16 rows, for ||L||_1: rows 64 r + 16 q .. of column c
// go to A's strict upper part, which nothing else uses before the
// leave-one-out gradient, at row c of column 64 r + q
__device__ inline double* lcol_part(const Slot& S, int r, int q) { return S.A + (size_t)(r * NB + q) * S.npad; }

__device__ inline double* diag_ptr(double* M, int kk, int ld) { return M + (size_t)kk * NB * ld + kk * NB; }

// panel p's columns of L (rows from the panel's first on) to memory; the
// running maximum of their magnitude
__device__ inline double store_panel(const ChainLds& sh, double* Ab, int ld, int p, double m, int l) {
  double v[16];
#pragma unroll
  for (int i = 0; i < 16; ++i) v[i] = sh.L[(16 * p + i) * CS + l];
  __builtin_amdgcn_sched_barrier(0);
  if (l >= 16 * p) {
#pragma unroll
    for (int i = 0; i < 16; ++i) Ab[(size_t)(16 * p + i) * ld + l] = v[i];
  }
#pragma unroll
  for (int i = 0; i < 16; ++i) m = (l >= 16 * p + i) ? fmax(m, fabs(v[i])) : m;
  return m;
}
// 16 columns (from c0) of T to memory, and their sums of magnitudes over each
// 16 rows (lcol_part)
__device__ inline void store_tile(const ChainLds& sh, const Slot& S, int kk, int ld, int c0, int l) {
  const int r = l & 15, g = l >> 4;
  double* A10 = S.A + (size_t)(kk - 1) * NB * ld + kk * NB;
  double v[16];
#pragma unroll
  for (int i = 0; i < 16; ++i) v[i] = sh.T[(c0 + i) * CS + l];
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int i = 0; i < 16; ++i) A10[(size_t)(c0 + i) * ld + l] = v[i];
  // lane (r, g): column c0 + r, rows 16 g ..
  double sum = 0.0;
#pragma unroll
  for (int i = 0; i < 16; ++i) sum += fabs(sh.T[(c0 + r) * CS + 16 * g + i]);
  lcol_part(S, kk, g)[(kk - 1) * NB + c0 + r] = sum;
}
// the inverse's 16-column block q above its diagonal block: zeros
__device__ inline void store_zeros(double* Wb, int ld, int q, int l) {
  if (l < 16 * q)
#pragma unroll
    for (int i = 0; i < 16; ++i) Wb[(size_t)(16 * q + i) * ld + l] = 0.0;
}
// row block i of the inverse to memory
__device__ inline void store_inverse(const ChainLds& sh, double* Wb, int ld, int i, int l) {
  const int c = l >> 4, r = 16 * i + (l & 15);
#pragma unroll
  for (int q = 0; q < 4; ++q)
    if (q <= i) {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int k = 16 * q + 4 * e + c;
        Wb[(size_t)k * ld + r] = sh.X[r * CS + k];
      }
    }
}
// what diag_block leaves in LDS of block kk (two waves, i = 0, 1): the last
// panel of L and the last two block rows of the inverse
__device__ inline void store_rest(const ChainLds& sh, const Slot& S, int kk, int ld, int i, int l) {
  double* Ab = diag_ptr(S.A, kk, ld);
  double* Wb = diag_ptr(S.W, kk, ld);
  if (i == 0) {
    const int c = 48 + (l >> 4), r = 48 + (l & 15);
#pragma unroll
    for (int e = 0; e < 4; ++e) Ab[(size_t)(c + 4 * e) * ld + r] = sh.L[(c + 4 * e) * CS + r];
  }
  store_inverse(sh, Wb, ld, 2 + i, l);
}

// the 16 column sums of a 16 x 16 block in MFMA result layout (lane: row
// l & 15, columns (l >> 4) + 4e) into dst[0 .. 15]
__device__ inline void lcol_store(const d4& t, double* dst, int l) {
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const double v = row16_sum(fabs(t[e]));
    if ((l & 15) == 0) dst[(l >> 4) + 4 * e] = v;
  }
}

// The second block's 16 x 16 tiles (of A - T T^T) by wave: U_TILE(w, 0) before
// its first panel (block column 0), U_TILE(w, 1) beside panel 0, U_TILE(w, 2)
// beside panel 1 (waves of the SIMDs that run no panel); (-1, -1): none
struct TileRc {
  int rb, cb;
};
__device__ inline TileRc u_tile(int w, int i) {
  if (i == 0) return (w < 4) ? TileRc{w, 0} : TileRc{-1, -1};
  if (i == 1) {
    if (w == 2) return TileRc{1, 1};
    if (w == 6) return TileRc{2, 1};
    if (w == 3) return TileRc{3, 1};
    if (w == 7) return TileRc{2, 2};
  } else {
    if (w == 2) return TileRc{3, 2};
    if (w == 3) return TileRc{3, 3};
  }
  return TileRc{-1, -1};
}
__device__ inline void u_update(ChainLds& sh, int w, int i, d4& D, int l) {
  const TileRc t = u_tile(w, i);
  if (t.rb < 0) return;
  tile_syrk<16>(D, sh.T, 0, t.rb, t.cb, l);
  tile_put(sh, t.rb, t.cb, D, l);
  if (i == 0 && w == 0) {  // block (0, 0) again, for diag_panel's repetition
#pragma unroll
    for (int e = 0; e < 4; ++e) sh.U[((l >> 4) + 4 * e) * CS + (l & 15)] = D[e];
  }
}

// Factor of sh.L in place and its inverse's lower 16 x 16 blocks into sh.X,
// both stored to the diagonal block kk of A and W but for store_rest's part.
// `given`: sh.L and sh.piv already hold a factor; only the inverse is formed.
// `behind`: the second block of a square; the rest of its update by T (D,
// u_tile), T's own stores and the first block's store_rest run beside its
// first panels.  Every wave passes the same barriers.
// Returns the condition estimate 64 max|L| max|L^-1| (PANEL_REFINE_COND).
__device__ inline double diag_block(ChainLds& sh, const Slot& S, int kk, bool given, bool behind, d4 (&D)[3], int w,
                                    int lane) {
  // one loop per role: the addresses and conditions of one role's work stay
  // out of the others' registers (above all out of wave 0's scalar ones)
  double m = 0.0;  // wave 4: max |L|; waves 5-7: max |L^-1|
  const int q = w - 5;
  d4 X[3], R;
  if (w == 0) {
#pragma unroll 1
    for (int p = 0; p < 4; ++p) {
      const int l = opaque(lane);
      if (given)
        given_inverse16(sh, p, l);
      else
        diag_panel(sh, p, false, l);
      __syncthreads();
      if (p < 3) {
        // panel p on the next panel's first tile
        if (!given) diag_tile_update(sh, p + 1, p + 1, p, l);
        __syncthreads();
      }
    }
  } else if (w < 4) {
#pragma unroll 1
    for (int p = 0; p < 4; ++p) {
      const int l = opaque(lane), k2 = opaque_s(kk), ld = opaque_s(S.npad);
      if (p == 0) {
        if (w == 1 && !given) diag_panel(sh, 0, true, l);
        if (w >= 2 && behind) u_update(sh, w, 1, D[1], l);
      } else {
        if (p == 1 && w >= 2 && behind) u_update(sh, w, 2, D[2], l);
        // panel p - 1 on the columns past panel p
        if (!given && p == 1) diag_tile_update(sh, w == 1 ? 2 : 3, w == 3 ? 3 : 2, 0, l);
        if (!given && p == 2 && w == 3) diag_tile_update(sh, 3, 3, 1, l);
        // the stores of T and of the inverse's zeros, where these waves idle
        if (behind && w == 1) store_tile(sh, S, k2, ld, 16 * (p - 1), l);
        if (behind && w == 2 && p == 2) store_tile(sh, S, k2, ld, 48, l);
        if (p == 3 && w > 1)
          for (int c = w - 1; c < 4; c += 2) store_zeros(diag_ptr(S.W, k2, ld), ld, c, l);
      }
      __syncthreads();
      if (p < 3) {
        // panel p on the next panel's other tiles
        if (!given && w < 3 && p + 1 + w < 4) diag_tile_update(sh, p + 1 + w, p + 1, p, l);
        __syncthreads();
      }
    }
  } else {
#pragma unroll
    for (int j = 0; j < 3; ++j) X[j] = d4{0.0, 0.0, 0.0, 0.0};
    R = d4{0.0, 0.0, 0.0, 0.0};
#pragma unroll 1
    for (int p = 0; p < 4; ++p) {
      const int l = opaque(lane), k2 = opaque_s(kk), ld = opaque_s(S.npad);
      if (p == 0) {
        if (behind) {
          if (w >= 6)
            u_update(sh, w, 1, D[1], l);
          else
            store_rest(sh, S, k2 - 1, ld, w - 4, l);
        }
      } else if (w == 4) {
        if (!given) diag_roots(sh, p - 1, l);
        m = store_panel(sh, diag_ptr(S.A, k2, ld), ld, p - 1, m, l);
        if (p > 1) store_inverse(sh, diag_ptr(S.W, k2, ld), ld, p - 2, l);
      } else {
        m = inverse_step(sh, p, q, X, R, m, l);
      }
      __syncthreads();
      if (p < 3) __syncthreads();
    }
  }
  const int l = opaque(lane), r = l & 15, g = l >> 4;
  if (w == 4) {
    if (!given) diag_roots(sh, 3, l);
    // the last panel of L and the last diagonal block of the inverse
    double x = 0.0;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int c = 48 + g + 4 * e;
      if (r >= g + 4 * e) m = fmax(m, fabs(sh.L[c * CS + 48 + r]));
      x = fmax(x, fabs(sh.X[(48 + r) * CS + c]));
    }
    m = wave_max(m);
    x = wave_max(x);
    if (l == 0) {
      sh.mx[0] = m;
      sh.mx[1] = x;
    }
  } else if (w > 4) {
    m = wave_max(max_abs(inverse_block(sh, 3, q, R, l), m));
    if (l == 0) sh.mx[w - 3] = m;
  }
  __syncthreads();
  const double cond = (double)NB * sh.mx[0] * fmax(fmax(sh.mx[1], sh.mx[2]), fmax(sh.mx[3], sh.mx[4]));
  if (w == 0 && l == 0) S.red[red_cond_off(S.nblk) + kk] = cond;
  return cond;
}

// sh.L, just written, is a given factor: zeros above its diagonal, the
// reciprocals of the diagonal; a non-positive or NaN entry there is a failure
__device__ inline void take_factor(ChainLds& sh, int tid) {
  __syncthreads();
  for (int i = tid; i < NB * NB; i += CH_TPB) {
    const int c = i / NB, r = i % NB;
    if (r < c) sh.L[c * CS + r] = 0.0;
    if (r == c) {
      const double v = sh.L[c * CS + c];
      sh.piv[c] = 1.0 / v;
      if (!(v > 0.0)) sh.bad = 1;
    }
  }
}

// t[i] += A X^T for column blocks C0, C1 (>= C0) of the inverse, whose rows end
// at the diagonal; x, y: the lane's first operands in the two LDS blocks
template <int C0, int C1>
__device__ inline void tile_times_inverse(d4 (&t)[2], const double* x, const double* y) {
  constexpr int S0 = 4 * (C0 + 1), S1 = 4 * (C1 + 1);
  double a0[S0], a1[S1], b[S1];
#pragma unroll
  for (int s = 0; s < S1; ++s) {
    b[s] = y[4 * s * CS];
    a1[s] = x[16 * C1 * CS + 4 * s];
    if (s < S0) a0[s] = x[16 * C0 * CS + 4 * s];
  }
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int s = 0; s < S1; ++s) {
    if (s < S0) t[0] = __builtin_amdgcn_mfma_f64_16x16x4f64(a0[s], b[s], t[0], 0, 0, 0);
    t[1] = __builtin_amdgcn_mfma_f64_16x16x4f64(a1[s], b[s], t[1], 0, 0, 0);
  }
}

// Blocks k and (two = 1) k + 1 of the diagonal, and the tile between them.  In
// factor mode both are given factors: only their inverses are formed.
// grid (nslots), 512 threads
__global__ __launch_bounds__(CH_TPB) void k_potrf_chain(const Slot* __restrict__ slots,
                                                        const SlotParams* __restrict__ params,
                                                        SlotOut* __restrict__ out, int k, int two) {
  const int b = blockIdx.x;
  const Slot S = slots[b];
  if (!slot_live(params[b], out[b]) || k >= S.nblk) return;
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int k0 = k * NB;
  const bool given = params[b].mode == MODE_FACTOR;
  const bool second = two != 0 && k + 1 < S.nblk;
  const bool tile = second && !given;
  __shared__ ChainLds sh;
  if (tid == 0) sh.bad = 0;
  const double* A00 = S.A + (size_t)k0 * S.npad + k0;
  d4 D[3];
  double v1[16];
  {
    const int l = tid & 63, r = l & 15, g = l >> 4, w = wave, ld = S.npad;
    double v0[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) v0[i] = gload(A00 + (size_t)(w + 8 * i) * ld + l);
    // the second diagonal block's tiles and (waves 4-7) the tile between: used
    // after the first block, so their loads run beside it
    if (tile) {
      if (w >= 4)
#pragma unroll
        for (int i = 0; i < 16; ++i) v1[i] = gload(A00 + (size_t)(16 * (w - 4) + i) * ld + NB + l);
#pragma unroll
      for (int i = 0; i < 3; ++i) {
        const TileRc t = u_tile(w, i);
        if (t.rb >= 0)
#pragma unroll
          for (int e = 0; e < 4; ++e)
            D[i][e] = gload(A00 + (size_t)(NB + 16 * t.cb + g + 4 * e) * ld + NB + 16 * t.rb + r);
      }
    }
    for (int i = tid; i < 16 * 16; i += CH_TPB) sh.eye[(i >> 4) * CS + (i & 15)] = ((i >> 4) == (i & 15)) ? 1.0 : 0.0;
#pragma unroll
    for (int i = 0; i < 8; ++i) sh.L[(w + 8 * i) * CS + l] = v0[i];
    if (l < 16) {  // block (0, 0) again, for diag_panel's repetition
      sh.U[w * CS + l] = v0[0];
      sh.U[(w + 8) * CS + l] = v0[1];
    }
  }
  if (given) take_factor(sh, tid);
  __syncthreads();
  if (sh.bad) {  // a given factor with a non-positive or NaN diagonal entry
    if (tid == 0) out[b].status = ST_CHOL_FAILED;
    return;
  }
  if (tile && wave >= 4)
#pragma unroll
    for (int i = 0; i < 16; ++i) sh.T[(16 * (wave - 4) + i) * CS + (tid & 63)] = v1[i];
#pragma unroll 1
  for (int kk = k;; ++kk) {
    const int l = opaque(tid & 63), r = l & 15, g = l >> 4, w = opaque_s(wave), ld = opaque_s(S.npad);
    const double cond = diag_block(sh, S, kk, given, kk > k && !given, D, w, l);
    if (sh.bad) {
      if (tid == 0) out[b].status = ST_CHOL_FAILED;
      return;
    }
    if (!second || kk > k) {
      if (w == 4 || w == 5) store_rest(sh, S, kk, ld, w - 4, l);
      return;
    }
    if (given) {
      if (w == 4 || w == 5) store_rest(sh, S, kk, ld, w - 4, l);
      __syncthreads();
      for (int c = w; c < NB; c += 8) sh.L[c * CS + l] = gload(A00 + (size_t)(NB + c) * ld + NB + l);
      take_factor(sh, tid);
      __syncthreads();
      if (sh.bad) {
        if (tid == 0) out[b].status = ST_CHOL_FAILED;
        return;
      }
      continue;
    }
    // the tile between: T(rows, c) = sum_{m <= c} A(rows, m) X(c, m).  Wave w
    // has row block w & 3 and column blocks {0, 3} or {1, 2} (equal K)
    const int rb = w & 3;
    d4 t[2];
    int cbs[2];
    cbs[0] = (w < 4) ? 0 : 1;
    cbs[1] = (w < 4) ? 3 : 2;
    auto times_inverse = [&] {
      const double* x = sh.X + r * CS + g;
      const double* y = sh.T + g * CS + 16 * rb + r;
      if (w < 4)
        tile_times_inverse<0, 3>(t, x, y);
      else
        tile_times_inverse<1, 2>(t, x, y);
    };
    auto put = [&](double* dst, const d4 (&x)[2]) {
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int e = 0; e < 4; ++e) dst[(16 * cbs[i] + g + 4 * e) * CS + 16 * rb + r] = x[i][e];
    };
    t[0] = t[1] = d4{0.0, 0.0, 0.0, 0.0};
    times_inverse();
    if (cond > PANEL_REFINE_COND) {
      // X += (A - X L^T) L^-T once (see k_potrf_rows)
      d4 res[2];
      put(sh.U, t);
      __syncthreads();
#pragma unroll
      for (int i = 0; i < 2; ++i) {
#pragma unroll
        for (int e = 0; e < 4; ++e) res[i][e] = sh.T[(16 * cbs[i] + g + 4 * e) * CS + 16 * rb + r];
        for (int s = 0; s < 4 * (cbs[i] + 1); ++s) {
          const int m = 4 * s + g, c = 16 * cbs[i] + r;
          const double lv = (c >= m) ? -sh.L[m * CS + c] : 0.0;
          res[i] = __builtin_amdgcn_mfma_f64_16x16x4f64(lv, sh.U[m * CS + 16 * rb + r], res[i], 0, 0, 0);
        }
      }
      __syncthreads();
      put(sh.T, res);
      __syncthreads();
      times_inverse();
    }
    __syncthreads();
    put(sh.T, t);
    __syncthreads();
    // the second diagonal block's first block column (the rest: diag_block)
    u_update(sh, w, 0, D[0], l);
    __syncthreads();
  }
}

hipError_t launch_potrf_chain(const Batch& B, int k, int nb) {
  if (nb < 1 || nb > 2) return hipErrorInvalidValue;
  hipLaunchKernelGGL(k_potrf_chain, dim3(B.nslots), dim3(CH_TPB), 0, B.stream, B.slots, B.params, B.out, k,
                     nb == 2 ? 1 : 0);
  return hipGetLastError();
}

// ---------------------------------------------------------------------------
// (2b) the rows below the square: L(r, j) = (A(r, j) - sum_{i < j} L(r, i)
// L(j, i)^T) L_jj^-T for blocks j = k (and k + 1), as products with the
// explicit inverse.  When a diagonal block is ill-conditioned (its estimate
// above PANEL_REFINE_COND) the product is refined once, X += (A - X L_jj^T)
// L_jj^-T: the product alone is accurate to cond(L_jj) eps relative to
// |L_jj^-1|, the refined one to the level of a substitution (dtrsm, as
// LAPACK's dpotrf uses).
// A workgroup has 16 RB rows and all the columns; wave w owns column block w
// of each 64.  The factors' operands are read straight from memory in MFMA
// layout (16 consecutive rows of 4 columns per load, each read by one wave
// of the workgroup); the rows' own blocks go through LDS, where the next
// product needs them as the other operand.
// RB: 1 while the launch leaves CUs idle (the fewest dependent MFMAs per
// workgroup), 4 for large launches (the factors are read once per 64 rows).
// grid (row groups, nslots), 256 threads
// ---------------------------------------------------------------------------
template <int RB>
__global__ __launch_bounds__(TPB) void k_potrf_rows(const Slot* __restrict__ slots,
                                                    const SlotParams* __restrict__ params,
                                                    SlotOut* __restrict__ out, int k, int nb) {
  const TileSlot ts = tile_slot();
  const int b = ts.slot;
  const Slot S = slots[b];
  const int row0 = (k + nb) * NB + ts.tile * 16 * RB;
  if (!slot_live(params[b], out[b]) || row0 >= S.npad || params[b].mode == MODE_FACTOR) return;
  const int tid = threadIdx.x, l = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6), r = l & 15, g = l >> 4;
  const int ld = S.npad;
  constexpr int RS = 16 * RB + 2;  // column stride of the LDS blocks
  __shared__ double sA[NB * RS];   // the current block, updated: [column][row]
  __shared__ double sX[NB * RS];   // the finished first block; refinement: the unrefined block
  const double* cond = S.red + red_cond_off(S.nblk);
  for (int j = 0; j < nb; ++j) {
    const int c0 = (k + j) * NB + 16 * w;  // first of this wave's columns
    double* Aj = S.A + (size_t)c0 * ld + row0;
    d4 acc[RB];
#pragma unroll
    for (int i = 0; i < RB; ++i)
#pragma unroll
      for (int e = 0; e < 4; ++e) acc[i][e] = gload(Aj + (size_t)(g + 4 * e) * ld + 16 * i + r);
    const double* Wj = S.W + (size_t)((k + j) * NB + g) * ld + c0 + r;
    const double* Lj = S.A + (size_t)((k + j) * NB + g) * ld + c0 + r;
    double op[16];
    if (j == 1) {
      const double* Lp = S.A + (size_t)(k * NB + g) * ld + c0 + r;
#pragma unroll
      for (int s = 0; s < 16; ++s) op[s] = -gload(Lp + (size_t)(4 * s) * ld);
#pragma unroll
      for (int s = 0; s < 16; ++s)
#pragma unroll
        for (int i = 0; i < RB; ++i)
          acc[i] = __builtin_amdgcn_mfma_f64_16x16x4f64(op[s], sX[(4 * s + g) * RS + 16 * i + r], acc[i], 0, 0, 0);
    }
    // L_jj^-1's operand (zero beyond this wave's columns)
#pragma unroll
    for (int s = 0; s < 16; ++s) op[s] = (s < 4 * (w + 1)) ? gload(Wj + (size_t)(4 * s) * ld) : 0.0;
#pragma unroll
    for (int i = 0; i < RB; ++i)
#pragma unroll
      for (int e = 0; e < 4; ++e) sA[(16 * w + g + 4 * e) * RS + 16 * i + r] = acc[i][e];
    __syncthreads();
    d4 x[RB];
#pragma unroll
    for (int i = 0; i < RB; ++i) x[i] = d4{0.0, 0.0, 0.0, 0.0};
    auto times_inverse = [&] {
#pragma unroll
      for (int s4 = 0; s4 < 4; ++s4)
        if (s4 <= w)
#pragma unroll
          for (int s = 4 * s4; s < 4 * s4 + 4; ++s)
#pragma unroll
            for (int i = 0; i < RB; ++i)
              x[i] = __builtin_amdgcn_mfma_f64_16x16x4f64(op[s], sA[(4 * s + g) * RS + 16 * i + r], x[i], 0, 0, 0);
    };
    times_inverse();
    if (cond[k + j] > PANEL_REFINE_COND) {
      // acc becomes the residual A - X L_jj^T
#pragma unroll
      for (int i = 0; i < RB; ++i)
#pragma unroll
        for (int e = 0; e < 4; ++e) sX[(16 * w + g + 4 * e) * RS + 16 * i + r] = x[i][e];
      __syncthreads();
      for (int s = 0; s < 4 * (w + 1); ++s) {
        const double lv = (16 * w + r >= 4 * s + g) ? -gload(Lj + (size_t)(4 * s) * ld) : 0.0;
#pragma unroll
        for (int i = 0; i < RB; ++i)
          acc[i] = __builtin_amdgcn_mfma_f64_16x16x4f64(lv, sX[(4 * s + g) * RS + 16 * i + r], acc[i], 0, 0, 0);
      }
#pragma unroll
      for (int i = 0; i < RB; ++i)
#pragma unroll
        for (int e = 0; e < 4; ++e) sA[(16 * w + g + 4 * e) * RS + 16 * i + r] = acc[i][e];
      __syncthreads();
      times_inverse();
    }
#pragma unroll
    for (int i = 0; i < RB; ++i) {
#pragma unroll
      for (int e = 0; e < 4; ++e) Aj[(size_t)(g + 4 * e) * ld + 16 * i + r] = x[i][e];
      const int row = row0 + 16 * i;
      lcol_store(x[i], lcol_part(S, row / NB, (row % NB) / 16) + c0, l);
    }
    if (j + 1 < nb) {
      // every wave is done with sX and sA
      __syncthreads();
#pragma unroll
      for (int i = 0; i < RB; ++i)
#pragma unroll
        for (int e = 0; e < 4; ++e) sX[(16 * w + g + 4 * e) * RS + 16 * i + r] = x[i][e];
      __syncthreads();
    }
  }
}

hipError_t launch_potrf_rows(const Batch& B, int k, int nb) {
  const int blocks = B.nblk_max - k - nb;
  if (blocks <= 0) return hipSuccess;
  if (nb < 1 || nb > 2) return hipErrorInvalidValue;
  // 16-row workgroups while they fit the chip at once (four per CU), else
  // 64-row ones, which read the square's inverse once for four times the rows:
  // all rows of a 64 x n = 1024 batch in two streams 340 us with the line at
  // 1024 workgroups, 346 with 16-row ones throughout, 423 with the line at 256
  const long long groups = 4LL * blocks * B.nslots;
  if (groups <= 1024)
    hipLaunchKernelGGL(k_potrf_rows<1>, dim3(4 * blocks, B.nslots), dim3(TPB), 0, B.stream, B.slots, B.params, B.out,
                       k, nb);
  else
    hipLaunchKernelGGL(k_potrf_rows<4>, dim3(blocks, B.nslots), dim3(TPB), 0, B.stream, B.slots, B.params, B.out, k,
                       nb);
  return hipGetLastError();
}

// ---------------------------------------------------------------------------
// (3a) L^-1 inside the 256 x 256 diagonal blocks: with the 64 x 64 diagonal
// inverses given, X_ij = -X_ii sum_{k = j}^{i-1} L_ik X_kj for i = j + 1 .. 3
// of block column j.  A workgroup has 16 columns of one block column and
// solves its (up to three) block rows one after the other, wave w rows 16 w ..
// of each; columns are independent, so one launch replaces the recursive
// doubling's four of its two smallest levels.
// grid (12 per 256 columns, nslots), 256 threads: workgroup -> group, block
// column j = 0 .. 2 (longest first), 16-column slice
// ---------------------------------------------------------------------------
constexpr int TB_S = 17;  // LDS row stride of a 64 x 16 slice
__global__ __launch_bounds__(TPB) void k_trtri_base(const Slot* __restrict__ slots,
                                                    const SlotParams* __restrict__ params,
                                                    SlotOut* __restrict__ out) {
  const TileSlot ts = tile_slot();
  const int b = ts.slot;
  const Slot S = slots[b];
  if (!slot_live(params[b], out[b])) return;
  const int per = gridDim.x / 3;  // 4 slices of every group
  const int j = ts.tile / per, rem = ts.tile % per;
  const int b0 = 4 * (rem >> 2), slice = rem & 3;
  const int jb = b0 + j, last = min(b0 + 4, S.nblk);
  if (jb + 1 >= last) return;
  const int tid = threadIdx.x, l = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6), r = l & 15, g = l >> 4;
  const int ld = S.npad, col0 = jb * NB + 16 * slice;
  __shared__ double sX[3][NB * TB_S];  // X_kj's slice, [row m][column]
  __shared__ double sS[NB * TB_S];     // the sum's
  // X_jj's slice
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int c = w + 4 * i;
    sX[0][l * TB_S + c] = gload(S.W + (size_t)(col0 + c) * ld + jb * NB + l);
  }
  __syncthreads();
  for (int ib = jb + 1; ib < last; ++ib) {
    const double* Lr = S.A + (size_t)g * ld + ib * NB + 16 * w + r;
    const double* Xi = S.W + (size_t)(ib * NB + g) * ld + ib * NB + 16 * w + r;
    double op[16];
    d4 acc = {0.0, 0.0, 0.0, 0.0};
    for (int kb = jb; kb < ib; ++kb) {
#pragma unroll
      for (int s = 0; s < 16; ++s) op[s] = gload(Lr + (size_t)(kb * NB + 4 * s) * ld);
      const double* x = sX[kb - jb];
#pragma unroll
      for (int s = 0; s < 16; ++s)
        acc = __builtin_amdgcn_mfma_f64_16x16x4f64(x[(4 * s + g) * TB_S + r], op[s], acc, 0, 0, 0);
    }
    // X_ii's operand: rows 16 w .., zero beyond the diagonal
#pragma unroll
    for (int s = 0; s < 16; ++s) op[s] = (s < 4 * (w + 1)) ? -gload(Xi + (size_t)(4 * s) * ld) : 0.0;
    // the sum: row 16 w + r, columns g + 4e
#pragma unroll
    for (int e = 0; e < 4; ++e) sS[(16 * w + r) * TB_S + g + 4 * e] = acc[e];
    __syncthreads();
    d4 x = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int s4 = 0; s4 < 4; ++s4)
      if (s4 <= w)
#pragma unroll
        for (int s = 4 * s4; s < 4 * s4 + 4; ++s)
          x = __builtin_amdgcn_mfma_f64_16x16x4f64(sS[(4 * s + g) * TB_S + r], op[s], x, 0, 0, 0);
#pragma unroll
    for (int e = 0; e < 4; ++e) S.W[(size_t)(col0 + g + 4 * e) * ld + ib * NB + 16 * w + r] = x[e];
    if (ib + 1 < last) {
#pragma unroll
      for (int e = 0; e < 4; ++e) sX[ib - jb][(16 * w + r) * TB_S + g + 4 * e] = x[e];
    }
    __syncthreads();
  }
}

hipError_t launch_trtri_base(const Batch& B) {
  if (B.nblk_max < 2) return hipSuccess;
  const int groups = (B.nblk_max + 3) / 4;
  hipLaunchKernelGGL(k_trtri_base, dim3(12 * groups, B.nslots), dim3(TPB), 0, B.stream, B.slots, B.params, B.out);
  return hipGetLastError();
}

}  // namespace lk
