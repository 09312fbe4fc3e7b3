// NestedKriging optimal ("NK") aggregation on gfx950, FP64.
//
// Reference: NestedKriging::predict_nk (src/lib/NestedKriging.cpp:353-465),
// after Rulliere, Durrande, Bachoc & Chevalier (Stat. Comput. 2018).  For a
// prediction point x and submodels g = 1..p (common prior sigma2 k(.,.;theta),
// constant trend beta0):
//   k_g(x)   = k(X_g, x)                       (n_g)
//   M_g(x)   = beta0 + k_g' R_g^-1 (y_g - beta0)
//   KM_gg    = k_g' R_g^-1 k_g + jitter
//   KM_ij    = (R_i^-1 k_i)' R_ij (R_j^-1 k_j)  (i != j, R_ij = k(X_i, X_j))
//   w        = KM^-1 diag(KM)
//   mean     = beta0 + w' (M - beta0),  var = sigma2 max(0, 1 - w' diag(KM))
// where R_g = k(X_g, X_g) + jitter I (NestedKriging.cpp:337-346).
//
// The dominant term is sum_{i<j} n_i n_j per point (N^2 q / 2 multiply-adds
// for q points): k_nk_pair forms R_ij on the fly from X (never stored) and
// contracts it on the FP64 MFMA against W_j = R_j^-1 k_j, then against W_i.
// A workgroup owns one group pair, a slice of its row tiles and a range of
// points; its sums stay in registers and the slices are added in order
// (deterministic, no atomics).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <type_traits>

#include <math.h>

#include "lk_device.hpp"
#include "lk_kernels.h"

namespace lk {

// The chunk's arrays C, U, W keep the points contiguous (row a of a group at
// a * qpad): every later reader takes 16 consecutive points per row.
// ---------------------------------------------------------------------------
// (1) C(a, t) = k(x_a - x_t; theta) for the group-ordered design rows a and
// the chunk's points t; zero on pad rows / pad points.  grid (qpad/64, Npad/64)
// ---------------------------------------------------------------------------
template <int DT>
__global__ __launch_bounds__(TPB) void k_nk_cross(NkArgs a) {
  const int t0 = blockIdx.x * NB, i0 = blockIdx.y * NB, tid = threadIdx.x;
  const NkGroup G = a.groups[a.tile_group[blockIdx.y]];
  const int d = a.d, qc = a.qc;
  const int nvalid = G.off + G.n;  // rows >= nvalid are the group's padding
  __shared__ double sXo[DT * NB];
  __shared__ double sXn[DT * NB];
  for (int q = tid; q < d * NB; q += TPB) {
    const int k = q / NB, r = q % NB;
    sXo[q] = a.Xg[(size_t)k * a.Npad + i0 + r];
    sXn[q] = (t0 + r < qc) ? a.Xc[(size_t)k * qc + t0 + r] : 0.0;
  }
  double it[DT];
#pragma unroll
  for (int k = 0; k < DT; ++k) it[k] = (k < d) ? 1.0 / a.theta[k] : 1.0;
  __syncthreads();
  const int jj = tid & 63, gt = t0 + jj;
  double dx[DT];
  for (int r = 0; r < NB / 4; ++r) {
    const int ii = (tid >> 6) + 4 * r, gi = i0 + ii;
    double v = 0.0;
    if (gi < nvalid && gt < qc) {
#pragma unroll
      for (int k = 0; k < DT; ++k) dx[k] = (k < d) ? sXo[k * NB + ii] - sXn[k * NB + jj] : 0.0;
      v = kern_rho<DT>(a.kernel, dx, it);
    }
    a.C[(size_t)gi * a.qpad + gt] = v;
  }
}

// (2) U_g = L_g^-1 C_g: tile (64 points, row tile of group g), K over the
// group's blocks up to the diagonal.  grid (qpad/64, Npad/64)
__global__ __launch_bounds__(TPB) void k_nk_trmm(NkArgs a) {
  const int t0 = blockIdx.x * NB, i0 = blockIdx.y * NB;
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, wr = w >> 1, wc = w & 1;
  const NkGroup G = a.groups[a.tile_group[blockIdx.y]];
  const int il = i0 - G.off, ld = a.qpad;
  __shared__ double sbuf[4 * KC * LDSS];
  d4 acc[2][2];
  acc_zero(acc);
  tile_mainloop<false, false, false>(a.C + (size_t)G.off * ld, ld, t0, a.Linv + G.loff, G.npad, il, 0, il + NB, sbuf,
                                     acc, tid, lane, wr, wc);
  acc_store(acc, a.U + (size_t)i0 * ld + t0, ld, lane, wr, wc);
}

// (3) W_g = L_g^-T U_g = R_g^-1 k_g, written over C (after k_nk_stats has
// used C): K over the group's blocks from the diagonal down.
__global__ __launch_bounds__(TPB) void k_nk_trmm_t(NkArgs a) {
  const int t0 = blockIdx.x * NB, i0 = blockIdx.y * NB;
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, wr = w >> 1, wc = w & 1;
  const NkGroup G = a.groups[a.tile_group[blockIdx.y]];
  const int il = i0 - G.off, ld = a.qpad;
  __shared__ double sbuf[4 * KC * LDSS];
  d4 acc[2][2];
  acc_zero(acc);
  tile_mainloop<false, true, false>(a.U + (size_t)G.off * ld, ld, t0, a.Linv + G.loff, G.npad, il, il, G.npad, sbuf,
                                    acc, tid, lane, wr, wc);
  acc_store(acc, a.C + (size_t)i0 * ld + t0, ld, lane, wr, wc);
}

// (4) per (point, group): M = beta0 + C_g' alpha_g, Kd = |U_g|^2.  Lane =
// point, the rows over the 16 waves (batches of 4), their sums added in wave
// order.  grid (qpad / 64, p)
constexpr int NK_ST_W = 16;
__global__ __launch_bounds__(64 * NK_ST_W) void k_nk_stats(NkArgs a) {
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int t = blockIdx.x * NB + lane, g = blockIdx.y;
  const NkGroup G = a.groups[g];
  const double* c = a.C + (size_t)G.off * a.qpad + t;
  const double* u = a.U + (size_t)G.off * a.qpad + t;
  const double* al = a.alpha + G.off;
  __shared__ double red[2][NK_ST_W][NB];
  double m = 0.0, s = 0.0;
  for (int i = 4 * w; i < G.n; i += 4 * NK_ST_W) {
    double cv[4], uv[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {  // rows beyond n are the group's padding: zero, as alpha is there
      cv[q] = gload(c + (size_t)(i + q) * a.qpad);
      uv[q] = gload(u + (size_t)(i + q) * a.qpad);
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      m = fma(cv[q], al[i + q], m);
      s = fma(uv[q], uv[q], s);
    }
  }
  red[0][w][lane] = m;
  red[1][w][lane] = s;
  __syncthreads();
  if (w < 2 && t < a.qc) {
    double v = red[w][0][lane];
#pragma unroll
    for (int q = 1; q < NK_ST_W; ++q) v += red[w][q][lane];
    if (w == 0)
      a.M[(size_t)t * a.p + g] = a.beta0 + v;
    else
      a.Kd[(size_t)t * a.p + g] = v;
  }
}

// (5) alpha_g = L_g^-T r_g (r_g = L_g^-1 (y_g - beta0), group-ordered): one
// wave per row, reading the row's column of L_g^-1 below the diagonal.
// grid (Npad / 4)
__global__ __launch_bounds__(TPB) void k_nk_alpha(NkArgs a, const double* __restrict__ r) {
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int row = blockIdx.x * 4 + w;
  if (row >= a.Npad) return;
  const NkGroup G = a.groups[a.tile_group[row / NB]];
  const int il = row - G.off;
  double s = 0.0;
  if (il < G.n) {
    const double* col = a.Linv + G.loff + (size_t)il * G.npad;
    for (int k = il + lane; k < G.n; k += 64) s = fma(col[k], r[G.off + k], s);
  }
  s = wave_sum(s);
  if (lane == 0) a.alpha[row] = s;
}

// ---------------------------------------------------------------------------
// (6) part(t) = sum_a W_i(a, t) sum_b R(x_a, x_b) W_j(b, t) for i < j over a
// slice of group i's 64-row tiles, written over U (done with by then) at
// row slice * npairs + pair; k_nk_solve adds the slices in order.  R is
// generated from X and never stored; acc(a, t) += R(a, b) W_j(b, t) on the
// MFMA, 64 rows a by 16 NBJ points per wave, then part(t) += W_i(a, t)
// acc(a, t).  W_j is read straight into the MFMA's operand registers: a wave
// owns its points, so nothing of it is shared, and 16 points of a row are
// one 128-byte line.
// ---------------------------------------------------------------------------
constexpr int NK_DR = 8;    // dimensions kept in registers; beyond, X_i's tile is in LDS
constexpr int NK_PKC = 16;  // rows of group j per chunk

// V covariances at once, of V points (coordinates xa(k, v)) with one (xb(k));
// c[k] is the kernel's scale over theta_k (uniform)
template <int DT, int KT, int V, class XA, class XB>
__device__ inline void nk_values(int d, const double* c, XA xa, XB xb, double (&out)[V]) {
  double s[V], pr[V];
#pragma unroll
  for (int v = 0; v < V; ++v) {
    s[v] = 0.0;
    pr[v] = 1.0;
  }
  auto dim = [&](int k) __attribute__((always_inline)) {
    const double xbk = xb(k), ck = c[k];
#pragma unroll
    for (int v = 0; v < V; ++v) {
      const double u = (xa(k, v) - xbk) * ck;
      if constexpr (KT == K_GAUSS) {
        s[v] = fma(u, u, s[v]);
      } else {
        s[v] += fabs(u);
        if constexpr (KT == K_MATERN32) pr[v] = fma(pr[v], fabs(u), pr[v]);
        if constexpr (KT == K_MATERN52) pr[v] = fma(pr[v], fabs(u) * fma(fabs(u), 1.0 / 3.0, 1.0), pr[v]);
      }
    }
  };
  if constexpr (DT <= NK_DR) {
#pragma unroll
    for (int k = 0; k < DT; ++k) {
      if (k > 0 && k >= d) break;
      dim(k);
    }
  } else {
#pragma unroll 4
    for (int k = 0; k < d; ++k) dim(k);
  }
#pragma unroll
  for (int v = 0; v < V; ++v) {
    const double e = exp(KT == K_GAUSS ? -0.5 * s[v] : -s[v]);
    out[v] = (KT == K_MATERN32 || KT == K_MATERN52) ? e * pr[v] : e;
  }
}

// a uniform value the compiler takes as new: addresses made from it are not
// computed ahead of the loop and kept in registers
__device__ inline int nk_fresh(int v) {
  asm volatile("" : "+s"(v));
  return v;
}
// here the value has arrived (the wait stands at this point and not, for
// every load behind it too, at each use after the branches join)
__device__ inline void nk_arrived(double v) { asm volatile("" : : "v"(v)); }

// uniform base and a lane's offset in bytes (one register, not a pointer)
__device__ inline double nk_load(const double* base, unsigned bytes) {
  return gload(reinterpret_cast<const double*>(reinterpret_cast<const char*>(base) + bytes));
}

// part of one wave -> its points' sums: add the four lanes (kq) of a point
__device__ inline double nk_fold(double v) {
  v += __shfl_xor(v, 16, 64);
  return v + __shfl_xor(v, 32, 64);
}

// (6a) many points: 128 NBJ points per 512-thread workgroup, 16 NBJ per wave;
// a chunk of R (64 x 16) is generated by all eight waves into LDS and used by
// all points.  Bound by the FP64 pipes, which the products (64 x 16 x 128 NBJ
// multiply-adds a chunk) share with the generation: at 512 points a value's
// ~45 vector instructions are 12 % of a chunk's time, at 128 points 36 %.
// What else the loop does: each operand is loaded a chunk ahead (W_j into the
// ring as its last use retires it, the chunk's coordinates into one register
// per lane, read back by v_readlane), two LDS buffers and one barrier per
// chunk, and the second wave of each SIMD runs half a chunk behind the first,
// so that one generates while the other multiplies.  64 rows x 64 points per
// wave: 128 accumulator registers, two waves per SIMD.  n = 20000 in 32
// groups, d = 5, 500 points: 3.77 ms, 53 TFLOP/s (a 64 x 128 tile of four
// waves with W_j staged through LDS and three barriers a chunk: 5.89 ms; the
// waves in step: 3.83 ms).  grid (npairs, slices, tiles), points tbase + 128
// NBJ blockIdx.z ..
template <int DT, int KT, int NBJ>
__global__ __launch_bounds__(512, 2) void k_nk_pair(NkArgs a, int tbase) {
  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r16 = lane & 15, kq = lane >> 4;
  const int2 pr = a.pairs[blockIdx.x];
  const NkGroup Gi = a.groups[pr.x], Gj = a.groups[pr.y];
  const int d = a.d, ld = a.qpad;
  const int nti = Gi.npad / NB, nch = (Gj.n + NK_PKC - 1) / NK_PKC;
  const int tile0 = nti * (int)blockIdx.y / a.nslice, tile1 = nti * ((int)blockIdx.y + 1) / a.nslice;
  __shared__ double sA[2][NK_PKC * LDSS];
  __shared__ double sX[DT > NK_DR ? DT * NB : 1];
  // a wave whose points lie beyond the chunk only helps to generate; block
  // starts beyond it are read at its last 16 points and dropped at the store
  const int tw = tbase + 128 * NBJ * (int)blockIdx.z + 16 * NBJ * w;
  const bool on = tw < a.qc;
  unsigned lo[NBJ];  // row kq, this lane's point
#pragma unroll
  for (int bj = 0; bj < NBJ; ++bj) lo[bj] = 8u * (kq * ld + min(tw + 16 * bj, ld - 16) + r16);
  double part[NBJ];
  d4 acc[4][NBJ];
#pragma unroll
  for (int bj = 0; bj < NBJ; ++bj) {
    part[bj] = 0.0;
#pragma unroll
    for (int bi = 0; bi < 4; ++bi) acc[bi][bj] = d4{0.0, 0.0, 0.0, 0.0};
  }
  const double* Wj = a.C + (size_t)Gj.off * ld;
  double ring[NK_PKC / 4][NBJ];  // the chunk's W_j operands, refilled as they are used
  auto load_ring = [&](int s, int b0) __attribute__((always_inline)) {
#pragma unroll
    for (int bj = 0; bj < NBJ; ++bj) ring[s][bj] = nk_load(Wj + (size_t)(b0 + 4 * s) * ld, lo[bj]);
  };
  double xa[DT > NK_DR ? 1 : DT];
  auto load_tile = [&](int tile) __attribute__((always_inline)) {
    const double* X = a.Xg + Gi.off + tile * NB;
    if constexpr (DT > NK_DR) {
      __syncthreads();
      for (int q = tid; q < d * NB; q += 512) sX[q] = X[(size_t)(q / NB) * a.Npad + q % NB];
      __syncthreads();
    } else {
#pragma unroll
      for (int k = 0; k < DT; ++k) xa[k] = nk_load(X + (size_t)min(k, d - 1) * a.Npad, 8u * lane);
#pragma unroll
      for (int k = 0; k < DT; ++k) nk_arrived(xa[k]);
    }
  };
  // rows b0 + w and b0 + w + 8 of the chunk by this wave, lane = row a; lane
  // 2 k + q holds coordinate k of row q of the pair, loaded a chunk ahead
  const unsigned xo = 8u * (min(lane >> 1, d - 1) * a.Npad + w + 8 * (lane & 1));
  double xb;
  auto load_b = [&](int b0) __attribute__((always_inline)) { xb = nk_load(a.Xg + Gj.off + b0, xo); };
  auto generate = [&](double* dst) __attribute__((always_inline)) {
    double v[2];
    nk_values<DT, KT, 2>(
        d, a.itheta, [&](int k, int q) { return readlane_d(xb, 2 * k + q); },
        [&](int k) {
          if constexpr (DT > NK_DR)
            return sX[k * NB + lane];
          else
            return xa[k];
        },
        v);
    dst[w * LDSS + lane] = v[0];
    dst[(w + 8) * LDSS + lane] = v[1];
  };
  // waves 4 .. 7 run half a chunk behind
  const bool late = DT <= NK_DR && w >= 4;
  // two instances of the loop, so that a wave without points carries no
  // branch around the others' loads
  auto run = [&](auto on_tag) __attribute__((always_inline)) {
    constexpr bool ON = decltype(on_tag)::value;
    load_tile(tile0);
    load_b(0);
    int gtile = tile0, gc = 0, gbuf = 0;  // what generate_next makes
    auto generate_next = [&]() __attribute__((always_inline)) {
      generate(sA[gbuf]);
      gbuf ^= 1;
      if (++gc == nch) {
        gc = 0;
        ++gtile;
        if (gtile < tile1) load_tile(gtile);
      }
      load_b(gc * NK_PKC);
    };
    if (!late) {
      generate_next();
      __syncthreads();
    }
    // (in the loop's order: a wait there then leaves the later ones in flight)
    if constexpr (ON) {
#pragma unroll
      for (int s = 0; s < NK_PKC / 4; ++s) {
        __builtin_amdgcn_sched_barrier(0);
        load_ring(s, 0);
      }
    }
    int buf = 0;
    for (int tile = tile0; tile < tile1; ++tile)
      for (int c = 0; c < nch; ++c, buf ^= 1) {
        const bool last = c + 1 == nch;
        const int bn = last ? 0 : (c + 1) * NK_PKC;
        if (gtile < tile1) generate_next();
        if (late) __syncthreads();
        if constexpr (ON) {
          double an[4];
          const double* pa = sA[buf] + kq * LDSS + r16;
#pragma unroll
          for (int q = 0; q < 4; ++q) an[q] = pa[16 * q];
#pragma unroll
          for (int s = 0; s < NK_PKC / 4; ++s) {
            double av[4];
#pragma unroll
            for (int q = 0; q < 4; ++q) {
              av[q] = an[q];
              if (s + 1 < NK_PKC / 4) an[q] = pa[4 * (s + 1) * LDSS + 16 * q];
            }
            __builtin_amdgcn_sched_barrier(0);  // the next step's operands are on their way
#pragma unroll
            for (int bj = 0; bj < NBJ; ++bj)
#pragma unroll
              for (int bi = 0; bi < 4; ++bi)
                acc[bi][bj] = __builtin_amdgcn_mfma_f64_16x16x4f64(av[bi], ring[s][bj], acc[bi][bj], 0, 0, 0);
            load_ring(s, bn);
          }
          if (last) {
            // lane (r16, kq), register e of block (bi, bj): row 16 bi + kq +
            // 4 e, point r16 of the block
            const double* Wi = a.C + ((size_t)Gi.off + nk_fresh(tile) * NB) * ld;
#pragma unroll
            for (int bj = 0; bj < NBJ; ++bj) {
              double wv[16];
#pragma unroll
              for (int q = 0; q < 16; ++q) wv[q] = nk_load(Wi + (size_t)(4 * q) * ld, lo[bj]);
#pragma unroll
              for (int bi = 0; bi < 4; ++bi) {
#pragma unroll
                for (int e = 0; e < 4; ++e) part[bj] = fma(acc[bi][bj][e], wv[4 * bi + e], part[bj]);
                acc[bi][bj] = d4{0.0, 0.0, 0.0, 0.0};
              }
              __builtin_amdgcn_sched_barrier(0);  // sixteen loads at a time: registers
            }
          }
        }
        if (!late) __syncthreads();
      }
    if (late) __syncthreads();
  };
  if (tile0 < tile1) {
    if (on)
      run(std::true_type{});
    else
      run(std::false_type{});
  }
  double* P = a.U + ((size_t)blockIdx.y * a.npairs + blockIdx.x) * ld;
#pragma unroll
  for (int bj = 0; bj < NBJ; ++bj) {
    const double v = nk_fold(part[bj]);
    const int t = tw + 16 * bj + r16;
    if (kq == 0 && t < a.qc) P[t] = v;
  }
}

// (6b) few points (<= 32): a value of R serves so few points that the time is
// its generation, so each wave generates its own operands in the MFMA's
// register layout (lane = row a r16, row b kq), four independent values a lane
// at a time.  The four waves take 16 of the 64 rows a each; group j's
// coordinates are in LDS, FB rows at a time, so that the loop has no barrier.
// A tile's products meet in LDS, where one wave per 16 points weights and adds
// them in (6a)'s order: the same sums, bit for bit.  A whole prediction, n =
// 20000 in 32 groups: 0.61 ms at 16 points, 0.87 through (6a); n = 3000 in 6
// groups 131 us and 145.  (The rows b over the waves, whose sums are not
// (6a)'s: 0.65 ms and 128 us.  The coordinates from memory, four times the
// loads of that: 1.08 ms.  The values through LDS, a barrier per chunk: 0.66.)
// grid (npairs, slices)
template <int DT, int KT, int NBJ>
__global__ __launch_bounds__(TPB, 3) void k_nk_pair_few(NkArgs a, int tbase) {
  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r16 = lane & 15, kq = lane >> 4;
  const int2 pr = a.pairs[blockIdx.x];
  const NkGroup Gi = a.groups[pr.x], Gj = a.groups[pr.y];
  const int d = a.d, ld = a.qpad;
  const int nti = Gi.npad / NB, nb = (Gj.n + NK_PKC - 1) / NK_PKC * NK_PKC;
  const int tile0 = nti * (int)blockIdx.y / a.nslice, tile1 = nti * ((int)blockIdx.y + 1) / a.nslice;
  constexpr int FB = DT > NK_DR ? NB : 256;  // rows b in LDS
  constexpr int DX = DT > NK_DR ? 1 : DT;
  __shared__ double sB[FB * DT];  // row b: its coordinates
  __shared__ double sX[DT > NK_DR ? DT * NB : 1];
  __shared__ d4 sAcc[4][NBJ][64];
  const unsigned lo = 8u * (kq * ld + r16);  // row kq, point r16
  const double* Wj = a.C + (size_t)Gj.off * ld + tbase;
  double part = 0.0;
  int have = -1;  // first of the rows in sB
  for (int tile = tile0; tile < tile1; ++tile) {
    const double* X = a.Xg + Gi.off + tile * NB;
    double xa[DX];
    if constexpr (DT <= NK_DR) {
#pragma unroll
      for (int k = 0; k < DT; ++k) xa[k] = nk_load(X + (size_t)min(k, d - 1) * a.Npad + 16 * w, 8u * r16);
    } else {
      __syncthreads();
      for (int q = tid; q < d * NB; q += TPB) sX[q] = X[(size_t)(q / NB) * a.Npad + q % NB];
      __syncthreads();
    }
    d4 acc[NBJ];
#pragma unroll
    for (int bj = 0; bj < NBJ; ++bj) acc[bj] = d4{0.0, 0.0, 0.0, 0.0};
    for (int s0 = 0; s0 < nb; s0 += FB) {
      if (have != s0) {
        __syncthreads();  // every wave is done with the rows before
        for (int q = tid; q < DT * FB; q += TPB) {
          const int k = q / FB, b = q % FB;
          if (k < d && s0 + b < Gj.npad) sB[b * DT + k] = a.Xg[(size_t)k * a.Npad + Gj.off + s0 + b];
        }
        have = s0;
        __syncthreads();
      }
      const int cend = min(FB, nb - s0);
      double x[DX][4];
      auto load_x = [&](int b) __attribute__((always_inline)) {
        if constexpr (DT <= NK_DR) {
#pragma unroll
          for (int q = 0; q < 4; ++q)
#pragma unroll
            for (int k = 0; k < DT; ++k) x[k][q] = sB[(b + 4 * q + kq) * DT + k];
        }
      };
      load_x(0);
#pragma unroll 1
      for (int b = 0; b < cend; b += NK_PKC) {
        double av[4], bv[4][NBJ];
#pragma unroll
        for (int s = 0; s < 4; ++s)
#pragma unroll
          for (int bj = 0; bj < NBJ; ++bj) bv[s][bj] = nk_load(Wj + (size_t)(s0 + b + 4 * s) * ld + 16 * bj, lo);
        __builtin_amdgcn_sched_barrier(0);  // they arrive while the values are made
        nk_values<DT, KT, 4>(
            d, a.itheta,
            [&](int k, int q) {
              if constexpr (DT > NK_DR)
                return sB[(b + 4 * q + kq) * DT + k];
              else
                return x[k][q];
            },
            [&](int k) {
              if constexpr (DT > NK_DR)
                return sX[k * NB + 16 * w + r16];
              else
                return xa[k];
            },
            av);
        load_x(min(b + NK_PKC, cend - NK_PKC));
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int s = 0; s < 4; ++s)
#pragma unroll
          for (int bj = 0; bj < NBJ; ++bj)
            acc[bj] = __builtin_amdgcn_mfma_f64_16x16x4f64(av[s], bv[s][bj], acc[bj], 0, 0, 0);
      }
    }
    __syncthreads();  // the tile before has been added
#pragma unroll
    for (int bj = 0; bj < NBJ; ++bj) sAcc[w][bj][lane] = acc[bj];
    __syncthreads();
    if (w < NBJ) {
      const double* Wi = a.C + ((size_t)Gi.off + nk_fresh(tile) * NB) * ld + tbase + 16 * w;
      double wv[16];
#pragma unroll
      for (int q = 0; q < 16; ++q) wv[q] = nk_load(Wi + (size_t)(4 * q) * ld, lo);
#pragma unroll
      for (int bi = 0; bi < 4; ++bi) {
        const d4 s = sAcc[bi][w][lane];
#pragma unroll
        for (int e = 0; e < 4; ++e) part = fma(s[e], wv[4 * bi + e], part);
      }
    }
  }
  const int t = tbase + 16 * w + r16;
  const double v = nk_fold(part);
  if (w < NBJ && kq == 0 && t < a.qc) a.U[((size_t)blockIdx.y * a.npairs + blockIdx.x) * ld + t] = v;
}

// ---------------------------------------------------------------------------
// (7) per point: KM = cross + diag(Kd + jitter); w = KM^-1 diag(KM) by
// Cholesky (arma::solve with likely_sympd); on a non-positive pivot, LU with
// partial pivoting on the same system (the general solver Armadillo falls
// back to).  One workgroup per point.  Bound by the chain of p columns and two
// substitutions, a few accesses to the factor each: it is in LDS up to
// NK_PLDS groups (32 groups, 500 points: 90 -> 62 us), in KF (global,
// L2) beyond.
// ---------------------------------------------------------------------------
constexpr int NK_PMAX = 2048;  // groups supported by the solve kernel (LDS vectors)
constexpr int NK_PLDS = 64;    // 33 KB: four workgroups per CU

template <bool LDS>
__global__ __launch_bounds__(TPB) void k_nk_solve(NkArgs a) {
  const int t = blockIdx.x, tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int p = a.p;
  const size_t pp = (size_t)p * p;
  double* K = a.KM + (size_t)t * pp;
  constexpr int PM = LDS ? NK_PLDS : NK_PMAX;
  __shared__ double sF[LDS ? NK_PLDS * NK_PLDS : 1];
  double* F = a.KF + (size_t)t * pp;
  if constexpr (LDS) F = sF;
  __shared__ double kM[PM];
  __shared__ double z[PM];
  __shared__ double sw[4];
  __shared__ int swi[4];
  __shared__ int spk;
  __shared__ int sflag;
  for (int i = tid; i < p; i += TPB) {
    const double v = a.Kd[(size_t)t * p + i] + a.jitter;
    K[(size_t)i * p + i] = v;
    kM[i] = v;
  }
  for (int q = tid; q < a.npairs; q += TPB) {
    const int2 pr = a.pairs[q];
    double v = a.U[(size_t)q * a.qpad + t];
    for (int z = 1; z < a.nslice; ++z) v += a.U[((size_t)z * a.npairs + q) * a.qpad + t];
    K[(size_t)pr.y * p + pr.x] = v;
    K[(size_t)pr.x * p + pr.y] = v;
  }
  __syncthreads();
  for (size_t q = tid; q < pp; q += TPB) F[q] = K[q];
  if (tid == 0) sflag = 0;
  __syncthreads();
  // right-looking Cholesky, lower triangle of F (column-major)
  for (int k = 0; k < p; ++k) {
    const double dkk = F[(size_t)k * p + k];
    if (!(dkk > 0.0)) {  // uniform: every thread read the same value
      if (tid == 0) sflag = 1;
      break;
    }
    const double r = sqrt(dkk);
    __syncthreads();  // every thread has read F(k, k)
    for (int i = k + tid; i < p; i += TPB) F[(size_t)k * p + i] = (i == k) ? r : F[(size_t)k * p + i] / r;
    __syncthreads();
    for (int j = k + 1 + w; j < p; j += 4) {
      const double ljk = F[(size_t)k * p + j];
      for (int i = j + lane; i < p; i += 64) F[(size_t)j * p + i] = fma(-F[(size_t)k * p + i], ljk, F[(size_t)j * p + i]);
    }
    __syncthreads();
  }
  __syncthreads();
  const bool chol_ok = sflag == 0;
  if (chol_ok) {
    // L z = kM (column sweep), then L' w = z
    for (int i = tid; i < p; i += TPB) z[i] = kM[i];
    __syncthreads();
    for (int k = 0; k < p; ++k) {
      const double zk = z[k] / F[(size_t)k * p + k];
      __syncthreads();
      if (tid == 0) z[k] = zk;
      for (int i = k + 1 + tid; i < p; i += TPB) z[i] = fma(-F[(size_t)k * p + i], zk, z[i]);
      __syncthreads();
    }
    for (int k = p - 1; k >= 0; --k) {
      const double wk = z[k] / F[(size_t)k * p + k];
      __syncthreads();
      if (tid == 0) z[k] = wk;
      for (int i = tid; i < k; i += TPB) z[i] = fma(-F[(size_t)i * p + k], wk, z[i]);
      __syncthreads();
    }
  } else {
    // LU with partial pivoting on a fresh copy of KM (row-wise elimination)
    for (size_t q = tid; q < pp; q += TPB) F[q] = K[q];
    for (int i = tid; i < p; i += TPB) z[i] = kM[i];
    if (tid == 0) sflag = 1;
    __syncthreads();
    for (int k = 0; k < p; ++k) {
      // pivot: largest |F(i, k)|, i >= k, first index on ties
      double best = -1.0;
      int bi = k;
      for (int i = k + tid; i < p; i += TPB) {
        const double v = fabs(F[(size_t)k * p + i]);
        if (v > best) {
          best = v;
          bi = i;
        }
      }
      for (int off = 32; off > 0; off >>= 1) {
        const double ob = __shfl_xor(best, off, 64);
        const int oi = __shfl_xor(bi, off, 64);
        if (ob > best || (ob == best && oi < bi)) {
          best = ob;
          bi = oi;
        }
      }
      if (lane == 0) {
        sw[w] = best;
        swi[w] = bi;
      }
      __syncthreads();
      if (tid == 0) {
        double b = sw[0];
        int ix = swi[0];
        for (int q = 1; q < 4; ++q)
          if (sw[q] > b || (sw[q] == b && swi[q] < ix)) {
            b = sw[q];
            ix = swi[q];
          }
        spk = ix;
        if (!(b > 0.0)) sflag = 2;
      }
      __syncthreads();
      if (sflag == 2) break;
      const int pk = spk;
      if (pk != k) {
        for (int j = tid; j < p; j += TPB) {
          const double u = F[(size_t)j * p + k];
          F[(size_t)j * p + k] = F[(size_t)j * p + pk];
          F[(size_t)j * p + pk] = u;
        }
        if (tid == 0) {
          const double u = z[k];
          z[k] = z[pk];
          z[pk] = u;
        }
      }
      __syncthreads();
      const double dkk = F[(size_t)k * p + k];
      for (int i = k + 1 + tid; i < p; i += TPB) F[(size_t)k * p + i] /= dkk;
      __syncthreads();
      for (int j = k + 1 + w; j < p; j += 4) {
        const double ukj = F[(size_t)j * p + k];
        for (int i = k + 1 + lane; i < p; i += 64) F[(size_t)j * p + i] = fma(-F[(size_t)k * p + i], ukj, F[(size_t)j * p + i]);
      }
      if (tid == 0) {
        const double zk = z[k];
        for (int i = k + 1; i < p; ++i) z[i] = fma(-F[(size_t)k * p + i], zk, z[i]);
      }
      __syncthreads();
    }
    if (sflag != 2) {
      for (int k = p - 1; k >= 0; --k) {
        const double wk = z[k] / F[(size_t)k * p + k];
        __syncthreads();
        if (tid == 0) z[k] = wk;
        for (int i = tid; i < k; i += TPB) z[i] = fma(-F[(size_t)k * p + i], wk, z[i]);
        __syncthreads();
      }
    }
  }
  __syncthreads();
  // mean and variance: fixed-order reductions
  double sm = 0.0, sv = 0.0;
  const double* Mt = a.M + (size_t)t * p;
  for (int i = tid; i < p; i += TPB) {
    sm = fma(z[i], Mt[i] - a.beta0, sm);
    sv = fma(z[i], kM[i], sv);
  }
  sm = wave_sum(sm);
  sv = wave_sum(sv);
  __shared__ double rs[2][4];
  if (lane == 0) {
    rs[0][w] = sm;
    rs[1][w] = sv;
  }
  __syncthreads();
  if (tid == 0) {
    const int st = sflag;
    if (st == 2) {
      a.out[t] = nan("");
      a.out[a.qc + t] = nan("");
    } else {
      const double m = (rs[0][0] + rs[0][1]) + (rs[0][2] + rs[0][3]);
      const double v = (rs[1][0] + rs[1][1]) + (rs[1][2] + rs[1][3]);
      a.out[t] = a.beta0 + m;
      a.out[a.qc + t] = a.sigma2 * fmax(0.0, 1.0 - v);
    }
    a.info[t] = st;
  }
}

// ---------------------------------------------------------------------------
// launchers
// ---------------------------------------------------------------------------
hipError_t launch_nk_prepare(const NkArgs& a, hipStream_t stream) {
  const dim3 grid(a.qpad / NB, a.Npad / NB);
  if (a.d <= 4)
    hipLaunchKernelGGL(k_nk_cross<4>, grid, dim3(TPB), 0, stream, a);
  else if (a.d <= 8)
    hipLaunchKernelGGL(k_nk_cross<8>, grid, dim3(TPB), 0, stream, a);
  else if (a.d <= 16)
    hipLaunchKernelGGL(k_nk_cross<16>, grid, dim3(TPB), 0, stream, a);
  else
    hipLaunchKernelGGL(k_nk_cross<32>, grid, dim3(TPB), 0, stream, a);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(k_nk_trmm, grid, dim3(TPB), 0, stream, a);
  if ((e = hipGetLastError()) != hipSuccess) return e;
  hipLaunchKernelGGL(k_nk_stats, dim3(a.qpad / NB, a.p), dim3(64 * NK_ST_W), 0, stream, a);
  if ((e = hipGetLastError()) != hipSuccess) return e;
  hipLaunchKernelGGL(k_nk_trmm_t, grid, dim3(TPB), 0, stream, a);
  return hipGetLastError();
}

// Slices of group i's row tiles, so that few pairs still cover the chip.  A
// point's sum is that of its slices in order, so their number depends on the
// pairs alone and never on the points: NK_WGS workgroups where 512 points or
// fewer are one launch of it (pair kernel at 496 pairs and 500 points 3.77 ms;
// 3.82 for 1024, 4.02 for 4096, where the start of each workgroup shows); with
// more points fewer, longer workgroups gained nothing (1000 points 7.96 ms a
// prediction against 8.29, 8192 points 61.7 against 61.4)
int nk_pair_slices(int npairs, int max_tiles) {
  if (npairs <= 0) return 1;
  return std::max(1, std::min(max_tiles, (NK_WGS + npairs - 1) / npairs));
}

hipError_t launch_nk_pairs(const NkArgs& args, hipStream_t stream) {
  if (args.npairs <= 0) return hipSuccess;
  if (args.qpad % NB != 0 || args.qc > args.qpad || args.nslice < 1) return hipErrorInvalidValue;
  NkArgs a = args;
  // the kernels' scale of |x - x'| / theta
  const double scale = a.kernel == K_MATERN32 ? SQRT3 : a.kernel == K_MATERN52 ? SQRT5 : 1.0;
  for (int k = 0; k < DMAX; ++k) a.itheta[k] *= scale;
  // one instance per (dimension bound, covariance kernel, points per wave):
  // the generation runs one kernel's code, not a branch per value
  auto run = [&](auto dtag, auto ktag, int tbase, int tiles, int nbj) {
    constexpr int DT = decltype(dtag)::value;
    constexpr int KT = decltype(ktag)::value;
    const dim3 grid(a.npairs, a.nslice, tiles);
    switch (nbj) {
      case 1: hipLaunchKernelGGL((k_nk_pair<DT, KT, 1>), grid, dim3(512), 0, stream, a, tbase); break;
      case 2: hipLaunchKernelGGL((k_nk_pair<DT, KT, 2>), grid, dim3(512), 0, stream, a, tbase); break;
      case 3: hipLaunchKernelGGL((k_nk_pair<DT, KT, 3>), grid, dim3(512), 0, stream, a, tbase); break;
      default: hipLaunchKernelGGL((k_nk_pair<DT, KT, 4>), grid, dim3(512), 0, stream, a, tbase); break;
    }
    return hipGetLastError();
  };
  auto run_few = [&](auto dtag, auto ktag, int tbase, int points) {
    constexpr int DT = decltype(dtag)::value;
    constexpr int KT = decltype(ktag)::value;
    const dim3 grid(a.npairs, a.nslice);
    if (points <= 16)
      hipLaunchKernelGGL((k_nk_pair_few<DT, KT, 1>), grid, dim3(TPB), 0, stream, a, tbase);
    else
      hipLaunchKernelGGL((k_nk_pair_few<DT, KT, 2>), grid, dim3(TPB), 0, stream, a, tbase);
    return hipGetLastError();
  };
  auto go = [&](auto dtag, auto ktag) {
    // whole tiles of 512 points, the rest in one launch of its own width
    const int tiles = a.qc / NK_QT, rest = a.qc % NK_QT;
    hipError_t e = hipSuccess;
    if (tiles > 0) e = run(dtag, ktag, 0, tiles, 4);
    if (e == hipSuccess && rest > NK_FEW) e = run(dtag, ktag, tiles * NK_QT, 1, (rest + 127) / 128);
    if (e == hipSuccess && rest > 0 && rest <= NK_FEW) e = run_few(dtag, ktag, tiles * NK_QT, rest);
    return e;
  };
  auto kern = [&](auto dtag) {
    switch (a.kernel) {
      case K_GAUSS: return go(dtag, std::integral_constant<int, K_GAUSS>{});
      case K_EXP: return go(dtag, std::integral_constant<int, K_EXP>{});
      case K_MATERN32: return go(dtag, std::integral_constant<int, K_MATERN32>{});
      default: return go(dtag, std::integral_constant<int, K_MATERN52>{});
    }
  };
  return a.d <= NK_DR ? kern(std::integral_constant<int, NK_DR>{}) : kern(std::integral_constant<int, DMAX>{});
}

hipError_t launch_nk_solve(const NkArgs& a, hipStream_t stream) {
  if (a.p > NK_PMAX) return hipErrorInvalidValue;
  if (a.p <= NK_PLDS)
    hipLaunchKernelGGL(k_nk_solve<true>, dim3(a.qc), dim3(TPB), 0, stream, a);
  else
    hipLaunchKernelGGL(k_nk_solve<false>, dim3(a.qc), dim3(TPB), 0, stream, a);
  return hipGetLastError();
}

hipError_t launch_nk_alpha(const NkArgs& a, const double* r, hipStream_t stream) {
  hipLaunchKernelGGL(k_nk_alpha, dim3(a.Npad / 4), dim3(TPB), 0, stream, a, r);
  return hipGetLastError();
}

}  // namespace lk
