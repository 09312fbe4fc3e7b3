// Device code of this repository run on the host, one fiber per lane: enough
// of the HIP language and of the gfx950 builtins for the kernels under test.
// Between two workgroup barriers the waves run one after the other in the
// order `wave_order`, and inside a wave the lanes run in `lane_order` between
// cross-lane operations.  Accesses that no barrier (lane: cross-lane operation
// or wave fence) orders give another result under some order and its reverse.
#pragma once
#include <math.h>
#include <stdint.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>
#include <ucontext.h>

#include <algorithm>
#include <functional>
#include <type_traits>
#include <vector>

namespace emu {
struct Dim {
  unsigned x = 1, y = 1, z = 1;
  Dim(unsigned a = 1, unsigned b = 1, unsigned c = 1) : x(a), y(b), z(c) {}
};
enum State { READY, LANE_OP, BARRIER, DONE };
struct Fiber {
  ucontext_t ctx;
  State state;
  unsigned ops;
  std::vector<char> stack;
};
constexpr int W = 64;
inline std::vector<Fiber> fibers;
inline std::vector<uint64_t> slots[2];  // a wave's operands of its last two operations
inline ucontext_t main_ctx;
inline int current;
inline std::function<void()> body;
inline std::vector<int> wave_order;
inline bool lanes_reversed = false;
inline Dim block_idx, thread_idx, grid_dim, block_dim;

inline void yield(State s) {
  fibers[current].state = s;
  swapcontext(&fibers[current].ctx, &main_ctx);
}
// every lane of the wave contributes v; returns the wave's 64 values
inline const uint64_t* exchange(uint64_t v) {
  const int k = fibers[current].ops++ & 1;
  slots[k][current] = v;
  yield(LANE_OP);
  return &slots[k][current / W * W];
}
inline void entry() {
  body();
  yield(DONE);
}
inline void run_workgroup(int threads) {
  if ((int)fibers.size() < threads) fibers.resize(threads);
  for (auto& s : slots) s.assign(threads, 0);
  for (int t = 0; t < threads; ++t) {
    Fiber& f = fibers[t];
    f.stack.resize(1 << 17);
    f.state = READY;
    f.ops = 0;
    getcontext(&f.ctx);
    f.ctx.uc_stack.ss_sp = f.stack.data();
    f.ctx.uc_stack.ss_size = f.stack.size();
    f.ctx.uc_link = nullptr;
    makecontext(&f.ctx, entry, 0);
  }
  for (bool live = true; live;) {
    for (int w : wave_order) {
      if (w * W >= threads) continue;
      for (bool again = true; again;) {
        int n[4] = {0, 0, 0, 0};
        for (int q = 0; q < W; ++q) {
          current = w * W + (lanes_reversed ? W - 1 - q : q);
          thread_idx = Dim(current, 0, 0);
          if (fibers[current].state == READY) swapcontext(&main_ctx, &fibers[current].ctx);
          ++n[fibers[current].state];
        }
        again = n[LANE_OP] > 0;
        if (again && n[LANE_OP] != W) {
          fprintf(stderr, "wave %d: a cross-lane operation that not every lane takes part in\n", w);
          abort();
        }
        if (again)
          for (int q = 0; q < W; ++q) fibers[w * W + q].state = READY;
      }
    }
    int done = 0, bar = 0;
    for (int t = 0; t < threads; ++t) (fibers[t].state == DONE ? done : bar) += 1;
    live = bar > 0;
    if (done > 0 && bar > 0) {
      fprintf(stderr, "a barrier that not every lane reaches\n");
      abort();
    }
    for (int t = 0; t < threads; ++t)
      if (fibers[t].state == BARRIER) fibers[t].state = READY;
  }
}
template <class K, class... A>
void launch(K kernel, Dim grid, Dim block, A... args) {
  grid_dim = grid;
  block_dim = block;
  if (wave_order.empty())
    for (int w = 0; w < 16; ++w) wave_order.push_back(w);
  for (unsigned y = 0; y < grid.y; ++y)
    for (unsigned x = 0; x < grid.x; ++x) {
      block_idx = Dim(x, y, 0);
      body = [&] { kernel(args...); };
      run_workgroup((int)block.x);
    }
}
inline uint64_t bits(double v) {
  uint64_t u;
  memcpy(&u, &v, 8);
  return u;
}
inline double number(uint64_t u) {
  double v;
  memcpy(&v, &u, 8);
  return v;
}
inline int lane() { return current % W; }

typedef double vec4 __attribute__((ext_vector_type(4)));
typedef unsigned vec2u __attribute__((ext_vector_type(2)));
// D(l >> 4 + 4e, l & 15) = C + sum_k P(., k) Q(k, .); P: lane -> (l & 15,
// l >> 4), Q: lane -> (l >> 4, l & 15)
inline vec4 mfma16x16x4(double p, double q, vec4 c) {
  uint64_t P[W], Q[W];
  memcpy(P, exchange(bits(p)), sizeof(P));
  memcpy(Q, exchange(bits(q)), sizeof(Q));
  const int l = lane();
  for (int e = 0; e < 4; ++e)
    for (int k = 0; k < 4; ++k)
      c[e] = ::fma(number(P[16 * k + (l >> 4) + 4 * e]), number(Q[16 * k + (l & 15)]), c[e]);
  return c;
}
inline int update_dpp(int v, int ctrl) {  // row_ror: 0x120 + n
  const int l = lane(), n = ctrl - 0x120;
  const uint64_t* s = exchange((uint32_t)v);
  return (int)(uint32_t)s[(l & 48) | ((l - n) & 15)];
}
// v_permlane{16,32}_swap of a register with itself: the even rows' (lower
// half's) values and the odd ones'
inline vec2u permlane_swap(unsigned v, int width) {
  const int l = lane();
  const uint64_t* s = exchange(v);
  return vec2u{(unsigned)s[l & ~width], (unsigned)s[l | width]};
}
inline int readlane(int v, int from) { return (int)(uint32_t)exchange((uint32_t)v)[from]; }
}  // namespace emu

#define __device__
#define __host__
#define __global__
#define __shared__ static
#define __launch_bounds__(...)
#define threadIdx (emu::thread_idx)
#define blockIdx (emu::block_idx)
#define gridDim (emu::grid_dim)
typedef emu::Dim dim3;
struct int2 {
  int x, y;
};
typedef int hipError_t;
typedef void* hipStream_t;
constexpr int hipSuccess = 0, hipErrorInvalidValue = 1;
inline int hipGetLastError() { return hipSuccess; }
#define hipLaunchKernelGGL(kernel, grid, block, lds, stream, ...) emu::launch(kernel, grid, block, __VA_ARGS__)

using std::max;
using std::min;
inline void __syncthreads() { emu::yield(emu::BARRIER); }
inline int __double2loint(double v) { return (int)(uint32_t)emu::bits(v); }
inline int __double2hiint(double v) { return (int)(uint32_t)(emu::bits(v) >> 32); }
inline double __hiloint2double(int hi, int lo) { return emu::number(((uint64_t)(uint32_t)hi << 32) | (uint32_t)lo); }
inline unsigned __float_as_uint(float v) {
  unsigned u;
  memcpy(&u, &v, 4);
  return u;
}
inline int __float_as_int(float v) { return (int)__float_as_uint(v); }
inline float __uint_as_float(unsigned u) {
  float v;
  memcpy(&v, &u, 4);
  return v;
}
inline float __int_as_float(int u) { return __uint_as_float((unsigned)u); }

#define __builtin_amdgcn_mfma_f64_16x16x4f64(p, q, c, x, y, z) emu::mfma16x16x4(p, q, c)
#define __builtin_amdgcn_update_dpp(old, v, ctrl, row, bank, bound) emu::update_dpp(v, ctrl)
#define __builtin_amdgcn_permlane16_swap(a, b, x, y) emu::permlane_swap(a, 16)
#define __builtin_amdgcn_permlane32_swap(a, b, x, y) emu::permlane_swap(a, 32)
#define __builtin_amdgcn_readlane(v, l) emu::readlane(v, l)
#define __builtin_amdgcn_readfirstlane(v) emu::readlane(v, 0)
#define __builtin_amdgcn_rsq(v) (1.0 / sqrt(v))
#define __builtin_amdgcn_sched_barrier(m)
#define __builtin_amdgcn_fence(order, scope)
#define __builtin_amdgcn_wave_barrier() ((void)emu::exchange(0))
// empty statements that only hide a value from the compiler
#define asm
#define volatile(...)
