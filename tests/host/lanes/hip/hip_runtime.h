// Lanes of a gfx950 workgroup on the CPU, for the host tests of the device headers (qex_amd/csrc/*.h): every thread
// of the workgroup is a fiber, and a barrier, a lane exchange or a ballot runs the others up to the same point.
// Between two such points the lanes run one after another, in lane order, so what one lane writes for another
// needs such a point in between, as it does from the compiler's view.
#pragma once
#include <math.h>
#include <stdint.h>
#include <string.h>
#include <ucontext.h>

#include <functional>
#include <vector>

#define __device__
#define __host__
#define __forceinline__ inline

struct double2 {
  double x, y;
};
struct int2 {
  int x, y;
};
inline double2 make_double2(double x, double y) { return {x, y}; }
inline int2 make_int2(int x, int y) { return {x, y}; }
inline int min(int a, int b) { return a < b ? a : b; }
inline int max(int a, int b) { return a > b ? a : b; }

namespace lanes {

struct Bar {
  int n = 0, count = 0, gen = 0;
};
struct Wave {
  std::vector<Bar> group[7];  // [k]: 64 >> k groups of 1 << k lanes
  uint64_t val[7][2][64];     // [k]: what the lanes exchange, alternating (a lane may be one exchange ahead)
};
struct Fiber {
  ucontext_t ctx;
  std::vector<char> stack;
  bool done = false;
  int turn[7] = {0, 0, 0, 0, 0, 0, 0};
};
struct Block {
  std::vector<Fiber> fibers;
  std::vector<Wave> waves;
  Bar all;
  ucontext_t main;
  int cur = 0, left = 0;
  std::function<void()> body;
};
inline Block*& block() {
  static Block* b = nullptr;
  return b;
}
inline void yield() {
  Block& b = *block();
  const int from = b.cur, n = (int)b.fibers.size();
  for (int k = 1; k <= n; ++k) {
    const int to = (from + k) % n;
    if (!b.fibers[to].done) {
      if (to == from) return;
      b.cur = to;
      swapcontext(&b.fibers[from].ctx, &b.fibers[to].ctx);
      return;
    }
  }
  swapcontext(&b.fibers[from].ctx, &b.main);
}
inline void wait(Bar& r) {
  const int gen = r.gen;
  if (++r.count == r.n) {
    r.count = 0;
    ++r.gen;
  } else {
    while (r.gen == gen) yield();
  }
}
inline int tid() { return block()->cur; }

// lane `src` of this wave's value, over groups of 1 << k lanes (only those take part)
inline uint64_t exchange(uint64_t x, int src, int k) {
  Block& b = *block();
  Wave& w = b.waves[b.cur >> 6];
  const int lane = b.cur & 63, p = b.fibers[b.cur].turn[k]++ & 1;
  w.val[k][p][lane] = x;
  wait(w.group[k][lane >> k]);
  return w.val[k][p][src & 63];
}

inline void enter() {
  Block& b = *block();
  b.body();
  b.fibers[b.cur].done = true;
  if (--b.left == 0)
    setcontext(&b.main);
  else
    yield();
}

// body() once by every thread of a workgroup of n threads (a multiple of 64)
inline void run(int n, std::function<void()> body) {
  Block b;
  block() = &b;
  b.body = body;
  b.fibers.resize(n);
  b.waves.resize(n / 64);
  b.all.n = n;
  b.left = n;
  for (Wave& w : b.waves)
    for (int k = 0; k < 7; ++k) {
      w.group[k].resize(64 >> k);
      for (Bar& g : w.group[k]) g.n = 1 << k;
    }
  for (Fiber& f : b.fibers) {
    f.stack.resize(256 * 1024);
    getcontext(&f.ctx);
    f.ctx.uc_stack.ss_sp = f.stack.data();
    f.ctx.uc_stack.ss_size = f.stack.size();
    f.ctx.uc_link = nullptr;
    makecontext(&f.ctx, (void (*)())enter, 0);
  }
  swapcontext(&b.main, &b.fibers[0].ctx);
  block() = nullptr;
}

struct Index3 {
  unsigned x, y, z;
};
inline uint64_t bits(double x) {
  uint64_t u;
  memcpy(&u, &x, 8);
  return u;
}
inline double value(uint64_t u) {
  double x;
  memcpy(&x, &u, 8);
  return x;
}

}  // namespace lanes

#define threadIdx (lanes::Index3{(unsigned)lanes::tid(), 0u, 0u})
#define blockDim (lanes::Index3{(unsigned)lanes::block()->fibers.size(), 1u, 1u})

inline void __syncthreads() { lanes::wait(lanes::block()->all); }
inline void __builtin_amdgcn_wave_barrier() { lanes::exchange(0, 0, 6); }
inline double __shfl(double x, int l, int) { return lanes::value(lanes::exchange(lanes::bits(x), l, 6)); }
inline int __shfl(int x, int l, int) { return (int)lanes::exchange((uint64_t)(uint32_t)x, l, 6); }
inline double __shfl_xor(double x, int m, int w) { return __shfl(x, (lanes::tid() & 63) ^ m, w); }
inline int __shfl_xor(int x, int m, int w) { return __shfl(x, (lanes::tid() & 63) ^ m, w); }
inline unsigned long long __ballot(bool p) {
  lanes::exchange(p, 0, 6);
  lanes::Block& b = *lanes::block();
  const int turn = (b.fibers[b.cur].turn[6] - 1) & 1;
  unsigned long long m = 0;
  for (int l = 0; l < 64; ++l) m |= (unsigned long long)b.waves[b.cur >> 6].val[6][turn][l] << l;
  return m;
}
inline bool __any(bool p) { return __ballot(p) != 0; }
inline int __builtin_amdgcn_readlane(int x, int l) { return __shfl(x, l, 64); }
inline int __builtin_amdgcn_readfirstlane(int x) { return __shfl(x, 0, 64); }
// the DPP moves in use: pairs, quads, half-row mirror, row mirror, row rotation
inline int __builtin_amdgcn_update_dpp(int, int x, int ctrl, int, int, bool) {
  const int l = lanes::tid() & 63;
  int src = l, k = 0;
  switch (ctrl) {
    case 0xB1: src = l ^ 1, k = 1; break;
    case 0x4E: src = l ^ 2, k = 2; break;
    case 0x141: src = l ^ 7, k = 3; break;
    case 0x140: src = l ^ 15, k = 4; break;
    default: __builtin_trap();
  }
  return (int)lanes::exchange((uint64_t)(uint32_t)x, src, k);
}
// hardware reciprocals: cut to 24 bits after the leading one, exact for 0 and infinity
inline double lanes_cut(double x) { return isfinite(x) ? lanes::value(lanes::bits(x) & ~((1ull << 28) - 1)) : x; }
inline double __builtin_amdgcn_rcp(double x) { return lanes_cut(1.0 / x); }
inline double __builtin_amdgcn_rsq(double x) { return lanes_cut(1.0 / sqrt(x)); }
inline int __builtin_amdgcn_frexp_exp(double x) {
  int e = 0;
  if (isfinite(x)) frexp(x, &e);
  return e;
}
inline unsigned __builtin_amdgcn_alignbit(unsigned hi, unsigned lo, unsigned s) {
  return (unsigned)((((uint64_t)hi << 32) | lo) >> (s & 31));
}
inline int __double2hiint(double x) { return (int)(lanes::bits(x) >> 32); }
inline int __double2loint(double x) { return (int)lanes::bits(x); }
inline double __hiloint2double(int h, int l) { return lanes::value(((uint64_t)(uint32_t)h << 32) | (uint32_t)l); }
inline long long __double_as_longlong(double x) { return (long long)lanes::bits(x); }
inline int __popc(unsigned x) { return __builtin_popcount(x); }
inline int __popcll(unsigned long long x) { return __builtin_popcountll(x); }
inline int __ffsll(long long x) { return __builtin_ffsll(x); }
inline int __clzll(long long x) { return x ? __builtin_clzll((unsigned long long)x) : 64; }
