// tiles.h -- a batch of B systems of N points each in launches whose kernels index points with int.
#pragma once
#include <hip/hip_runtime.h>

namespace qextile {

// Points of a launch: with the tiles past the end that the last round of its workgroups addresses, below 2^31.  One
// launch with 64-bit point numbers instead costs k_adj_mlp registers (15 spilled instead of 11, a training
// step 5.46 -> 5.50 ms), and only batches of millions of systems take a second one.
#ifndef QEX_TILE_POINTS
#define QEX_TILE_POINTS (1l << 30)
#endif
inline int systems_per_launch(int N) { return (int)(QEX_TILE_POINTS / N > 0 ? QEX_TILE_POINTS / N : 1); }

// f(first system, systems) for each launch
template <class F>
void for_launches(int B, int N, F f) {
  const int per = systems_per_launch(N);
  for (int s0 = 0; s0 < B;) {
    const int n = B - s0 < per ? B - s0 : per;
    f(s0, n);
    s0 += n;
  }
}

}  // namespace qextile
