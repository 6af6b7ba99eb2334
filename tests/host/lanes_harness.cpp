// The device headers on emulated lanes (lanes/hip/hip_runtime.h), as functions for ctypes.
#include <hip/hip_runtime.h>

#include "symeig.h"

extern "C" {

// A (n x n, symmetric) -> w ascending, Z (n x n, row-major, column j belongs to w[j]); nvec as in qexeig::symeig
void host_symeig(int n, const double* A, int nvec, double* w, double* Z) {
  const int S = n + 1;
  std::vector<double> m((size_t)2 * n * S), f((size_t)3 * n * n);
  qexeig::Smem sh{};
  for (int i = 0; i < n; ++i)
    for (int j = 0; j < n; ++j) m[i * S + j] = A[i * n + j];
  double* z = m.data() + (size_t)n * S;
  lanes::run(512, [&] { qexeig::symeig(n, m.data(), z, S, w, f.data(), sh, nvec); });
  for (int i = 0; i < n; ++i)
    for (int j = 0; j < n; ++j) Z[i * n + j] = z[i * S + j];
}

}  // extern "C"
