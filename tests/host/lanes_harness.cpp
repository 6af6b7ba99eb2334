// The device headers on emulated lanes (lanes/hip/hip_runtime.h), as functions for ctypes.
#include <hip/hip_runtime.h>

#include "symeig.h"
#include "symeig_lds.h"

namespace {

template <class Smem, class F>
void solve(int threads, int n, const double* A, double* Z, int* perm, F f) {
  const int S = n + 1;
  std::vector<double> m((size_t)2 * n * S), scratch((size_t)3 * n * n);
  Smem sh{};
  for (int& p : sh.perm) p = -1;
  for (int i = 0; i < n; ++i)
    for (int j = 0; j < n; ++j) m[i * S + j] = A[i * n + j];
  double* z = m.data() + (size_t)n * S;
  lanes::run(threads, [&] { f(m.data(), z, S, scratch.data(), sh); });
  for (int i = 0; i < n; ++i) {
    perm[i] = sh.perm[i];
    for (int j = 0; j < n; ++j) Z[i * n + j] = z[i * S + j];
  }
}

}  // namespace

extern "C" {

// A (n x n, symmetric) -> w ascending, Z (n x n, row-major, column j belongs to w[j]); nvec as in symeig;
// perm: the order of the solver's slots (-1: not set)
void host_symeig(int n, const double* A, int nvec, double* w, double* Z, int* perm) {
  solve<qexeig::Smem>(512, n, A, Z, perm, [&](double* a, double* z, int S, double* f, qexeig::Smem& sh) {
    qexeig::symeig(n, a, z, S, w, f, sh, nvec);
  });
}
void host_symeig_lds(int n, const double* A, int nvec, double* w, double* Z, int* perm) {
  solve<qexeig_lds::Smem>(1024, n, A, Z, perm, [&](double* a, double* z, int S, double* f, qexeig_lds::Smem& sh) {
    qexeig_lds::symeig(n, a, z, S, w, f, sh, nvec);
  });
}

}  // extern "C"
