// The device headers on emulated lanes (lanes/hip/hip_runtime.h), as functions for ctypes.
#include <hip/hip_runtime.h>

#include "eigen1d.h"
#include "symeig.h"
#include "symeig_lds.h"
#include "tiles.h"

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

// the pentadiagonal A = diag(a) + b + c and the workspace of its solves
struct Band {
  int N, kt;
  double b, c, hnorm;
  std::vector<double> a, ap, F;
  Band(int n, const double* diag, double b_, double c_) : N(n), kt((n - 2) / 2), b(b_), c(c_), a(diag, diag + n), ap(n) {
    double m = 0.0;
    for (int t = 0; t < n; ++t) {
      ap[qexband::side_pos(t, n, kt)] = a[t];
      m = fmax(m, fabs(a[t]));
    }
    hnorm = m + 2.0 * (fabs(b) + fabs(c));
    F.resize(qexband::wave_doubles(n));
  }
};

}  // namespace

extern "C" {

// eigenvalues of A below sigma: by the two-sided pivots, and by one wave's substructured factorisation
int host_sturm(int N, const double* a, double b, double c, double sigma) {
  Band m(N, a, b, c);
  const int kt = m.kt;
  const qexband::Side t = qexband::sturm_side(m.ap.data(), 1, kt, b, c, sigma);
  const qexband::Side u = qexband::sturm_side(m.ap.data() + kt + 2, 1, N - 2 - kt, b, c, sigma);
  return qexband::sturm_join(t, u, a[kt], a[kt + 1], b, c, sigma);
}
int host_wave_count(int N, const double* a, double b, double c, double sigma) {
  Band m(N, a, b, c);
  int n = 0;
  lanes::run(64, [&] { n = qexband::wave_solve<false>(m.a.data(), nullptr, N, b, c, sigma, m.F.data()); });
  return n;
}
// y <- (A - sigma)^-1 y by one wave; by the pivoted elimination
int host_wave_solve(int N, const double* a, double* y, double b, double c, double sigma) {
  Band m(N, a, b, c);
  int n = 0;
  lanes::run(64, [&] { n = qexband::wave_solve<true>(m.a.data(), y, N, b, c, sigma, m.F.data()); });
  return n;
}
void host_pivoted_solve(int N, const double* a, double* y, double b, double c, double sigma) {
  Band m(N, a, b, c);
  std::vector<double> R((size_t)5 * N);
  qexband::pivoted_solve(a, y, R.data(), N, b, c, sigma, qexband::EPS * m.hnorm);
}
// the j-th eigenvalue from the vector y: refinement and, with near, the index; 1 if found
int host_refine(int N, const double* a, double* y, double b, double c, int j, double lo, double hi, int near, double* rho) {
  Band m(N, a, b, c);
  int ok = 0;
  lanes::run(64, [&] {
    double r = 0.0;
    bool found = qexband::refine_eigenvalue(m.a.data(), y, m.F.data(), N, b, c, lo, hi, near != 0, &r);
    if (found && near)
      for (int above = 0; above < 2; ++above)
        found = qexband::confirm_side(m.a.data(), m.F.data(), N, b, c, m.hnorm, j, r, above) && found;
    if (threadIdx.x == 0) {
      ok = found;
      *rho = r;
    }
  });
  return ok;
}
// the launches of a batch: first system and number of systems of each; returns how many
int host_launches(int B, int N, int max, int* first, int* n) {
  int k = 0;
  qextile::for_launches(B, N, [&](int s0, int m) {
    if (k < max) {
      first[k] = s0;
      n[k] = m;
    }
    ++k;
  });
  return k;
}
// two twisted inverse-iteration solves at sigma from y
void host_twisted(int N, const double* a, double* y, double b, double c, double sigma) {
  Band m(N, a, b, c);
  std::vector<double> yp(N), part(256);
  for (int t = 0; t < N; ++t) yp[qexband::side_pos(t, N, m.kt)] = y[t];
  lanes::run(256, [&] {
    qexband::twisted_inverse_iteration<256>(m.ap.data(), yp.data(), m.F.data(), N, m.kt, b, c, sigma, qexband::EPS * m.hnorm,
                                            [&](double x) {
                                              part[threadIdx.x] = x;
                                              __syncthreads();
                                              double s = 0.0;
                                              for (double p : part) s += p;
                                              __syncthreads();
                                              return s;
                                            });
  });
  for (int t = 0; t < N; ++t) y[t] = yp[qexband::side_pos(t, N, m.kt)];
}

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
