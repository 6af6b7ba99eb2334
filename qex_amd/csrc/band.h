// band.h -- symmetric pentadiagonal eigen-kernels shared by the gfx950 eigensolver.
//
// A = diag(a) + b (first off-diagonals) + c (second off-diagonals), the 5-point-stencil
// Kohn-Sham Hamiltonian of the 1D grid.
#pragma once
#include <hip/hip_runtime.h>
#include <math.h>

#define QEX_HD __host__ __device__

namespace qexband {

// 1/d to double precision: the hardware reciprocal (relative error <= 5e-8 on gfx950) and one
// Newton step (relative error ~2e-15) on the device.
QEX_HD inline double rcp64(double d) {
#if defined(__HIP_DEVICE_COMPILE__)
  const double r = __builtin_amdgcn_rcp(d);
  return fma(r, fma(-d, r, 1.0), r);
#else
  return 1.0 / d;
#endif
}

// 1 if the sign bit of x is set (also for -0.0), else 0 -- without a compare/VCC round trip.
QEX_HD inline int sign_bit(double x) {
#if defined(__HIP_DEVICE_COMPILE__)
  return (int)(((unsigned)__double2hiint(x)) >> 31);
#else
  return signbit(x) ? 1 : 0;
#endif
}

// 1/d clamped to [-RMAX, RMAX]: a pivot smaller than 1/RMAX in magnitude acts as +-1/RMAX
// (an O(1e-60) perturbation of one diagonal entry) and no inf/NaN can enter a recurrence.
constexpr double RMAX = 1e60;
QEX_HD inline double rcp_clamped(double d) { return fmin(fmax(rcp64(d), -RMAX), RMAX); }

// ---- two-sided elimination ------------------------------------------------------------------
// The rows of A - sigma are eliminated from the top (rows 0 .. k-1) and from the bottom (rows
// N-1 .. k+2) at the same time.  Neither side touches the other's rows: a top row couples to rows
// <= k+1 and a bottom row to rows >= k, so both only update the 2x2 block of the middle pair
// (k, k+1), and A - sigma = P diag(D_top, M, D_bottom) P^T.  Each side runs the recurrence of the
// LDL^T pivots over its own rows, with u_i = l_i d_i:
//   d_i = (a_i - sigma) - u_{i-1}^2 / d_{i-1} - c^2 / d_{i-2},   u_i = b - c u_{i-1} / d_{i-1},
// read with stride st = +1 from the side's first row or st = -1; the inertia of A - sigma is that of the
// pivots plus that of M.
struct Side {
  double r1, r2, u1;  // 1/d of the side's last two pivots, Schur off-diagonal u of its last row
  int neg;            // negative pivots
};

// Sturm count of one side (rows >= 0 rows, a = the side's first row).  The diagonal is read 8 entries at a time so the
// LDS latency is paid once per chunk.
QEX_HD inline Side sturm_side(const double* __restrict__ a, int st, int rows, double b, double c, double sigma) {
  const double nc2 = -c * c, nc = -c;
  double rm1 = 0.0, rm2 = 0.0, um1 = 0.0;
  int cnt = 0;
  auto step = [&](double ai) {
    const double p = fma(nc2, rm2, ai - sigma);
    const double d = fma(-um1 * um1, rm1, p);
    cnt += sign_bit(d);
    const double u = fma(nc * rm1, um1, b);
    rm2 = rm1;
    rm1 = rcp_clamped(d);
    um1 = u;
  };
  int i = 0;
  for (; i + 8 <= rows; i += 8) {
    double av[8];
#pragma unroll
    for (int q = 0; q < 8; ++q) av[q] = a[st * (i + q)];
#pragma unroll
    for (int q = 0; q < 8; ++q) step(av[q]);
  }
  for (; i < rows; ++i) step(a[st * i]);
  return Side{rm1, rm2, um1, cnt};
}

// The middle block M of the pair (k, k+1) from the two sides; ak, ak1 = diagonal of rows k, k+1.
QEX_HD inline void middle_block(const Side& t, const Side& u, double ak, double ak1, double b, double c, double sigma,
                                double& m00, double& m01, double& m11) {
  const double c2 = c * c;
  m00 = (ak - sigma) - t.u1 * t.u1 * t.r1 - c2 * t.r2 - c2 * u.r1;
  m11 = (ak1 - sigma) - c2 * t.r1 - u.u1 * u.u1 * u.r1 - c2 * u.r2;
  m01 = b - c * t.u1 * t.r1 - c * u.u1 * u.r1;
}

// Number of eigenvalues below sigma from the two sides and the inertia of M.
QEX_HD inline int sturm_join(const Side& t, const Side& u, double ak, double ak1, double b, double c, double sigma) {
  double m00, m01, m11;
  middle_block(t, u, ak, ak1, b, c, sigma, m00, m01, m11);
  const double det = m00 * m11 - m01 * m01;
  const int neg = det < 0.0 ? 1 : (det > 0.0 ? (m00 < 0.0 ? 2 : 0) : (m00 + m11 < 0.0 ? 1 : 0));
  return t.neg + u.neg + neg;
}

// Forward state of one side of a solve: the Side of the factorisation plus the multipliers and
// forward-solve values of its last two rows, which enter the middle right-hand side.
struct SideZ {
  Side s;
  double l1, m1, m2, z1, z2;  // l, m of the last row, m of the row before; z of the last two rows
};

// Solve of the middle pair: M [x_k, x_k+1] = [y_k, y_k+1] minus both sides' forward terms, M by
// a 2x2 LDL^T with the pivots clamped to +-tiny like the sides' pivots.
QEX_HD inline void middle_solve(const Side& t, const Side& u, const SideZ& zt, const SideZ& zu, double ak, double ak1,
                                double yk, double yk1, double b, double c, double sigma, double tiny, double& xk,
                                double& xk1) {
  double m00, m01, m11;
  middle_block(t, u, ak, ak1, b, c, sigma, m00, m01, m11);
  const double r0 = yk - (zt.l1 * zt.z1 + zt.m2 * zt.z2) - zu.m1 * zu.z1;
  const double r1 = yk1 - zt.m1 * zt.z1 - (zu.l1 * zu.z1 + zu.m2 * zu.z2);
  double p0 = m00;
  if (fabs(p0) < tiny) p0 = p0 < 0.0 ? -tiny : tiny;
  const double l = m01 / p0;
  double p1 = m11 - l * m01;
  if (fabs(p1) < tiny) p1 = p1 < 0.0 ? -tiny : tiny;
  xk1 = (r1 - l * r0) / p1;
  xk = r0 / p0 - l * xk1;
}

// One thread: y <- (A - sigma)^-1 y by Gaussian elimination with partial pivoting (bandwidth 2,
// fill to 4).  The three active rows (columns i .. i + 4) are in registers; each finished row of U (5 entries)
// goes to R and its right-hand side to y, then the back substitution.  Pivots below tiny become +-tiny.
// (k_adj_eig falls back to it.)
QEX_HD __attribute__((noinline)) inline void pivoted_solve(const double* a, double* y, double* R, int N, double b, double c, double sigma,
                                                           double tiny) {
  auto band = [&](int row, int col) -> double {  // entry of A - sigma (zero outside the matrix)
    if (row >= N || col < 0 || col >= N) return 0.0;
    const int d = col - row;
    return d == 0 ? a[row] - sigma : (d == 1 || d == -1) ? b : (d == 2 || d == -2) ? c : 0.0;
  };
  double r0[5], r1[5], r2[5];
  for (int c = 0; c < 5; ++c) {
    r0[c] = band(0, c);
    r1[c] = band(1, c);
    r2[c] = band(2, c);
  }
  double y0 = y[0], y1 = N > 1 ? y[1] : 0.0, y2 = N > 2 ? y[2] : 0.0;
  for (int i = 0; i < N; ++i) {
    // pivot among the (existing) rows i, i+1, i+2 in column i
    int pr = 0;
    double best = fabs(r0[0]);
    if (i + 1 < N && fabs(r1[0]) > best) {
      best = fabs(r1[0]);
      pr = 1;
    }
    if (i + 2 < N && fabs(r2[0]) > best) pr = 2;
    if (pr == 1) {
      for (int c = 0; c < 5; ++c) {
        const double t1 = r0[c];
        r0[c] = r1[c];
        r1[c] = t1;
      }
      const double ty = y0;
      y0 = y1;
      y1 = ty;
    } else if (pr == 2) {
      for (int c = 0; c < 5; ++c) {
        const double t1 = r0[c];
        r0[c] = r2[c];
        r2[c] = t1;
      }
      const double ty = y0;
      y0 = y2;
      y2 = ty;
    }
    if (fabs(r0[0]) < tiny) r0[0] = r0[0] < 0.0 ? -tiny : tiny;
    const double ip = 1.0 / r0[0];
    const double l1 = r1[0] * ip, l2 = r2[0] * ip;
    for (int c = 1; c < 5; ++c) {
      r1[c] = fma(-l1, r0[c], r1[c]);
      r2[c] = fma(-l2, r0[c], r2[c]);
    }
    y1 = fma(-l1, y0, y1);
    y2 = fma(-l2, y0, y2);
    for (int c = 0; c < 5; ++c) R[(size_t)i * 5 + c] = r0[c];
    y[i] = y0;
    // advance: rows i+1, i+2 shift one column left; row i+3 enters
    for (int c = 0; c < 4; ++c) {
      r0[c] = r1[c + 1];
      r1[c] = r2[c + 1];
    }
    r0[4] = 0.0;
    r1[4] = 0.0;
    for (int c = 0; c < 5; ++c) r2[c] = band(i + 3, i + 1 + c);
    y0 = y1;
    y1 = y2;
    y2 = i + 3 < N ? y[i + 3] : 0.0;
  }
  for (int i = N - 1; i >= 0; --i) {
    double v = y[i];
    for (int c = 1; c < 5 && i + c < N; ++c) v = fma(-R[(size_t)i * 5 + c], y[i + c], v);
    y[i] = v / R[(size_t)i * 5];
  }
}

}  // namespace qexband
