// eigen1d.h -- what one workgroup does for one eigenpair of the 1D Kohn-Sham operator (k_eigen in qex1d.hip): the
// eigenvalue by Rayleigh-quotient steps of one wave, the multisection bracket, and the two twisted
// inverse-iteration solves.
#pragma once
#include "band_wave.h"

namespace qexband {

constexpr double EPS = 2.220446049250313e-16;

template <int CTRL>
__device__ __forceinline__ double dpp_f64(double x) {
  const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(x), CTRL, 0xf, 0xf, false);
  const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(x), CTRL, 0xf, 0xf, false);
  return __hiloint2double(hi, lo);
}

__device__ __forceinline__ double read_lane(double x, int l) {
  return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(x), l),
                          __builtin_amdgcn_readlane(__double2loint(x), l));
}

// Sum over the 64 lanes (all active), the same value in every lane: DPP moves within each row of
// 16 lanes (pairs, quads, half-row mirror, row mirror), then the four row sums in a fixed order.
__device__ __forceinline__ double wave_sum(double x) {
  x += dpp_f64<0xB1>(x);   // quad_perm [1, 0, 3, 2]
  x += dpp_f64<0x4E>(x);   // quad_perm [2, 3, 0, 1]
  x += dpp_f64<0x141>(x);  // row_half_mirror
  x += dpp_f64<0x140>(x);  // row_mirror
  return (read_lane(x, 0) + read_lane(x, 16)) + (read_lane(x, 32) + read_lane(x, 48));
}

// The same where every lane needs the very same bits (control flow): not contracted, since a product fused
// into its own lane's first addition, but rounded on its way to the others, would make the lanes' sums differ.
__device__ __forceinline__ double wave_sum_same(double x) {
#pragma clang fp contract(off)
  x += dpp_f64<0xB1>(x);
  x += dpp_f64<0x4E>(x);
  x += dpp_f64<0x141>(x);
  x += dpp_f64<0x140>(x);
  return (read_lane(x, 0) + read_lane(x, 16)) + (read_lane(x, 32) + read_lane(x, 48));
}

// y <- (A - sigma)^-1 y / |.| on one wave
__device__ __forceinline__ void inverse_step(const double* a, double* y, double* F, int N, double b, double c, double sigma) {
  const int m = wave_rows(N), r0 = (threadIdx.x & 63) * m, r1 = min(N, r0 + m);
  wave_solve<true>(a, y, N, b, c, sigma, F);
  double n2 = 0.0;
  for (int i = r0; i < r1; ++i) n2 = fma(y[i], y[i], n2);
  const double sc = 1.0 / sqrt(wave_sum_same(n2));
  for (int i = r0; i < r1; ++i) y[i] *= sc;
  wave_lds_order();
}

// An eigenvalue by Rayleigh-quotient iteration on one wave (all 64 lanes) from the vector in y, until the residual
// |A y - rho y| is 1e-8; the quotient's error is the residual's square over the gap to the next eigenvalue.
//   near: at most 3 solves, the first with y's own quotient as shift.  Of a pair closer than 2e-8 any mixture has
//     such a residual, and another eigenvalue may be nearer: confirm_side has to say that it is the j-th.
//   else: [slo, shi] is known to hold the j-th eigenvalue and no other, with the neighbours well away; the shift
//     is its middle until the quotient lies inside.
// false if that does not end; the caller brackets the eigenvalue further.
__device__ bool refine_eigenvalue(const double* a, double* y, double* F, int N, double b, double c, double slo, double shi,
                                  bool near, double* rho_out) {
  const int m = wave_rows(N), r0 = (threadIdx.x & 63) * m, r1 = min(N, r0 + m);
  auto hy = [&](int i) {
    double v = a[i] * y[i];
    if (i >= 1) v = fma(b, y[i - 1], v);
    if (i + 1 < N) v = fma(b, y[i + 1], v);
    if (i >= 2) v = fma(c, y[i - 2], v);
    if (i + 2 < N) v = fma(c, y[i + 2], v);
    return v;
  };
  auto quotient = [&]() {
    double q = 0.0;
    for (int i = r0; i < r1; ++i) q = fma(y[i], hy(i), q);
    return wave_sum_same(q);
  };
  double sigma = near ? quotient() : 0.5 * (slo + shi);
  for (int it = 0; it < (near ? 3 : 6); ++it) {
    inverse_step(a, y, F, N, b, c, sigma);
    const double rho = quotient();
    if (rho >= slo && rho <= shi) {
      double r2 = 0.0;
      for (int i = r0; i < r1; ++i) {
        const double d = fma(-rho, y[i], hy(i));
        r2 = fma(d, d, r2);
      }
      if (wave_sum_same(r2) <= 1e-16 * fmax(1.0, rho * rho)) {
        *rho_out = rho;
        return true;
      }
      sigma = rho;
    }
  }
  return false;
}

// One side of "the j-th eigenvalue lies within tau of rho", by the number of eigenvalues below rho + tau (above)
// or rho - tau; a wave.  tau is the quotient's error at a gap of 1e-5 and the rounding of a count.
__device__ __forceinline__ bool confirm_side(const double* a, double* F, int N, double b, double c, double hnorm, int j,
                                             double rho, bool above) {
  const double tau = 1e-11 * fmax(1.0, fabs(rho)) + 64.0 * EPS * hnorm;
  return wave_solve<false>(a, nullptr, N, b, c, above ? rho + tau : rho - tau, F) == j + (above ? 1 : 0);
}

// Multisection bracket of the j-th eigenvalue: NS shifts per round, both ends included; first = index of the
// first shift with more than j eigenvalues below it (NS: none).
struct Bracket {
  double lo, hi, gl, gu;
  __device__ __forceinline__ double step(int NS) const { return (hi - lo) / (double)(NS - 1); }
  __device__ __forceinline__ double shift(int me, int NS, double st) const { return me == NS - 1 ? hi : fma((double)me, st, lo); }
  __device__ __forceinline__ bool small(double hnorm) const {
    return hi - lo <= 1e-9 * fmax(1.0, fabs(0.5 * (lo + hi))) + 64.0 * EPS * hnorm;
  }
  // the next bracket; false if it does not change (rounding floor).  An eigenvalue outside: the adjacent
  // interval 256 times as wide (clipped to the Gershgorin bounds), so a missed warm start costs about one round
  __device__ __forceinline__ bool narrow(int first, int NS, double st) {
    const double wide = 256.0 * (hi - lo);
    double nlo, nhi;
    if (first == 0) {
      nhi = lo;
      nlo = fmax(gl, lo - wide);
      if (!(nlo < lo)) nlo = lo > gl ? gl : lo;
    } else if (first == NS) {
      nlo = hi;
      nhi = fmin(gu, hi + wide);
      if (!(nhi > hi)) nhi = hi < gu ? gu : hi;
    } else {
      nlo = first - 1 == 0 ? lo : fma((double)(first - 1), st, lo);
      nhi = first == NS - 1 ? hi : fma((double)first, st, lo);
    }
    const bool moved = nlo != lo || nhi != hi;
    lo = nlo;
    hi = nhi;
    return moved;
  }
};

// Order of the rows for the two-sided chains: the top rows 0 .. kt - 1, the middle pair kt, kt + 1, then the bottom
// rows from N - 1 up to kt + 2, so that both sides walk forward (LDS reads at constant offsets from one
// address; with a per-lane direction every operand's address took its own instructions)
__device__ __forceinline__ int side_pos(int t, int N, int kt) { return t <= kt + 1 ? t : N + 1 + kt - t; }

// Inverse iteration without pivoting, by the whole workgroup: one LDL^T factorisation of A - sigma (L unit lower
// triangular with the multipliers l_i, m_i of a row's two neighbours; pivots below tiny act as +-tiny), twisted
// at rows kt, kt + 1 (the top rows eliminated downwards by lane 0, the bottom rows upwards by lane 1), and two
// solves from y, normalised after each; ap and y in the order of side_pos; sum(x) adds x over the workgroup.
// The recurrences are chains of what one wave can issue (7 cycles an instruction), so a chain carries only what
// it must: wave 0 factorises a chunk of rows (pivots r and off-diagonals u) while wave 1 forms the
// multipliers of the chunk before with all its lanes and runs the forward solve; z / d is a parallel pass;
// the back substitution is two FMAs a row.  A single wave doing all of it took 29 + 17 us at N = 513.
// F: 5 N doubles: (r, u) and (l, m) per row, z.
template <int NT, class Sum>
__device__ __forceinline__ void twisted_inverse_iteration(const double* ap, double* y, double* F, int N, int kt, double b,
                                                          double c, double sigma, double tiny, Sum sum) {
  constexpr int CH = 32;
  const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int kb = N - 2 - kt;
  double2* ru = reinterpret_cast<double2*>(F);
  double2* lm = ru + N;
  double* z = reinterpret_cast<double*>(lm + N);
  for (int t = tid; t < N; t += NT) z[t] = ap[t] - sigma;
  __syncthreads();
  // this lane's side: rows of them from position r0 on
  const bool bot = lane & 1;
  const int rows = bot ? kb : kt, r0 = bot ? kt + 2 : 0;
  const double c2 = c * c, rtiny = 1.0 / tiny;
  // forward solve of a row range: z_i = y_i - l_{i-1} z_{i-1} - m_{i-2} z_{i-2}
  double z1 = 0.0, z2 = 0.0, lm1 = 0.0, mm1 = 0.0, mm2 = 0.0;
  auto forward = [&](int i0, int i1) {
    auto step = [&](double* zp, double yi, double2 q) {
      const double zi = fma(-mm2, z2, fma(-lm1, z1, yi));
      *zp = zi;
      z2 = z1;
      z1 = zi;
      mm2 = mm1;
      mm1 = q.y;
      lm1 = q.x;
    };
    const double* yp = y + r0 + i0;
    const double2* qp = lm + r0 + i0;
    double* zp = z + r0 + i0;
    int n = i1 - i0;
    for (; n >= 8; n -= 8, yp += 8, qp += 8, zp += 8) {
      double yv[8];
      double2 qv[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        yv[u] = yp[u];
        qv[u] = qp[u];
      }
#pragma unroll
      for (int u = 0; u < 8; ++u) step(zp + u, yv[u], qv[u]);
    }
    for (; n > 0; --n, ++yp, ++qp, ++zp) step(zp, *yp, *qp);
  };
  double rm1 = 0.0, rm2 = 0.0, um1 = 0.0;
  auto factor = [&](int i0, int i1) {
    auto step = [&](double2* p, double as) {
      const double d = fma(-um1 * um1, rm1, fma(-c2, rm2, as));
      const double r = fmin(fmax(rcp64(d), -rtiny), rtiny);
      const double u = fma(-c * rm1, um1, b);
      *p = make_double2(r, u);
      rm2 = rm1;
      rm1 = r;
      um1 = u;
    };
    const double* zp = z + r0 + i0;
    double2* p = ru + r0 + i0;
    int n = i1 - i0;
    for (; n >= 8; n -= 8, zp += 8, p += 8) {
      double av[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) av[u] = zp[u];
#pragma unroll
      for (int u = 0; u < 8; ++u) step(p + u, av[u]);
    }
    for (; n > 0; --n, ++zp, ++p) step(p, *zp);
  };
  const int nch = (max(kt, kb) + CH - 1) / CH;
  for (int ch = 0; ch <= nch; ++ch) {
    if (wv == 0 && ch < nch) {
      if (lane < 2) factor(ch * CH, min(rows, ch * CH + CH));
    } else if (wv == 1 && ch > 0) {
      const int i = (ch - 1) * CH + (lane & (CH - 1));
      const bool lower = lane >= CH;
      if (i < (lower ? kb : kt)) {
        const int row = lower ? kt + 2 + i : i;
        const double2 q = ru[row];
        lm[row] = make_double2(q.y * q.x, c * q.x);
      }
      __builtin_amdgcn_wave_barrier();
      if (lane < 2) forward((ch - 1) * CH, min(rows, ch * CH));
    }
    __syncthreads();
  }
  for (int it = 0; it < 2; ++it) {
    // the middle pair, by every thread: the state of both sides from their last two rows
    double xk, xk1;
    {
      auto side = [&](int n, int e0) {
        SideZ q{};
        if (n >= 1) {
          const double2 p = ru[e0 + n - 1], w = lm[e0 + n - 1];
          q.s.r1 = p.x;
          q.s.u1 = p.y;
          q.l1 = w.x;
          q.m1 = w.y;
          q.z1 = z[e0 + n - 1];
        }
        if (n >= 2) {
          q.s.r2 = ru[e0 + n - 2].x;
          q.m2 = lm[e0 + n - 2].y;
          q.z2 = z[e0 + n - 2];
        }
        return q;
      };
      const SideZ zt = side(kt, 0), zb = side(kb, kt + 2);
      middle_solve(zt.s, zb.s, zt, zb, ap[kt], ap[kt + 1], y[kt], y[kt + 1], b, c, sigma, tiny, xk, xk1);
    }
    __syncthreads();
    for (int t = tid; t < N; t += NT)
      if (t < kt || t > kt + 1) z[t] *= ru[t].x;  // z / d
    __syncthreads();
    if (tid < 2) {
      // back substitution of a side toward its outer end
      double x1 = bot ? xk1 : xk, x2 = bot ? xk : xk1;
      auto step = [&](double* yp, double w, double2 q) {
        const double xi = fma(-q.y, x2, fma(-q.x, x1, w));
        *yp = xi;
        x2 = x1;
        x1 = xi;
      };
      int n = rows;
      double* yp = y + r0 + n - 8;
      const double* wp = z + r0 + n - 8;
      const double2* qp = lm + r0 + n - 8;
      for (; n >= 8; n -= 8, yp -= 8, wp -= 8, qp -= 8) {
        double w8[8];
        double2 qv[8];
#pragma unroll
        for (int u = 7; u >= 0; --u) {
          w8[u] = wp[u];
          qv[u] = qp[u];
        }
#pragma unroll
        for (int u = 7; u >= 0; --u) step(yp + u, w8[u], qv[u]);
      }
      for (; n > 0; --n) step(y + r0 + n - 1, z[r0 + n - 1], lm[r0 + n - 1]);
      if (tid == 0) {
        y[kt] = xk;
        y[kt + 1] = xk1;
      }
    }
    __syncthreads();
    double nrm = 0.0;
    for (int t = tid; t < N; t += NT) {
      const double x = y[side_pos(t, N, kt)];
      nrm = fma(x, x, nrm);
    }
    const double sc = 1.0 / sqrt(sum(nrm));
    for (int t = tid; t < N; t += NT) y[t] *= sc;
    __syncthreads();
    if (it == 0) {
      z1 = z2 = lm1 = mm1 = mm2 = 0.0;
      if (tid < 2) forward(0, rows);
      __syncthreads();
    }
  }
}

}  // namespace qexband
