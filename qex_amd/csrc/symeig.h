// symeig.h -- dense symmetric eigensolver for one workgroup (n <= 96, FP64).
//
//   1. Householder tridiagonalisation with the matrix in registers (each thread a cyclic patch): for
//      k = 0..n-3 the reflector H_k = I - tau v v^T annihilates column k below the subdiagonal; the
//      trailing block becomes A - v w^T - w v^T with p = tau A v, w = p - (tau / 2)(v^T p) v.  d / e collect
//      the tridiagonal.
//   2. T, scaled by a power of two to norm 1..2, splits into unreduced blocks where
//      |e_k| <= eps (|d_k| + |d_k+1|).
//   3. Eigenvalues: multisection on Sturm counts (sign changes of the leading minors of T - x), three
//      lanes per eigenvalue, a fixed number of rounds (interval / 7 per round).
//   4. Eigenvectors of T: two inverse iterations (LDL^T pivots of T - lam, pivots smaller than
//      eps |T| replaced by +-eps |T|) from a fixed pseudo-random start, two lanes per vector; eigenvalues
//      of one block closer than 1e-5 |T| form a cluster, whose vectors are orthogonalised after every
//      solve.  Rayleigh quotients give the eigenvalues.
//   5. Ascending sort and back-transformation Z <- H_0 ... H_{n-3} Y, four lanes per column.
// All reductions run in a fixed order: the result does not depend on timing.
//
// What bounds it: every stage is a chain of dependent steps of one workgroup, so its time is
// barriers and latencies, not arithmetic.  Hence the matrix stays in registers (one barrier and a
// few LDS words per Householder step; the LDS-resident form took three barriers over 16 waves and
// re-read the block), the counts need no reciprocal and no barrier, and a column of the
// back-transformation stays in four lanes' registers from the first reflector to the last.
#pragma once
#include <hip/hip_runtime.h>
#include <math.h>

namespace qexeig {

constexpr double EPS = 2.220446049250313e-16;
constexpr int MAXN = 96;
// eigenvalues of a block closer than CLUSTER |T| are orthogonalised against each other: two inverse
// iterations leave vectors eps / gap apart from orthogonal, 1e-11 at this gap
constexpr double CLUSTER = 1e-5;
constexpr int NT_MIN = 512;  // threads the solver needs (it uses the first 512 of the workgroup)

// f(0), ..., f(N - 1) with compile-time indices (register arrays stay in registers)
template <int I>
struct Index {
  static constexpr int value = I;
};
template <int I, int N, class F>
__device__ __forceinline__ void static_for(F&& f) {
  if constexpr (I < N) {
    f(Index<I>{});
    static_for<I + 1, N>(f);
  }
}

// one DPP move of a double (both halves)
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

// Sum over the 64 lanes (all active), the same value in every lane: DPP within each row of 16
// lanes (pairs, quads, half-row mirror, row mirror), then the four row sums in a fixed order.
// No contraction in these sums: a product fused into its lane's first addition, but rounded on its way to
// the neighbour, would make the lanes' sums differ.
__device__ __forceinline__ double wave_sum(double x) {
#pragma clang fp contract(off)
  x += dpp_f64<0xB1>(x);   // quad_perm [1, 0, 3, 2]
  x += dpp_f64<0x4E>(x);   // quad_perm [2, 3, 0, 1]
  x += dpp_f64<0x141>(x);  // row_half_mirror
  x += dpp_f64<0x140>(x);  // row_mirror
  return (read_lane(x, 0) + read_lane(x, 16)) + (read_lane(x, 32) + read_lane(x, 48));
}

__device__ __forceinline__ double wave_max(double x) {
  x = fmax(x, dpp_f64<0xB1>(x));
  x = fmax(x, dpp_f64<0x4E>(x));
  x = fmax(x, dpp_f64<0x141>(x));
  x = fmax(x, dpp_f64<0x140>(x));
  return fmax(fmax(read_lane(x, 0), read_lane(x, 16)), fmax(read_lane(x, 32), read_lane(x, 48)));
}

// sum over an aligned group of 4 / 8 lanes, the same value in each of them
__device__ __forceinline__ double group4_sum(double x) {
#pragma clang fp contract(off)
  x += dpp_f64<0xB1>(x);
  x += dpp_f64<0x4E>(x);
  return x;
}
__device__ __forceinline__ double group8_sum(double x) {
#pragma clang fp contract(off)
  x = group4_sum(x);
  x += dpp_f64<0x141>(x);
  return x;
}

// Shared state of the solver (static LDS besides the two n x S matrices).
struct Smem {
  double d[MAXN], e[MAXN], lam[MAXN], rq[MAXN], tau[MAXN], nv[MAXN];
  double p[2][MAXN + 40], col[2][MAXN + 40];  // exchanged per step (alternating): p = tau A v and a column of A
  double2 de[MAXN + 8];              // (d_i, e_{i-1}^2) for the Sturm counts
  int bs[MAXN], bt[MAXN], perm[MAXN];
  unsigned long long cut[2];
  unsigned char need[MAXN];  // slot's vector wanted (nvec < n: its eigenvalue ranks below nvec)
};

// 1/d: hardware reciprocal refined by one Newton step (relative error ~1e-15)
__device__ __forceinline__ double rcp_nr(double d) {
  const double r = __builtin_amdgcn_rcp(d);
  return fma(r, fma(-d, r, 1.0), r);
}

// Running minors of T - x, p_i = (d_i - x) p_{i-1} - e_{i-1}^2 p_{i-2}, whose sign changes count the
// eigenvalues below x.  No division, so a row is one dependent FMA (a pivot recurrence has a reciprocal, a
// Newton step and two clamps in the chain).  T is scaled to norm 1..2 and e^2 floored at 1e-60, so 8 rows
// change a minor by less than 1e-250 .. 1e6 and two neighbouring minors never vanish together;
// rescale() divides both by a power of two every 8 rows.
struct Minors {
  double p0 = 0.0, p1 = 1.0;
  unsigned bits = 0;
  __device__ __forceinline__ void step(double2 de, double x) {
    const double pn = fma(de.x - x, p1, -(de.y * p0));
    p0 = p1;
    p1 = pn;
    bits = __builtin_amdgcn_alignbit(bits, (unsigned)__double2hiint(pn), 31);  // bits << 1 | sign
  }
  // sign changes of the last m <= 16 rows
  __device__ __forceinline__ int changes(int m) const { return __popc((bits ^ (bits >> 1)) & ((1u << m) - 1u)); }
  __device__ __forceinline__ void rescale() {
    const int ex = -__builtin_amdgcn_frexp_exp(fmax(fabs(p0), fabs(p1)));
    p0 = ldexp(p0, ex);
    p1 = ldexp(p1, ex);
  }
};

// eigenvalues of rows s..t-1 of T below x and below y, (d_i, e_{i-1}^2) in LDS.  Two shifts a lane: one leaves
// the pipeline idle between dependent operations and reads LDS for half the arithmetic.
__device__ __forceinline__ int2 sturm_count2(const double2* de, int s, int t, double x, double y) {
  Minors m, l;
  int2 c = make_int2(0, 0);
  int j = s;
  for (; j + 8 <= t; j += 8) {
    double2 v[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) v[u] = de[j + u];
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      m.step(v[u], x);
      l.step(v[u], y);
    }
    c.x += m.changes(8);
    c.y += l.changes(8);
    m.rescale();
    l.rescale();
  }
  const int left = t - j;
  for (; j < t; ++j) {
    m.step(de[j], x);
    l.step(de[j], y);
  }
  return make_int2(c.x + m.changes(left), c.y + l.changes(left));
}

// deterministic start vector entry in [-1, 1)
__device__ __forceinline__ double start_entry(int slot, int i) {
  unsigned x = 2654435761u * (unsigned)(slot + 1) ^ (40503u * (unsigned)(i + 7));
  x ^= x >> 13;
  x *= 0x5bd1e995u;
  x ^= x >> 15;
  return (double)(x & 0xFFFFFF) / 8388608.0 - 1.0;
}

// A pair of lanes: column `col` of Y <- (T_block - lam)^-1 b, rows s..t-1.  The even lane eliminates from
// the top, the odd one (bot) from the bottom, to the row h = (s + t) / 2, which they solve together; each
// then substitutes back outward over its own half (half the dependent chain of a one-sided solve).  The
// inverse pivots 1/D_i (|1/D| <= rmax) are kept in column `col` of Dm.  FIRST: b is the start vector, and the
// pivots are computed along with the elimination; else b = scale * Y and the pivots are read.  Returns
// |x|^2 in both lanes.  The operands of 8 rows are in flight per LDS wait.
template <bool FIRST>
__device__ __forceinline__ double ldl_solve(const double* d, const double* e, int s, int t, bool bot, double lam,
                                            double rmax, double* Dm, double* Y, int S, int col, double scale) {
  const int h = (s + t) >> 1, m = bot ? t - 1 - h : h - s;  // rows of this side
  const int i0 = bot ? t - 1 : s, st = bot ? -1 : 1;
  const double* ec = bot ? e - 1 : e;  // ec[i] couples row i to its neighbour toward h
  double y = 0.0, qi = 0.0, ep = 0.0;
  auto fwd = [&](int i, double di, double ei, double bi, double ri) {
    // l = e / D of the row before; D_i = d_i - lam - e l; y_i = b_i - l y
    const double l = ep * qi;
    y = fma(-l, y, bi);
    if (FIRST) {
      qi = fmin(fmax(rcp_nr(fma(-ep, l, di - lam)), -rmax), rmax);
      Dm[i * S + col] = qi;
    } else {
      qi = ri;
    }
    Y[i * S + col] = y;
    ep = ei;
  };
  int k = 0;
  for (; k + 8 <= m; k += 8) {
    double dv[8], ev[8], bv[8], rv[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const int i = i0 + st * (k + u);
      ev[u] = ec[i];
      dv[u] = FIRST ? d[i] : 0.0;
      bv[u] = FIRST ? start_entry(col, i) : scale * Y[i * S + col];
      rv[u] = FIRST ? 0.0 : Dm[i * S + col];
    }
#pragma unroll
    for (int u = 0; u < 8; ++u) fwd(i0 + st * (k + u), dv[u], ev[u], bv[u], rv[u]);
  }
  for (; k < m; ++k) {
    const int i = i0 + st * k;
    fwd(i, FIRST ? d[i] : 0.0, ec[i], FIRST ? start_entry(col, i) : scale * Y[i * S + col], FIRST ? 0.0 : Dm[i * S + col]);
  }
  // row h, in both lanes (a side without rows contributes l = 0)
  const double l = ep * qi, el = ep * l, ly = l * y;
  const double bh = FIRST ? start_entry(col, h) : scale * Y[h * S + col];  // (read before the exchange: one lane then writes it)
  const double elo = dpp_f64<0xB1>(el), lyo = dpp_f64<0xB1>(ly);
  const double qh = FIRST ? fmin(fmax(rcp_nr((d[h] - lam) - (bot ? elo + el : el + elo)), -rmax), rmax) : Dm[h * S + col];
  double x = (bh - (bot ? lyo + ly : ly + lyo)) * qh;
  double n0 = bot ? 0.0 : x * x;
  if (!bot) {
    if (FIRST) Dm[h * S + col] = qh;
    Y[h * S + col] = x;
  }
  // outward: x_i = y_i / D_i - (e / D_i) x of the row toward h
  k = m - 1;
  for (; k - 7 >= 0; k -= 8) {
    double yv[8], lv[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const int i = i0 + st * (k - u);
      const double r = Dm[i * S + col];
      yv[u] = Y[i * S + col] * r;
      lv[u] = ec[i] * r;
    }
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      x = fma(-lv[u], x, yv[u]);
      n0 = fma(x, x, n0);
      Y[(i0 + st * (k - u)) * S + col] = x;
    }
  }
  for (; k >= 0; --k) {
    const int i = i0 + st * k;
    const double r = Dm[i * S + col];
    x = fma(-(ec[i] * r), x, Y[i * S + col] * r);
    n0 = fma(x, x, n0);
    Y[i * S + col] = x;
  }
  return n0 + dpp_f64<0xB1>(n0);
}

// 1/sqrt(d) to double precision (NaN for d <= 0)
__device__ __forceinline__ double rsqrt_nr(double d) {
  double y = __builtin_amdgcn_rsq(d);
  y = fma(y, fma(-0.5 * d * y, y, 0.5), y);
  return fma(y, fma(-0.5 * d * y, y, 0.5), y);
}

// exponent of the power of two above |x| (0 for 0, infinities and NaN), where 2^-exponent is a normal number
__device__ __forceinline__ int exponent(double x) {
  const int ex = x > 0.0 ? __builtin_amdgcn_frexp_exp(x) : 0;
  return min(max(ex, -1000), 1000);
}

// Householder tridiagonalisation of A (n x n in LDS, row stride S).  NC >= ceil(n / 8).
// Thread (r, c) = (tid / 8, tid % 8) of 512 holds A[r + 64 i][c + 8 j] in registers: row sums cross 8
// lanes (three DPP steps), and two waves per SIMD fill each other's dependency stalls (four waves of
// 32 x 8 patches: 1.03 us a step at n = 80, bound by the instructions one wave issues).  One barrier per
// step: every thread keeps the column x being reduced for its rows and columns; its rows of p = tau A v
// and column q of A as it still is go to LDS together, and after the barrier every thread forms its part
// of the updated column q, the next x, itself.  Row k of V (stride 8 NC, zero padded, over A's own LDS)
// receives v_k; sh.d, sh.e, sh.tau the rest.
// A is scaled by a power of two to a largest element of 1/2 .. 1, and a column whose squared norm below the subdiagonal is
// under TAIL is taken as reduced: with both, the squares and tau = 2 / |v|^2 neither overflow nor underflow,
// whatever A's norm and however weakly its blocks are coupled.  Returns the exponent: T is that of A / 2^ex.
constexpr double TAIL = 1e-280;
template <int NC>
__device__ __forceinline__ int tridiagonalise(int n, double* A, int S, Smem& sh) {
  constexpr int NR = (NC + 7) / 8, SP = 8 * NC;
  const int tid = threadIdx.x, r = tid >> 3, c = tid & 7;
  double a[NR][NC];
#pragma unroll
  for (int i = 0; i < NR; ++i)
#pragma unroll
    for (int j = 0; j < NC; ++j) {
      const int row = r + 64 * i, col = c + 8 * j;
      a[i][j] = row < n && col < n ? A[row * S + col] : 0.0;
    }
  // x = column 0 below the diagonal, at this thread's columns, rows and at row q = 1
  double xc[NC], xr[NR], x0 = A[S];
#pragma unroll
  for (int j = 0; j < NC; ++j) {
    const int col = c + 8 * j;
    xc[j] = col >= 1 && col < n ? A[col * S] : 0.0;
  }
#pragma unroll
  for (int i = 0; i < NR; ++i) {
    const int row = r + 64 * i;
    xr[i] = row >= 1 && row < n ? A[row * S] : 0.0;
  }
  double amax = 0.0;
#pragma unroll
  for (int i = 0; i < NR; ++i)
#pragma unroll
    for (int j = 0; j < NC; ++j) amax = fmax(amax, fabs(a[i][j]));
  amax = wave_max(amax);
  if ((tid & 63) == 0) sh.nv[tid >> 6] = amax;
  __syncthreads();  // A is in registers; its LDS takes V
#pragma unroll
  for (int k = 0; k < NT_MIN / 64; ++k) amax = fmax(amax, sh.nv[k]);
  const int ex = exponent(amax);
  const double scale = ldexp(1.0, -ex);
#pragma unroll
  for (int i = 0; i < NR; ++i) {
    xr[i] *= scale;
#pragma unroll
    for (int j = 0; j < NC; ++j) a[i][j] *= scale;
  }
#pragma unroll
  for (int j = 0; j < NC; ++j) xc[j] *= scale;
  x0 *= scale;
  if (tid == 0) sh.d[0] = a[0][0];
  static_for<0, NC>([&](auto block) {
    constexpr int jb = decltype(block)::value, ib = jb / 8;
#pragma unroll 1
    for (int c0 = 0; c0 < 8; ++c0) {
      const int q = 8 * jb + c0;  // reduces column q - 1 to rows <= q
      if (q < 1) continue;
      if (q > n - 2) break;
      double* pb = sh.p[q & 1];
      double* ab = sh.col[q & 1];
      double* vrow = A + (size_t)(q - 1) * SP;
      double tail;
      {
        const double t = c == c0 ? 0.0 : xc[jb];
        tail = t * t;
#pragma unroll
        for (int j = jb + 1; j < NC; ++j) tail = fma(xc[j], xc[j], tail);
      }
      tail = group8_sum(tail);
      const bool skip = !(tail > TAIL);
      const double s2 = fma(x0, x0, tail), nx = s2 * rsqrt_nr(s2);
      const double alpha = x0 >= 0.0 ? -nx : nx;
      const double v0 = skip ? 0.0 : x0 - alpha;
      const double tau = skip ? 0.0 : rcp_nr(nx * (nx + fabs(x0)));
      double u[NR];
#pragma unroll
      for (int i = ib; i < NR; ++i) {
        u[i] = 0.0;
#pragma unroll
        for (int j = jb + 1; j < NC; ++j) u[i] = fma(a[i][j], xc[j], u[i]);
      }
      if (c == c0) xc[jb] = v0;  // x becomes v
      if (r == (q & 63)) xr[ib] = v0;
#pragma unroll
      for (int i = ib; i < NR; ++i) u[i] = tau * group8_sum(fma(a[i][jb], xc[jb], u[i]));
      if (c == c0) {
#pragma unroll
        for (int i = 0; i < NR; ++i) {
          const int row = r + 64 * i;
          if (row < 8 * NC) {
            if (i >= ib) {
              pb[row] = u[i];
              ab[row] = a[i][jb];
            }
            vrow[row] = i < ib ? 0.0 : xr[i];
          }
        }
      }
      if (tid == 0) {
        sh.e[q - 1] = skip ? x0 : alpha;
        sh.tau[q - 1] = tau;
      }
      __syncthreads();
      double wc[NC], nc[NC], nr[NR];
      const double pq = pb[q], pq1 = pb[q + 1], aq1 = ab[q + 1], vq1 = vrow[q + 1];
      double vp = 0.0;
#pragma unroll
      for (int j = jb; j < NC; ++j) {
        wc[j] = pb[c + 8 * j];
        nc[j] = ab[c + 8 * j];
        vp = fma(xc[j], wc[j], vp);
      }
#pragma unroll
      for (int i = ib; i < NR; ++i) nr[i] = ab[r + 64 * i];
      const double K = 0.5 * tau * group8_sum(vp);
      const double wq = fma(-K, v0, pq);
      if (tid == 0) sh.d[q] = fma(-v0, wq, fma(-wq, v0, ab[q]));
      x0 = fma(-vq1, wq, fma(-fma(-K, vq1, pq1), v0, aq1));
#pragma unroll
      for (int j = jb; j < NC; ++j) wc[j] = fma(-K, xc[j], wc[j]);
#pragma unroll
      for (int i = ib; i < NR; ++i) {
        const double wr = fma(-K, xr[i], u[i]);
#pragma unroll
        for (int j = jb; j < NC; ++j) a[i][j] = fma(-xr[i], wc[j], fma(-wr, xc[j], a[i][j]));
        xr[i] = fma(-xr[i], wq, fma(-wr, v0, nr[i]));
      }
      if (r + 64 * ib <= q) xr[ib] = 0.0;  // (rows of later blocks lie below q)
#pragma unroll
      for (int j = jb; j < NC; ++j) xc[j] = fma(-xc[j], wq, fma(-wc[j], v0, nc[j]));
      if (c <= c0) xc[jb] = 0.0;
    }
  });
  if (tid == 0) sh.e[n - 2] = x0;
#pragma unroll
  for (int i = 0; i < NR; ++i)
#pragma unroll
    for (int j = 0; j < NC; ++j)
      if (r + 64 * i == n - 1 && c + 8 * j == n - 1) sh.d[n - 1] = a[i][j];
  __syncthreads();
  return ex;
}

// X = L^-T (upper triangle, row-major n x n) of the Cholesky factorisation S = L L^T, both in registers: thread
// (r, c) of 32 x 8 holds the elements [r + 32 i][c + 8 j] (the other waves only take part in the barriers); step k eliminates below the diagonal of S and applies the same row operations to
// W = I, which ends as L^-1; column k of S and row k of W go to LDS, one barrier a step (a
// barrier and an LDS or L2 pass per division, column and update took 226 us from LDS, 450 us from L2).
template <int NC>
__device__ __forceinline__ void inverse_cholesky(int n, const double* Sm, double* X, Smem& sh) {
  constexpr int NR = (NC + 3) / 4;
  const int tid = threadIdx.x;
  if (__builtin_amdgcn_readfirstlane(tid >> 6) >= 4) {
    for (int k = 0; k <= n; ++k) __syncthreads();
    return;
  }
  const int r = tid >> 3, c = tid & 7;
  double a[NR][NC], w[NR][NC];
#pragma unroll
  for (int i = 0; i < NR; ++i)
#pragma unroll
    for (int j = 0; j < NC; ++j) {
      const int row = r + 32 * i, col = c + 8 * j;
      a[i][j] = row < n && col < n ? Sm[row * n + col] : 0.0;
      w[i][j] = row == col ? 1.0 : 0.0;
    }
  static_for<0, NC>([&](auto block) {
    constexpr int jb = decltype(block)::value, ib = jb / 4;
#pragma unroll 1
    for (int c0 = 0; c0 < 8; ++c0) {
      const int k = 8 * jb + c0;
      if (k >= n) break;
      double* cb = sh.col[k & 1];
      double* rb = sh.p[k & 1];
      if (c == c0) {
#pragma unroll
        for (int i = ib; i < NR; ++i) cb[r + 32 * i] = a[i][jb];
      }
      if (r == (k & 31)) {
#pragma unroll
        for (int j = 0; j <= jb; ++j) rb[c + 8 * j] = w[ib][j];
      }
      __syncthreads();
      const double rs = rsqrt_nr(cb[k]);
      double lc[NC], wk[NC];
#pragma unroll
      for (int j = jb; j < NC; ++j) lc[j] = cb[c + 8 * j] * rs;
#pragma unroll
      for (int j = 0; j <= jb; ++j) wk[j] = rb[c + 8 * j] * rs;
#pragma unroll
      for (int i = ib; i < NR; ++i) {
        const int row = r + 32 * i;
        const double lr = row > k ? cb[row] * rs : 0.0;
#pragma unroll
        for (int j = jb; j < NC; ++j) a[i][j] = fma(-lr, lc[j], a[i][j]);
#pragma unroll
        for (int j = 0; j <= jb; ++j) w[i][j] = row == k ? wk[j] : fma(-lr, wk[j], w[i][j]);
      }
    }
  });
#pragma unroll
  for (int i = 0; i < NR; ++i)
#pragma unroll
    for (int j = 0; j < NC; ++j) {
      const int row = r + 32 * i, col = c + 8 * j;
      if (row < n && col < n) X[col * n + row] = row >= col ? w[i][j] : 0.0;
    }
  __syncthreads();
}

// f<NC>() of the size class of n
template <class F>
__device__ __forceinline__ void by_size(int n, F&& f) {
  if (n <= 16)
    f(Index<2>{});
  else if (n <= 32)
    f(Index<4>{});
  else if (n <= 64)
    f(Index<8>{});
  else
    f(Index<12>{});
}

// Z <- H_0 ... H_{n-3} Y: column c of the result from column perm[c] of Y (in Z), scaled by nv.
// Four lanes hold a column, lane q the rows 8 i + 2 q + {0, 1}; the next reflector's LDS reads are in
// flight during the current one.  (Two columns per lane group halve those reads but leave three waves:
// 26 us against 20 at n = 80.)  V (n - 2 rows of stride 8 NC) is read into the LDS of both matrices once
// every column is in registers.
template <int NC>
__device__ __forceinline__ void back_transform(int n, int nvec, double* A, double* Z, int S, const double* f, Smem& sh) {
  constexpr int SP = 8 * NC;
  const int tid = threadIdx.x, nt = blockDim.x, c = tid >> 2, q4 = tid & 3;
  const bool act = c < nvec;
  double2 z[NC];
  {
    const int sl = act ? sh.perm[c] : 0;
    const double sc = act ? sh.nv[sl] : 0.0;
#pragma unroll
    for (int i = 0; i < NC; ++i) {
      const int row = 8 * i + 2 * q4;
      z[i].x = act && row < n ? sc * Z[row * S + sl] : 0.0;
      z[i].y = act && row + 1 < n ? sc * Z[(row + 1) * S + sl] : 0.0;
    }
  }
  __syncthreads();
  for (int idx = tid; idx < (n - 2) * SP; idx += nt) A[idx] = f[idx];
  __syncthreads();
  if (__builtin_amdgcn_readfirstlane(c & ~15) < nvec) {  // (16 columns a wave)
    static_for<0, NC>([&](auto block) {
      constexpr int jb = NC - 1 - decltype(block)::value;
      const int kt = min(8 * jb + 6, n - 3), kb = max(8 * jb - 1, 0);  // reflectors k with k + 1 in this block
      if (kt < kb) return;
      const double2* v = reinterpret_cast<const double2*>(A) + q4;
      double2 vn[NC], vv[NC];
#pragma unroll
      for (int i = jb; i < NC; ++i) vn[i] = v[kt * (SP / 2) + 4 * i];
      double tau_n = sh.tau[kt];
#pragma unroll 1
      for (int k = kt; k >= kb; --k) {
        const double tau = tau_n;
        const int kn = max(k - 1, kb);
        double s0 = 0.0, s1 = 0.0;
#pragma unroll
        for (int i = jb; i < NC; ++i) {
          vv[i] = vn[i];
          vn[i] = v[kn * (SP / 2) + 4 * i];
        }
        tau_n = sh.tau[kn];
#pragma unroll
        for (int i = jb; i < NC; ++i) {
          s0 = fma(vv[i].x, z[i].x, s0);
          s1 = fma(vv[i].y, z[i].y, s1);
        }
        const double s = tau * group4_sum(s0 + s1);
#pragma unroll
        for (int i = jb; i < NC; ++i) {
          z[i].x = fma(-s, vv[i].x, z[i].x);
          z[i].y = fma(-s, vv[i].y, z[i].y);
        }
      }
    });
  }
  __syncthreads();
  if (c < n) {
#pragma unroll
    for (int i = 0; i < NC; ++i) {
      const int row = 8 * i + 2 * q4;
      if (row < n) Z[row * S + c] = z[i].x;
      if (row + 1 < n) Z[(row + 1) * S + c] = z[i].y;
    }
  }
  __syncthreads();
}

// A: n x n symmetric in LDS (row stride S = n + 1, 16-byte aligned, destroyed), directly followed in LDS by
// Z: n x n output, column j = eigenvector of the j-th smallest eigenvalue; w: ascending eigenvalues (any
// memory).  f: global scratch of 3 n^2 doubles (the reflectors: (n - 2) 8 NC <= 3 n^2, and <= 2 n S of
// LDS, with NC = 2, 4, 8, 12 for n <= 16, 32, 64, 96).  Must be called by every thread of the workgroup
// (blockDim.x a multiple of 64, >= NT_MIN).
// nvec < n: only the eigenvectors of the nvec smallest eigenvalues (ranked by their multisection
// values, whole clusters) are computed and back-transformed, into columns 0..nvec-1 of Z, exactly as
// the full solve computes them (the other columns are zero); the other eigenvalues are the
// multisection values (not refined).
__device__ __forceinline__ void symeig(int n, double* A, double* Z, int S, double* w, double* f, Smem& sh,
                                       int nvec = 1 << 30) {
  if (nvec > n) nvec = n;
  const int tid = threadIdx.x, nt = blockDim.x, lane = tid & 63, wv = tid >> 6, nw = nt >> 6;
  if (n == 1) {
    if (tid == 0) {
      w[0] = A[0];
      Z[0] = 1.0;
    }
    __syncthreads();
    return;
  }
  // ---- 1. tridiagonalisation ----
  int ex = 0;  // T and the eigenvalues below are those of A / 2^ex
  by_size(n, [&](auto nc) {
    constexpr int NC = decltype(nc)::value;
    ex = tridiagonalise<NC>(n, A, S, sh);
    // V to scratch: the pivots of phase 4 take its place
    for (int idx = tid; idx < (n - 2) * 8 * NC; idx += nt) f[idx] = A[idx];
  });
  // ---- 2. norm, scaling, unreduced blocks ----
  double scale;  // a power of two
  {
    double nrm = 0.0;  // every wave by itself
    for (int i = lane; i < n; i += 64)
      nrm = fmax(nrm, fabs(sh.d[i]) + (i > 0 ? fabs(sh.e[i - 1]) : 0.0) + (i < n - 1 ? fabs(sh.e[i]) : 0.0));
    nrm = wave_max(nrm);
    const int et = nrm > 0.0 ? exponent(nrm) - 1 : 0;
    scale = ldexp(1.0, -et);
    ex += et;
  }
  __syncthreads();
  if (wv < 2) {
    const int k = tid;  // 0 .. 127
    double dk = 0.0, ek = 0.0;
    bool cut = false;
    if (k < n) {
      dk = sh.d[k] * scale;
      ek = k < n - 1 ? sh.e[k] * scale : 0.0;
      cut = k == n - 1 || fabs(ek) <= EPS * (fabs(dk) + fabs(sh.d[k + 1] * scale));
    }
    const unsigned long long m = __ballot(cut);
    if (lane == 0) sh.cut[wv] = m;
    if (k < n) {
      sh.lam[k] = cut ? 0.0 : ek;  // (parked until every d, e is read)
      sh.rq[k] = dk;
    }
  }
  __syncthreads();
  if (tid < n) {
    const int k = tid;
    const double ek = sh.lam[k], dk = sh.rq[k], em = k > 0 ? sh.lam[k - 1] : 0.0;
    sh.d[k] = dk;
    sh.e[k] = ek;
    sh.de[k] = make_double2(dk, fmax(em * em, 1e-60));
    const unsigned long long m0 = sh.cut[0], m1 = sh.cut[1];
    // block of row k: after the last cut below k, up to the first cut at or above k
    const unsigned long long b1 = k > 64 ? m1 & ((1ull << (k - 64)) - 1) : 0ull;
    const unsigned long long b0 = k < 64 ? m0 & ((1ull << k) - 1) : m0;
    sh.bs[k] = b1 ? 128 - __clzll((long long)b1) : b0 ? 64 - __clzll((long long)b0) : 0;
    const unsigned long long a0 = k < 64 ? m0 >> k : 0ull;
    const unsigned long long a1 = k < 64 ? m1 : m1 >> (k - 64);
    sh.bt[k] = a0 ? k + __ffsll((long long)a0) : (k < 64 ? 64 : k) + __ffsll((long long)a1);
  }
  __syncthreads();
  // ---- 3. eigenvalues by multisection: lanes 3 v .. 3 v + 2 of a wave for its slot v, no barriers ----
  // 7^-18 of a width <= 4: 2^-48 of the norm.  Three lanes of two shifts each: with n = 80 four waves, one
  // per SIMD (more lanes per eigenvalue share the SIMDs and gain fewer bits per unit of time).
  {
    const int v = lane / 3, g = lane - 3 * v, slot = wv * 21 + v;
    const bool act = v < 21 && slot < n;
    if (__any(act)) {
      double lo = 0.0, hi = 0.0;
      int s = 0, t = 0, li = 0;
      if (act) {
        s = sh.bs[slot];
        t = sh.bt[slot];
        li = slot - s;
        lo = 1e300;
        hi = -1e300;
        for (int j = s; j < t; ++j) {
          const double r = (j > s ? fabs(sh.e[j - 1]) : 0.0) + fabs(sh.e[j]);
          lo = fmin(lo, sh.d[j] - r);
          hi = fmax(hi, sh.d[j] + r);
        }
        const double span = fmax(hi - lo, EPS);
        lo -= 1e-12 * span;
        hi += 1e-12 * span;
      }
      for (int r = 0; r < 18; ++r) {
        const double wd = (hi - lo) * (1.0 / 7.0);
        const int2 c = act ? sturm_count2(sh.de, s, t, fma(wd, (double)(2 * g + 1), lo), fma(wd, (double)(2 * g + 2), lo))
                           : make_int2(0, 0);
        const unsigned long long m0 = __ballot(act && c.x <= li), m1 = __ballot(act && c.y <= li);
        const int below = __popcll((m0 >> (lane - g)) & 7ull) + __popcll((m1 >> (lane - g)) & 7ull);
        lo = fma(wd, (double)below, lo);
        hi = lo + wd;
      }
      if (act && g == 0) sh.lam[slot] = 0.5 * (lo + hi);
    }
  }
  __syncthreads();
  // wanted vectors: every slot when nvec = n; else the slots whose multisection value ranks below
  // nvec (ties by slot), and the rest of their clusters
  const double ctol = CLUSTER;
  for (int i = tid; i < n; i += nt) {
    int r = 0;
    if (nvec < n)
      for (int j = 0; j < n; ++j) r += (sh.lam[j] < sh.lam[i]) || (sh.lam[j] == sh.lam[i] && j < i);
    sh.need[i] = r < nvec;
  }
  // ---- 4. eigenvectors of T (column `slot` of Z holds the block's rows) ----
  for (int idx = tid; idx < n * n; idx += nt) Z[(idx / n) * S + idx % n] = 0.0;
  __syncthreads();
  // 16 vectors a wave, two lanes each: the lanes of a wave read neighbouring columns
  const int slot = (tid >> 6) * 16 + (lane >> 1);
  const bool vact = lane < 32 && slot < n, bot = lane & 1;
  int bs = 0, bt = 0;
  bool want = false;
  if (vact) {
    bs = sh.bs[slot];
    bt = sh.bt[slot];
    // the cluster's slots: neighbours closer than ctol
    int a = slot, b = slot;
    while (a > bs && sh.lam[a] - sh.lam[a - 1] < ctol) --a;
    while (b + 1 < bt && sh.lam[b + 1] - sh.lam[b] < ctol) ++b;
    for (int q = a; q <= b; ++q) want = want || sh.need[q];
  }
  // Orthonormalises the vectors of each cluster of two or more (a wave per cluster), in slot order
  auto orthogonalise = [&](int passes) {
    for (int a = wv; a < n; a += nw) {
      const int s = sh.bs[a], t = sh.bt[a];
      if (a > s && sh.lam[a] - sh.lam[a - 1] < ctol) continue;  // not a cluster's first
      int last = a;
      while (last + 1 < t && sh.lam[last + 1] - sh.lam[last] < ctol) ++last;
      if (last == a) continue;
      bool any = false;
      for (int q = a; q <= last; ++q) any = any || sh.need[q];
      if (!any) continue;
      const int i0 = s + lane, i1 = s + lane + 64;
      for (int p = a; p <= last; ++p) {
        double y0 = i0 < t ? Z[i0 * S + p] * sh.nv[p] : 0.0, y1 = i1 < t ? Z[i1 * S + p] * sh.nv[p] : 0.0;
        for (int pass = 0; pass < passes; ++pass)
          for (int b = a; b < p; ++b) {
            const double z0 = i0 < t ? Z[i0 * S + b] : 0.0, z1 = i1 < t ? Z[i1 * S + b] : 0.0;
            const double dp = wave_sum(fma(y0, z0, y1 * z1));
            y0 = fma(-dp, z0, y0);
            y1 = fma(-dp, z1, y1);
          }
        const double in = 1.0 / sqrt(wave_sum(fma(y0, y0, y1 * y1)));
        if (i0 < t) Z[i0 * S + p] = y0 * in;
        if (i1 < t) Z[i1 * S + p] = y1 * in;
        __builtin_amdgcn_wave_barrier();
        if (lane == 0) sh.nv[p] = 1.0;
      }
    }
  };
  const double rmax = 1.0 / (EPS * 2.0);
  if (vact) {
    double nv = 1.0;
    if (want) {
      if (bt - bs == 1)
        Z[bs * S + slot] = 1.0;
      else
        nv = 1.0 / sqrt(ldl_solve<true>(sh.d, sh.e, bs, bt, bot, sh.lam[slot], rmax, A, Z, S, slot, 1.0));
    }
    sh.nv[slot] = nv;
  }
  __syncthreads();
  orthogonalise(1);
  __syncthreads();
  if (vact && want && bt - bs > 1) {
    const double nv = sh.nv[slot];
    sh.nv[slot] = 1.0 / sqrt(ldl_solve<false>(sh.d, sh.e, bs, bt, bot, sh.lam[slot], rmax, A, Z, S, slot, nv));
  }
  __syncthreads();
  orthogonalise(2);
  __syncthreads();
  // Rayleigh quotients z^T T z / z^T z (the eigenvalue to ~eps |T|): four lanes per vector
  {
    const int c = tid >> 2, q4 = tid & 3;
    double num = 0.0, den = 0.0;
    if (c < n) {
      for (int i = q4; i < n; i += 4) {
        const double zi = Z[i * S + c], zn = i + 1 < n ? Z[(i + 1) * S + c] : 0.0;
        num = fma(zi, fma(sh.d[i], zi, 2.0 * sh.e[i] * zn), num);
        den = fma(zi, zi, den);
      }
    }
    num = group4_sum(num);
    den = group4_sum(den);
    if (c < n && q4 == 0) {
      sh.rq[c] = ldexp(den > 0.0 ? num / den : sh.lam[c], ex);  // no vector: the multisection value
      sh.nv[c] = den > 0.0 ? 1.0 / sqrt(den) : 0.0;
    }
  }
  __syncthreads();
  // ---- 5. sort ascending (rank; ties by slot), back-transform ----
  for (int i = tid; i < n; i += nt) {
    // (a NaN ranks with the infinities: perm is a permutation whatever the input holds)
    auto key = [&](int j) { return sh.rq[j] == sh.rq[j] ? sh.rq[j] : HUGE_VAL; };
    const double ki = key(i);
    int r = 0;
    for (int j = 0; j < n; ++j) r += key(j) < ki || (key(j) == ki && j < i);
    sh.perm[r] = i;
    w[r] = sh.rq[i];
  }
  __syncthreads();
  by_size(n, [&](auto nc) { back_transform<decltype(nc)::value>(n, nvec, A, Z, S, f, sh); });
}

}  // namespace qexeig
