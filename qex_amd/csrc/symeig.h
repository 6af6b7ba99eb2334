// symeig.h -- dense symmetric eigensolver for one workgroup (n <= 96, FP64).
//
//   1. Householder tridiagonalisation with the matrix in registers (256 threads, each a cyclic
//      patch): for k = 0..n-3 the reflector H_k = I - tau v v^T annihilates column k below the
//      subdiagonal; the trailing block becomes A - v w^T - w v^T with p = tau A v,
//      w = p - (tau / 2)(v^T p) v.  The rows v_k go to global scratch, d / e collect the tridiagonal.
//   2. T, scaled by a power of two to norm 1..2, splits into unreduced blocks where
//      |e_k| <= eps (|d_k| + |d_k+1|).
//   3. Eigenvalues: multisection on Sturm counts (sign changes of the leading minors of T - x), three
//      lanes per eigenvalue, a fixed number of rounds (interval / 4 per round).
//   4. Eigenvectors of T: two inverse iterations (LDL^T pivots of T - lam, pivots smaller than
//      eps |T| replaced by +-eps |T|) from a fixed pseudo-random start, one lane per vector; eigenvalues
//      of one block closer than 1e-5 |T| form a cluster, whose vectors are orthogonalised after every
//      solve.  Rayleigh quotients give the eigenvalues.
//   5. Ascending sort and back-transformation Z <- H_0 ... H_{n-3} Y, four lanes per column.
// All reductions run in a fixed order: the result does not depend on timing.
//
// What bounds it: every stage is a chain of dependent steps of one workgroup, so its time is
// barriers and latencies, not arithmetic.  Hence the matrix stays in registers (two barriers and a
// few LDS words per Householder step; the LDS-resident form took three barriers over 16 waves and
// re-read the block), the counts need no reciprocal and no barrier, and a column of the
// back-transformation stays in four lanes' registers from the first reflector to the last.
#pragma once
#include <hip/hip_runtime.h>

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
__device__ __forceinline__ double wave_sum(double x) {
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
  x += dpp_f64<0xB1>(x);
  x += dpp_f64<0x4E>(x);
  return x;
}
__device__ __forceinline__ double group8_sum(double x) {
  x = group4_sum(x);
  x += dpp_f64<0x141>(x);
  return x;
}

// Shared state of the solver (static LDS besides the two n x S matrices).
struct Smem {
  double d[MAXN], e[MAXN], lam[MAXN], rq[MAXN], tau[MAXN], nv[MAXN];
  double x[MAXN + 8], p[MAXN + 8];   // column being reduced; p = tau A v
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

// Number of eigenvalues of rows s..t-1 of T below x: the sign changes of the leading minors
// p_i = (d_i - x) p_{i-1} - e_{i-1}^2 p_{i-2}.  No division, so a row is one dependent FMA (a pivot
// recurrence needs a reciprocal, a Newton step and two clamps in the chain: 60 cycles a row against
// 16).  T is scaled to norm 1..2 and e^2 floored at 1e-60, so 8 rows change a minor by less than
// 1e-250 .. 1e6 and both minors never vanish together; they are rescaled by a power of two every 8 rows.
__device__ __forceinline__ int sturm_count(const double2* de, int s, int t, double x) {
  double p0 = 0.0, p1 = 1.0;
  unsigned bits = 0, c = 0;
  auto step = [&](double2 v) {
    const double pn = fma(v.x - x, p1, -(v.y * p0));
    p0 = p1;
    p1 = pn;
    bits = __builtin_amdgcn_alignbit(bits, (unsigned)__double2hiint(pn), 31);  // bits << 1 | sign
  };
  int j = s;
  for (; j + 8 <= t; j += 8) {
    double2 v[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) v[u] = de[j + u];
#pragma unroll
    for (int u = 0; u < 8; ++u) step(v[u]);
    c += __popc((bits ^ (bits >> 1)) & 0xFFu);
    const int ex = -__builtin_amdgcn_frexp_exp(fmax(fabs(p0), fabs(p1)));
    p0 = ldexp(p0, ex);
    p1 = ldexp(p1, ex);
  }
  const int left = t - j;
  for (; j < t; ++j) step(de[j]);
  return (int)(c + __popc((bits ^ (bits >> 1)) & ((1u << left) - 1u)));
}

// deterministic start vector entry in [-1, 1)
__device__ __forceinline__ double start_entry(int slot, int i) {
  unsigned x = 2654435761u * (unsigned)(slot + 1) ^ (40503u * (unsigned)(i + 7));
  x ^= x >> 13;
  x *= 0x5bd1e995u;
  x ^= x >> 15;
  return (double)(x & 0xFFFFFF) / 8388608.0 - 1.0;
}

// One thread: column `col` of Y <- (T_block - lam)^-1 b, rows s..t-1, with the inverse pivots 1/D_i
// of T_block - lam (|1/D| <= rmax) in column `col` of Dm.  FIRST: b is the start vector, and the
// pivots are computed along with the forward solve; else b = scale * Y and the pivots are read.
// Returns |x|^2.  The operands of 8 rows are in flight per LDS wait.
template <bool FIRST>
__device__ __forceinline__ double ldl_solve(const double* d, const double* e, int s, int t, double lam, double rmax,
                                            double* Dm, double* Y, int S, int col, double scale) {
  double y = 0.0, qi = 0.0, ep = 0.0;
  auto fwd = [&](int i, double di, double ei, double bi, double ri) {
    // row i: l = e_{i-1} / D_{i-1}; D_i = d_i - lam - e_{i-1} l; y_i = b_i - l y_{i-1}
    const double l = ep * qi;
    y = fma(-l, y, bi);
    if (FIRST) {
      const double q = fma(-ep, l, di - lam);
      qi = fmin(fmax(rcp_nr(q), -rmax), rmax);
      Dm[i * S + col] = qi;
    } else {
      qi = ri;
    }
    Y[i * S + col] = y;
    ep = ei;
  };
  int i = s;
  for (; i + 8 <= t; i += 8) {
    double dv[8], ev[8], bv[8], rv[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      ev[u] = e[i + u];
      if (FIRST) {
        dv[u] = d[i + u];
        bv[u] = start_entry(col, i + u);
        rv[u] = 0.0;
      } else {
        dv[u] = 0.0;
        bv[u] = scale * Y[(i + u) * S + col];
        rv[u] = Dm[(i + u) * S + col];
      }
    }
#pragma unroll
    for (int u = 0; u < 8; ++u) fwd(i + u, dv[u], ev[u], bv[u], rv[u]);
  }
  for (; i < t; ++i)
    fwd(i, d[i], e[i], FIRST ? start_entry(col, i) : scale * Y[i * S + col], FIRST ? 0.0 : Dm[i * S + col]);
  // x_i = y_i / D_i - (e_i / D_i) x_{i+1}; e_{t-1} = 0 at a block's end
  double x = 0.0, n0 = 0.0;
  i = t - 1;
  for (; i - 7 >= s; i -= 8) {
    double yv[8], rv[8], lv[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      rv[u] = Dm[(i - u) * S + col];
      yv[u] = Y[(i - u) * S + col] * rv[u];
      lv[u] = e[i - u] * rv[u];
    }
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      x = fma(-lv[u], x, yv[u]);
      n0 = fma(x, x, n0);
      Y[(i - u) * S + col] = x;
    }
  }
  for (; i >= s; --i) {
    const double r = Dm[i * S + col];
    x = fma(-(e[i] * r), x, Y[i * S + col] * r);
    n0 = fma(x, x, n0);
    Y[i * S + col] = x;
  }
  return n0;
}

// Householder tridiagonalisation of A (n x n in LDS, row stride S; only read).  NC >= ceil(n / 8).
// Threads 0..255: thread (r, c) = (tid / 8, tid % 8) holds A[r + 32 i][c + 8 j] in registers; the other
// waves only take part in the barriers.  32 x 8 rather than 16 x 16: row sums then cross 8 lanes (three
// DPP steps for 3 rows) instead of 16 (four steps for 6 rows).  Per step: the owners of column k put it
// in LDS | every thread forms v, tau and its rows of p = tau A v | p in LDS | rank-2 update.
// Row k of f (stride 8 NC, zero padded) receives v_k; sh.d, sh.e, sh.tau the rest.
template <int NC>
__device__ __forceinline__ void tridiagonalise(int n, const double* A, int S, double* f, Smem& sh) {
  constexpr int NR = (NC + 3) / 4, SP = 8 * NC;
  const int tid = threadIdx.x;
  if (__builtin_amdgcn_readfirstlane(tid >> 6) >= 4) {
    __syncthreads();
    for (int q = 1; q <= n - 2; ++q) {
      __syncthreads();
      __syncthreads();
    }
    __syncthreads();
    return;
  }
  const int r = tid >> 3, c = tid & 7;
  double a[NR][NC];
#pragma unroll
  for (int i = 0; i < NR; ++i)
#pragma unroll
    for (int j = 0; j < NC; ++j) {
      const int row = r + 32 * i, col = c + 8 * j;
      a[i][j] = row < n && col < n ? A[row * S + col] : 0.0;
    }
  // column 0 below the diagonal
  if (c == 0) {
#pragma unroll
    for (int i = 0; i < NR; ++i) sh.x[r + 32 * i] = r + 32 * i >= 1 ? a[i][0] : 0.0;
    if (r == 0) sh.d[0] = a[0][0];
  }
  __syncthreads();
  static_for<0, NC>([&](auto block) {
    constexpr int jb = decltype(block)::value, ib = jb / 4;
    for (int c0 = 0; c0 < 8; ++c0) {
      const int q = 8 * jb + c0;  // reduces column q - 1 to rows <= q
      if (q < 1) continue;
      if (q > n - 2) break;
      double vc[NC], vr[NR];
#pragma unroll
      for (int j = jb; j < NC; ++j) vc[j] = sh.x[c + 8 * j];
#pragma unroll
      for (int i = ib; i < NR; ++i) vr[i] = sh.x[r + 32 * i];
      const double x0 = sh.x[q];
      double tail = 0.0;
      {
        const double t = c == c0 ? 0.0 : vc[jb];
        tail = t * t;
#pragma unroll
        for (int j = jb + 1; j < NC; ++j) tail = fma(vc[j], vc[j], tail);
      }
      tail = group8_sum(tail);
      const bool skip = !(tail > 0.0);
      const double nx = sqrt(fma(x0, x0, tail));
      const double alpha = x0 >= 0.0 ? -nx : nx;
      const double v0 = skip ? 0.0 : x0 - alpha;
      const double tau = skip ? 0.0 : rcp_nr(nx * (nx + fabs(x0)));
      double u[NR];
#pragma unroll
      for (int i = ib; i < NR; ++i) {
        u[i] = 0.0;
#pragma unroll
        for (int j = jb + 1; j < NC; ++j) u[i] = fma(a[i][j], vc[j], u[i]);
      }
      if (c == c0) vc[jb] = v0;
      if (r == (q & 31)) vr[ib] = v0;
#pragma unroll
      for (int i = ib; i < NR; ++i) {
        u[i] = tau * group8_sum(fma(a[i][jb], vc[jb], u[i]));
        if (c == 0) sh.p[r + 32 * i] = u[i];
      }
#pragma unroll
      for (int j = 0; j < NC; ++j)
        if (r == j) f[(size_t)(q - 1) * SP + c + 8 * j] = j < jb ? 0.0 : vc[j];
      if (tid == 0) {
        sh.e[q - 1] = skip ? x0 : alpha;
        sh.tau[q - 1] = tau;
      }
      __syncthreads();
      double wc[NC];
      double vp = 0.0;
#pragma unroll
      for (int j = jb; j < NC; ++j) {
        wc[j] = sh.p[c + 8 * j];
        vp = fma(vc[j], wc[j], vp);
      }
      const double K = 0.5 * tau * group8_sum(vp);
#pragma unroll
      for (int j = jb; j < NC; ++j) wc[j] = fma(-K, vc[j], wc[j]);
#pragma unroll
      for (int i = ib; i < NR; ++i) {
        const double wr = fma(-K, vr[i], u[i]);
#pragma unroll
        for (int j = jb; j < NC; ++j) a[i][j] = fma(-vr[i], wc[j], fma(-wr, vc[j], a[i][j]));
      }
      // column q, the next one, and d_q (x was last read before the barrier above)
      if (c == c0) {
#pragma unroll
        for (int i = ib; i < NR; ++i) {
          const int row = r + 32 * i;
          sh.x[row] = row > q ? a[i][jb] : 0.0;
          if (row == q) sh.d[q] = a[i][jb];
        }
      }
      __syncthreads();
    }
  });
  if (tid == 0) sh.e[n - 2] = sh.x[n - 1];
#pragma unroll
  for (int i = 0; i < NR; ++i)
#pragma unroll
    for (int j = 0; j < NC; ++j)
      if (r + 32 * i == n - 1 && c + 8 * j == n - 1) sh.d[n - 1] = a[i][j];
  __syncthreads();
}

// Z <- H_0 ... H_{n-3} Y: column c of the result from column perm[c] of Y (in Z), scaled by nv.
// Four lanes hold a column: lane q the rows 8 i + 2 q + {0, 1}.  V (n - 2 rows of stride 8 NC) is
// read into the LDS of both matrices once every column is in registers.
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
      for (int c0 = 7; c0 >= 0; --c0) {
        const int k = 8 * jb + c0 - 1;  // rows > k
        if (k > n - 3) continue;
        if (k < 0) break;
        const double2* v = reinterpret_cast<const double2*>(A + (size_t)k * SP) + q4;
        double2 vv[NC];
        double acc0 = 0.0, acc1 = 0.0;
#pragma unroll
        for (int i = jb; i < NC; ++i) {
          vv[i] = v[4 * i];
          acc0 = fma(vv[i].x, z[i].x, acc0);
          acc1 = fma(vv[i].y, z[i].y, acc1);
        }
        const double s = sh.tau[k] * group4_sum(acc0 + acc1);
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
  if (n <= 16)
    tridiagonalise<2>(n, A, S, f, sh);
  else if (n <= 32)
    tridiagonalise<4>(n, A, S, f, sh);
  else if (n <= 64)
    tridiagonalise<8>(n, A, S, f, sh);
  else
    tridiagonalise<12>(n, A, S, f, sh);
  // ---- 2. norm, scaling, unreduced blocks ----
  double scale, unscale;  // powers of two
  {
    double nrm = 0.0;  // every wave by itself
    for (int i = lane; i < n; i += 64)
      nrm = fmax(nrm, fabs(sh.d[i]) + (i > 0 ? fabs(sh.e[i - 1]) : 0.0) + (i < n - 1 ? fabs(sh.e[i]) : 0.0));
    nrm = wave_max(nrm);
    int ex = nrm > 0.0 ? __builtin_amdgcn_frexp_exp(nrm) - 1 : 0;
    ex = ex < -1000 ? -1000 : ex > 1000 ? 1000 : ex;
    scale = ldexp(1.0, -ex);
    unscale = ldexp(1.0, ex);
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
  // 4^-25 of a width <= 4: 2^-48 of the norm.  Three lanes each: with n = 80 four waves, one per SIMD
  // (more lanes per eigenvalue share the SIMDs and gain fewer bits per unit of time).
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
      for (int r = 0; r < 25; ++r) {
        const double wd = 0.25 * (hi - lo);
        const int c = act ? sturm_count(sh.de, s, t, fma(wd, (double)(g + 1), lo)) : 0;
        const unsigned long long m = __ballot(act && c <= li);
        const int below = __popcll((m >> (lane - g)) & 7ull);
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
  // 16 vectors a wave: lanes of one wave read neighbouring columns
  const int slot = (tid >> 6) * 16 + lane;
  const bool vact = lane < 16 && slot < n;
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
    sh.nv[slot] = 1.0;
    if (want) {
      if (bt - bs == 1)
        Z[bs * S + slot] = 1.0;
      else
        sh.nv[slot] = 1.0 / sqrt(ldl_solve<true>(sh.d, sh.e, bs, bt, sh.lam[slot], rmax, A, Z, S, slot, 1.0));
    }
  }
  __syncthreads();
  orthogonalise(1);
  __syncthreads();
  if (vact && want && bt - bs > 1)
    sh.nv[slot] =
        1.0 / sqrt(ldl_solve<false>(sh.d, sh.e, bs, bt, sh.lam[slot], rmax, A, Z, S, slot, sh.nv[slot]));
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
      sh.rq[c] = (den > 0.0 ? num / den : sh.lam[c]) * unscale;  // no vector: the multisection value
      sh.nv[c] = den > 0.0 ? 1.0 / sqrt(den) : 0.0;
    }
  }
  __syncthreads();
  // ---- 5. sort ascending (rank; ties by slot), back-transform ----
  for (int i = tid; i < n; i += nt) {
    int r = 0;
    for (int j = 0; j < n; ++j) r += (sh.rq[j] < sh.rq[i]) || (sh.rq[j] == sh.rq[i] && j < i);
    sh.perm[r] = i;
    w[r] = sh.rq[i];
  }
  __syncthreads();
  if (n <= 16)
    back_transform<2>(n, nvec, A, Z, S, f, sh);
  else if (n <= 32)
    back_transform<4>(n, nvec, A, Z, S, f, sh);
  else if (n <= 64)
    back_transform<8>(n, nvec, A, Z, S, f, sh);
  else
    back_transform<12>(n, nvec, A, Z, S, f, sh);
}

}  // namespace qexeig
