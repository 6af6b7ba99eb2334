// band_wave.h -- one wave (64 lanes) solves (A - sigma) x = y for the symmetric pentadiagonal A of band.h
// and counts the eigenvalues of A below sigma, by substructuring:
//
//   Lane p owns m rows (m odd, 64 m >= N), the last two of them its separators.  It eliminates its
//   m - 2 interior rows in order (LDL^T with the fill towards the two separators of lane p - 1 as two
//   extra columns), which leaves a block tridiagonal system of 2 x 2 blocks over the lanes; that is
//   solved by cyclic reduction (6 levels, lane p - h and p + h by lane exchange), and the interior
//   rows follow by back substitution.
//
// A dependent chain of N rows at about 90 cycles a row (the two-sided elimination: N / 2) becomes m rows and
// 12 exchange levels: 4 us instead of 17..29 us at N = 513.  As in band.h there is no pivoting: this
// is LDL^T of a symmetric permutation of A - sigma (nested dissection order), small pivots are clamped, and
// the pivots' signs give the inertia.  Callers check the eigenpair by its residual and index.
#pragma once
#include "band.h"

namespace qexband {

constexpr int WAVE_F = 5;  // doubles of LDS per row for the factors
// rows per lane: odd (lanes then read LDS at an odd stride), >= 5
QEX_HD inline int wave_rows(int N) {
  const int m = (N + 63) / 64 | 1;
  return m < 5 ? 5 : m;
}
QEX_HD inline size_t wave_doubles(int N) { return (size_t)WAVE_F * wave_rows(N) * 64; }

// 2 x 2 symmetric block [p q; q s]
struct Sym2 {
  double p, q, s;
};
struct Vec2 {
  double x, y;
};
struct Mat2 {
  double xx, xy, yx, yy;  // row-major
};

__device__ __forceinline__ double lane_get(double x, int l) { return __shfl(x, l, 64); }
__device__ __forceinline__ Sym2 lane_get(Sym2 a, int l) { return {lane_get(a.p, l), lane_get(a.q, l), lane_get(a.s, l)}; }
__device__ __forceinline__ Vec2 lane_get(Vec2 a, int l) { return {lane_get(a.x, l), lane_get(a.y, l)}; }
__device__ __forceinline__ Mat2 lane_get(Mat2 a, int l) {
  return {lane_get(a.xx, l), lane_get(a.xy, l), lane_get(a.yx, l), lane_get(a.yy, l)};
}
__device__ __forceinline__ Sym2 inverse(Sym2 d) {
  const double r = rcp_clamped(fma(d.p, d.s, -(d.q * d.q)));
  return {d.s * r, -d.q * r, d.p * r};
}
// D x = z by elimination with row pivoting: the last block of a singular A - sigma keeps its regular direction (the
// determinant's rounding would scale it)
__device__ __forceinline__ Vec2 solve(Sym2 d, Vec2 z) {
  const bool sw = fabs(d.p) < fabs(d.q);
  const double a = sw ? d.q : d.p, b = sw ? d.s : d.q, c = sw ? d.p : d.q, e = sw ? d.q : d.s;
  const double za = sw ? z.y : z.x, zb = sw ? z.x : z.y;
  const double r = rcp_clamped(a), l = c * r;
  const double y = fma(-l, za, zb) * rcp_clamped(fma(-l, b, e));
  return {fma(-b, y, za) * r, y};
}
// negative eigenvalues of the block: signs of p and of det / p
__device__ __forceinline__ int negatives(Sym2 d) {
  const int a = sign_bit(d.p);
  return a + (a ^ sign_bit(fma(d.p, d.s, -(d.q * d.q))));
}
__device__ __forceinline__ Vec2 mul(Sym2 a, Vec2 v) { return {fma(a.p, v.x, a.q * v.y), fma(a.q, v.x, a.s * v.y)}; }
__device__ __forceinline__ Vec2 mul(Mat2 a, Vec2 v) { return {fma(a.xx, v.x, a.xy * v.y), fma(a.yx, v.x, a.yy * v.y)}; }
__device__ __forceinline__ Vec2 tmul(Mat2 a, Vec2 v) { return {fma(a.xx, v.x, a.yx * v.y), fma(a.xy, v.x, a.yy * v.y)}; }
__device__ __forceinline__ Mat2 mul(Sym2 a, Mat2 b) {
  return {fma(a.p, b.xx, a.q * b.yx), fma(a.p, b.xy, a.q * b.yy), fma(a.q, b.xx, a.s * b.yx), fma(a.q, b.xy, a.s * b.yy)};
}
__device__ __forceinline__ Mat2 mul(Mat2 a, Sym2 b) {
  return {fma(a.xx, b.p, a.xy * b.q), fma(a.xx, b.q, a.xy * b.s), fma(a.yx, b.p, a.yy * b.q), fma(a.yx, b.q, a.yy * b.s)};
}
__device__ __forceinline__ Mat2 mul(Mat2 a, Mat2 b) {
  return {fma(a.xx, b.xx, a.xy * b.yx), fma(a.xx, b.xy, a.xy * b.yy), fma(a.yx, b.xx, a.yy * b.yx), fma(a.yx, b.xy, a.yy * b.yy)};
}

// What the lanes of a wave wrote to LDS before, all of them read after: the LDS executes one wave's accesses in
// issue order, so only the compiler must be kept from moving them across this point.
__device__ __forceinline__ void wave_lds_order() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_wave_barrier();
  asm volatile("" ::: "memory");
}

// Every lane of the wave calls this.  a, y: LDS, N doubles each; F: LDS, wave_doubles(N) doubles.
// SOLVE: y <- (A - sigma)^-1 y.  Returns the number of eigenvalues of A below sigma (the same in every lane).
// Each lane reads and writes only its own rows of y and F; lanes that go on to read others' rows call
// wave_lds_order first.
template <bool SOLVE>
__device__ __forceinline__ int wave_solve(const double* a, double* y, int N, double b, double c, double sigma, double* F) {
  const int p = threadIdx.x & 63, m = wave_rows(N), k = m - 2, row0 = p * m;
  const double c2 = c * c;
  double* Fl = F + p;           // l_i                 (row i of lane p at [i * 64])
  double* Fm = Fl + 64 * m;     // m_i = c / d_i
  double* Fz = Fm + 64 * m;     // z_i / d_i
  double* G1 = Fz + 64 * m;     // fill towards the previous lane's separators, over d_i
  double* G2 = G1 + 64 * m;
  // rows past N are decoupled by a diagonal of 1e100
  auto diag = [&](int i) { return row0 + i < N ? a[row0 + i] - sigma : 1e100; };
  auto rhs = [&](int i) { return SOLVE && row0 + i < N ? y[row0 + i] : 0.0; };
  double rm1 = 0.0, rm2 = 0.0, um1 = 0.0, lm1 = 0.0, mm1 = 0.0, mm2 = 0.0;
  double z1 = 0.0, z2 = 0.0;
  Vec2 g1{0.0, 0.0}, g2{0.0, 0.0};  // fill of the last two rows (first row: c, b; second: 0, c)
  Sym2 SL{0.0, 0.0, 0.0};
  Vec2 ZL{0.0, 0.0};
  int neg = 0;
  for (int i = 0; i < k; ++i) {
    const double d = fma(-um1 * um1, rm1, fma(-c2, rm2, diag(i)));
    neg += sign_bit(d);
    const double r = rcp_clamped(d), u = fma(-c * rm1, um1, b);
    Vec2 g{fma(-mm2, g2.x, -(lm1 * g1.x)), fma(-mm2, g2.y, -(lm1 * g1.y))};
    if (i == 0 && p > 0) g = {c, b};
    if (i == 1 && p > 0) g.y += c;
    const double gx = g.x * r, gy = g.y * r;
    SL = {fma(g.x, gx, SL.p), fma(g.x, gy, SL.q), fma(g.y, gy, SL.s)};
    const double l = u * r, mm = c * r;
    if (SOLVE) {
      const double z = fma(-mm2, z2, fma(-lm1, z1, rhs(i)));
      ZL = {fma(gx, z, ZL.x), fma(gy, z, ZL.y)};
      Fl[64 * i] = l;
      Fm[64 * i] = mm;
      Fz[64 * i] = z * r;
      G1[64 * i] = gx;
      G2[64 * i] = gy;
      z2 = z1;
      z1 = z;
    }
    g2 = g1;
    g1 = g;
    mm2 = mm1;
    mm1 = mm;
    lm1 = l;
    rm2 = rm1;
    rm1 = r;
    um1 = u;
  }
  // the separators' block, its coupling E to the previous lane's, and the right-hand side
  Sym2 D{fma(-um1 * um1, rm1, fma(-c2, rm2, diag(k))), fma(-c * rm1, um1, b), fma(-c2, rm1, diag(k + 1))};
  if (row0 + k + 1 >= N) D.q = 0.0;  // (row k + 1 is padding)
  Mat2 E{fma(-mm2, g2.x, -(lm1 * g1.x)), fma(-mm2, g2.y, -(lm1 * g1.y)), -(mm1 * g1.x), -(mm1 * g1.y)};
  Vec2 Zr{0.0, 0.0};
  if (SOLVE) Zr = {fma(-mm2, z2, fma(-lm1, z1, rhs(k))), fma(-mm1, z1, rhs(k + 1))};
  {
    const Sym2 s = lane_get(SL, p + 1);
    const bool in = p < 63;
    D = {D.p - (in ? s.p : 0.0), D.q - (in ? s.q : 0.0), D.s - (in ? s.s : 0.0)};
    if (SOLVE) {
      const Vec2 z = lane_get(ZL, p + 1);
      Zr = {Zr.x - (in ? z.x : 0.0), Zr.y - (in ? z.y : 0.0)};
    }
  }
  // cyclic reduction: at level h the lanes p = h - 1 (mod 2 h) are eliminated into p - h and p + h
  Mat2 Wk{0.0, 0.0, 0.0, 0.0}, Gk[6];
  Vec2 vk{0.0, 0.0};
#pragma unroll
  for (int t = 0; t < 6; ++t) {
    const int h = 1 << t;
    const bool mine = (p & (2 * h - 1)) == h - 1;           // eliminated at this level
    const bool stays = (p & (2 * h - 1)) == 2 * h - 1;      // its neighbours are
    const Sym2 I = inverse(D);
    const Mat2 W = mul(I, E);
    const Vec2 v = SOLVE ? solve(D, Zr) : Vec2{0.0, 0.0};
    if (mine) {
      neg += negatives(D);
      if (SOLVE) {
        Wk = W;
        vk = v;
      }
    }
    // what the left neighbour p - h receives: E^T W, E^T v
    const Sym2 SLp{fma(E.xx, W.xx, E.yx * W.yx), fma(E.xx, W.xy, E.yx * W.yy), fma(E.xy, W.xy, E.yy * W.yy)};
    const int lo = p - h, hi = p + h;
    const Sym2 Il = lane_get(I, lo), Sr = lane_get(SLp, hi);
    const Mat2 Wl = lane_get(W, lo);
    const bool right = hi < 64;
    const Mat2 G = mul(E, Il);  // E D_l^-1
    Gk[t] = G;
    Sym2 Dn{D.p - fma(G.xx, E.xx, G.xy * E.xy), D.q - fma(G.xx, E.yx, G.xy * E.yy), D.s - fma(G.yx, E.yx, G.yy * E.yy)};
    if (right) Dn = {Dn.p - Sr.p, Dn.q - Sr.q, Dn.s - Sr.s};
    if (SOLVE) {
      const Vec2 vl = lane_get(v, lo), zr = lane_get(tmul(E, v), hi);
      const Vec2 q = mul(E, vl);
      Vec2 zn{Zr.x - q.x, Zr.y - q.y};
      if (right) zn = {zn.x - zr.x, zn.y - zr.y};
      if (stays) Zr = zn;
    }
    const Mat2 En = mul(E, Wl);
    if (stays) {
      D = Dn;
      E = {-En.xx, -En.xy, -En.yx, -En.yy};
    }
  }
  if (p == 63) neg += negatives(D);
  int total = 0;
#pragma unroll
  for (int bit = 0; bit < 6; ++bit) total += __popcll(__ballot((neg >> bit) & 1)) << bit;
  if (!SOLVE) return total;
  // back through the levels: x_e = v_e - W_e x_(e-h) - (E_r D_e^-1)^T x_r, r = e + h
  Vec2 x = solve(D, Zr);  // (lane 63)
#pragma unroll
  for (int t = 5; t >= 0; --t) {
    const int h = 1 << t;
    const bool mine = (p & (2 * h - 1)) == h - 1;
    const Vec2 xl = lane_get(x, p - h), xr = lane_get(tmul(Gk[t], x), p + h);
    const Vec2 w = mul(Wk, xl);
    const bool left = p >= h;
    if (mine) x = {vk.x - (left ? w.x : 0.0) - xr.x, vk.y - (left ? w.y : 0.0) - xr.y};
  }
  // interior rows, from the separators of this lane and of the previous one
  Vec2 xs = lane_get(x, p - 1);
  if (p == 0) xs = {0.0, 0.0};
  double x1 = x.x, x2 = x.y;
  auto put = [&](int i, double v) {
    if (row0 + i < N) y[row0 + i] = v;
  };
  put(k, x.x);
  put(k + 1, x.y);
  for (int i = k - 1; i >= 0; --i) {
    const double q = fma(-G1[64 * i], xs.x, fma(-G2[64 * i], xs.y, Fz[64 * i]));
    const double xi = fma(-Fm[64 * i], x2, fma(-Fl[64 * i], x1, q));
    put(i, xi);
    x2 = x1;
    x1 = xi;
  }
  return total;
}

}  // namespace qexband
