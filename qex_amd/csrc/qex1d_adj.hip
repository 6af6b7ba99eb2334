// qex1d_adj.hip -- reverse pass of the batched 1D Kohn-Sham scan loop with respect to the
// parameters of a windowed LocalMLP XC functional (the gradient that jax.grad takes through
// jit_scf.kohn_sham in qedft/train/od/train.py:250-323).
//
// Given the forward outputs of qex1d_kohn_sham (stored densities, v_H, v_xc and the orbitals of
// every iteration) and cotangents of the stored energies and densities, iteration k is reversed
// as (n_k: input density, n_out: unmixed output, psi_j: occupied orbitals, 2-norm 1):
//   k_adj_mix        nbar_k, dbar (the mixing n_k+1 = n_k + alpha_k mean(last m differences))
//   energy           nob += c (-v_KS + v_H(n_out) + v_xc(n_out) + v_ext), thetabar += c dF(n_out)/dtheta,
//                    c = dE_k dx (the eigenvalue sum and -dx v_KS.n_out cancel at fixed n_out)
//   k_adj_eig        vbar = sum_j occ_j (2/dx) psi_j * y_j with y_j = -(H - eps_j)^-1 Q (nob psi_j)
//                    (Q projects out the occupied orbitals) minus the pairs of occupied orbitals with unequal occupations
//   Hartree + XC     nbar += dx U vbar + H_F vbar, thetabar += d(vbar . grad F)/dtheta, F = sum e(n) n
// The MLP terms come from reverse mode over the network's forward and forward-tangent passes on tiles of
// points (FP64 matrix instructions); each workgroup accumulates its parameter partials in registers and
// adds them to its own slot, and the slots are summed in a fixed order.
// A GLOBAL_MLP functional (amplitude encoded: E_xc = dx f(n), v_xc = dx grad f) takes the same
// steps with F = f in the energy and F = dx f in the potential, through k_adj_gmlp (one workgroup
// per system); under reflection its functional sees the unflipped densities (the forward flips only
// the density passed on), so only the mixing cotangents are flipped.
#include <hip/hip_runtime.h>

#include <math.h>
#include <stdarg.h>
#include <stdio.h>
#include <string.h>

#include <type_traits>

#include "band_wave.h"
#include "prof.h"
#include "qex.h"
#include "tiles.h"

namespace {

constexpr int NT = 256;
constexpr int ADJ_WG = 256;     // workgroups of the MLP adjoint launch = parameter-partial slots
constexpr int HMAX = 64;        // hidden width
constexpr int WMAXW = QEX1D_MAX_MLP_WINDOW;
thread_local char g_erra[512] = "";

int faila(int code, const char* fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(g_erra, sizeof(g_erra), fmt, ap);
  va_end(ap);
  return code;
}

__device__ __forceinline__ double wsum(double x) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) x += __shfl_xor(x, o, 64);
  return x;
}

__device__ double bsum(double x, double* red) {
  x = wsum(x);
  const int w = threadIdx.x >> 6, l = threadIdx.x & 63;
  __syncthreads();
  if (l == 0) red[w] = x;
  __syncthreads();
  double s = 0.0;
  for (int q = 0; q < (int)(blockDim.x >> 6); ++q) s += red[q];
  __syncthreads();
  return s;
}

__device__ double bmax(double x, double* red) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) x = fmax(x, __shfl_xor(x, o, 64));
  const int w = threadIdx.x >> 6, l = threadIdx.x & 63;
  __syncthreads();
  if (l == 0) red[w] = x;
  __syncthreads();
  double s = 0.0;
  for (int q = 0; q < (int)(blockDim.x >> 6); ++q) s = fmax(s, red[q]);
  __syncthreads();
  return s;
}

// activation and its first two derivatives
__device__ void act3(int act, double z, double* a, double* d1, double* d2) {
  switch (act) {
    case QEX_ACT_SILU: {
      const double s = 1.0 / (1.0 + exp(-z));
      *a = z * s;
      *d1 = s * (1.0 + z * (1.0 - s));
      *d2 = s * (1.0 - s) * (2.0 + z * (1.0 - 2.0 * s));
      break;
    }
    case QEX_ACT_TANH: {
      const double t = tanh(z);
      *a = t;
      *d1 = 1.0 - t * t;
      *d2 = -2.0 * t * (1.0 - t * t);
      break;
    }
    case QEX_ACT_SOFTPLUS: {
      const double s = 1.0 / (1.0 + exp(-z));
      *a = z > 0.0 ? z + log1p(exp(-z)) : log1p(exp(z));
      *d1 = s;
      *d2 = s * (1.0 - s);
      break;
    }
    case QEX_ACT_SIGMOID: {
      const double s = 1.0 / (1.0 + exp(-z));
      *a = s;
      *d1 = s * (1.0 - s);
      *d2 = s * (1.0 - s) * (1.0 - 2.0 * s);
      break;
    }
    case QEX_ACT_RELU:
      *a = z > 0.0 ? z : 0.0;
      *d1 = z > 0.0 ? 1.0 : 0.0;
      *d2 = 0.0;
      break;
    default: {  // GELU, tanh form
      const double k = 0.7978845608028654, c = 0.044715;
      const double t = tanh(k * (z + c * z * z * z));
      const double du = k * (1.0 + 3.0 * c * z * z);
      const double s2 = 1.0 - t * t;
      *a = 0.5 * z * (1.0 + t);
      *d1 = 0.5 * (1.0 + t) + 0.5 * z * s2 * du;
      *d2 = s2 * du + 0.5 * z * (-2.0 * t * s2 * du * du + s2 * k * 6.0 * c * z);
      break;
    }
  }
}

// output transform of the network (QEX1D_MLP_OUTPUT_*) and its first two derivatives
__device__ __forceinline__ double out3(int kind, double y, double* d1, double* d2) {
  if (kind == QEX1D_MLP_OUTPUT_NEGATIVITY) {  // -swish(y)
    const double s = 1.0 / (1.0 + exp(-y));
    *d1 = -(s * (1.0 + y * (1.0 - s)));
    *d2 = -(s * (1.0 - s) * (2.0 + y * (1.0 - 2.0 * s)));
    return -y * s;
  }
  *d1 = 1.0;
  *d2 = 0.0;
  return y;
}

struct Adj {
  int B, N, T, K, M, W, H1, H2, NL, act, P, mlpout, reflect, sgs;
  const int* win;  // [B][2] reflection window (reflect)
  double dx, norm;
  int w1, b1, w2, b2, w3, b3;  // parameter offsets (w2/b2 unused when NL == 1)
  const double* table;
  const double* vext;
  const double* n0;
  const int* ne;
  const double* mlp;
  const double* dens;  // [B][T][N] stored (mixed) densities
  const double* vh;    // [B][T][N] v_H(n_k)
  const double* vxc;   // [B][T][N] v_xc(n_k)
  const double* orb;   // [B][T][K][N]
  const double* dE;    // [B][T] or null
  const double* dn;    // [B][T][N] or null
  // workspace
  double* nbar;  // [B][N]
  double* nob;   // [B][N]
  double* nout;  // [B][N]
  double* vbar;  // [B][N]
  double* tmp;   // [B][N]
  double* dbar;  // [B][T][N]
  double* xbar;  // [B][N][W]
  double* fv;    // [B][N]
  double* fdv;   // [B][N]
  double* thp;   // [ADJ_WG][P]
};

__device__ __forceinline__ const double* input_density(const Adj& a, int s, int k) {
  return k == 0 ? a.n0 + (size_t)s * a.N : a.dens + ((size_t)s * a.T + k - 1) * a.N;
}

__device__ __forceinline__ double occupation(int ne, int j) { return j < (ne + 1) / 2 ? (double)min(2, ne - 2 * j) : 0.0; }

__global__ void k_zero_a(double* p, long n) {
  for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x) p[i] = 0.0;
}

// mixing and difference cotangents; one workgroup per system
__global__ __launch_bounds__(NT) void k_adj_mix(Adj a, int k, double alpha_k) {
  const int s = blockIdx.x, N = a.N, T = a.T;
  const int cnt = min(a.M, k + 1);
  const double wgt = alpha_k / (double)cnt;
  const bool stopped = k <= a.sgs;  // the state of this iteration is a constant: no cotangent reaches it
  for (int t = threadIdx.x; t < N; t += NT) {
    double g = stopped ? 0.0 : a.nbar[(size_t)s * N + t];
    if (a.dn && !stopped) g += a.dn[((size_t)s * T + k) * N + t];
    for (int j = k - cnt + 1; j <= k; ++j) a.dbar[((size_t)s * T + j) * N + t] += wgt * g;
    const double dk = a.dbar[((size_t)s * T + k) * N + t];
    a.nob[(size_t)s * N + t] = dk;
    a.nbar[(size_t)s * N + t] = g - dk;
    // unmixed output density of iteration k from its orbitals
    double no = 0.0;
    const int ne = a.ne[s];
    for (int j = 0; j < (ne + 1) / 2; ++j) {
      const double x = a.orb[(((size_t)s * T + k) * a.K + j) * N + t];
      no = fma(occupation(ne, j), x * x, no);
    }
    a.nout[(size_t)s * N + t] = no / a.dx;
  }
}

// x[s] <- S x[s] in place: the flip-and-average map inside the system's reflection window (S is
// symmetric and idempotent, so it is also its own adjoint)
__global__ void k_sym_inplace(Adj a, double* x) {
  const long idx = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= (long)a.B * a.N) return;
  const int s = (int)(idx / a.N), i = (int)(idx % a.N);
  const int lo = a.win[2 * s], hi = a.win[2 * s + 1];
  const int m = (i >= lo && i <= hi) ? lo + hi - i : i;
  if (i < m) {
    double* r = x + (size_t)s * a.N;
    const double v = 0.5 * (r[i] + r[m]);
    r[i] = v;
    r[m] = v;
  }
}

// dst[s] += S c[s] + d[s] (d optional)
__global__ void k_sym_add(Adj a, double* dst, const double* c, const double* d) {
  const long idx = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= (long)a.B * a.N) return;
  const int s = (int)(idx / a.N), i = (int)(idx % a.N);
  const int lo = a.win[2 * s], hi = a.win[2 * s + 1];
  const int m = (i >= lo && i <= hi) ? lo + hi - i : i;
  dst[idx] += 0.5 * (c[idx] + c[(size_t)s * a.N + m]) + (d ? d[idx] : 0.0);
}

// dst[s] = S src[s]
__global__ void k_sym_copy(Adj a, double* dst, const double* src) {
  const long idx = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= (long)a.B * a.N) return;
  const int s = (int)(idx / a.N), i = (int)(idx % a.N);
  const int lo = a.win[2 * s], hi = a.win[2 * s + 1];
  const int m = (i >= lo && i <= hi) ? lo + hi - i : i;
  dst[idx] = 0.5 * (src[idx] + src[(size_t)s * a.N + m]);
}

// out[s] = dx * U in[s] (Toeplitz interaction matrix from its first row)
__global__ __launch_bounds__(NT) void k_toeplitz(int N, double dx, const double* table, const double* in,
                                                 double* out) {
  extern __shared__ double sm[];
  const int s = blockIdx.y;
  double* tab = sm;
  double* x = sm + N;
  for (int t = threadIdx.x; t < N; t += NT) {
    tab[t] = table[t];
    x[t] = in[(size_t)s * N + t];
  }
  __syncthreads();
  const int i = blockIdx.x * NT + threadIdx.x;
  if (i >= N) return;
  double acc = 0.0;
  for (int j = 0; j < N; ++j) acc = fma(tab[abs(i - j)], x[j], acc);
  out[(size_t)s * N + i] = dx * acc;
}

typedef double d4_t __attribute__((ext_vector_type(4)));
__device__ __forceinline__ d4_t mfma64(double a, double b, d4_t c) {
  return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}

// sum over the 16 lanes of a DPP row, in every lane of it
template <int ROT>
__device__ __forceinline__ double row_rotated(double x) {
  const int lo = __builtin_amdgcn_mov_dpp(__double2loint(x), 0x120 + ROT, 0xf, 0xf, true);
  const int hi = __builtin_amdgcn_mov_dpp(__double2hiint(x), 0x120 + ROT, 0xf, 0xf, true);
  return __hiloint2double(hi, lo);
}
__device__ __forceinline__ double row_sum(double x) {
  x += row_rotated<8>(x);
  x += row_rotated<4>(x);
  x += row_rotated<2>(x);
  return x + row_rotated<1>(x);
}

// MLP second-order adjoint.  Per point p = (s, i): x = window(xin[s])_i / norm, tangent
// xt = window(tin[s])_i / norm, fbar = sf[s] * F1[s][i], fdbar = F2[s][i].
// Outputs per point: xbar (dPhi/dx), f, fdot; parameter gradient of Phi = fbar f + fdbar fdot
// added to the workgroup's slot.  TAN = false: without tangents (Phi = fbar f, no tin, F2 and fdot).
//
// Every product is a tile of FP64 matrix instructions.  A group of 4 waves takes 32 rows: 16 points and their
// tangents, or (TAN = false) 32 points; wave w owns the units 16 w .. 16 w + 15 of each layer, so a weight
// fragment serves both row blocks, and value and tangent of a unit meet in one lane.  The partial sums of dW1
// and dW2 stay in registers over all tiles of a group; weights, activations and adjoints are in LDS
// (stride 66: the operand reads of a product along a row touch all banks once).
// A workgroup holds two groups (two waves a SIMD), and there are at most as many workgroups as CUs, since each adds its
// parameter partials to memory once per launch.
// One point per wave with one lane per unit (weights from LDS for every multiply, 0.25 flop a byte) took 255 us for
// 32 x 513 points of a 17-64-64-1 network; as matrix products 64 us with tangents and 52 without, of which 14
// and 7 are the matrix instructions at peak: bound by the barriers between the phases and the activations.
// The LDS (153 KB for every network) leaves a CU to one workgroup.  Beside two streams that are never out of batches
// of 48 molecules a training step takes 11.5 ms (5.5 alone) with FP32-grid molecules and 15.2 with FP64 ones; the
// 97 KB kernel of one point a wave took 28.6 and 26.0 (17.2 alone), so the workgroups do get their CUs.
// MFMA operand layout (16x16x4, one wave): lane l supplies A[l%16][l/16] and B[l/16][l%16]; it receives
// D[4v + l/16][l%16] in element v.
constexpr int AG = 2;              // groups of a workgroup
constexpr int ANT = AG * 256;      // its threads
constexpr int AS = 66;             // LDS row stride (doubles)
constexpr int AROWS = 32;          // rows of a tile
constexpr int AW1 = (WMAXW + 3) / 4 * 4;  // rows of W1 in LDS
constexpr int AXL = (AW1 + 7) / 8;  // window entries a thread fetches
constexpr int ATILE = 3 * AROWS * AS + 4 * AROWS + AROWS;  // LDS of a group (doubles)
constexpr size_t ADJ_MLP_LDS = (size_t)(AW1 * AS + HMAX * AS + AG * ATILE) * 8;
static_assert(ADJ_MLP_LDS <= 160 * 1024, "LDS of a CU");
// (the parameter partials take the place of the tiles at the end)
static_assert(WMAXW * HMAX + HMAX * HMAX + 3 * HMAX + 1 <= AW1 * AS + AG * ATILE, "parameters fit in LDS");
template <int NL, bool TAN>
__global__ __launch_bounds__(ANT) void k_adj_mlp(Adj a, const double* xin, const double* tin, const double* F1,
                                                 const double* sf, const double* F2) {
  extern __shared__ double sm[];
  constexpr int PTS = TAN ? 16 : 32;  // points of a tile
  const int tid = threadIdx.x, grp = tid >> 8, t = tid & 255, wv = t >> 6, l = t & 63, lr = l & 15, lk = l >> 4;
  const int W = a.W, H1 = a.H1, H2 = a.H2, HL = NL == 2 ? H2 : H1, N = a.N, h = W / 2;
  double* sW1 = sm;                      // W1, row o at o * AS, rows to a multiple of 4 and all columns zero filled
  double* sW2 = sW1 + AW1 * AS;          // W2 (NL == 2), zero filled
  double* sX = sW2 + (NL == 2 ? HMAX * AS : 0) + grp * ATILE;  // window and tangent window
  double* sA = sX + AROWS * AS;          // activations of layer 1, then its adjoints
  double* sZ = sA + AROWS * AS;          // adjoints of layer 2
  double* sY = sZ + AROWS * AS;          // output partials of the 4 waves
  double* sF = sY + 4 * AROWS;           // fbar, fdbar
  // weights into LDS, a thread's loads in flight together
  auto copy = [&](double* dst, int w, int rows, int cols, auto padded) {
    constexpr int total = decltype(padded)::value, M = (total * HMAX + ANT - 1) / ANT;
    double v[M];
#pragma unroll
    for (int e = 0; e < M; ++e) {
      const int q = tid + e * ANT, r = q / HMAX, u = q % HMAX;
      v[e] = r < rows && u < cols ? a.mlp[w + r * cols + u] : 0.0;
    }
#pragma unroll
    for (int e = 0; e < M; ++e) {
      const int q = tid + e * ANT;
      if (q < total * HMAX) dst[q / HMAX * AS + q % HMAX] = v[e];
    }
  };
  copy(sW1, a.w1, W, H1, std::integral_constant<int, AW1>{});
  const int col = wv * 16 + lr;
  if constexpr (NL == 2) copy(sW2, a.w2, H1, H2, std::integral_constant<int, HMAX>{});
  const double b1 = col < H1 ? a.mlp[a.b1 + col] : 0.0, b2 = NL == 2 && col < H2 ? a.mlp[a.b2 + col] : 0.0;
  const double w3 = col < HL ? a.mlp[a.w3 + col] : 0.0, b3 = a.mlp[a.b3];
  const d4_t zero = {0.0, 0.0, 0.0, 0.0};
  constexpr int RB1 = (WMAXW + 15) / 16;
  d4_t gW1[RB1], gW2[NL == 2 ? 4 : 1];
#pragma unroll
  for (int rb = 0; rb < RB1; ++rb) gW1[rb] = zero;
#pragma unroll
  for (int rb = 0; rb < (NL == 2 ? 4 : 1); ++rb) gW2[rb] = zero;
  double gb1 = 0.0, gb2 = 0.0, gW3 = 0.0, gb3 = 0.0;
  const double inorm = 1.0 / a.norm;
  const int npts = a.B * N, ntile = (npts + PTS - 1) / PTS;
  // inputs of a tile: 8 threads a row
  const int frow = t >> 3, fo = t & 7;
  double nx[AXL], nf;
  auto fetch = [&](int tile) {
    const int p = tile * PTS + (TAN ? frow & 15 : frow);
    const bool in = tile < ntile && p < npts;
    const int s = in ? p / N : 0, i = p - s * N;
    const double* src = (TAN && frow >= 16 ? tin : xin) + (size_t)s * N;
#pragma unroll
    for (int q = 0; q < AXL; ++q) {
      const int o = fo + 8 * q, x = i + o - h;
      nx[q] = in && o < W && x >= 0 && x < N ? src[x] * inorm : 0.0;
    }
    nf = 0.0;
    if (in && fo == 0) nf = TAN && frow >= 16 ? F2[p] : sf[s] * F1[p];
  };
  const int G = gridDim.x;
  fetch(blockIdx.x + G * grp);
  // (both groups run the rounds of the first one)
  for (int round = 0; blockIdx.x + G * AG * round < ntile; ++round) {
    const int tile = blockIdx.x + G * (AG * round + grp);
#pragma unroll
    for (int q = 0; q < AXL; ++q)
      if (fo + 8 * q < AW1) sX[frow * AS + fo + 8 * q] = nx[q];
    if (fo == 0) sF[frow] = nf;
    __syncthreads();
    fetch(tile + G * AG);
    // ---- layer 1 ----
    d4_t z0 = zero, z1 = zero;
#pragma unroll 1
    for (int q = 0; 4 * q < W; ++q) {
        const int k = 4 * q + lk;
        const double b = sW1[k * AS + col];
        z0 = mfma64(sX[lr * AS + k], b, z0);
        z1 = mfma64(sX[(16 + lr) * AS + k], b, z1);
      }
    // TAN: z0 the pre-activations and z1 their tangents; else both pre-activations
    double aL[2][4], p1[2][4], q1[4], t1[4];  // activations, act' (block 1: unused with TAN), act'', tangents
    auto activate = [&](double bias, d4_t y0, d4_t y1, double (&av)[2][4], double (&d1)[2][4], double (&d2)[4], double (&zt)[4]) {
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        double e2;
        act3(a.act, y0[v] + bias, &av[0][v], &d1[0][v], &e2);
        if (TAN) {
          d2[v] = e2;
          zt[v] = y1[v];
          av[1][v] = d1[0][v] * y1[v];
        } else {
          act3(a.act, y1[v] + bias, &av[1][v], &d1[1][v], &e2);
        }
      }
    };
    activate(b1, z0, z1, aL, p1, q1, t1);
    double p2[2][4], q2[4], t2[4];
    if constexpr (NL == 2) {
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        sA[(4 * v + lk) * AS + col] = col < H1 ? aL[0][v] : 0.0;
        sA[(16 + 4 * v + lk) * AS + col] = col < H1 ? aL[1][v] : 0.0;
      }
      __syncthreads();
      z0 = z1 = zero;
#pragma unroll 4
      for (int q = 0; 4 * q < H1; ++q) {
          const double b = sW2[(4 * q + lk) * AS + col];
          z0 = mfma64(sA[lr * AS + 4 * q + lk], b, z0);
          z1 = mfma64(sA[(16 + lr) * AS + 4 * q + lk], b, z1);
        }
      activate(b2, z0, z1, aL, p2, q2, t2);
    }
    // ---- output: the units of a wave in one DPP row, the waves through LDS ----
#pragma unroll
    for (int rb = 0; rb < 2; ++rb)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const double y = row_sum(aL[rb][v] * w3);
        if (lr == 0) sY[wv * AROWS + rb * 16 + 4 * v + lk] = y;
      }
    __syncthreads();
    // adjoints of the last hidden layer: zb[0] of the values, zb[1] of the tangents (else of the points 16 .. 31)
    double zb[2][4];
    const double(&pl)[2][4] = NL == 2 ? p2 : p1;
    const double(&ql)[4] = NL == 2 ? q2 : q1;
    const double(&tl)[4] = NL == 2 ? t2 : t1;
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int r = 4 * v + lk;
      auto raw = [&](int row) { return (sY[row] + sY[AROWS + row]) + (sY[2 * AROWS + row] + sY[3 * AROWS + row]); };
      double g1, g2;
      if (TAN) {
        const int p = tile * PTS + r;
        const double fbar = sF[r], fdbar = sF[16 + r], yd = raw(16 + r);
        const double f = out3(a.mlpout, raw(r) + b3, &g1, &g2);
        // reverse through the transform: ybar = fbar g' + fdbar g'' yd, ydbar = fdbar g'
        const double ybar = fma(fbar, g1, fdbar * g2 * yd), ydbar = fdbar * g1;
        if (wv == 0 && lr == 0) {
          if (tile < ntile && p < npts) {
            a.fv[p] = f;
            a.fdv[p] = g1 * yd;
          }
          gb3 += ybar;
        }
        gW3 = fma(ybar, aL[0][v], fma(ydbar, aL[1][v], gW3));
        const double hb = ybar * w3, hdb = ydbar * w3;
        zb[0][v] = fma(hb, pl[0][v], hdb * ql[v] * tl[v]);
        zb[1][v] = hdb * pl[0][v];
      } else {
#pragma unroll
        for (int rb = 0; rb < 2; ++rb) {
          const int row = rb * 16 + r, p = tile * PTS + row;
          const double f = out3(a.mlpout, raw(row) + b3, &g1, &g2);
          const double ybar = sF[row] * g1;
          if (wv == 0 && lr == 0) {
            if (tile < ntile && p < npts) a.fv[p] = f;
            gb3 += ybar;
          }
          gW3 = fma(ybar, aL[rb][v], gW3);
          zb[rb][v] = ybar * w3 * pl[rb][v];
        }
      }
    }
    if constexpr (NL == 2) {
#pragma unroll
      for (int rb = 0; rb < 2; ++rb)
#pragma unroll
        for (int v = 0; v < 4; ++v) sZ[(rb * 16 + 4 * v + lk) * AS + col] = zb[rb][v];
#pragma unroll
      for (int v = 0; v < 4; ++v) gb2 += TAN ? zb[0][v] : zb[0][v] + zb[1][v];
      __syncthreads();
      // dW2 += a1^T zb (rows of values and tangents in one sum); adjoints of a1 = zb W2^T
#pragma unroll 2
      for (int q = 0; q < AROWS / 4; ++q) {
        const double b = sZ[(4 * q + lk) * AS + col];
#pragma unroll
        for (int rb = 0; rb < 4; ++rb)
          if (16 * rb < H1) gW2[rb] = mfma64(sA[(4 * q + lk) * AS + rb * 16 + lr], b, gW2[rb]);
      }
      z0 = z1 = zero;
#pragma unroll 4
      for (int q = 0; 4 * q < H2; ++q) {
          const double b = sW2[col * AS + 4 * q + lk];
          z0 = mfma64(sZ[lr * AS + 4 * q + lk], b, z0);
          z1 = mfma64(sZ[(16 + lr) * AS + 4 * q + lk], b, z1);
        }
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        if (TAN) {
          zb[0][v] = fma(z0[v], p1[0][v], z1[v] * q1[v] * t1[v]);
          zb[1][v] = z1[v] * p1[0][v];
        } else {
          zb[0][v] = z0[v] * p1[0][v];
          zb[1][v] = z1[v] * p1[1][v];
        }
      }
      __syncthreads();  // every wave has read the activations
    }
#pragma unroll
    for (int rb = 0; rb < 2; ++rb)
#pragma unroll
      for (int v = 0; v < 4; ++v) sA[(rb * 16 + 4 * v + lk) * AS + col] = col < H1 ? zb[rb][v] : 0.0;
#pragma unroll
    for (int v = 0; v < 4; ++v) gb1 += TAN ? zb[0][v] : zb[0][v] + zb[1][v];
    __syncthreads();
    // dW1 += x^T zb; window cotangents = zb W1^T
#pragma unroll 2
    for (int q = 0; q < AROWS / 4; ++q) {
      const double b = sA[(4 * q + lk) * AS + col];
#pragma unroll
      for (int rb = 0; rb < RB1; ++rb)
        if (16 * rb < W) gW1[rb] = mfma64(sX[(4 * q + lk) * AS + rb * 16 + lr], b, gW1[rb]);
    }
    if (wv * 16 < W) {
      z0 = z1 = zero;
#pragma unroll 4
      for (int q = 0; 4 * q < H1; ++q) {
          const double b = col < W ? sW1[col * AS + 4 * q + lk] : 0.0;
          z0 = mfma64(sA[lr * AS + 4 * q + lk], b, z0);
          if (!TAN) z1 = mfma64(sA[(16 + lr) * AS + 4 * q + lk], b, z1);
        }
#pragma unroll
      for (int rb = 0; rb < (TAN ? 1 : 2); ++rb)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const int p = tile * PTS + rb * 16 + 4 * v + lk;
          if (col < W && tile < ntile && p < npts) a.xbar[(size_t)p * W + col] = rb ? z1[v] : z0[v];
        }
    }
    __syncthreads();
  }
  // the groups add their partials into LDS one after another, then the sum goes to the
  // workgroup's slot (slots are owned: no races; a fixed order)
  auto over_rows = [&](double x) {
    x += __shfl_xor(x, 16, 64);
    return x + __shfl_xor(x, 32, 64);
  };
  gb1 = over_rows(gb1);
  gb2 = over_rows(gb2);
  gW3 = over_rows(gW3);
  gb3 = over_rows(gb3);
  double* r = sm;
  for (int g = 0; g < AG; ++g) {
    if (grp == g) {
      auto put = [&](int at, double x) { r[at] = g == 0 ? x : r[at] + x; };
#pragma unroll
      for (int rb = 0; rb < RB1; ++rb)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const int o = rb * 16 + 4 * v + lk;
          if (o < W && col < H1) put(a.w1 + o * H1 + col, gW1[rb][v]);
        }
      if constexpr (NL == 2) {
#pragma unroll
        for (int rb = 0; rb < 4; ++rb)
#pragma unroll
          for (int v = 0; v < 4; ++v) {
            const int k = rb * 16 + 4 * v + lk;
            if (k < H1 && col < H2) put(a.w2 + k * H2 + col, gW2[rb][v]);
          }
        if (lk == 0 && col < H2) put(a.b2 + col, gb2);
      }
      if (lk == 0 && col < H1) put(a.b1 + col, gb1);
      if (lk == 0 && col < HL) put(a.w3 + col, gW3);
      if (t == 0) put(a.b3, gb3);
    }
    __syncthreads();
  }
  double* g = a.thp + (size_t)blockIdx.x * a.P;
  for (int q0 = tid; q0 < a.P; q0 += 8 * ANT) {  // (8 loads in flight)
    double v[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = q0 + e * ANT < a.P ? g[q0 + e * ANT] : 0.0;
#pragma unroll
    for (int e = 0; e < 8; ++e)
      if (q0 + e * ANT < a.P) g[q0 + e * ANT] = v[e] + r[q0 + e * ANT];
  }
}

// Global-network second-order adjoint (GLOBAL_MLP: f(n) = g(MLP(n / norm)), one scalar per
// system).  Per system s: x = xin[s] / norm, tangent xt = tin[s] / norm (zero without tin),
// Phi = sf[s] f + fd fdot (sf null: 0; fdot = grad f . tin).  dst[s][i] += dPhi/dn_i (+ A2[s][i]);
// the parameter gradient of Phi is added to slot blockIdx.x.  A workgroup takes systems blockIdx.x,
// blockIdx.x + gridDim.x, ... in order, so each slot is written by one workgroup in a fixed order.
// Hidden widths <= 64: unit u of a layer is lane u of a wave; the input layer's sums over the N
// grid points are split over the 4 waves and combined in a fixed order.
// Bound by the latency of the weights' loads and of the partials' updates: 16 in flight a thread, 44 -> 26 us a launch
// for 5 systems (257-64-64-1).
template <int NL>
__global__ __launch_bounds__(NT) void k_adj_gmlp(Adj a, const double* xin, const double* tin, const double* sf,
                                                 double fd, const double* A2, double* dst) {
  extern __shared__ double sm[];
  constexpr int NW = NT / 64;
  const int N = a.N, H1 = a.H1, H2 = a.H2, HL = NL == 2 ? H2 : H1;
  const int t = threadIdx.x, u = t & 63, q = t >> 6;
  double* x = sm;                 // N
  double* xd = x + N;             // N
  double* part = xd + N;          // 2 x NW x 64
  double* h1 = part + 2 * NW * 64;  // activations, tangents, act', act'' and the two adjoints, 6 x 64
  double* h2 = h1 + 6 * 64;         // the same for layer 2
  double* sc = h2 + 6 * 64;         // scalars: fbar', fdbar'
  const double* W1 = a.mlp + a.w1;
  const double* W2 = a.mlp + a.w2;
  const double* W3 = a.mlp + a.w3;
  const double in = 1.0 / a.norm;
  double* g = a.thp + (size_t)blockIdx.x * a.P;
  for (int s = blockIdx.x; s < a.B; s += gridDim.x) {
    for (int i = t; i < N; i += NT) {
      x[i] = xin[(size_t)s * N + i] * in;
      xd[i] = tin ? tin[(size_t)s * N + i] * in : 0.0;
    }
    __syncthreads();
    // layer 1: z = b1 + W1^T x, zd = W1^T xd, the grid points split over the waves
    {
      double acc = 0.0, accd = 0.0;
      if (u < H1)
#pragma unroll 16
        for (int i = q; i < N; i += NW) {
          const double w = W1[(size_t)i * H1 + u];
          acc = fma(x[i], w, acc);
          accd = fma(xd[i], w, accd);
        }
      part[q * 64 + u] = acc;
      part[(NW + q) * 64 + u] = accd;
    }
    __syncthreads();
    if (t < H1) {
      double z = a.mlp[a.b1 + t], zd = 0.0;
      for (int w = 0; w < NW; ++w) {
        z += part[w * 64 + t];
        zd += part[(NW + w) * 64 + t];
      }
      double av, d1, d2;
      act3(a.act, z, &av, &d1, &d2);
      h1[t] = av;
      h1[64 + t] = d1 * zd;
      h1[128 + t] = d1;
      h1[192 + t] = d2;
      h1[256 + t] = zd;
    }
    __syncthreads();
    if (NL == 2 && t < H2) {
      double z = a.mlp[a.b2 + t], zd = 0.0;
#pragma unroll 16
      for (int v = 0; v < H1; ++v) {
        const double w = W2[v * H2 + t];
        z = fma(h1[v], w, z);
        zd = fma(h1[64 + v], w, zd);
      }
      double av, d1, d2;
      act3(a.act, z, &av, &d1, &d2);
      h2[t] = av;
      h2[64 + t] = d1 * zd;
      h2[128 + t] = d1;
      h2[192 + t] = d2;
      h2[256 + t] = zd;
    }
    __syncthreads();
    const double* hl = NL == 2 ? h2 : h1;
    if (t == 0) {
      double y = a.mlp[a.b3], yd = 0.0;
#pragma unroll 16
      for (int v = 0; v < HL; ++v) {
        y = fma(hl[v], W3[v], y);
        yd = fma(hl[64 + v], W3[v], yd);
      }
      double g1, g2;
      (void)out3(a.mlpout, y, &g1, &g2);
      const double fb = sf ? sf[s] : 0.0;
      sc[0] = fb * g1 + fd * g2 * yd;  // cotangent of y
      sc[1] = fd * g1;                 // cotangent of yd
      g[a.b3] += sc[0];
    }
    __syncthreads();
    const double yb = sc[0], ydb = sc[1];
    // last hidden layer: its adjoints (zb, zdb) from the output layer
    double* hL = NL == 2 ? h2 : h1;
    if (t < HL) {
      const double w = W3[t];
      g[a.w3 + t] += hL[t] * yb + hL[64 + t] * ydb;
      const double hb = yb * w, hdb = ydb * w;
      hL[320 + t] = hb * hL[128 + t] + hdb * hL[192 + t] * hL[256 + t];  // zb
      hL[256 + t] = hdb * hL[128 + t];                                 // zdb (zd no longer needed)
    }
    __syncthreads();
    if (NL == 2) {
      // W2 (H1 x H2): lane u = row, waves over the columns
      if (u < H1)
      {
        double w[HMAX / NW];
#pragma unroll
        for (int e = 0; e < HMAX / NW; ++e) w[e] = q + e * NW < H2 ? g[a.w2 + u * H2 + q + e * NW] : 0.0;
#pragma unroll
        for (int e = 0; e < HMAX / NW; ++e) {
          const int v = q + e * NW;
          if (v < H2) g[a.w2 + u * H2 + v] = w[e] + (h1[u] * h2[320 + v] + h1[64 + u] * h2[256 + v]);
        }
      }
      if (t < H2) g[a.b2 + t] += h2[320 + t];
      __syncthreads();
      if (t < H1) {
        double hb = 0.0, hdb = 0.0;
#pragma unroll 16
        for (int v = 0; v < H2; ++v) {
          const double w = W2[t * H2 + v];
          hb = fma(w, h2[320 + v], hb);
          hdb = fma(w, h2[256 + v], hdb);
        }
        const double zb = hb * h1[128 + t] + hdb * h1[192 + t] * h1[256 + t];
        h1[256 + t] = hdb * h1[128 + t];
        h1[320 + t] = zb;
      }
      __syncthreads();
    }
    // layer 1: W1 (N x H1), b1, and the input cotangent
    if (u < H1)
      for (int i0 = q; i0 < N; i0 += 16 * NW) {  // (16 loads in flight)
        double w[16];
#pragma unroll
        for (int e = 0; e < 16; ++e) w[e] = i0 + e * NW < N ? g[a.w1 + (size_t)(i0 + e * NW) * H1 + u] : 0.0;
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          const int i = i0 + e * NW;
          if (i < N) g[a.w1 + (size_t)i * H1 + u] = w[e] + (x[i] * h1[320 + u] + xd[i] * h1[256 + u]);
        }
      }
    if (t < H1) g[a.b1 + t] += h1[320 + t];
    for (int i = t; i < N; i += NT) {
      double xb = 0.0;
#pragma unroll 16
      for (int v = 0; v < H1; ++v) xb = fma(W1[(size_t)i * H1 + v], h1[320 + v], xb);
      double r = xb * in;
      if (A2) r += A2[(size_t)s * N + i];
      dst[(size_t)s * N + i] += r;
    }
    __syncthreads();
  }
}

// dst[s][i] += sa[s] * (A1[s][i] + F[s][i]) + A2[s][i] + window^T(xbar)_i / norm (A1, A2 optional)
__global__ void k_adj_gather(Adj a, double* dst, const double* A1, const double* A2, const double* F,
                             const double* sa) {
  const long idx = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= (long)a.B * a.N) return;
  const int s = (int)(idx / a.N), i = (int)(idx % a.N), N = a.N, W = a.W, h = W / 2;
  double acc = 0.0;
  for (int o = 0; o < W; ++o) {
    const int q = i - o + h;  // point whose window slot o reads n_i
    if (q >= 0 && q < N) acc += a.xbar[((size_t)s * N + q) * W + o];
  }
  double v = acc / a.norm;
  const double c = sa ? sa[s] : 1.0;
  double direct = F[idx];
  if (A1) direct += A1[idx];
  v = fma(c, direct, v);
  if (A2) v += A2[idx];
  dst[idx] += v;
}

// energy term: nob += c (-(v_H(n_k) + v_xc(n_k)) + v_H(n_out)) with c = dE dx (the v_xc(n_out) part
// is added by k_adj_gather from the MLP pass at n_out)
__global__ void k_adj_energy(Adj a, int k, const double* cs) {
  const long idx = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= (long)a.B * a.N) return;
  const int s = (int)(idx / a.N), i = (int)(idx % a.N);
  const size_t kk = ((size_t)s * a.T + k) * a.N + i;
  a.nob[idx] += cs[s] * (a.tmp[idx] - a.vh[kk] - a.vxc[kk]);
}

__global__ void k_adj_scales(Adj a, int k, double* cs, double* ones) {
  const int s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= a.B) return;
  cs[s] = (a.dE && k > a.sgs) ? a.dE[(size_t)s * a.T + k] * a.dx : 0.0;
  ones[s] = 1.0;
}

// eigen adjoint, one workgroup per system.
//
// Bound by the dependent chain of the banded solves.  One thread eliminating with partial pivoting takes 0.7 us a
// row; the substructured solve of one wave (band_wave.h) takes 5 us at N = 513 but does not pivot, so each solution
// is refined on its residual inside the complement of the occupied orbitals until that is at the rounding of
// (H - eps_j) x, and a system where SOLVES of them do not get there goes to the pivoted elimination.
// One occupied orbital: N = 513 (32 systems) 386 -> 22 us a launch, N = 257 190 -> 15 us; one solve is at rounding
// there, so most of what is left is latency of the projections and loads.
// LDS: H diagonal, r, y, vbar, x, w and the factors of the wave (the rows of U of the pivoted elimination).
constexpr int SOLVES = 5;
size_t adj_eig_lds(int N) { return ((size_t)6 * N + qexband::wave_doubles(N)) * 8; }
__global__ __launch_bounds__(NT) void k_adj_eig(Adj a, int k, double Td, double Tb, double Tc) {
  extern __shared__ double sm[];
  __shared__ double red[NT / 64];
  __shared__ double eps[QEX1D_MAX_ELECTRONS / 2 + 1];
  const int s = blockIdx.x, N = a.N, T = a.T;
  double* hd = sm;       // N
  double* r = hd + N;    // N
  double* y = r + N;     // N
  double* vb = y + N;    // N
  double* x = vb + N;    // N
  double* w = x + N;     // N
  double* F = w + N;     // factors
  const int ne = a.ne[s], nocc = (ne + 1) / 2;
  const double* vxc = a.vxc + ((size_t)s * T + k) * N;
  const double* vh = a.vh + ((size_t)s * T + k) * N;
  const double* ve = a.vext + (size_t)s * N;
  const double* psi = a.orb + ((size_t)s * T + k) * a.K * N;
  const double* nob = a.nob + (size_t)s * N;
  double hmax = 0.0;
  for (int t = threadIdx.x; t < N; t += NT) {
    const double h = Td + ve[t] + vh[t] + vxc[t];
    hd[t] = h;
    hmax = fmax(hmax, fabs(h));
    vb[t] = 0.0;
  }
  hmax = bmax(hmax, red);
  // (H p)_t of a vector in memory or LDS
  auto apply = [&](const double* p, int t) {
    double hx = hd[t] * p[t];
    if (t >= 1) hx = fma(Tb, p[t - 1], hx);
    if (t + 1 < N) hx = fma(Tb, p[t + 1], hx);
    if (t >= 2) hx = fma(Tc, p[t - 2], hx);
    if (t + 2 < N) hx = fma(Tc, p[t + 2], hx);
    return hx;
  };
  // eigenvalues as Rayleigh quotients of the stored orbitals
  for (int j = 0; j < nocc; ++j) {
    const double* pj = psi + (size_t)j * N;
    double q = 0.0;
    for (int t = threadIdx.x; t < N; t += NT) q = fma(pj[t], apply(pj, t), q);
    q = bsum(q, red);
    if (threadIdx.x == 0) eps[j] = q;
  }
  __syncthreads();
  const double hnorm = hmax + 2.0 * fabs(Tb) + 2.0 * fabs(Tc), rounding = 2.220446049250313e-16 * hnorm;
  // v <- Q v, the occupied orbitals projected out one after another
  auto project = [&](double* v) {
    for (int b = 0; b < nocc; ++b) {
      const double* pb = psi + (size_t)b * N;
      double d = 0.0;
      for (int t = threadIdx.x; t < N; t += NT) d = fma(pb[t], v[t], d);
      d = bsum(d, red);
      for (int t = threadIdx.x; t < N; t += NT) v[t] = fma(-d, pb[t], v[t]);
    }
  };
  for (int j = 0; j < nocc; ++j) {
    const double* pj = psi + (size_t)j * N;
    const double oj = occupation(ne, j), ej = eps[j];
    // rhs = Q r
    for (int t = threadIdx.x; t < N; t += NT) {
      const double v = nob[t] * pj[t];
      r[t] = v;
      y[t] = v;
      x[t] = 0.0;
    }
    project(y);
    for (int t = threadIdx.x; t < N; t += NT) w[t] = y[t];
    bool solved = false;
    for (int it = 0; it < SOLVES && !solved; ++it) {
      __syncthreads();
      if (threadIdx.x < 64) qexband::wave_solve<true>(hd, w, N, Tb, Tc, ej, F);
      __syncthreads();
      project(w);
      double xx = 0.0, rr = 0.0;
      for (int t = threadIdx.x; t < N; t += NT) {
        x[t] += w[t];
        xx = fma(x[t], x[t], xx);
      }
      __syncthreads();
      for (int t = threadIdx.x; t < N; t += NT) w[t] = fma(ej, x[t], y[t]) - apply(x, t);
      project(w);
      for (int t = threadIdx.x; t < N; t += NT) rr = fma(w[t], w[t], rr);
      rr = bsum(rr, red);
      xx = bsum(xx, red);
      solved = rr <= 16.0 * rounding * rounding * xx;
    }
    if (!solved) {
      // (the solution's component along psi_j is projected out)
      for (int t = threadIdx.x; t < N; t += NT) x[t] = y[t];
      __syncthreads();
      if (threadIdx.x == 0) qexband::pivoted_solve(hd, x, F, N, Tb, Tc, ej, rounding);
    }
    __syncthreads();
    // x <- Q x; y_j = -x - sum over occupied b with occ_b != occ_j of psi_b (psi_b . r) / (eps_b - eps_j)
    for (int b = 0; b < nocc; ++b) {
      const double* pb = psi + (size_t)b * N;
      double d = 0.0, dr = 0.0;
      for (int t = threadIdx.x; t < N; t += NT) {
        d = fma(pb[t], x[t], d);
        dr = fma(pb[t], r[t], dr);
      }
      d = bsum(d, red);
      dr = bsum(dr, red);
      const double ob = occupation(ne, b);
      const double extra = (b != j && ob != oj) ? dr / (eps[b] - ej) : 0.0;
      // the final y_j = -(Q x) - sum extra psi_b  ->  accumulate as x - d psi_b + extra psi_b, negated below
      for (int t = threadIdx.x; t < N; t += NT) x[t] = fma(extra - d, pb[t], x[t]);
    }
    const double sc = -oj * 2.0 / a.dx;
    for (int t = threadIdx.x; t < N; t += NT) vb[t] = fma(sc * pj[t], x[t], vb[t]);
    __syncthreads();
  }
  for (int t = threadIdx.x; t < N; t += NT) a.vbar[(size_t)s * N + t] = vb[t];
}

// the input densities n_k of all systems, contiguous [B][N]
__global__ void k_adj_gather_input(Adj a, int k, double* dst) {
  const long idx = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= (long)a.B * a.N) return;
  const int s = (int)(idx / a.N), i = (int)(idx % a.N);
  dst[idx] = input_density(a, s, k)[i];
}

// grad[q] = sum over slots of thp[slot][q]: 32 parameters per workgroup, 8 interleaved partial
// sums each, combined in a fixed order
__global__ __launch_bounds__(256) void k_adj_reduce(int P, const double* thp, double* grad) {
  __shared__ double red[8][33];
  const int t = threadIdx.x, q = blockIdx.x * 32 + (t & 31), part = t >> 5;
  double g = 0.0;
  if (q < P)
    for (int sl = part; sl < ADJ_WG; sl += 8) g += thp[(size_t)sl * P + q];
  red[part][t & 31] = g;
  __syncthreads();
  if (t < 32 && q < P) {
    double v = 0.0;
    for (int k = 0; k < 8; ++k) v += red[k][t];
    grad[q] = v;
  }
}

size_t al(size_t x) { return (x + 255) & ~(size_t)255; }

struct LayA {
  size_t nbar, nob, nout, vbar, tmp, dbar, xbar, fv, fdv, thp, cs, ones, total;
};

int adj_check(const qex1d_problem* p) {
  if (!p) return faila(QEX_E_BADARG, "null problem");
  if (p->batch < 1 || p->num_grids < 5 || p->num_grids > QEX1D_MAX_GRIDS || !(p->dx > 0.0) || p->num_iterations < 1 ||
      p->max_electrons < 1 || p->max_electrons > QEX1D_MAX_ELECTRONS || p->num_mixing_iterations < 1)
    return faila(QEX_E_BADARG, "bad problem sizes");
  // with density_mse_converge_tolerance < 0 (checked below) the two loop kinds differ only in the
  // reflection window, which the reverse pass takes per system
  if (p->loop != QEX1D_LOOP_SCAN && p->loop != QEX1D_LOOP_PYTHON) return faila(QEX_E_BADARG, "bad loop kind");
  if (!(p->density_mse_converge_tolerance < 0.0))
    return faila(QEX_E_UNSUPPORTED, "the reverse pass needs density_mse_converge_tolerance < 0 (no frozen states)");
  const bool glob = p->xc_kind == QEX1D_XC_GLOBAL_MLP;
  if (p->xc_kind != QEX1D_XC_LOCAL_MLP && !glob)
    return faila(QEX_E_UNSUPPORTED, "the reverse pass needs a LOCAL_MLP or GLOBAL_MLP functional");
  if (p->mlp_layers != 2 && p->mlp_layers != 3)
    return faila(QEX_E_UNSUPPORTED, "the reverse pass supports 1 or 2 hidden layers");
  if (glob) {
    if (p->mlp_widths[0] != p->num_grids) return faila(QEX_E_BADARG, "GLOBAL_MLP input width must be num_grids");
  } else if (p->mlp_widths[0] < 1 || p->mlp_widths[0] > WMAXW || p->mlp_widths[0] % 2 == 0) {
    return faila(QEX_E_UNSUPPORTED, "window must be odd and <= %d", WMAXW);
  }
  for (int l = 1; l < p->mlp_layers; ++l)
    if (p->mlp_widths[l] < 1 || p->mlp_widths[l] > HMAX)
      return faila(QEX_E_UNSUPPORTED, "hidden widths must be in [1, %d] for the reverse pass", HMAX);
  if (p->mlp_widths[p->mlp_layers] != 1) return faila(QEX_E_UNSUPPORTED, "MLP output width must be 1");
  if (p->mlp_activation < 0 || p->mlp_activation > QEX_ACT_GELU_TANH || !(p->mlp_norm != 0.0))
    return faila(QEX_E_BADARG, "bad activation or norm");
  if (p->mlp_output != QEX1D_MLP_OUTPUT_LINEAR && p->mlp_output != QEX1D_MLP_OUTPUT_NEGATIVITY)
    return faila(QEX_E_BADARG, "bad mlp_output");
  if (p->stop_gradient_iterations < 0) return faila(QEX_E_BADARG, "stop_gradient_iterations must be >= 0");
  return QEX_OK;
}

int param_count(const qex1d_problem* p) {
  int n = 0;
  for (int l = 0; l < p->mlp_layers; ++l) n += p->mlp_widths[l] * p->mlp_widths[l + 1] + p->mlp_widths[l + 1];
  return n;
}

LayA layout_adj(const qex1d_problem* p) {
  LayA L{};
  size_t off = 0;
  const size_t B = p->batch, N = p->num_grids, T = p->num_iterations;
  const size_t W = p->xc_kind == QEX1D_XC_GLOBAL_MLP ? 0 : p->mlp_widths[0];  // window cotangents (local only)
  auto take = [&](size_t b) {
    const size_t o = off;
    off = al(off + b);
    return o;
  };
  L.nbar = take(B * N * 8);
  L.nob = take(B * N * 8);
  L.nout = take(B * N * 8);
  L.vbar = take(B * N * 8);
  L.tmp = take(B * N * 8);
  L.dbar = take(B * T * N * 8);
  L.xbar = take(B * N * W * 8);
  L.fv = take(B * N * 8);
  L.fdv = take(B * N * 8);
  L.thp = take((size_t)ADJ_WG * param_count(p) * 8);
  L.cs = take(B * 8);
  L.ones = take(B * 8);
  L.total = off;
  return L;
}

}  // namespace

extern "C" {

const char* qex1d_vjp_last_error(void) { return g_erra; }

size_t qex1d_kohn_sham_vjp_workspace_bytes(const qex1d_problem* p) {
  if (adj_check(p) != QEX_OK) return 0;
  return layout_adj(p).total;
}

int qex1d_kohn_sham_vjp(const qex1d_problem* p, const qex1d_inputs* in, const qex1d_outputs* fwd,
                        const double* d_total_energy, const double* d_density, double* d_xc_params, void* workspace,
                        size_t workspace_bytes, void* stream_) {
  int rc = adj_check(p);
  if (rc) return rc;
  if (!in || !fwd || !d_xc_params) return faila(QEX_E_BADARG, "null inputs, forward outputs or gradient");
  if (!in->interaction_table || !in->external_potential || !in->initial_density || !in->num_electrons ||
      !in->xc_params)
    return faila(QEX_E_BADARG, "missing forward inputs");
  if (!fwd->density || !fwd->hartree_potential || !fwd->xc_potential || !fwd->orbitals)
    return faila(QEX_E_BADARG, "the forward outputs density, hartree_potential, xc_potential and orbitals are required");
  if (p->reflect && !in->reflect_window) return faila(QEX_E_BADARG, "reflection needs reflect_window");
  const size_t need = layout_adj(p).total;
  if (!workspace || workspace_bytes < need) return faila(QEX_E_WORKSPACE, "workspace too small: need %zu", need);
  hipStream_t st = (hipStream_t)stream_;
  const LayA L = layout_adj(p);
  char* ws = (char*)workspace;
  Adj a{};
  a.B = p->batch;
  a.N = p->num_grids;
  a.T = p->num_iterations;
  a.K = p->max_electrons / 2 + 1;
  a.M = p->num_mixing_iterations;
  a.W = p->mlp_widths[0];
  a.NL = p->mlp_layers - 1;
  a.H1 = p->mlp_widths[1];
  a.H2 = a.NL == 2 ? p->mlp_widths[2] : 0;
  a.act = p->mlp_activation;
  a.mlpout = p->mlp_output;
  a.reflect = p->reflect ? 1 : 0;
  a.win = in->reflect_window;
  a.sgs = p->stop_gradient_iterations - 1;  // last stopped iteration (-1: none)
  a.P = param_count(p);
  a.dx = p->dx;
  a.norm = p->mlp_norm;
  int off = 0;
  a.w1 = off;
  off += a.W * a.H1;
  a.b1 = off;
  off += a.H1;
  if (a.NL == 2) {
    a.w2 = off;
    off += a.H1 * a.H2;
    a.b2 = off;
    off += a.H2;
  }
  a.w3 = off;
  off += a.NL == 2 ? a.H2 : a.H1;
  a.b3 = off;
  a.table = in->interaction_table;
  a.vext = in->external_potential;
  a.n0 = in->initial_density;
  a.ne = in->num_electrons;
  a.mlp = in->xc_params;
  a.dens = fwd->density;
  a.vh = fwd->hartree_potential;
  a.vxc = fwd->xc_potential;
  a.orb = fwd->orbitals;
  a.dE = d_total_energy;
  a.dn = d_density;
  a.nbar = (double*)(ws + L.nbar);
  a.nob = (double*)(ws + L.nob);
  a.nout = (double*)(ws + L.nout);
  a.vbar = (double*)(ws + L.vbar);
  a.tmp = (double*)(ws + L.tmp);
  a.dbar = (double*)(ws + L.dbar);
  a.xbar = (double*)(ws + L.xbar);
  a.fv = (double*)(ws + L.fv);
  a.fdv = (double*)(ws + L.fdv);
  a.thp = (double*)(ws + L.thp);
  double* cs = (double*)(ws + L.cs);
  double* ones = (double*)(ws + L.ones);
  const long BN = (long)a.B * a.N;
  const double s2 = -0.5 / (a.dx * a.dx);
  const double Td = s2 * -2.5, Tb = s2 * (4.0 / 3.0), Tc = s2 * (-1.0 / 12.0);
  const size_t eig_lds = adj_eig_lds(a.N);
  const bool glob = p->xc_kind == QEX1D_XC_GLOBAL_MLP;
  const size_t gmlp_lds = (2 * (size_t)a.N + 2 * (NT / 64) * 64 + 12 * 64 + 8) * 8;
  if (eig_lds > 64 * 1024)
    (void)hipFuncSetAttribute((const void*)k_adj_eig, hipFuncAttributeMaxDynamicSharedMemorySize, (int)eig_lds);
  if (!glob) {
    const void* fns[4] = {(const void*)k_adj_mlp<1, false>, (const void*)k_adj_mlp<1, true>,
                          (const void*)k_adj_mlp<2, false>, (const void*)k_adj_mlp<2, true>};
    for (const void* f : fns) (void)hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, (int)ADJ_MLP_LDS);
  }
  auto mlp = [&](const double* xin, const double* tin, const double* F1, const double* sf, const double* F2) {
    qexprof::Scope ps(qexprof::K_ADJ_MLP, st);
    qextile::for_launches(a.B, a.N, [&](int s0, int n) {
      const size_t p0 = (size_t)s0 * a.N;
      Adj q = a;
      q.B = n;
      q.fv += p0;
      q.fdv += p0;
      q.xbar += p0 * a.W;
      const long tiles = ((long)n * a.N + (tin ? 15 : 31)) / (tin ? 16 : 32);
      const dim3 grid((unsigned)(tiles < ADJ_WG ? tiles : ADJ_WG)), block(ANT);
      auto launch = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, grid, block, ADJ_MLP_LDS, st, q, xin + p0, tin ? tin + p0 : nullptr, F1 + p0, sf + s0,
                           F2 ? F2 + p0 : nullptr);
      };
      if (a.NL == 2 && tin)
        launch(k_adj_mlp<2, true>);
      else if (a.NL == 2)
        launch(k_adj_mlp<2, false>);
      else if (tin)
        launch(k_adj_mlp<1, true>);
      else
        launch(k_adj_mlp<1, false>);
    });
  };
  // the global network: one workgroup per system (at most ADJ_WG, each then taking several in turn)
  const unsigned gG = (unsigned)(a.B < ADJ_WG ? a.B : ADJ_WG);
  auto gmlp = [&](const double* xin, const double* tin, const double* sf, double fd, const double* A2, double* dst) {
    qexprof::Scope ps(qexprof::K_ADJ_MLP, st);
    if (a.NL == 2)
      hipLaunchKernelGGL(k_adj_gmlp<2>, dim3(gG), dim3(NT), gmlp_lds, st, a, xin, tin, sf, fd, A2, dst);
    else
      hipLaunchKernelGGL(k_adj_gmlp<1>, dim3(gG), dim3(NT), gmlp_lds, st, a, xin, tin, sf, fd, A2, dst);
  };
  const unsigned gBN = (unsigned)((BN + NT - 1) / NT);
  // alpha_k as the forward computes it
  double alphas[4096];
  if (a.T > 4096) return faila(QEX_E_UNSUPPORTED, "too many iterations");
  double al_k = p->alpha;
  for (int k = 0; k < a.T; ++k) {
    alphas[k] = al_k;
    al_k *= p->alpha_decay;
  }
  {
    hipLaunchKernelGGL(k_zero_a, dim3(256), dim3(NT), 0, st, a.nbar, BN);
    hipLaunchKernelGGL(k_zero_a, dim3(256), dim3(NT), 0, st, a.dbar, BN * a.T);
    hipLaunchKernelGGL(k_zero_a, dim3(1024), dim3(NT), 0, st, a.thp, (long)ADJ_WG * a.P);
    // with one mixing difference nothing reaches the stopped iterations; with more,
    // the differences of those iterations still enter later mixes and are reversed
    const int k_end = a.M == 1 ? (a.sgs >= 0 ? a.sgs + 1 : 0) : 0;
    for (int k = a.T - 1; k >= k_end; --k) {
      hipLaunchKernelGGL(k_adj_mix, dim3(a.B), dim3(NT), 0, st, a, k, alphas[k]);
      hipLaunchKernelGGL(k_adj_scales, dim3((a.B + 63) / 64), dim3(64), 0, st, a, k, cs, ones);
      // with reflection the density passed on is S n_raw: its cotangent maps to S dbar_k on n_raw
      if (a.reflect) hipLaunchKernelGGL(k_sym_inplace, dim3(gBN), dim3(NT), 0, st, a, a.nob);
      // energy: v_H(n_raw) and the MLP at the XC density of the energy (n_raw, or S n_raw with reflection)
      hipLaunchKernelGGL(k_toeplitz, dim3((a.N + NT - 1) / NT, a.B), dim3(NT), (size_t)2 * a.N * 8, st, a.N, a.dx,
                         a.table, a.nout, a.tmp);
      hipLaunchKernelGGL(k_adj_energy, dim3(gBN), dim3(NT), 0, st, a, k, cs);
      if (glob) {
        // dx f(n_raw): nob += c grad f(n_raw), thetabar += c df/dtheta (no flip of the XC input)
        gmlp(a.nout, nullptr, cs, 0.0, nullptr, a.nob);
      } else if (a.reflect) {
        // dx F(S n_raw): nob += c S grad F(S n_raw) (vbar and tmp are free until the eigen adjoint)
        hipLaunchKernelGGL(k_sym_copy, dim3(gBN), dim3(NT), 0, st, a, a.vbar, a.nout);
        mlp(a.vbar, nullptr, a.vbar, cs, nullptr);
        hipLaunchKernelGGL(k_zero_a, dim3(256), dim3(NT), 0, st, a.tmp, BN);
        hipLaunchKernelGGL(k_adj_gather, dim3(gBN), dim3(NT), 0, st, a, a.tmp, nullptr, nullptr, a.fv, cs);
        hipLaunchKernelGGL(k_sym_add, dim3(gBN), dim3(NT), 0, st, a, a.nob, a.tmp, nullptr);
      } else {
        mlp(a.nout, nullptr, a.nout, cs, nullptr);
        hipLaunchKernelGGL(k_adj_gather, dim3(gBN), dim3(NT), 0, st, a, a.nob, nullptr, nullptr, a.fv, cs);
      }
      // eigen adjoint: nob -> vbar
      {
        qexprof::Scope ps(qexprof::K_ADJ_EIG, st);
        hipLaunchKernelGGL(k_adj_eig, dim3(a.B), dim3(NT), eig_lds, st, a, k, Td, Tb, Tc);
      }
      // Hartree and XC: nbar += dx U vbar + H_F vbar
      hipLaunchKernelGGL(k_toeplitz, dim3((a.N + NT - 1) / NT, a.B), dim3(NT), (size_t)2 * a.N * 8, st, a.N, a.dx,
                         a.table, a.vbar, a.tmp);
      // the input densities n_k of all systems, gathered contiguously into nout (free again)
      hipLaunchKernelGGL(k_adj_gather_input, dim3(gBN), dim3(NT), 0, st, a, k, a.nout);
      if (glob) {
        // v_xc = dx grad f: nbar += dx U vbar + dx H_f vbar, thetabar += dx d(vbar . grad f)/dtheta
        gmlp(a.nout, a.vbar, nullptr, a.dx, a.tmp, a.nbar);
      } else if (a.reflect) {
        // v_xc(n) = S grad F(S n): the second-order adjoint at (S n, S vbar), its n-cotangent mapped by S
        hipLaunchKernelGGL(k_sym_inplace, dim3(gBN), dim3(NT), 0, st, a, a.nout);
        hipLaunchKernelGGL(k_sym_inplace, dim3(gBN), dim3(NT), 0, st, a, a.vbar);
        mlp(a.nout, a.vbar, a.vbar, ones, a.nout);
        hipLaunchKernelGGL(k_zero_a, dim3(256), dim3(NT), 0, st, a.nob, BN);
        hipLaunchKernelGGL(k_adj_gather, dim3(gBN), dim3(NT), 0, st, a, a.nob, nullptr, nullptr, a.fdv, ones);
        hipLaunchKernelGGL(k_sym_add, dim3(gBN), dim3(NT), 0, st, a, a.nbar, a.nob, a.tmp);
      } else {
        mlp(a.nout, a.vbar, a.vbar, ones, a.nout);
        hipLaunchKernelGGL(k_adj_gather, dim3(gBN), dim3(NT), 0, st, a, a.nbar, nullptr, a.tmp, a.fdv, ones);
      }
    }
    hipLaunchKernelGGL(k_adj_reduce, dim3((a.P + 31) / 32), dim3(256), 0, st, a.P, a.thp, d_xc_params);
  }
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return faila(QEX_E_LAUNCH, "qex1d_kohn_sham_vjp: %s", hipGetErrorString(e));
  return QEX_OK;
}

}  // extern "C"
