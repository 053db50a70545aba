// Learned initial guesses for the implicit radiation solve and the u2p W
// inversion: a small MLP
// (11 -> 128 -> 128 -> 128 -> 4, GELU in tanh form) that maps the
// dimensionless local state of a cell to corrections of the plain Newton
// start.  A gas network corrects (u, u~^1..3), a radiation network
// (E, F~^1..3); the solve picks one per cell.  A W network (kind 2)
// predicts the start of the W Newton iteration of u2p.  Training is FP32 (forward,
// backward and Adam kernels below, deterministic reductions); inference runs
// the weights in BF16 on the matrix cores (v_mfma_f32_16x16x16_bf16, FP32
// accumulation).
//
// Parameters: one FP32 vector W1[128][11], b1, W2[128][128], b2, W3[128][128],
// b3, W4[4][128], b4 (row-major W[out][in]).  Normalisation: feature mean and
// std (11 + 11), target mean and std (4 + 4).
//
// Features of a cell: log10 rho, log10(u/rho), log10(E/u), gas u~^i (3),
// radiation-frame u~^i (3), log10(dt kappa_abs), log10(dt kappa_es).
// Targets between the converged energy-equation lab-frame state (x*) and the
// initial state (x0) of the network's four primitives: log(x*_0 / x0_0) and
// asinh((x*_i - x0_i) / VSCALE) for the three velocity components.
#include <hip/hip_runtime.h>
#include <math.h>
#include <type_traits>
#include "koral_hip.h"
#include "dev_cell.hpp"
#include "capi_util.hpp"

using namespace kd;

namespace {

constexpr int NIN = 11, NH = 128, NOUT = 4;
constexpr int OW1 = 0, OB1 = OW1 + NH * NIN, OW2 = OB1 + NH, OB2 = OW2 + NH * NH, OW3 = OB2 + NH,
              OB3 = OW3 + NH * NH, OW4 = OB3 + NH, OB4 = OW4 + NOUT * NH, NPARAM = OB4 + NOUT;
constexpr int NNORM = 2 * NIN + 2 * NOUT;  // feature mean, std, target mean, std
constexpr int BMAX = 4096;                 // largest training batch
constexpr float C_GELU = 0.7978845608028654f;
// velocity-like targets are asinh(delta / VSCALE): linear below VSCALE,
// logarithmic above, so changes from 1e-10 to 1 carry comparable weight
constexpr double VSCALE = 1e-6;

__device__ __forceinline__ float gelu(float z)
{
  return 0.5f * z * (1.f + tanhf(C_GELU * (z + 0.044715f * z * z * z)));
}

// ---------------------------------------------------------------------------
// features and targets
// ---------------------------------------------------------------------------
template <int MAG>
__global__ void __launch_bounds__(256) k_features(koral_params P, long n, const double *__restrict__ pp,
                                                  const double *__restrict__ dt, const float *__restrict__ norm,
                                                  float *__restrict__ feat)
{
  constexpr int EE = Lay<MAG, 1>::EE;
  long c = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= n) return;
  const double rho = pp[0 * n + c], u = pp[1 * n + c], E = pp[EE * n + c], d = dt[c];
  double f[NIN];
  f[0] = log10(rho);
  f[1] = log10(u / rho);
  f[2] = log10(E / u);
  f[3] = pp[2 * n + c];
  f[4] = pp[3 * n + c];
  f[5] = pp[4 * n + c];
  f[6] = pp[(EE + 1) * n + c];
  f[7] = pp[(EE + 2) * n + c];
  f[8] = pp[(EE + 3) * n + c];
  f[9] = log10(d * kappa_abs(P, rho, u));
  f[10] = log10(d * kappa_es(P, rho));
#pragma unroll
  for (int k = 0; k < NIN; k++) {
    float v = (float)f[k];
    if (norm) v = (v - norm[k]) / norm[NIN + k];
    feat[k * n + c] = v;
  }
}

__global__ void __launch_bounds__(256) k_targets(long n, int base, const double *__restrict__ p0,
                                                 const double *__restrict__ p1, float *__restrict__ t)
{
  long c = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= n) return;
  t[c] = (float)log(p1[base * n + c] / p0[base * n + c]);
#pragma unroll
  for (int i = 1; i < NOUT; i++)
    t[i * n + c] = (float)asinh((p1[(base + i) * n + c] - p0[(base + i) * n + c]) / VSCALE);
}

// The W network (kind 2): features of a point of the u2p W inversion from
// its conserved state uu and the guess pp (the primitives the inversion
// starts from), and the target log(W1 / W0) between the solution pp1 and
// the guess pp0.  W = (rho + Gamma u) gamma^2, the start u2p.c:2094-2112
// computes from a primitive state.
template <int MAG>
__device__ __forceinline__ double plain_W(const koral_params &P, const double *p, const Geom &g)
{
  return (p[0] + P.gamma * p[1]) * (1. + qsq_of(p[2], p[3], p[4], g));
}

template <int MAG>
__device__ __forceinline__ void load_mhd(const double *__restrict__ a, long n, long c, double *x)
{
  constexpr int NVM = 6 + 3 * MAG;
#pragma unroll
  for (int k = 0; k < 9; k++) x[k] = k < NVM ? a[k * n + c] : 0.;
}

template <int MAG>
__global__ void __launch_bounds__(256) k_u2p_features(koral_params P, long n, const double *__restrict__ uu,
                                                      const double *__restrict__ pp, const double *__restrict__ g20,
                                                      const double *__restrict__ G20, const float *__restrict__ norm,
                                                      float *__restrict__ feat)
{
  long c = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= n) return;
  Geom g;
  load_geom(g, [&](int k) { return g20[k * n + c]; }, [&](int k) { return G20[k * n + c]; });
  double p[9], U[9], U0[9];
  load_mhd<MAG>(pp, n, c, p);
  load_mhd<MAG>(uu, n, c, U);
  p2u_mhd<MAG, 0>(P, p, U0, g);
  const double rho = p[0], u = p[1];
  double bsq = 0.;
  if (MAG) {
    double ucon[4], ucov[4], bcon[4], bcov[4];
    relr_to_4vel(p[2], p[3], p[4], ucon, ucov, g);
    bcon4(p[6], p[7], p[8], ucon, ucov, bcon);
    lower(bcon, bcov, g);
    bsq = dot4(bcon, bcov);
  }
  double f[NIN];
  f[0] = log10(u / rho);
  f[1] = log10(bsq / rho + 1e-30);
#pragma unroll
  for (int i = 0; i < 3; i++) f[2 + i] = p[2 + i] * sqrt(g.g[1 + i][1 + i]);
  f[5] = log(U[0] / U0[0]);
  f[6] = asinh((U[1] - U0[1]) / fabs(U0[1]));
  const double s2 = fabs(U0[0]) + fabs(U0[1]);
#pragma unroll
  for (int i = 0; i < 3; i++) f[7 + i] = asinh((U[2 + i] - U0[2 + i]) / s2);
  f[10] = log10(plain_W<MAG>(P, p, g) / rho);
#pragma unroll
  for (int k = 0; k < NIN; k++) {
    float v = (float)f[k];
    if (norm) v = (v - norm[k]) / norm[NIN + k];
    feat[k * n + c] = v;
  }
}

template <int MAG>
__global__ void __launch_bounds__(256) k_u2p_targets(koral_params P, long n, const double *__restrict__ p0,
                                                     const double *__restrict__ p1, const double *__restrict__ g20,
                                                     const double *__restrict__ G20, float *__restrict__ t)
{
  long c = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= n) return;
  Geom g;
  load_geom(g, [&](int k) { return g20[k * n + c]; }, [&](int k) { return G20[k * n + c]; });
  double a[9], b[9];
  load_mhd<MAG>(p0, n, c, a);
  load_mhd<MAG>(p1, n, c, b);
  t[c] = (float)log(plain_W<MAG>(P, b, g) / plain_W<MAG>(P, a, g));
#pragma unroll
  for (int i = 1; i < NOUT; i++) t[i * n + c] = 0.f;
}

template <int MAG>
__global__ void __launch_bounds__(256) k_u2p_guess(koral_params P, long n, const double *__restrict__ pp,
                                                   const double *__restrict__ g20, const double *__restrict__ G20,
                                                   const float *__restrict__ y, const float *__restrict__ norm,
                                                   double *__restrict__ W0)
{
  long c = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= n) return;
  Geom g;
  load_geom(g, [&](int k) { return g20[k * n + c]; }, [&](int k) { return G20[k * n + c]; });
  double p[9];
  load_mhd<MAG>(pp, n, c, p);
  const double t = (double)y[c] * norm[2 * NIN + NOUT] + norm[2 * NIN];
  const double w = plain_W<MAG>(P, p, g) * exp(t);
  W0[c] = (isfinite(w) && w > 0.) ? w : 0.;
}

// ---------------------------------------------------------------------------
// FP32 training kernels.  A step of B samples is three launches: k_mlp_pass
// (forward, loss, and backward to every layer's dZ), k_mlp_grad (weight and
// bias gradients, summed over chunks of CHUNK samples) and k_mlp_reduce (the
// chunks' sum in a fixed order, and the Adam update).  All products run on the
// FP32 matrix cores (v_mfma_f32_16x16x4_f32: lane l holds A[l%16][l/16],
// B[l/16][l%16] and D[4(l/16)..+3][l%16]; FP32 products and sums).  A step of
// 4096 samples is 0.9 GFLOP, 6 us at the matrix cores' rate; with one thread
// per output and a launch per layer it took 290 us (16 launches), most of it
// re-reading operands.
// ---------------------------------------------------------------------------
typedef float f32x4 __attribute__((ext_vector_type(4)));
constexpr int TILE = 16;    // samples of a k_mlp_pass block: 4096 samples give each CU one
constexpr int CHUNK = 64;   // samples of a k_mlp_grad block
constexpr int SMAX = BMAX / CHUNK;
constexpr int HS = 20;      // LDS row stride of a [feature][TILE] activation tile: the four
                            // quarters of a wave read rows 4 apart, 16 banks from each other

__device__ __forceinline__ f32x4 mfma4(float a, float b, f32x4 c)
{
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// a = gelu(z) and its derivative from one tanh
__device__ __forceinline__ void gelu_both(float z, float &a, float &d)
{
  float t = tanhf(C_GELU * (z + 0.044715f * z * z * z));
  a = 0.5f * z * (1.f + t);
  d = 0.5f * (1.f + t) + 0.5f * z * (1.f - t * t) * C_GELU * (1.f + 3.f * 0.044715f * z * z);
}

// A lane's weights of two 16-row tiles of W h (W [128][128], rows o and
// o + 16): lane quarter q takes inputs 16 j + 4 q + r, one 16-byte load each j.
// They are loaded a layer ahead, so that no layer waits for them.
struct RowsW {
  f32x4 w[2][NH / 16];
};
__device__ __forceinline__ void load_rows(const float *__restrict__ W, int o, int q, RowsW &k)
{
#pragma unroll
  for (int j = 0; j < NH / 16; j++)
#pragma unroll
    for (int t = 0; t < 2; t++) k.w[t][j] = *(const f32x4 *)(W + (o + 16 * t) * NH + 16 * j + 4 * q);
}
// the same of W^T h: columns i and i + 16 of W
__device__ __forceinline__ void load_cols(const float *__restrict__ W, int i, int q, RowsW &k)
{
#pragma unroll
  for (int j = 0; j < NH / 16; j++)
#pragma unroll
    for (int r = 0; r < 4; r++)
#pragma unroll
      for (int t = 0; t < 2; t++) k.w[t][j][r] = W[(16 * j + 4 * q + r) * NH + i + 16 * t];
}
__device__ __forceinline__ void dense(const RowsW &k, const float (*h)[HS], int q, int b, f32x4 acc[2])
{
#pragma unroll
  for (int j = 0; j < NH / 16; j++)
#pragma unroll
    for (int r = 0; r < 4; r++) {
      const float x = h[16 * j + 4 * q + r][b];
      acc[0] = mfma4(k.w[0][j][r], x, acc[0]);
      acc[1] = mfma4(k.w[1][j][r], x, acc[1]);
    }
}

// activations and gradients of a training batch, [feature][sample] with
// stride BMAX
struct TrainBufs {
  float *A[3], *dZ[3], *dY, *lpart;
};

// A batch of B samples: column b of the batch is column idx[b] of X [11][N] and
// T [4][N], or column b itself without idx (N = B then).  A training loop over
// shuffled samples passes the permutation and keeps its pairs in place: the
// kernels gather the 60 bytes of a sample themselves.
struct Batch {
  const float *X, *T;
  long N;
  const long *idx;
  __device__ __forceinline__ long col(int b) const { return idx ? idx[b] : (long)b; }
};

// One block takes TILE samples through the whole network: wave w holds the
// output rows 32 w..32 w + 31 of each hidden layer, the activations pass
// through LDS, the weights come from L2.  TRAIN: the squared error, and the
// backward pass; samples past B leave zeros.
template <bool TRAIN>
__global__ void __launch_bounds__(256) k_mlp_pass(const float *__restrict__ th, Batch bt, int B,
                                                  float *__restrict__ Yout, TrainBufs tb)
{
  __shared__ float h[2][NH][HS];
  __shared__ float part[4][NOUT][TILE];
  __shared__ float dy[NOUT][TILE];
  __shared__ float sq[NOUT * TILE];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, q = lane >> 4, c = lane & 15;
  const int b0 = blockIdx.x * TILE, bs = b0 + c;  // this lane's sample
  const bool live = bs < B;
  const long xc = live ? bt.col(bs) : 0;
  if (TRAIN && b0 >= B) {
    for (int k = threadIdx.x; k < NH * TILE; k += 256) {
      const long at = (long)(k / TILE) * BMAX + b0 + k % TILE;
#pragma unroll
      for (int l = 0; l < 3; l++) tb.A[l][at] = tb.dZ[l][at] = 0.f;
    }
    if (threadIdx.x < NOUT * TILE) tb.dY[(long)(threadIdx.x / TILE) * BMAX + b0 + threadIdx.x % TILE] = 0.f;
    if (threadIdx.x == 0) tb.lpart[blockIdx.x] = 0.f;
    return;
  }
  const int row = 32 * wave;
  float gp[3][2][4];  // gelu' of this lane's rows of each hidden layer
  f32x4 acc[2];
  auto hidden = [&](int l, float (*dst)[HS]) {
#pragma unroll
    for (int t = 0; t < 2; t++)
#pragma unroll
      for (int r = 0; r < 4; r++) {
        const int o = row + 16 * t + 4 * q + r;
        float a;
        gelu_both(acc[t][r], a, gp[l][t][r]);
        dst[o][c] = a;
        if (TRAIN) tb.A[l][(long)o * BMAX + bs] = live ? a : 0.f;
      }
  };
  auto bias = [&](int ob) {
#pragma unroll
    for (int t = 0; t < 2; t++)
#pragma unroll
      for (int r = 0; r < 4; r++) acc[t][r] = th[ob + row + 16 * t + 4 * q + r];
  };
  RowsW wa, wb;
  load_rows(th + OW2, row + c, q, wa);
  // layer 1: 11 inputs, the twelfth of the three K = 4 products is zero
  bias(OB1);
#pragma unroll
  for (int j = 0; j < 3; j++) {
    const int k = 4 * j + q;
    const float x = (k < NIN && live) ? bt.X[k * bt.N + xc] : 0.f;
#pragma unroll
    for (int t = 0; t < 2; t++)
      acc[t] = mfma4(k < NIN ? th[OW1 + (row + 16 * t + c) * NIN + k] : 0.f, x, acc[t]);
  }
  hidden(0, h[0]);
  load_rows(th + OW3, row + c, q, wb);
  __syncthreads();
  bias(OB2);
  dense(wa, h[0], q, c, acc);
  hidden(1, h[1]);
  if (TRAIN) load_cols(th + OW3, row + c, q, wa);
  __syncthreads();
  bias(OB3);
  dense(wb, h[1], q, c, acc);
  hidden(2, h[0]);
  if (TRAIN) load_cols(th + OW2, row + c, q, wb);
  __syncthreads();
  // output layer: each wave a quarter of the inputs
  {
    f32x4 y = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int j = 0; j < 2; j++)
#pragma unroll
      for (int r = 0; r < 4; r++) {
        const int k = row + 16 * j + 4 * q + r;
        y = mfma4(c < NOUT ? th[OW4 + c * NH + k] : 0.f, h[0][k][c], y);
      }
    if (q == 0)
#pragma unroll
      for (int r = 0; r < 4; r++) part[wave][r][c] = y[r];
  }
  __syncthreads();
  if (threadIdx.x < NOUT * TILE) {
    const int o = threadIdx.x / TILE, b = threadIdx.x % TILE;
    const float y = th[OB4 + o] + part[0][o][b] + part[1][o][b] + part[2][o][b] + part[3][o][b];
    const bool in = b0 + b < B;
    if (Yout && in) Yout[(long)o * B + b0 + b] = y;
    if (TRAIN) {
      const float r = in ? y - bt.T[o * bt.N + bt.col(b0 + b)] : 0.f;
      const float d = 2.f * r * (1.f / (float)(NOUT * B));
      dy[o][b] = d;
      sq[threadIdx.x] = r * r;
      tb.dY[(long)o * BMAX + b0 + b] = d;
    }
  }
  if (!TRAIN) return;
  __syncthreads();
  if (threadIdx.x == 0) {
    float s = 0.f;
    for (int k = 0; k < NOUT * TILE; k++) s += sq[k];
    tb.lpart[blockIdx.x] = s;
  }
  // dZ of a hidden layer from dA in acc
  auto back = [&](int l, float (*dst)[HS]) {
#pragma unroll
    for (int t = 0; t < 2; t++)
#pragma unroll
      for (int r = 0; r < 4; r++) {
        const int i = row + 16 * t + 4 * q + r;
        const float d = acc[t][r] * gp[l][t][r];
        dst[i][c] = d;
        tb.dZ[l][(long)i * BMAX + bs] = live ? d : 0.f;
      }
  };
#pragma unroll
  for (int t = 0; t < 2; t++) acc[t] = mfma4(th[OW4 + q * NH + row + 16 * t + c], dy[q][c], f32x4{0.f, 0.f, 0.f, 0.f});
  back(2, h[1]);
  __syncthreads();
  acc[0] = acc[1] = f32x4{0.f, 0.f, 0.f, 0.f};
  dense(wa, h[1], q, c, acc);
  back(1, h[0]);
  __syncthreads();
  acc[0] = acc[1] = f32x4{0.f, 0.f, 0.f, 0.f};
  dense(wb, h[0], q, c, acc);
  back(0, h[1]);
}

// Gradients over one chunk of samples, gpart[chunk][NPARAM]: blockIdx.y 0..3 the
// halves (64 outputs) of layers 2 and 3, a wave 32 x 64 weights; 4 the first
// and the last layer.
__global__ void __launch_bounds__(256, 1) k_mlp_grad(Batch bt, int B, TrainBufs tb, float *__restrict__ gpart)
{
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, q = lane >> 4, c = lane & 15;
  const int s0 = blockIdx.x * CHUNK;
  float *g = gpart + (long)blockIdx.x * NPARAM;
  // D tile of the weights W[rows][cols] at (o0, i0)
  auto store = [&](int ow, int width, int o0, int i0, int rows, int cols, const f32x4 &d) {
#pragma unroll
    for (int r = 0; r < 4; r++) {
      const int o = o0 + 4 * q + r, i = i0 + c;
      if (o < rows && i < cols) g[ow + o * width + i] = d[r];
    }
  };
  // sum over the chunk of row o0 + c's gradients from the lanes' parts
  auto store_bias = [&](int ob, int rows, float sum) {
    sum += __shfl_xor(sum, 16);
    sum += __shfl_xor(sum, 32);
    if (q == 0 && c < rows) g[ob + c] = sum;
  };
  if (blockIdx.y < 4) {
    const int l = blockIdx.y < 2 ? 1 : 2;
    const float *dz = tb.dZ[l], *a = tb.A[l - 1];
    const int o0 = 64 * (blockIdx.y & 1) + 32 * (wave >> 1), i0 = 64 * (wave & 1);
    f32x4 acc[2][4];
    float sum[2] = {0.f, 0.f};
#pragma unroll
    for (int t = 0; t < 2; t++)
#pragma unroll
      for (int u = 0; u < 4; u++) acc[t][u] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int j = 0; j < CHUNK / 16; j++) {
      const int b = s0 + 16 * j + 4 * q;
      f32x4 x[2], y[4];
#pragma unroll
      for (int t = 0; t < 2; t++) x[t] = *(const f32x4 *)(dz + (long)(o0 + 16 * t + c) * BMAX + b);
#pragma unroll
      for (int u = 0; u < 4; u++) y[u] = *(const f32x4 *)(a + (long)(i0 + 16 * u + c) * BMAX + b);
#pragma unroll
      for (int r = 0; r < 4; r++)
#pragma unroll
        for (int t = 0; t < 2; t++) {
          sum[t] += x[t][r];
#pragma unroll
          for (int u = 0; u < 4; u++) acc[t][u] = mfma4(x[t][r], y[u][r], acc[t][u]);
        }
    }
    const int ow = l == 1 ? OW2 : OW3, ob = l == 1 ? OB2 : OB3;
#pragma unroll
    for (int t = 0; t < 2; t++) {
#pragma unroll
      for (int u = 0; u < 4; u++) store(ow, NH, o0 + 16 * t, i0 + 16 * u, NH, NH, acc[t][u]);
      if ((wave & 1) == 0) store_bias(ob + o0 + 16 * t, 16, sum[t]);
    }
    return;
  }
  f32x4 a1[2], a4[2];
  float sum1[2] = {0.f, 0.f}, sum4 = 0.f;
#pragma unroll
  for (int t = 0; t < 2; t++) a1[t] = a4[t] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int w0 = 32 * wave;
#pragma unroll
  for (int j = 0; j < CHUNK / 16; j++) {
    const int b = s0 + 16 * j + 4 * q;
    f32x4 x1[2], y4[2], x4 = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int t = 0; t < 2; t++) {
      x1[t] = *(const f32x4 *)(tb.dZ[0] + (long)(w0 + 16 * t + c) * BMAX + b);
      y4[t] = *(const f32x4 *)(tb.A[2] + (long)(w0 + 16 * t + c) * BMAX + b);
    }
    if (c < NOUT) x4 = *(const f32x4 *)(tb.dY + (long)c * BMAX + b);
#pragma unroll
    for (int r = 0; r < 4; r++) {
      const float y1 = (c < NIN && b + r < B) ? bt.X[c * bt.N + bt.col(b + r)] : 0.f;
      sum4 += x4[r];
#pragma unroll
      for (int t = 0; t < 2; t++) {
        sum1[t] += x1[t][r];
        a1[t] = mfma4(x1[t][r], y1, a1[t]);
        a4[t] = mfma4(x4[r], y4[t][r], a4[t]);
      }
    }
  }
#pragma unroll
  for (int t = 0; t < 2; t++) {
    store(OW1, NIN, w0 + 16 * t, 0, NH, NIN, a1[t]);
    store_bias(OB1 + w0 + 16 * t, 16, sum1[t]);
    store(OW4, NH, 0, w0 + 16 * t, NOUT, NH, a4[t]);
  }
  if (wave == 0) store_bias(OB4, NOUT, sum4);
}

// g = the chunks' sum; adam: the Adam update of th.  The last block
// sums the loss over the nb blocks of k_mlp_pass.
__global__ void __launch_bounds__(256) k_mlp_reduce(float *__restrict__ th, const float *__restrict__ gpart, int chunks,
                                                    float *__restrict__ g, float *__restrict__ m,
                                                    float *__restrict__ v, bool adam, float lr, float b1, float b2,
                                                    float c1, float c2, float eps, const float *__restrict__ lpart,
                                                    int nb, int B, float *__restrict__ loss)
{
  if (blockIdx.x == gridDim.x - 1) {
    __shared__ float red[256];
    red[threadIdx.x] = (int)threadIdx.x < nb ? lpart[threadIdx.x] : 0.f;
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
      if ((int)threadIdx.x < w) red[threadIdx.x] += red[threadIdx.x + w];
      __syncthreads();
    }
    if (threadIdx.x == 0) *loss = red[0] * (1.f / (float)(NOUT * B));
    return;
  }
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= NPARAM) return;
  float gk = 0.f;
#pragma unroll 8
  for (int q = 0; q < chunks; q++) gk += gpart[(long)q * NPARAM + k];
  g[k] = gk;
  if (!adam) return;
  float mk = b1 * m[k] + (1.f - b1) * gk;
  float vk = b2 * v[k] + (1.f - b2) * gk * gk;
  m[k] = mk;
  v[k] = vk;
  th[k] -= lr * (mk / c1) / (sqrtf(vk / c2) + eps);
}
static_assert(BMAX / TILE <= 256, "k_mlp_reduce sums one loss part per thread");
static_assert(BMAX % CHUNK == 0 && CHUNK % TILE == 0, "tiles fill chunks");

// ---------------------------------------------------------------------------
// BF16 matrix-core inference
// ---------------------------------------------------------------------------
typedef short bf16x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ unsigned short f2bf(float x)
{
  unsigned u = __float_as_uint(x);
  u += 0x7fffu + ((u >> 16) & 1u);  // round to nearest even
  return (unsigned short)(u >> 16);
}

// Weights in BF16 in the order the matrix cores' lanes read them (see
// k_mlp_infer): a fragment is a 16 x 16 block of W[out][in], lane l's four
// values W[16 ot + l%16][16 kc + 4 (l/16)..+3] next to each other and the
// lanes in order, so a wave reads a fragment as 512 consecutive bytes (rows
// of W lie 256 bytes apart: 16 lanes would meet in the same LDS banks).  W1
// is padded to 16 inputs, W4 to 16 outputs, with zeros.
constexpr int FRAG = 256;  // values of a fragment
constexpr int PW1 = 0, PW2 = PW1 + NH * 16, PW3 = PW2 + NH * NH, PW4 = PW3 + NH * NH, NPACK = PW4 + 16 * NH;

__global__ void __launch_bounds__(256) k_pack_bf16(const float *__restrict__ th, unsigned short *__restrict__ wp)
{
  int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= NPACK) return;
  // row and column of value k of its fragment
  const int l = (k % FRAG) / 4, ro = l % 16, co = 4 * (l / 16) + k % 4;
  float v = 0.f;
  if (k < PW2) {
    const int o = 16 * ((k - PW1) / FRAG) + ro;
    v = co < NIN ? th[OW1 + o * NIN + co] : 0.f;
  } else if (k < PW4) {
    const int base = k < PW3 ? PW2 : PW3, f = (k - base) / FRAG;
    v = th[(k < PW3 ? OW2 : OW3) + (16 * (f / 8) + ro) * NH + 16 * (f % 8) + co];
  } else {
    v = ro < NOUT ? th[OW4 + ro * NH + 16 * ((k - PW4) / FRAG) + co] : 0.f;
  }
  wp[k] = f2bf(v);
}

// Each wave takes CT tiles of 16 cells through the network.  For D = A B on
// the 16x16x16 BF16 matrix core, lane l holds A[l%16][4(l/16)..+3] and
// B[4(l/16)..+3][l%16] and receives D[4(l/16)..+3][l%16].  A is a block of
// the weights [out][in], B the activations [in][cell], so D holds the outputs
// of one cell per lane as four consecutive inputs of the next layer: exactly
// its B operand, and the activations never leave the registers.  The weights
// sit in LDS (74 KB: two blocks of eight waves a CU) and a fragment read
// serves CT tiles.  Bound by the 384 tanh of a cell (FP32 VALU), not by the
// products: 2^20 cells take 423 us (1645 us with activations through LDS and
// conflicting weight reads; two tiles a wave 435 us at two waves per SIMD,
// 902 us at four, spilling).
constexpr int CT = 1;
constexpr int INFER_WAVES = 8;
__global__ void __launch_bounds__(64 * INFER_WAVES, 4) k_mlp_infer(const unsigned short *__restrict__ wp,
                                                                   const float *__restrict__ th,
                                                                   const float *__restrict__ feat, long n,
                                                                   float *__restrict__ out)
{
  __shared__ __align__(16) unsigned short sw[NPACK];
  __shared__ __align__(16) float sb[3 * NH + 16];
  for (int k = threadIdx.x; k < NPACK / 8; k += blockDim.x) ((uint4 *)sw)[k] = ((const uint4 *)wp)[k];
  for (int k = threadIdx.x; k < 3 * NH + 16; k += blockDim.x) {
    float v = 0.f;
    if (k < NH) v = th[OB1 + k];
    else if (k < 2 * NH) v = th[OB2 + k - NH];
    else if (k < 3 * NH) v = th[OB3 + k - 2 * NH];
    else if (k - 3 * NH < NOUT) v = th[OB4 + k - 3 * NH];
    sb[k] = v;
  }
  __syncthreads();
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int col = lane & 15, kq = 4 * (lane >> 4);
  auto frag = [&](int base, int f) { return *(const bf16x4 *)&sw[base + f * FRAG + 4 * lane]; };
  const long step = (long)gridDim.x * INFER_WAVES * 16 * CT;
  for (long c0 = ((long)blockIdx.x * INFER_WAVES + wave) * 16 * CT; c0 < n; c0 += step) {
    bf16x4 x[CT], h[CT][NH / 16];
    // inputs: 11 features, zero padded
#pragma unroll
    for (int t = 0; t < CT; t++) {
      const long c = c0 + 16 * t + col;
#pragma unroll
      for (int q = 0; q < 4; q++) {
        const int k = kq + q;
        const float v = (c < n && k < NIN) ? feat[k * n + c] : 0.f;
        x[t][q] = (short)f2bf(v);
      }
    }
    auto activate = [&](const f32x4 &acc, const float *bias, int ot) {
      const f32x4 b = *(const f32x4 *)&bias[16 * ot + kq];
      bf16x4 v;
#pragma unroll
      for (int r = 0; r < 4; r++) v[r] = (short)f2bf(gelu(acc[r] + b[r]));
      return v;
    };
#pragma unroll
    for (int ot = 0; ot < NH / 16; ot++) {
      const bf16x4 w = frag(PW1, ot);
#pragma unroll
      for (int t = 0; t < CT; t++) {
        f32x4 acc = {0.f, 0.f, 0.f, 0.f};
        acc = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(w, x[t], acc, 0, 0, 0);
        h[t][ot] = activate(acc, sb, ot);
      }
    }
    // layers 2 and 3: one copy of the code (it holds 32 inlined tanh)
#pragma unroll 1
    for (int layer = 0; layer < 2; layer++) {
      bf16x4 hn[CT][NH / 16];
      const int base = layer == 0 ? PW2 : PW3;
#pragma unroll
      for (int ot = 0; ot < NH / 16; ot++) {
        // the weights of one row of fragments in flight at a time
        compiler_fence();
        f32x4 acc[CT];
#pragma unroll
        for (int t = 0; t < CT; t++) acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int kc = 0; kc < NH / 16; kc++) {
          const bf16x4 w = frag(base, 8 * ot + kc);
#pragma unroll
          for (int t = 0; t < CT; t++)
            acc[t] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(w, h[t][kc], acc[t], 0, 0, 0);
        }
#pragma unroll
        for (int t = 0; t < CT; t++) hn[t][ot] = activate(acc[t], sb + (layer + 1) * NH, ot);
      }
#pragma unroll
      for (int t = 0; t < CT; t++)
#pragma unroll
        for (int ot = 0; ot < NH / 16; ot++) h[t][ot] = hn[t][ot];
    }
    // output layer: 128 -> 4 (padded to 16)
#pragma unroll
    for (int t = 0; t < CT; t++) {
      f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int kc = 0; kc < NH / 16; kc++)
        acc = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(frag(PW4, kc), h[t][kc], acc, 0, 0, 0);
      const long c = c0 + 16 * t + col;
      if (kq == 0 && c < n) {
#pragma unroll
        for (int o = 0; o < NOUT; o++) out[o * n + c] = acc[o] + sb[3 * NH + o];
      }
    }
  }
}

// guess (u, u~^i) = plain start corrected by the de-normalised outputs;
// non-finite or non-positive guesses fall back to the plain start
__global__ void __launch_bounds__(256) k_guess(long n, int base, const double *__restrict__ pp,
                                               const float *__restrict__ y, const float *__restrict__ norm,
                                               double *__restrict__ gx)
{
  long c = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= n) return;
  double t[NOUT];
#pragma unroll
  for (int j = 0; j < NOUT; j++) t[j] = (double)y[j * n + c] * norm[2 * NIN + NOUT + j] + norm[2 * NIN + j];
  const double x0 = pp[base * n + c], x1 = pp[(base + 1) * n + c], x2 = pp[(base + 2) * n + c],
               x3 = pp[(base + 3) * n + c];
  const double g0 = x0 * exp(t[0]);
  const double g1 = x1 + VSCALE * sinh(t[1]), g2 = x2 + VSCALE * sinh(t[2]), g3 = x3 + VSCALE * sinh(t[3]);
  const bool ok = isfinite(g0) && g0 > 0. && isfinite(g1) && isfinite(g2) && isfinite(g3);
  gx[0 * n + c] = ok ? g0 : x0;
  gx[1 * n + c] = ok ? g1 : x1;
  gx[2 * n + c] = ok ? g2 : x2;
  gx[3 * n + c] = ok ? g3 : x3;
}

// the gate network (kind 3) scores whether a learned try will solve a cell;
// a cell scored below thr gets no learned try: its gas start becomes NaN,
// which the learned solve reads as "start the chain at once"
__global__ void __launch_bounds__(256) k_gate(long n, const float *__restrict__ y, const float *__restrict__ norm,
                                              float thr, double *__restrict__ gxg)
{
  long c = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= n) return;
  const float score = y[c] * norm[2 * NIN + NOUT] + norm[2 * NIN];
  if (!(score >= thr)) gxg[c] = __builtin_nan("");
}

inline dim3 grid1(long n) { return dim3((unsigned)((n + 255) / 256)); }

}  // namespace

// ---------------------------------------------------------------------------
// the network object
// ---------------------------------------------------------------------------
struct koral_hip_mlp {
  int kind = 0;  // 0: gas primitives (u, u~^i), 1: radiation primitives (E, F~^i)
  float *th = nullptr, *m = nullptr, *v = nullptr, *g = nullptr, *norm = nullptr;
  unsigned short *wp = nullptr;
  bool packed = false;
  int step = 0;
  TrainBufs tb{};
  float *gpart = nullptr, *loss = nullptr;
  void *mem = nullptr;  // one allocation holds them all
  // f(ptr, count) for every device buffer
  template <class F>
  void buffers(F &&f)
  {
    f(th, (size_t)NPARAM);
    f(this->m, (size_t)NPARAM);
    f(v, (size_t)NPARAM);
    f(g, (size_t)NPARAM);
    f(norm, (size_t)NNORM);
    f(wp, (size_t)NPACK);
    for (int k = 0; k < 3; k++) f(tb.A[k], (size_t)NH * BMAX);
    for (int k = 0; k < 3; k++) f(tb.dZ[k], (size_t)NH * BMAX);
    f(tb.dY, (size_t)NOUT * BMAX);
    f(tb.lpart, (size_t)(BMAX / TILE));
    f(gpart, (size_t)SMAX * NPARAM);
    f(loss, (size_t)1);
  }
  int alloc()
  {
    size_t bytes = 0;
    auto padded = [](size_t b) { return (b + 255) & ~(size_t)255; };
    buffers([&](auto *&p, size_t n) { bytes += padded(n * sizeof(*p)); });
    int rc = check_hip(hipMalloc(&mem, bytes), "hipMalloc mlp");
    if (rc) return rc;
    char *at = (char *)mem;
    buffers([&](auto *&p, size_t n) {
      p = (std::remove_reference_t<decltype(p)>)at;
      at += padded(n * sizeof(*p));
    });
    return 0;
  }
  ~koral_hip_mlp()
  {
    if (mem) (void)hipFree(mem);
  }
};

namespace {

int pack(koral_hip_mlp *m, hipStream_t s)
{
  if (!m->packed) {
    k_pack_bf16<<<grid1(NPACK), 256, 0, s>>>(m->th, m->wp);
    m->packed = true;
  }
  return check_launch("mlp pack");
}

// loss and gradient of the mean squared error of a batch into m->loss and
// m->g, and with adam the update of step m->step
int train(koral_hip_mlp *m, const Batch &bt, int B, bool adam, float lr, hipStream_t s)
{
  const int chunks = (B + CHUNK - 1) / CHUNK, nb = chunks * (CHUNK / TILE);
  const double b1 = 0.9, b2 = 0.999;
  const float c1 = (float)(1. - pow(b1, m->step)), c2 = (float)(1. - pow(b2, m->step));
  k_mlp_pass<true><<<nb, 256, 0, s>>>(m->th, bt, B, nullptr, m->tb);
  k_mlp_grad<<<dim3(chunks, 5), 256, 0, s>>>(bt, B, m->tb, m->gpart);
  k_mlp_reduce<<<(NPARAM + 255) / 256 + 1, 256, 0, s>>>(m->th, m->gpart, chunks, m->g, m->m, m->v, adam, lr, (float)b1,
                                                        (float)b2, c1, c2, 1e-8f, m->tb.lpart, nb, B, m->loss);
  return check_launch("mlp train");
}

int read_loss(koral_hip_mlp *m, float *loss, hipStream_t s)
{
  if (!loss) return 0;
  int rc = check_hip(hipMemcpyAsync(loss, m->loss, sizeof(float), hipMemcpyDeviceToHost, s), "loss");
  return rc ? rc : check_hip(hipStreamSynchronize(s), "sync");
}

}  // namespace

extern "C" {

int koral_hip_mlp_nparam(void) { return NPARAM; }

int koral_hip_mlp_create(int kind, koral_hip_mlp **out)
{
  if (!out || kind < 0 || kind > 3) return set_error(KORAL_E_ARG, "mlp_create: bad arguments");
  auto *m = new koral_hip_mlp();
  m->kind = kind;
  int rc = m->alloc();
  if (!rc) rc = check_hip(hipMemset(m->m, 0, NPARAM * sizeof(float)), "memset");
  if (!rc) rc = check_hip(hipMemset(m->v, 0, NPARAM * sizeof(float)), "memset");
  if (rc) {
    delete m;
    return rc;
  }
  *out = m;
  return 0;
}

int koral_hip_mlp_destroy(koral_hip_mlp *m)
{
  if (m) {
    (void)hipDeviceSynchronize();
    delete m;
  }
  return 0;
}

int koral_hip_mlp_set(koral_hip_mlp *m, const float *theta, const float *norm)
{
  if (!m || !theta || !norm) return set_error(KORAL_E_ARG, "mlp_set: bad arguments");
  int rc = check_hip(hipMemcpy(m->th, theta, NPARAM * sizeof(float), hipMemcpyHostToDevice), "mlp_set");
  if (!rc) rc = check_hip(hipMemcpy(m->norm, norm, NNORM * sizeof(float), hipMemcpyHostToDevice), "mlp_set");
  if (!rc) rc = check_hip(hipMemset(m->m, 0, NPARAM * sizeof(float)), "memset");
  if (!rc) rc = check_hip(hipMemset(m->v, 0, NPARAM * sizeof(float)), "memset");
  m->step = 0;
  m->packed = false;
  return rc;
}

int koral_hip_mlp_get(koral_hip_mlp *m, float *theta, float *norm)
{
  if (!m) return set_error(KORAL_E_ARG, "mlp_get: null");
  int rc = check_hip(hipDeviceSynchronize(), "sync");
  if (!rc && theta) rc = check_hip(hipMemcpy(theta, m->th, NPARAM * sizeof(float), hipMemcpyDeviceToHost), "mlp_get");
  if (!rc && norm) rc = check_hip(hipMemcpy(norm, m->norm, NNORM * sizeof(float), hipMemcpyDeviceToHost), "mlp_get");
  return rc;
}

int koral_hip_mlp_features(const koral_params *P, const koral_hip_mlp *m, long n, const double *pp,
                           const double *dt, float *feat, void *stream)
{
  if (check_params(P) || !P->rad || n < 0 || !pp || !dt || !feat) return set_error(KORAL_E_ARG, "mlp_features");
  if (n == 0) return 0;
  hipStream_t s = (hipStream_t)stream;
  const float *norm = m ? m->norm : nullptr;
  if (P->mag)
    k_features<1><<<grid1(n), 256, 0, s>>>(*P, n, pp, dt, norm, feat);
  else
    k_features<0><<<grid1(n), 256, 0, s>>>(*P, n, pp, dt, norm, feat);
  return check_launch("mlp_features");
}

int koral_hip_mlp_kind(const koral_hip_mlp *m) { return m ? m->kind : -1; }

int koral_hip_mlp_targets(int kind, long n, int nv, const double *pp0, const double *pp1, float *targ,
                          void *stream)
{
  if (n < 0 || !pp0 || !pp1 || !targ || kind < 0 || kind > 1 || (kind == 1 && nv < 10))
    return set_error(KORAL_E_ARG, "mlp_targets: bad arguments");
  if (n == 0) return 0;
  k_targets<<<grid1(n), 256, 0, (hipStream_t)stream>>>(n, kind == 0 ? 1 : nv - 4, pp0, pp1, targ);
  return check_launch("mlp_targets");
}

int koral_hip_mlp_u2p_features(const koral_params *P, const koral_hip_mlp *m, long n, const double *uu,
                               const double *pp, const double *g20, const double *G20, float *feat, void *stream)
{
  if (check_params(P) || n < 0 || !uu || !pp || !g20 || !G20 || !feat || (m && m->kind != 2))
    return set_error(KORAL_E_ARG, "mlp_u2p_features: bad arguments");
  if (n == 0) return 0;
  hipStream_t s = (hipStream_t)stream;
  const float *norm = m ? m->norm : nullptr;
  if (P->mag)
    k_u2p_features<1><<<grid1(n), 256, 0, s>>>(*P, n, uu, pp, g20, G20, norm, feat);
  else
    k_u2p_features<0><<<grid1(n), 256, 0, s>>>(*P, n, uu, pp, g20, G20, norm, feat);
  return check_launch("mlp_u2p_features");
}

int koral_hip_mlp_u2p_targets(const koral_params *P, long n, const double *pp0, const double *pp1,
                              const double *g20, const double *G20, float *targ, void *stream)
{
  if (check_params(P) || n < 0 || !pp0 || !pp1 || !g20 || !G20 || !targ)
    return set_error(KORAL_E_ARG, "mlp_u2p_targets: bad arguments");
  if (n == 0) return 0;
  hipStream_t s = (hipStream_t)stream;
  if (P->mag)
    k_u2p_targets<1><<<grid1(n), 256, 0, s>>>(*P, n, pp0, pp1, g20, G20, targ);
  else
    k_u2p_targets<0><<<grid1(n), 256, 0, s>>>(*P, n, pp0, pp1, g20, G20, targ);
  return check_launch("mlp_u2p_targets");
}

int koral_hip_mlp_u2p_guess(const koral_params *P, const koral_hip_mlp *m, long n, const double *pp,
                            const double *g20, const double *G20, const float *Y, double *W0, void *stream)
{
  if (check_params(P) || n < 0 || !m || m->kind != 2 || !pp || !g20 || !G20 || !Y || !W0)
    return set_error(KORAL_E_ARG, "mlp_u2p_guess: bad arguments");
  if (n == 0) return 0;
  hipStream_t s = (hipStream_t)stream;
  if (P->mag)
    k_u2p_guess<1><<<grid1(n), 256, 0, s>>>(*P, n, pp, g20, G20, Y, m->norm, W0);
  else
    k_u2p_guess<0><<<grid1(n), 256, 0, s>>>(*P, n, pp, g20, G20, Y, m->norm, W0);
  return check_launch("mlp_u2p_guess");
}

int koral_hip_mlp_forward(koral_hip_mlp *m, const float *X, int B, float *Y, void *stream)
{
  if (!m || !X || !Y || B < 1 || B > BMAX) return set_error(KORAL_E_ARG, "mlp_forward: bad arguments");
  hipStream_t s = (hipStream_t)stream;
  k_mlp_pass<false><<<(B + TILE - 1) / TILE, 256, 0, s>>>(m->th, Batch{X, nullptr, B, nullptr}, B, Y, m->tb);
  return check_launch("mlp_forward");
}

int koral_hip_mlp_grad(koral_hip_mlp *m, const float *X, const float *T, int B, float *grad, float *loss,
                       void *stream)
{
  if (!m || !X || !T || B < 1 || B > BMAX) return set_error(KORAL_E_ARG, "mlp_grad: bad arguments");
  hipStream_t s = (hipStream_t)stream;
  int rc = train(m, Batch{X, T, B, nullptr}, B, false, 0.f, s);
  if (!rc && grad)
    rc = check_hip(hipMemcpyAsync(grad, m->g, NPARAM * sizeof(float), hipMemcpyDeviceToDevice, s), "copy");
  return rc ? rc : read_loss(m, loss, s);
}

int koral_hip_mlp_train_step(koral_hip_mlp *m, const float *X, const float *T, int B, float lr, float *loss,
                             void *stream)
{
  return koral_hip_mlp_train_step_at(m, X, T, B, nullptr, B, lr, loss, stream);
}

int koral_hip_mlp_train_step_at(koral_hip_mlp *m, const float *X, const float *T, long N, const long *idx, int B,
                                float lr, float *loss, void *stream)
{
  if (!m || !X || !T || B < 1 || B > BMAX || N < 1 || (!idx && N != B))
    return set_error(KORAL_E_ARG, "mlp_train_step: bad arguments");
  hipStream_t s = (hipStream_t)stream;
  m->step++;
  int rc = train(m, Batch{X, T, N, idx}, B, true, lr, s);
  m->packed = false;
  return rc ? rc : read_loss(m, loss, s);
}

int koral_hip_mlp_infer(koral_hip_mlp *m, const float *feat, long n, float *Y, void *stream)
{
  if (!m || !feat || !Y || n < 0) return set_error(KORAL_E_ARG, "mlp_infer: bad arguments");
  if (n == 0) return 0;
  hipStream_t s = (hipStream_t)stream;
  int rc = pack(m, s);
  if (rc) return rc;
  const long per = 16L * CT * INFER_WAVES;
  long blocks = (n + per - 1) / per;
  if (blocks > 512) blocks = 512;
  k_mlp_infer<<<(unsigned)blocks, 64 * INFER_WAVES, 0, s>>>(m->wp, m->th, feat, n, Y);
  return check_launch("mlp_infer");
}

int koral_hip_mlp_gate(koral_hip_mlp *m, long n, const float *Y, float thr, double *gxg, void *stream)
{
  if (!m || m->kind != 3 || n < 0 || !Y || !gxg) return set_error(KORAL_E_ARG, "mlp_gate: bad arguments");
  if (n == 0) return 0;
  k_gate<<<grid1(n), 256, 0, (hipStream_t)stream>>>(n, Y, m->norm, thr, gxg);
  return check_launch("mlp_gate");
}

int koral_hip_mlp_guess(koral_hip_mlp *m, long n, int nv, const double *pp, const float *Y, double *gx,
                        void *stream)
{
  if (!m || n < 0 || !pp || !Y || !gx || (m->kind == 1 && nv < 10))
    return set_error(KORAL_E_ARG, "mlp_guess: bad arguments");
  if (n == 0) return 0;
  k_guess<<<grid1(n), 256, 0, (hipStream_t)stream>>>(n, m->kind == 0 ? 1 : nv - 4, pp, Y, m->norm, gx);
  return check_launch("mlp_guess");
}

}  // extern "C"
