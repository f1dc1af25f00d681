// Hand-written kernels of the transport-surrogate MLP: 64 -> kH -> kH -> kH -> 64 (kH = 256)
// (55 inputs / 55 outputs zero-padded to 64), GELU (tanh form) on the hidden layers.
//
// Training (FP32 master weights): FP32-MFMA GEMMs with the bias, GELU and GELU's derivative in their
// epilogues, weight and bias gradients of a layer in one launch with the gradient handed down,
// masked-MSE gradient, Adam.
// Inference: BF16 weights packed into MFMA fragment order (kx_mlp_wave.h) and the
// wave-level forward pass of kx_mlp_wave.h, 64 states per wavefront.
//
// Parameter block (FP32, contiguous): W1[kH][64] b1[kH] W2[kH][kH] b2[kH]
// W3[kH][kH] b3[kH] W4[64][kH] b4[64].
#include <hip/hip_runtime.h>

#include <cstdint>

#include "../../include/kinetix_mi.h"
#include "kx_mlp_wave.h"

namespace {

using kxmlp::kIn;
using kxmlp::kH;
using kxmlp::kOut;
using kxmlp::kValidOut;
using kxmlp::kW1;
using kxmlp::kB1;
using kxmlp::kW2;
using kxmlp::kB2;
using kxmlp::kW3;
using kxmlp::kB3;
using kxmlp::kW4;
using kxmlp::kB4;
using kxmlp::kParams;
constexpr int kWeightsBf16 = kxmlp::kFragTotal;

__device__ __forceinline__ float gelu(float x)
{
  const float u = 0.7978845608028654f * (x + 0.044715f * x * x * x);
  return 0.5f * x * (1.0f + tanhf(u));
}

__device__ __forceinline__ float gelu_grad(float x)
{
  const float x2 = x * x;
  const float u = 0.7978845608028654f * (x + 0.044715f * x2 * x);
  const float th = tanhf(u);
  return 0.5f * (1.0f + th) + 0.5f * x * (1.0f - th * th) * 0.7978845608028654f * (1.0f + 3.0f * 0.044715f * x2);
}

__device__ __forceinline__ uint16_t to_bf16(float f)
{
  uint32_t u = __float_as_uint(f);
  if ((u & 0x7f800000u) == 0x7f800000u) return (uint16_t)((u >> 16) | ((u & 0xffff) ? 0x40 : 0));
  u += 0x7fffu + ((u >> 16) & 1u);      // round to nearest even
  return (uint16_t)(u >> 16);
}

// ---- training GEMMs on FP32 MFMA (v_mfma_f32_32x32x2_f32, 16x16x4): full FP32 products and sums
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x4t __attribute__((ext_vector_type(4)));
// in the caller's arrays, which are aligned as float
typedef float f32x4u __attribute__((ext_vector_type(4), aligned(4)));

// What a GEMM tile does with its result c at (row, col):
//   BIAS_GELU  Z = c + bias[col], H = gelu(Z)          (hidden layer forward)
//   BIAS       Z = c + bias[col]                       (output layer forward)
//   GELU_BACK  Z = c * gelu'(Zin)                      (gradient before the activation)
enum Epilogue { BIAS_GELU, BIAS, GELU_BACK };

struct GemmArgs {
  const float* A;      // M x K row-major
  const float* B;      // N x K (forward: W) or, transposed, K x N (backward: W again)
  int N, K;
  const float* bias;   // N, or null
  const float* Zin;    // M x N, GELU_BACK
  float* Z;            // M x N
  float* H;            // M x N, BIAS_GELU
};

// One (32 WM) x (32 WN) tile of C = A op(B)^T: WM x WN wavefronts of 32 x 32. K runs in chunks of 32
// staged in LDS as [row][k] (rows padded to 36 floats: 16 B reads without bank conflicts),
// the next chunk's global loads in flight during the products. A lane's 16 B hold k = 8 q + 4 h
// .. + 3 (h = lane / 32), so product e of the four takes k = 8 q + e and 8 q + 4 + e from the
// two halves: the same permutation of k in A and B.
constexpr int kBK = 32, kLd = kBK + 4;
template <int WM, int WN>
constexpr int gemm_lds() { return 32 * (WM + WN) * kLd; }

template <int WM, int WN, bool TB, Epilogue EPI>
__device__ __forceinline__ void gemm_tile(const GemmArgs& g, int tm, int tn, float* lds)
{
  constexpr int TH = 64 * WM * WN, MT = 32 * WM, NT = 32 * WN;
  constexpr int LA = MT * kBK / 4 / TH, LB = NT * kBK / 4 / TH;
  static_assert(LA >= 1 && LB >= 1 && MT * kBK / 4 % TH == 0 && NT * kBK / 4 % TH == 0, "whole loads");
  float* As = lds;                 // [MT][kLd]
  float* Bs = lds + MT * kLd;      // [NT][kLd]
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, i = lane & 31, h = lane >> 5;
  const int wm = w / WN, wn = w % WN, m0 = tm * MT, n0 = tn * NT;
  f32x4t ra[LA], rb[LB];
  auto load = [&](int k0) {
#pragma unroll
    for (int r = 0; r < LA; ++r) {
      const int e = threadIdx.x + r * TH;
      ra[r] = *(const f32x4u*)(g.A + (size_t)(m0 + e / (kBK / 4)) * g.K + k0 + 4 * (e % (kBK / 4)));
    }
#pragma unroll
    for (int r = 0; r < LB; ++r) {
      const int e = threadIdx.x + r * TH;
      if (TB) rb[r] = *(const f32x4u*)(g.B + (size_t)(k0 + e / (NT / 4)) * g.N + n0 + 4 * (e % (NT / 4)));
      else rb[r] = *(const f32x4u*)(g.B + (size_t)(n0 + e / (kBK / 4)) * g.K + k0 + 4 * (e % (kBK / 4)));
    }
  };
  auto store = [&]() {
#pragma unroll
    for (int r = 0; r < LA; ++r) {
      const int e = threadIdx.x + r * TH;
      *(f32x4t*)(As + (e / (kBK / 4)) * kLd + 4 * (e % (kBK / 4))) = ra[r];
    }
#pragma unroll
    for (int r = 0; r < LB; ++r) {
      const int e = threadIdx.x + r * TH;
      if (TB) {
#pragma unroll
        for (int q = 0; q < 4; ++q) Bs[(4 * (e % (NT / 4)) + q) * kLd + e / (NT / 4)] = rb[r][q];
      } else {
        *(f32x4t*)(Bs + (e / (kBK / 4)) * kLd + 4 * (e % (kBK / 4))) = rb[r];
      }
    }
  };
  f32x16 acc = {};
  load(0);
  for (int k0 = 0; k0 < g.K; k0 += kBK) {
    __syncthreads();
    store();
    __syncthreads();
    if (k0 + kBK < g.K) load(k0 + kBK);
#pragma unroll
    for (int q = 0; q < kBK / 8; ++q) {
      const f32x4t a = *(const f32x4t*)(As + (32 * wm + i) * kLd + 8 * q + 4 * h);
      const f32x4t b = *(const f32x4t*)(Bs + (32 * wn + i) * kLd + 8 * q + 4 * h);
#pragma unroll
      for (int e = 0; e < 4; ++e) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a[e], b[e], acc, 0, 0, 0);
    }
  }
  // element r of a lane: row 8 (r / 4) + 4 h + r % 4, column i
  const int col = n0 + 32 * wn + i;
  const float bias = EPI != GELU_BACK ? g.bias[col] : 0.0f;
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    const size_t o = (size_t)(m0 + 32 * wm + 8 * (r >> 2) + 4 * h + (r & 3)) * g.N + col;
    if (EPI == GELU_BACK) {
      g.Z[o] = acc[r] * gelu_grad(g.Zin[o]);
    } else {
      const float z = acc[r] + bias;
      g.Z[o] = z;
      if (EPI == BIAS_GELU) g.H[o] = gelu(z);
    }
  }
}

template <int WM, int WN, Epilogue EPI>
__global__ void __launch_bounds__(64 * WM * WN) gemm_forward(GemmArgs g)
{
  __shared__ __attribute__((aligned(16))) float lds[gemm_lds<WM, WN>()];
  gemm_tile<WM, WN, false, EPI>(g, blockIdx.y, blockIdx.x, lds);
}

// Weight gradient of one layer, dW[m][n] = sum_b dZ[b][m] X[b][n], db[m] = sum_b dZ[b][m].
struct GradArgs {
  const float* dZ;     // batch x M
  const float* X;      // batch x N
  int batch, M, N;
  float* dW;           // M x N
  float* db;           // M
};

// x[0] + .. + x[K - 1], in pairs
template <int K, class V>
__device__ __forceinline__ V pairwise(const V* x)
{
  if constexpr (K == 1) return x[0];
  else return pairwise<K / 2>(x) + pairwise<K - K / 2>(x + K / 2);
}

// A (16 RM) x 16 tile of dW per workgroup, the batch split over its WAVES wavefronts and summed in
// wavefront order through LDS: deterministic, and no workspace beyond the caller's. The
// operands are read in MFMA layout straight from memory (lane l: row l / 16 of four, RM
// consecutive columns from RM (l % 16)), two batches of U steps of 4 rows in flight: the operands
// come from other XCDs' L2s, ~2 us away (one batch of 8: 78 us for a hidden layer's launch at
// batch 8,192, two of 16: 49). Tiles of column 0 add up db: pairwise within a batch of loads and
// over wavefronts and rows (at batch 8,192 within 4.2e-8 of the FP64 sums, as 256 strided sums and a
// tree; one running sum per lane, added in wavefront order: 1.2e-7, and no faster).
template <int RM, int WAVES>
constexpr int grad_lds() { return WAVES * 64 * (4 * RM + RM); }

template <int RM, int WAVES>
__device__ __forceinline__ void grad_tile(const GradArgs& g, int tile, float* lds)
{
  typedef float vec __attribute__((ext_vector_type(RM)));
  typedef float vecu __attribute__((ext_vector_type(RM), aligned(4)));
  constexpr int U = WAVES > 8 ? 8 : 16;        // rows of 4 per batch of loads; two batches in flight
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, i = lane & 15, q = lane >> 4;
  const int tn = g.N / 16, m0 = (tile / tn) * 16 * RM, n0 = (tile % tn) * 16;
  const int steps = g.batch / (4 * WAVES);                      // per wavefront
  const float* a = g.dZ + (size_t)(4 * steps * w + q) * g.M + m0 + RM * i;
  const float* b = g.X + (size_t)(4 * steps * w + q) * g.N + n0 + i;
  f32x4t acc[RM];
  vec bs;
#pragma unroll
  for (int e = 0; e < RM; ++e) { acc[e] = (f32x4t){0.f, 0.f, 0.f, 0.f}; bs[e] = 0.f; }
  int s = 0;
  vec va[2][U];
  float vb[2][U];
  auto load = [&](vec (&va)[U], float (&vb)[U], int at) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      va[u] = *(const vecu*)(a + (size_t)4 * (at + u) * g.M);
      vb[u] = b[(size_t)4 * (at + u) * g.N];
    }
  };
  auto products = [&](const vec (&va)[U], const float (&vb)[U]) {
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int e = 0; e < RM; ++e)
        acc[e] = __builtin_amdgcn_mfma_f32_16x16x4f32(va[u][e], vb[u], acc[e], 0, 0, 0);
    bs += pairwise<U>(va);
  };
  if (U <= steps) load(va[0], vb[0], 0);
  for (; s + 2 * U <= steps; s += 2 * U) {
    load(va[1], vb[1], s + U);
    products(va[0], vb[0]);
    __builtin_amdgcn_sched_barrier(0);
    if (s + 3 * U <= steps) load(va[0], vb[0], s + 2 * U);
    products(va[1], vb[1]);
    __builtin_amdgcn_sched_barrier(0);
  }
  if (s + U <= steps) { products(va[0], vb[0]); s += U; }
  vec t0 = {}, t1 = {};                           // the rest of the rows: even and odd ones
  for (; s < steps; ++s) {
    const vec ta = *(const vecu*)(a + (size_t)4 * s * g.M);
    const float tb = b[(size_t)4 * s * g.N];
#pragma unroll
    for (int e = 0; e < RM; ++e)
      acc[e] = __builtin_amdgcn_mfma_f32_16x16x4f32(ta[e], tb, acc[e], 0, 0, 0);
    const vec t = t0 + ta;
    t0 = t1;
    t1 = t;
  }
  bs += t0 + t1;
  float* red = lds;                               // [wave][RM * 4][64]
  float* redb = lds + WAVES * 64 * 4 * RM;        // [wave][RM][64]
#pragma unroll
  for (int e = 0; e < RM; ++e) {
#pragma unroll
    for (int r = 0; r < 4; ++r) red[(w * 4 * RM + 4 * e + r) * 64 + lane] = acc[e][r];
    redb[(w * RM + e) * 64 + lane] = bs[e];
  }
  __syncthreads();
  for (int t = threadIdx.x; t < 256 * RM; t += 64 * WAVES) {
    float v = 0.0f;
    for (int k = 0; k < WAVES; ++k) v += red[k * 256 * RM + t];
    const int l = t & 63, e = t >> 8, r = (t >> 6) & 3;        // element r of lane l, block e
    g.dW[(size_t)(m0 + RM * (4 * (l >> 4) + r) + e) * g.N + n0 + (l & 15)] = v;
  }
  if (n0 == 0 && threadIdx.x < 16 * RM) {
    const int e = threadIdx.x >> 4, c = threadIdx.x & 15;
    float v[4 * WAVES];
#pragma unroll
    for (int k = 0; k < WAVES; ++k)
#pragma unroll
      for (int r = 0; r < 4; ++r) v[4 * k + r] = redb[(k * RM + e) * 64 + 16 * r + c];
    g.db[m0 + RM * c + e] = pairwise<4 * WAVES>(v);
  }
}

// One layer backwards in one launch: the first n_grad workgroups take tiles of its weight
// gradient, the others tiles of the gradient handed to the layer below (dZ W * gelu'). The
// long batch sums start first and share the chip with the other product. Bound: the weight
// gradient's reads (each 32 x 16 tile reads both operands' columns over the whole batch); the
// two products' FP32 MFMA time is 14 us of the 49.
constexpr int kWN = kH % 128 ? 2 : 4;            // hidden-layer tiles: 64 rows x 32 kWN columns
constexpr int kTileWaves = 2 * kWN;

template <int RM>
__global__ void __launch_bounds__(64 * kTileWaves) layer_backward(GradArgs gr, GemmArgs ge, int n_grad, int tiles_n)
{
  constexpr int L0 = grad_lds<RM, kTileWaves>(), L1 = gemm_lds<2, kWN>();
  __shared__ __attribute__((aligned(16))) float lds[L0 > L1 ? L0 : L1];
  const int b = blockIdx.x;
  if (b < n_grad) grad_tile<RM, kTileWaves>(gr, b, lds);
  else gemm_tile<2, kWN, true, GELU_BACK>(ge, (b - n_grad) / tiles_n, (b - n_grad) % tiles_n, lds);
}

template <int RM, int WAVES>
__global__ void __launch_bounds__(64 * WAVES) layer_grad(GradArgs gr)
{
  __shared__ float lds[grad_lds<RM, WAVES>()];
  grad_tile<RM, WAVES>(gr, blockIdx.x, lds);
}

// dY = 2 (Y - T) / (M * valid) on the first `valid` columns, 0 on the padding; per-block
// partial sums of the squared error go to part[blockIdx.x].
__global__ void __launch_bounds__(256) mse_grad(int M, int N, int valid, const float* __restrict__ Y,
                                                const float* __restrict__ T, float* __restrict__ dY,
                                                float* __restrict__ part)
{
  __shared__ float red[256];
  const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
  float se = 0.0f;
  if (i < (size_t)M * N) {
    const int col = (int)(i % N);
    const float d = (col < valid) ? Y[i] - T[i] : 0.0f;
    dY[i] = 2.0f * d / ((float)M * (float)valid);
    se = d * d;
  }
  red[threadIdx.x] = se;
  __syncthreads();
  for (int s = 128; s > 0; s >>= 1) {
    if (threadIdx.x < s) red[threadIdx.x] += red[threadIdx.x + s];
    __syncthreads();
  }
  if (threadIdx.x == 0) part[blockIdx.x] = red[0];
}

__global__ void __launch_bounds__(256) adam(int n, float* __restrict__ w, const float* __restrict__ g,
                                            float* __restrict__ m, float* __restrict__ v, float lr,
                                            float b1, float b2, float eps, float c1, float c2)
{
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  const float gi = g[i];
  const float mi = b1 * m[i] + (1.0f - b1) * gi;
  const float vi = b2 * v[i] + (1.0f - b2) * gi * gi;
  m[i] = mi;
  v[i] = vi;
  w[i] -= lr * (mi * c1) / (sqrtf(vi * c2) + eps);
}

// BF16 weights in MFMA fragment order: fragment (ob, kb) of layer l, lane i + 16 g,
// element e = W_l[16 ob + i][kphi(kb, g, e)] (kx_mlp_wave.h).
__global__ void __launch_bounds__(256) pack_bf16(const float* __restrict__ p, uint16_t* __restrict__ wb)
{
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= kWeightsBf16) return;
  int base, K, w;
  if (i < kxmlp::kF2)      { base = kxmlp::kF1; K = kIn; w = kW1; }
  else if (i < kxmlp::kF3) { base = kxmlp::kF2; K = kH;  w = kW2; }
  else if (i < kxmlp::kF4) { base = kxmlp::kF3; K = kH;  w = kW3; }
  else                     { base = kxmlp::kF4; K = kH;  w = kW4; }
  const int local = i - base, e = local & 7, lane = (local >> 3) & 63, frag = local >> 9;
  const int KB = K / 32, kb = frag % KB, ob = frag / KB;
  const int row = 16 * ob + (lane & 15), col = kxmlp::kphi(kb, lane >> 4, e);
  wb[i] = to_bf16(p[w + row * K + col]);
}

// BF16-MFMA inference of n states (row-major FP32 X and Y, n x 64): 4 waves x 64 states
// per workgroup; the inputs go through LDS once to reach the MFMA fragment layout.
constexpr int kXS = 68;       // LDS row stride (bf16) of the staged inputs

__global__ void __launch_bounds__(256, 1) mlp_infer_bf16(const uint16_t* __restrict__ wb,
                                                         const float* __restrict__ p, int n_states,
                                                         const float* __restrict__ X, float* __restrict__ Y)
{
  __shared__ __attribute__((aligned(16))) uint16_t xs[4][64 * kXS];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const long long s0 = (long long)blockIdx.x * 256 + wv * 64;
  // stage the wave's 64 input rows as BF16 (each pass reads one 256-B row, coalesced)
  for (int e = lane; e < 64 * kIn; e += 64) {
    const int row = e >> 6, col = e & 63;
    const float x = (s0 + row < n_states) ? X[(s0 + row) * kIn + col] : 0.0f;
    xs[wv][row * kXS + col] = to_bf16(x);
  }
  __syncthreads();
  kxmlp::f32x4 y[kOut / 16][4];
  kxmlp::forward<kXS>(wb, p, xs[wv], y, lane);
  const int j = lane & 15, g = lane >> 4;
#pragma unroll
  for (int sb = 0; sb < 4; ++sb) {
    const long long s = s0 + 16 * sb + j;
    if (s < n_states) {
#pragma unroll
      for (int ob = 0; ob < kOut / 16; ++ob)
        *(kxmlp::f32x4*)(Y + s * kOut + 16 * ob + 4 * g) = y[ob][sb];
    }
  }
}

typedef short bf16x4 __attribute__((ext_vector_type(4)));
typedef float floatx4 __attribute__((ext_vector_type(4)));

// Self-test of the BF16 MFMA layout: D = A B for closed-form 16x16 A and B.
__global__ void __launch_bounds__(64) bf16_layout_probe(float* __restrict__ d)
{
  const int l = threadIdx.x, i = l & 15, g = l >> 4;
  bf16x4 a, b;
  for (int e = 0; e < 4; ++e) {
    const int k = 4 * g + e;
    a[e] = (short)to_bf16((float)(i + 16 * k + 1) / 16.0f);      // A[i][k]
    b[e] = (short)to_bf16((float)((k + 1) * 3 + i));             // B[k][j = i]
  }
  floatx4 acc = {0.f, 0.f, 0.f, 0.f};
  acc = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, acc, 0, 0, 0);
  for (int r = 0; r < 4; ++r) d[(4 * g + r) * 16 + i] = acc[r];
}

// Self-test of the v_mfma_f32_16x16x32_bf16 layout the inference path relies on:
// A[i][k] in element k % 8 of lane i + 16 (k / 8), B[k][j] likewise with j, D as above;
// small integer entries so that every product and sum is exact.
__global__ void __launch_bounds__(64) bf16_k32_layout_probe(float* __restrict__ d)
{
  const int l = threadIdx.x, i = l & 15, g = l >> 4;
  kxmlp::u32x4 a, b;
  for (int h = 0; h < 4; ++h) {
    uint32_t wa = 0, wbv = 0;
    for (int q = 0; q < 2; ++q) {
      const int k = 8 * g + 2 * h + q;
      wa |= (uint32_t)to_bf16((float)((i * 7 + k * 3) % 17 - 8)) << (16 * q);     // A[i][k]
      wbv |= (uint32_t)to_bf16((float)((k * 5 + i * 11) % 13 - 6)) << (16 * q);   // B[k][j = i]
    }
    a[h] = wa;
    b[h] = wbv;
  }
  kxmlp::f32x4 acc = {0.f, 0.f, 0.f, 0.f};
  acc = kxmlp::mfma(a, b, acc);
  for (int r = 0; r < 4; ++r) d[(4 * g + r) * 16 + i] = acc[r];
}

inline int grid1(size_t n) { return (int)((n + 255) / 256); }

int hip_status() { return hipGetLastError() == hipSuccess ? KX_OK : KX_ERR_HIP; }

}  // namespace

extern "C" {

int kx_mlp_width(void) { return kH; }
int kx_mlp_n_params(void) { return kParams; }
int kx_mlp_n_weights_bf16(void) { return kWeightsBf16; }

int kx_selftest_mfma_bf16_layout(float* d_out, void* stream)
{
  if (!d_out) return KX_ERR_INVALID_ARG;
  hipLaunchKernelGGL(bf16_layout_probe, dim3(1), dim3(64), 0, (hipStream_t)stream, d_out);
  return hip_status();
}

int kx_selftest_mfma_bf16_k32_layout(float* d_out, void* stream)
{
  if (!d_out) return KX_ERR_INVALID_ARG;
  hipLaunchKernelGGL(bf16_k32_layout_probe, dim3(1), dim3(64), 0, (hipStream_t)stream, d_out);
  return hip_status();
}

// acts (FP32, 6 blocks of B x kH = Z1 H1 Z2 H2 Z3 H3 and Y (B x 64) at the end)
int kx_mlp_forward(const float* p, int B, const float* X, float* acts, void* stream)
{
  if (!p || !X || !acts || B <= 0 || B % 64) return KX_ERR_INVALID_ARG;
  hipStream_t s = (hipStream_t)stream;
  const size_t L = (size_t)B * kH;
  float *Z1 = acts, *H1 = Z1 + L, *Z2 = H1 + L, *H2 = Z2 + L, *Z3 = H2 + L, *H3 = Z3 + L, *Yo = H3 + L;
  const dim3 gH(kH / (32 * kWN), B / 64), bH(64 * kTileWaves), gO(kOut / 64, B / 64);
  const GemmArgs l1{X, p + kW1, kH, kIn, p + kB1, nullptr, Z1, H1}, l2{H1, p + kW2, kH, kH, p + kB2, nullptr, Z2, H2};
  const GemmArgs l3{H2, p + kW3, kH, kH, p + kB3, nullptr, Z3, H3}, l4{H3, p + kW4, kOut, kH, p + kB4, nullptr, Yo, nullptr};
  hipLaunchKernelGGL((gemm_forward<2, kWN, BIAS_GELU>), gH, bH, 0, s, l1);
  hipLaunchKernelGGL((gemm_forward<2, kWN, BIAS_GELU>), gH, bH, 0, s, l2);
  hipLaunchKernelGGL((gemm_forward<2, kWN, BIAS_GELU>), gH, bH, 0, s, l3);
  hipLaunchKernelGGL((gemm_forward<2, 2, BIAS>), gO, dim3(256), 0, s, l4);
  return hip_status();
}

// Gradient of the masked MSE (first 55 outputs) w.r.t. all parameters, written to g
// (same layout as p). work: 2 x B x kH floats. loss_part: ceil(B*64/256) floats.
int kx_mlp_backward(const float* p, int B, const float* X, const float* acts, const float* T,
                    float* g, float* work, float* loss_part, void* stream)
{
  if (!p || !X || !acts || !T || !g || !work || !loss_part || B <= 0 || B % 64)
    return KX_ERR_INVALID_ARG;
  hipStream_t s = (hipStream_t)stream;
  const size_t L = (size_t)B * kH;
  const float *Z1 = acts, *H1 = Z1 + L, *Z2 = H1 + L, *H2 = Z2 + L, *Z3 = H2 + L, *H3 = Z3 + L, *Yo = H3 + L;
  float *dA = work, *dB = work + L;       // dZ of alternate layers (B x kH each)
  float* dY = dB;                          // B x 64 fits in dB
  hipLaunchKernelGGL(mse_grad, dim3(grid1((size_t)B * kOut)), dim3(256), 0, s, B, kOut, kValidOut, Yo, T, dY, loss_part);
  // layers 4, 3, 2: the weight gradient and the gradient before the next activation down
  const GradArgs w4{dY, H3, B, kOut, kH, g + kW4, g + kB4}, w3{dA, H2, B, kH, kH, g + kW3, g + kB3};
  const GradArgs w2{dB, H1, B, kH, kH, g + kW2, g + kB2}, w1{dA, X, B, kH, kIn, g + kW1, g + kB1};
  const GemmArgs x3{dY, p + kW4, kH, kOut, nullptr, Z3, dA, nullptr}, x2{dA, p + kW3, kH, kH, nullptr, Z2, dB, nullptr};
  const GemmArgs x1{dB, p + kW2, kH, kH, nullptr, Z1, dA, nullptr};
  constexpr int tn = kH / (32 * kWN);
  const dim3 bH(64 * kTileWaves);
  const int nx = (B / 64) * tn, n4 = (kOut / 16) * (kH / 16), nh = (kH / 32) * (kH / 16);
  hipLaunchKernelGGL(layer_backward<1>, dim3(n4 + nx), bH, 0, s, w4, x3, n4, tn);
  hipLaunchKernelGGL(layer_backward<2>, dim3(nh + nx), bH, 0, s, w3, x2, nh, tn);
  hipLaunchKernelGGL(layer_backward<2>, dim3(nh + nx), bH, 0, s, w2, x1, nh, tn);
  // layer 1
  hipLaunchKernelGGL((layer_grad<1, 16>), dim3((kH / 16) * (kIn / 16)), dim3(1024), 0, s, w1);
  return hip_status();
}

int kx_mlp_adam(float* p, const float* g, float* m, float* v, float lr, float b1, float b2,
                float eps, int step, void* stream)
{
  if (!p || !g || !m || !v || step < 1) return KX_ERR_INVALID_ARG;
  const float c1 = 1.0f / (1.0f - powf(b1, (float)step));
  const float c2 = 1.0f / (1.0f - powf(b2, (float)step));
  hipLaunchKernelGGL(adam, dim3(grid1(kParams)), dim3(256), 0, (hipStream_t)stream, kParams, p, g, m, v,
                     lr, b1, b2, eps, c1, c2);
  return hip_status();
}

int kx_mlp_pack_bf16(const float* p, uint16_t* wb, void* stream)
{
  if (!p || !wb) return KX_ERR_INVALID_ARG;
  hipLaunchKernelGGL(pack_bf16, dim3(grid1(kWeightsBf16)), dim3(256), 0, (hipStream_t)stream, p, wb);
  return hip_status();
}

// Y[n][64] = MLP(X[n][64]) with BF16 weights/activations and FP32 accumulation.
int kx_mlp_infer_bf16(const uint16_t* wb, const float* p, int n, const float* X, float* Y, void* stream)
{
  if (!wb || !p || n < 0 || (n > 0 && (!X || !Y))) return KX_ERR_INVALID_ARG;
  if (n == 0) return KX_OK;
  hipLaunchKernelGGL(mlp_infer_bf16, dim3((n + 255) / 256), dim3(256), 0, (hipStream_t)stream,
                     wb, p, n, X, Y);
  return hip_status();
}

}  // extern "C"
