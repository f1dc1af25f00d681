// Mixture-averaged transport (FP64), four lanes per state: the wave-level routine of
// kx_bk2_fp64, kx_bk2_fp64_pstate and kx_bk2_fp64_queue, with the pair tables in LDS or, beyond 72
// species, their rows streamed through it (kinetix/core/mix_transport.py:261-471; benchmark/okl/transportProps.okl:11-47).
//
// A wavefront takes 16 states: lane l works on state l % 16, and lane group g = l / 16 owns the
// species 4 m + g (slot m). Why this layout:
//  * the pair fits D'_kj(ln T) of 16 pairs and 16 states are one v_mfma_f64_16x16x4_f64 (the
//    quartic's four powers of t = ln T - t0 are the K index, its constant term the initial
//    accumulator); row 4 c + g of block (m, j) is the pair (4 m + c, 4 j + g), so element c of
//    a lane is the pair of species 4 m + c with the lane's own species of slot j;
//  * one coefficient read from LDS serves 16 states, not one lane: with one state per lane
//    every pair's five coefficients were broadcast to each wavefront again, and LDS bandwidth,
//    not arithmetic, set the time;
//  * each unordered pair is evaluated once: the lane adds it to its own slot's sum and to a
//    partial sum of species 4 m + c, which the four lane groups reduce-scatter once per m.
// The reciprocals of two blocks share one v_rcp_f64 (a tree of products).
//
// The Wilke rule uses that C1_kj + C2_kj eta_k / eta_j = (W_j / (8 (W_k + W_j)))^(1/4) (u_k + u_j) / u_j
// with u = eta W^(-1/4): S_k = sum_j a_j M_kj (u_k + u_j)^2, a_j = x_j sqrt(W_j) / u_j^2, with the
// positive definite matrix M_kj = (8 (W_k + W_j))^(-1/2), a smooth function of W_k + W_j: its
// pivoted Cholesky factor L reaches FP64 rounding at rank 13-16 for the combustion mechanisms here (up
// to 93 g/mol; octane to dodecane 17-18), and at 21 of 22 where masses spread over a factor of 300
// (ranks beyond 16 take a second block of z). Entries of L L^T are within 1e-15 of M; by
// Cauchy-Schwarz the products' magnitudes sum to at most twice M_kj, so nothing cancels badly.
// S = u^2 L(L^T a) + 2 u L(L^T a u) + L(L^T a u^2) is then six thin products per 16 states, all on MFMA.
//
// Bound: FP64 issue. v_mfma_f64 and FP64 VALU instructions do not overlap on this chip (32 v_fma
// and 2 v_mfma take the sum of their times), so per 16 states the ~18k cycles of the pair blocks
// (per block 68 for the MFMA, 110 for the reciprocals and sums) and ~12k of the rest are the
// floor of this form; eight wavefronts per CU reach it. Measured against one state per lane
// (pair constants broadcast from LDS by every wavefront): GRI-3.0, 4,194,304 states 7.30 ->
// 3.62 ms, 1,000 states 222 -> 18.6 us; NH3Konnov_edit, 100,003 states 97 -> 61 us. At 12 and
// 16 wavefronts per workgroup the registers spill: 0.97 and 1.13 ms for 1,048,576 states
// against 0.91. With the pair rows streamed (160 species, 524,288 states): 3.07 ms against 9.14 for
// 64-state tiles with a row per wavefront and LDS atomics; 162 registers spill, most of them once.
//
// The table (gen/emit_bk2_quad.py) holds the fits about t0, the middle of the fit window: the
// same polynomials with far smaller cancelling terms than in powers of ln T.
#pragma once
#include <hip/hip_runtime.h>
#include "kx_rcp.h"

namespace kxquad {

typedef double f64x4 __attribute__((ext_vector_type(4)));
typedef double f64x2 __attribute__((ext_vector_type(2)));
typedef unsigned u32x2 __attribute__((ext_vector_type(2)));

// swap of lanes [32, 64) of a with lanes [0, 32) of b / of the odd 16-lane rows of a with the
// even rows of b
__device__ __forceinline__ void swap32(double& a, double& b)
{
  const u32x2 A = __builtin_bit_cast(u32x2, a), B = __builtin_bit_cast(u32x2, b);
  const u32x2 lo = __builtin_amdgcn_permlane32_swap(A[0], B[0], false, false);
  const u32x2 hi = __builtin_amdgcn_permlane32_swap(A[1], B[1], false, false);
  a = __builtin_bit_cast(double, (u32x2){lo[0], hi[0]});
  b = __builtin_bit_cast(double, (u32x2){lo[1], hi[1]});
}

__device__ __forceinline__ void swap16(double& a, double& b)
{
  const u32x2 A = __builtin_bit_cast(u32x2, a), B = __builtin_bit_cast(u32x2, b);
  const u32x2 lo = __builtin_amdgcn_permlane16_swap(A[0], B[0], false, false);
  const u32x2 hi = __builtin_amdgcn_permlane16_swap(A[1], B[1], false, false);
  a = __builtin_bit_cast(double, (u32x2){lo[0], hi[0]});
  b = __builtin_bit_cast(double, (u32x2){lo[1], hi[1]});
}

// the value of every lane group, in every lane of the state
__device__ __forceinline__ void bcast4(double v, double (&out)[4])
{
  double a = v, b = v;
  swap32(a, b);                       // a: rows 0 1 0 1, b: rows 2 3 2 3
  out[0] = a; out[1] = a;
  swap16(out[0], out[1]);
  out[2] = b; out[3] = b;
  swap16(out[2], out[3]);
}

// sum over the lane groups of p[g], in lane group g
__device__ __forceinline__ double reduce_scatter4(const double (&p)[4])
{
  double a = p[0], b = p[2], c = p[1], d = p[3];
  swap32(a, b);
  swap32(c, d);
  double q0 = a + b, q1 = c + d;      // lower half: sums of p0 / p1 over g, g + 2; upper: p2 / p3
  swap16(q0, q1);
  return q0 + q1;
}

// sum over the four lanes of a state, in all of them
__device__ __forceinline__ double sum4(double v)
{
  double a = v, b = v;
  swap32(a, b);
  v = a + b;
  a = v; b = v;
  swap16(a, b);
  return a + b;
}

// reciprocals of a block's four positive fits of moderate exponent (their products stay
// normal), from q = 1 / (product of the four)
__device__ __forceinline__ void rcp4(const f64x4& d, double ab, double cd, double q, double (&r)[4])
{
  const double ra = q * cd, rc = q * ab;
  r[0] = ra * d[1];
  r[1] = ra * d[0];
  r[2] = rc * d[3];
  r[3] = rc * d[2];
}

__device__ __forceinline__ f64x4 mfma(double a, double b, const f64x4& c)
{
  return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}

// The sums S[0..m] are needed as values here: without this the compiler defers their additions
// to the end of the kernel and keeps every reciprocal alive until then (2,400 spilled VGPRs).
template <int NB>
__device__ __forceinline__ void pin(double (&S)[NB], int m)
{
#pragma unroll
  for (int j = 0; j < NB; ++j)
    if (j <= m) asm volatile("" : "+v"(S[j]));
}

// f(0), f(1) .. f(N - 1) with compile-time arguments: the pair rows index register arrays, and
// the unroller gives up on 40 of them
template <int... I>
struct Seq {};
template <int N, int... I>
struct MakeSeq : MakeSeq<N - 1, N - 1, I...> {};
template <int... I>
struct MakeSeq<0, I...> { typedef Seq<I...> type; };
template <int V>
struct Int { static constexpr int value = V; };
template <class F, int... I>
__device__ __forceinline__ void each(Seq<I...>, F&& f) { (f(Int<I>()), ...); }

// Table offsets (doubles) for N species and Wilke factors of KR groups of four ranks; see
// gen/emit_bk2_quad.py for the contents. Rows of pair blocks first (row m: 64 (m + 1) doubles of
// A operands, 16 (m + 1) of constants), then the species part.
template <int N, int KR>
struct Layout {
  static constexpr int NB = (N + 3) / 4, SG = (NB + 3) / 4, RB = (KR + 3) / 4;
  static constexpr int row(int m) { return 40 * m * (m + 1); }
  static constexpr int kSpecies = row(NB);
  static constexpr int kWilT = 0, kWil = kWilT + 64 * NB * RB, kViscA = kWil + 64 * SG * KR;
  static constexpr int kViscC = kViscA + 64 * SG, kCondA = kViscC + 16 * SG;
  static constexpr int kCondC = kCondA + 64 * SG, kRcpW = kCondC + 16 * SG;
  static constexpr int kW = kRcpW + 4 * NB, kSqW = kW + 4 * NB;
  static constexpr int kSpeciesSize = (kSqW + 4 * NB + 1) & ~1;
  static constexpr int kSize = kSpecies + kSpeciesSize;
  static constexpr int kRowMax = 80 * NB;                    // the last row
};

// copy of (part of) the table to LDS by the whole workgroup, 16 B per lane, 8 loads in flight
template <int SIZE, int THREADS>
__device__ __forceinline__ void stage(double* dst, const double* __restrict__ src)
{
  constexpr int n = SIZE / 2, batch = 8;
  const f64x2* s = (const f64x2*)src;
  f64x2* d = (f64x2*)dst;
  for (int b = threadIdx.x; b < n; b += batch * THREADS) {
    f64x2 t[batch];
#pragma unroll
    for (int r = 0; r < batch; ++r) t[r] = s[min(b + r * THREADS, n - 1)];
#pragma unroll
    for (int r = 0; r < batch; ++r) if (b + r * THREADS < n) d[b + r * THREADS] = t[r];
  }
  __syncthreads();
}

// Transport of the wavefront's 16 states; lane l: state l % 16 (index id), species group
// l / 16. store(D, rho) is called once with D_km of the lane's species 4 m + g in D[m] (all lanes;
// the caller masks lanes without a state). Returns mu and lambda in all four lanes of a state.
//
// STAGE > 0 (the workgroup's threads): the pair rows do not fit the LDS and are streamed through
// two row buffers, the next row's global loads in flight during a row; every wavefront of the
// workgroup makes the call together (one barrier per row), those without states with busy =
// false. `rows` is then the two buffers and `grows` the table in global memory; else `rows` holds
// every row.
template <int N, int KR, bool RCP, int STAGE, class Store>
__device__ __forceinline__ void states16(const double* tab, double* rows,
                                         const double* __restrict__ grows, bool busy,
                                         const double* __restrict__ state,
                                         long long id, long long offsetT, long long offset,
                                         double Tref, double p, double t0, double rcpR, int lane,
                                         double& mu, double& lambda, Store&& store)
{
  typedef Layout<N, KR> L;
  constexpr int NB = L::NB;
  // opaque per call: the caller's loop over units would otherwise hoist the table reads
  // (thousands of registers) out of itself
  asm volatile("" : "+v"(lane));
  const int g = lane >> 4;
  const double T = Tref * state[id];
  double X[NB], S[NB];
  const double* y = state + id + offsetT + g * offset;        // species 4 m + g at y + 4 m offset
#pragma unroll
  for (int m = 0; m < NB; ++m)
    X[m] = 4 * m + 3 < N || 4 * m + g < N ? y[4 * m * offset] : 0.0;
  const double rcpT = 1.0 / T, sqrT = sqrt(T);
  const double t = log(T) - t0, tt = t * t;
  const double B = (g & 1 ? tt : t) * (g & 2 ? tt : 1.0);     // t^(g + 1)
  double part = 0.0;
#pragma unroll
  for (int m = 0; m < NB; ++m) {
    X[m] = fmax(0.0, X[m]) * tab[L::kRcpW + 4 * m + g];       // 1/W is 0 for the padding species
    part += X[m];
  }
  const double Mbar = 1.0 / sum4(part);
#pragma unroll
  for (int m = 0; m < NB; ++m) { X[m] *= Mbar; S[m] = 0.0; }

  // ---- diffusion: S_k = sum_{j != k} x_j / D'_kj
  each(typename MakeSeq<NB>::type(), [&](auto mc) __attribute__((always_inline)) {
    constexpr int m = decltype(mc)::value;
    __builtin_amdgcn_sched_barrier(0);
    const double* row = rows + (STAGE ? (m & 1) * L::kRowMax : L::row(m));
    constexpr int PF = STAGE ? (L::kRowMax / 2 + STAGE - 1) / STAGE : 1;
    f64x2 ahead[PF];
    constexpr int n_ahead = 40 * (m + 2);                        // 16 B pieces of row m + 1
    if (STAGE) {
      __syncthreads();                   // row m written; the other buffer's row read by all
      if (m + 1 < NB) {
#pragma unroll
        for (int r = 0; r < PF; ++r)
          if (r * STAGE < n_ahead)
            ahead[r] = ((const f64x2*)(grows + L::row(m + 1)))[min((int)threadIdx.x + r * STAGE, n_ahead - 1)];
      }
    }
    if (!STAGE || busy) {
    double xk[4], q[4] = {0.0, 0.0, 0.0, 0.0};
    bcast4(X[m], xk);
#pragma unroll
    for (int j = 0; j <= m; j += 2) {
      if (STAGE) __builtin_amdgcn_sched_barrier(0);            // 160 registers hold X and S
      const bool two = j < m;                                  // blocks (m, j) and (m, j + 1)
      f64x4 d0 = *(const f64x4*)(row + 64 * (m + 1) + 16 * j + 4 * g), d1 = {1.0, 1.0, 1.0, 1.0};
      d0 = mfma(row[64 * j + lane], B, d0);
      if (two) {
        d1 = *(const f64x4*)(row + 64 * (m + 1) + 16 * (j + 1) + 4 * g);
        d1 = mfma(row[64 * (j + 1) + lane], B, d1);
      }
      double r0[4] = {d0[0], d0[1], d0[2], d0[3]}, r1[4] = {d1[0], d1[1], d1[2], d1[3]};
      if (!RCP) {
        const double ab = d0[0] * d0[1], cd = d0[2] * d0[3], p0 = ab * cd;
        if (two) {
          const double ef = d1[0] * d1[1], gh = d1[2] * d1[3], p1 = ef * gh;
          const double v = kx_rcp(p0 * p1);
          rcp4(d0, ab, cd, v * p1, r0);
          rcp4(d1, ef, gh, v * p0, r1);
        } else {
          rcp4(d0, ab, cd, kx_rcp(p0), r0);
        }
      }
      // row pair (4 m + c, own species of the slot); the diagonal block (slot m) holds both
      // orders of its pairs: own sum only, k = j left out
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        if (j < m) { S[j] += xk[c] * r0[c]; q[c] += X[j] * r0[c]; }
        else S[m] += xk[c] * (c == g ? 0.0 : r0[c]);
        if (two) {
          if (j + 1 < m) { S[j + 1] += xk[c] * r1[c]; q[c] += X[j + 1] * r1[c]; }
          else S[m] += xk[c] * (c == g ? 0.0 : r1[c]);
        }
      }
    }
    if (m) S[m] += reduce_scatter4(q);
    pin<NB>(S, m);
    }
    if (STAGE && m + 1 < NB) {
      f64x2* next = (f64x2*)(rows + ((m + 1) & 1) * L::kRowMax);
#pragma unroll
      for (int r = 0; r < PF; ++r)
        if (r * STAGE < n_ahead && (int)threadIdx.x + r * STAGE < n_ahead) next[threadIdx.x + r * STAGE] = ahead[r];
    }
  });
  if (STAGE && !busy) return;
  __builtin_amdgcn_sched_barrier(0);
  const double TsqrT = T * sqrT, rho = p * rcpR * rcpT * Mbar, pMbar = p * Mbar;
#pragma unroll
  for (int m = 0; m < NB; ++m)
    S[m] = TsqrT * (Mbar - tab[L::kW + 4 * m + g] * X[m]) / (pMbar * S[m]);     // D_km
  store(S, rho);

  // ---- conductivity, then u_k (in U) and a_k = x_k sqrt(W_k) / u_k^2 (in A)
  double s1 = 0.0, s2 = 0.0, U[NB], A[NB];
#pragma unroll
  for (int h = 0; h < L::SG; ++h) {
    __builtin_amdgcn_sched_barrier(0);
    f64x4 l = *(const f64x4*)(tab + L::kCondC + 16 * h + 4 * g);
    l = mfma(tab[L::kCondA + 64 * h + lane], B, l);
    f64x4 u = *(const f64x4*)(tab + L::kViscC + 16 * h + 4 * g);
    u = mfma(tab[L::kViscA + 64 * h + lane], B, u);
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      const int m = 4 * h + c;
      if (m < NB) {
        s1 += X[m] * l[c];
        s2 += X[m] * kx_rcp(l[c]);
        U[m] = u[c];
        A[m] = X[m] * tab[L::kSqW + 4 * m + g] * kx_rcp(u[c] * u[c]);
      }
    }
  }
  s1 = sum4(s1);
  s2 = sum4(s2);
  lambda = sqrT * (0.5 * (s1 + 1.0 / s2));

  // ---- viscosity (Wilke): z = L^T (a, a u, a u^2), element e of a lane: rank 16 h + 4 e + g
  constexpr int RB = L::RB;
  f64x4 z[3][RB];
#pragma unroll
  for (int h = 0; h < RB; ++h) {
    z[0][h] = z[1][h] = z[2][h] = (f64x4){0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int m = 0; m < NB; ++m) {
      const double a = tab[L::kWilT + 64 * (RB * m + h) + lane];
      const double au = A[m] * U[m];
      z[0][h] = mfma(a, A[m], z[0][h]);
      z[1][h] = mfma(a, au, z[1][h]);
      z[2][h] = mfma(a, au * U[m], z[2][h]);
    }
  }
  double vis = 0.0;
#pragma unroll
  for (int h = 0; h < L::SG; ++h) {
    __builtin_amdgcn_sched_barrier(0);
    f64x4 y[3];
    y[0] = y[1] = y[2] = (f64x4){0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int q = 0; q < KR; ++q) {
      const double a = tab[L::kWil + 64 * (KR * h + q) + lane];
#pragma unroll
      for (int v = 0; v < 3; ++v) y[v] = mfma(a, z[v][q >> 2][q & 3], y[v]);
    }
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      const int m = 4 * h + c;
      if (m < NB) {
        double s = y[2][c] + U[m] * (2.0 * y[1][c] + U[m] * y[0][c]);
        if (4 * m + 3 >= N) s = 4 * m + g < N ? s : 1.0;         // padding species: a = 0
        const double uu = U[m] * U[m];
        vis += A[m] * (uu * uu) * kx_rcp(s);                     // x_k eta_k^2 / S_k
      }
    }
  }
  mu = sqrT * sum4(vis);
}

// Unit (16 states) of iteration `it` for wavefront w of workgroup b: whole rounds of the grid
// take neighbouring units per workgroup (their rows share cache lines); the last, partial
// round is spread over the workgroups first, so a small call runs on as many CUs as it has
// units.
__device__ __forceinline__ long long unit_of(long long units, int it, int waves, int w)
{
  const long long G = gridDim.x, b = blockIdx.x, base = it * G * waves;
  return units - base >= G * waves ? base + b * waves + w : base + b + G * w;
}

// The plain kernel over states [0, n_eff); STAGED: `rows` is two row buffers (states16).
template <int N, int KR, bool RCP, int WAVES, bool PSTATE, bool STAGED>
__device__ __forceinline__ void plain(const double* tab, double* rows, const double* __restrict__ grows,
                                      long long n_eff, long long offsetT,
                                      long long offset, const double* __restrict__ p_state,
                                      double pressure, const double* __restrict__ state,
                                      double* __restrict__ conductivity,
                                      double* __restrict__ viscosity, double* __restrict__ rhoD,
                                      double* __restrict__ Dkm, double Tref, double t0, double rcpR)
{
  constexpr int NB = Layout<N, KR>::NB;
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const long long units = (n_eff + 15) / 16;
#pragma unroll 1
  for (int it = 0;; ++it) {
    const long long u0 = unit_of(units, it, WAVES, w);
    const bool busy = u0 < units;
    if (STAGED ? unit_of(units, it, WAVES, 0) >= units : !busy) break;   // staged: whole workgroups
    const long long u = busy ? u0 : 0;
    const long long id0 = 16 * u + (lane & 15);
    const bool live = busy && id0 < n_eff;
    const long long id = id0 < n_eff ? id0 : 16 * u;   // lanes past the end redo the first state, store nothing
    if (STAGED) {
      __syncthreads();                                 // the last call's rows read by all
      for (int e = threadIdx.x; e < 80; e += 64 * WAVES) rows[e] = grows[e];
    }
    const double p = PSTATE ? p_state[id] : pressure;
    double mu, lambda;
    const long long own = id + (lane >> 4) * offset;       // species 4 m + g at own + 4 m offset
    states16<N, KR, RCP, STAGED ? 64 * WAVES : 0>(tab, rows, grows, busy, state, id, offsetT, offset,
                     Tref, p, t0, rcpR, lane, mu, lambda, [&](const double (&D)[NB], double rho) {
                       if (!live) return;
#pragma unroll
                       for (int m = 0; m < NB; ++m)
                         if (4 * m + 3 < N || 4 * m + (lane >> 4) < N) {
                           rhoD[own + 4 * m * offset] = rho * D[m];
                           if (PSTATE) Dkm[own + 4 * m * offset] = D[m];
                         }
                     });
    if (live && lane < 16) {
      viscosity[id] = mu;
      conductivity[id] = lambda;
    }
  }
}

// The surrogate's plain pass over the queue: entries [0, n_audit) are audit samples, then the
// out-of-hull states up to `valid`. Reads each state in place and overwrites its outputs; an
// audit entry the surrogate answered (flag 0) first compares mu, lambda and rho*D_k with its
// values, and counts in counters[1] if any is off (or NaN).
template <int N, int KR, bool RCP, int WAVES>
__device__ __forceinline__ void queued(const double* tab, double* rows, long long valid, int n_audit,
                                       const int* __restrict__ queue, int* __restrict__ counters,
                                       const int* __restrict__ flags, double tol, double tol_rhoD,
                                       long long offsetT, long long offset,
                                       const double* __restrict__ p_state,
                                       const double* __restrict__ state,
                                       double* __restrict__ conductivity,
                                       double* __restrict__ viscosity, double* __restrict__ rhoD,
                                       double* __restrict__ Dkm, double Tref, double t0, double rcpR)
{
  constexpr int NB = Layout<N, KR>::NB;
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const long long units = (valid + 15) / 16;
#pragma unroll 1
  for (int it = 0;; ++it) {
    const long long u = unit_of(units, it, WAVES, w);
    if (u >= units) break;
    const long long slot = 16 * u + (lane & 15);
    const bool live = slot < valid;
    const long long id = queue[live ? slot : 16 * u];    // dead lanes redo a valid state, store nothing
    const bool audit = live && slot < n_audit && flags[id] == 0;
    const long long own = id + (lane >> 4) * offset;
    double mu, lambda, bad = 0.0;
    states16<N, KR, RCP, 0>(tab, rows, nullptr, true, state, id, offsetT, offset, Tref, p_state[id], t0,
                         rcpR, lane, mu, lambda, [&](const double (&D)[NB], double rho) {
                           if (!live) return;
#pragma unroll
                           for (int m = 0; m < NB; ++m)
                             if (4 * m + 3 < N || 4 * m + (lane >> 4) < N) {
                               double* r = rhoD + own + 4 * m * offset;
                               const double v = rho * D[m];
                               if (!(fabs(*r / v - 1.0) <= tol_rhoD)) bad = 1.0;
                               *r = v;
                             }
                           if (Dkm) {
#pragma unroll
                             for (int m = 0; m < NB; ++m)
                               if (4 * m + 3 < N || 4 * m + (lane >> 4) < N)
                                 Dkm[own + 4 * m * offset] = D[m];
                           }
                         });
    bad = sum4(bad);
    if (live && lane < 16) {
      if (audit) {
        const double ev = fabs(viscosity[id] / mu - 1.0), el = fabs(conductivity[id] / lambda - 1.0);
        if (!(ev <= tol) || !(el <= tol) || bad > 0.0) atomicAdd(counters + 1, 1);
      }
      viscosity[id] = mu;
      conductivity[id] = lambda;
    }
  }
}

}  // namespace kxquad
