// Fused per-edge passes of the training path (second_order.py), which differentiates the forces once more: the
// first-order value aggregation, the segmented-softmax attention weights, each with its gradient and the gradient
// of that gradient, and the sum of a per-edge tensor with two gathered per-atom ones.  Composed from single
// segment and elementwise kernels these were half of a step: every value row gathered three times (once per
// component of the edge vector) and some sixty passes over [E, 128] tensors per layer.
#include <type_traits>

#include "common.h"
#include "../../include/e2v2.h"

namespace e2v2 {
namespace {

constexpr int kTC = 256, kTH = 128, kTR = 9;   // channels, heads, irreps rows
constexpr int kTWaves = 4, kTThreads = 64 * kTWaves;

__device__ __forceinline__ float4 ld4(const float* p) { return *reinterpret_cast<const float4*>(p); }
__device__ __forceinline__ void st4(float* p, float4 v) { *reinterpret_cast<float4*>(p) = v; }
__device__ __forceinline__ float4 f4(float x) { return make_float4(x, x, x, x); }
__device__ __forceinline__ float4 add4(float4 a, float4 b) {
  return make_float4(a.x + b.x, a.y + b.y, a.z + b.z, a.w + b.w);
}
__device__ __forceinline__ float4 mul4(float4 a, float4 b) {
  return make_float4(a.x * b.x, a.y * b.y, a.z * b.z, a.w * b.w);
}
__device__ __forceinline__ float4 fma4(float4 a, float4 b, float4 c) {
  return make_float4(fmaf(a.x, b.x, c.x), fmaf(a.y, b.y, c.y), fmaf(a.z, b.z, c.z), fmaf(a.w, b.w, c.w));
}
__device__ __forceinline__ float sum4(float4 a) { return (a.x + a.y) + (a.z + a.w); }

// ---------------------------------------------------------------------------
// First-order value aggregation.  With S = sum_e sum_k sum_c w[e, h(c)] u[e, k] sum_r g[k, r, row_e, c] v[r, col_e, c]
// (h(c) = c mod 128, k the component of the unit edge vector u, r the irreps row) the aggregation is dS/dg, its
// input gradients dS/dv, dS/dw, dS/du, and since S is linear in each operand the second-order pass is sums of the
// same three forms with one operand replaced by its cotangent: each kernel below takes both terms at once.
// Lane l of a wavefront owns channels 4 l .. 4 l + 3 (a gathered row is one contiguous 1 KB load); the four
// wavefronts of a row's (column's) workgroup take its edges in turn and add their sums in LDS in a fixed order.
// They are bound by the gathered rows (9 KB an edge; 27 KB for dS/dv, whose rows are g's): 1,500 atoms, 128 k edges:
// dS/dv 227 us (three reductions of g before: 282 us and the products w u_k), dS/dw and dS/du 122 us (three dots
// and the sums over heads: 207 us and three passes over [E, 128]), both second-order terms of the aggregation 252 us.
struct EdgeW {          // weights w[e, 128] times u[e, 3]; w NULL: no such term
  const float* w;
  const float* u;
};

__device__ __forceinline__ void add_weights(const EdgeW& W, int64_t e, int h4, float4 (&c)[3], bool first) {
  if (!W.w) {
    if (first) c[0] = c[1] = c[2] = f4(0.f);
    return;
  }
  const float4 w = ld4(W.w + e * kTH + h4);
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    const float4 u = f4(W.u[3 * e + k]);
    c[k] = first ? mul4(w, u) : fma4(w, u, c[k]);
  }
}

// Adds the wavefronts' kN quads: (w0 + w2) + (w1 + w3), left in wavefront 0.  red: [2][kN][64] float4.
template <int kN>
__device__ __forceinline__ void add_waves(float4 (*red)[kN][64], float4 (&acc)[kN], int wave, int lane) {
  auto put = [&](int b) {
#pragma unroll
    for (int i = 0; i < kN; ++i) red[b][i][lane] = acc[i];
  };
  auto add = [&](int b) {
#pragma unroll
    for (int i = 0; i < kN; ++i) acc[i] = add4(acc[i], red[b][i][lane]);
  };
  if (wave >= 2) put(wave - 2);
  __syncthreads();
  if (wave < 2) add(wave);
  __syncthreads();
  if (wave == 1) put(0);
  __syncthreads();
  if (wave == 0) add(0);
}

// a[k][r][i][c] = sum over the edges of row i of (w1 u1_k + w2 u2_k) v[r][j][c] (+ w3 u3_k v2[r][j][c])
template <bool kSecond>
__global__ __launch_bounds__(kTThreads, 2) void k_so2_agg(const int32_t* __restrict__ row_ptr,
                                                          const int32_t* __restrict__ col, int n, EdgeW W1, EdgeW W2,
                                                          const float* __restrict__ v, EdgeW W3,
                                                          const float* __restrict__ v2, float* __restrict__ a) {
  __shared__ float4 red[2][3 * kTR][64];
  const int i = xcd_row(blockIdx.x, n);
  if (i >= n) return;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int c = 4 * lane, h4 = c & (kTH - 1);
  const size_t rs = (size_t)n * kTC;
  float4 acc[3 * kTR];
#pragma unroll
  for (int q = 0; q < 3 * kTR; ++q) acc[q] = f4(0.f);
  const int e1 = row_ptr[i + 1];
  for (int64_t e = row_ptr[i] + wave; e < e1; e += kTWaves) {
    const size_t off = (size_t)col[e] * kTC + c;
    float4 x[kTR], cw[3];
#pragma unroll
    for (int r = 0; r < kTR; ++r) x[r] = ld4(v + r * rs + off);
    add_weights(W1, e, h4, cw, true);
    if constexpr (kSecond) add_weights(W2, e, h4, cw, false);
#pragma unroll
    for (int k = 0; k < 3; ++k)
#pragma unroll
      for (int r = 0; r < kTR; ++r) acc[k * kTR + r] = fma4(cw[k], x[r], acc[k * kTR + r]);
    if constexpr (kSecond) {
      if (v2) {
#pragma unroll
        for (int r = 0; r < kTR; ++r) x[r] = ld4(v2 + r * rs + off);
        add_weights(W3, e, h4, cw, true);
#pragma unroll
        for (int k = 0; k < 3; ++k)
#pragma unroll
          for (int r = 0; r < kTR; ++r) acc[k * kTR + r] = fma4(cw[k], x[r], acc[k * kTR + r]);
      }
    }
  }
  add_waves<3 * kTR>(red, acc, wave, lane);
  if (wave == 0) {
#pragma unroll
    for (int q = 0; q < 3 * kTR; ++q) st4(a + q * rs + (size_t)i * kTC + c, acc[q]);
  }
}

// dv[r][j][c] = sum over the edges of column j of sum_k (w1 u1_k + w2 u2_k) g[k][r][i][c]
template <bool kSecond>
__global__ __launch_bounds__(kTThreads, 2) void k_so2_dv(const int32_t* __restrict__ key_ptr,
                                                         const int32_t* __restrict__ key_eid,
                                                         const int32_t* __restrict__ edge_row, int n, EdgeW W1,
                                                         EdgeW W2, const float* __restrict__ g,
                                                         float* __restrict__ dv) {
  __shared__ float4 red[2][kTR][64];
  const int j = xcd_row(blockIdx.x, n);
  if (j >= n) return;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int c = 4 * lane, h4 = c & (kTH - 1);
  const size_t rs = (size_t)n * kTC;
  float4 acc[kTR];
#pragma unroll
  for (int r = 0; r < kTR; ++r) acc[r] = f4(0.f);
  const int p1 = key_ptr[j + 1];
  for (int p = key_ptr[j] + wave; p < p1; p += kTWaves) {
    const int64_t e = key_eid[p];
    const float* gr = g + (size_t)edge_row[e] * kTC + c;
    float4 x[3 * kTR], cw[3];
#pragma unroll
    for (int q = 0; q < 3 * kTR; ++q) x[q] = ld4(gr + q * rs);
    add_weights(W1, e, h4, cw, true);
    if constexpr (kSecond) add_weights(W2, e, h4, cw, false);
#pragma unroll
    for (int k = 0; k < 3; ++k)
#pragma unroll
      for (int r = 0; r < kTR; ++r) acc[r] = fma4(cw[k], x[k * kTR + r], acc[r]);
  }
  add_waves<kTR>(red, acc, wave, lane);
  if (wave == 0) {
#pragma unroll
    for (int r = 0; r < kTR; ++r) st4(dv + r * rs + (size_t)j * kTC + c, acc[r]);
  }
}

// With P_k[c] = sum_r g[k][r][i][c] v[r][j][c] and Q_k the same of v2:
// dw[e, h] = sum over the head's two channels of sum_k (u1_k P_k + u2_k Q_k), du[e, k] = sum_c w1 P_k + w2 Q_k.
// The row's 27 g quads stay in registers over its edges.
template <bool kSecond>
__global__ __launch_bounds__(kTThreads, 2) void k_so2_dw(const int32_t* __restrict__ row_ptr,
                                                         const int32_t* __restrict__ col, int n, EdgeW W1,
                                                         const float* __restrict__ v, EdgeW W2,
                                                         const float* __restrict__ v2, const float* __restrict__ g,
                                                         float* __restrict__ dw, float* __restrict__ du) {
  const int i = xcd_row(blockIdx.x, n);
  if (i >= n) return;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int c = 4 * lane, h4 = c & (kTH - 1);
  const size_t rs = (size_t)n * kTC;
  const int e0 = row_ptr[i], e1 = row_ptr[i + 1];
  if (e0 + wave >= e1) return;
  float4 gq[3 * kTR];
#pragma unroll
  for (int q = 0; q < 3 * kTR; ++q) gq[q] = ld4(g + q * rs + (size_t)i * kTC + c);
  for (int64_t e = e0 + wave; e < e1; e += kTWaves) {
    const size_t off = (size_t)col[e] * kTC + c;
    float4 s = f4(0.f);
    float d[3] = {0.f, 0.f, 0.f};
    auto term = [&](const float* vv, const float* w, const float* u) {
      float4 x[kTR];
#pragma unroll
      for (int r = 0; r < kTR; ++r) x[r] = ld4(vv + r * rs + off);
      const float4 ww = w ? ld4(w + e * kTH + h4) : f4(0.f);
#pragma unroll
      for (int k = 0; k < 3; ++k) {
        float4 P = f4(0.f);
#pragma unroll
        for (int r = 0; r < kTR; ++r) P = fma4(gq[k * kTR + r], x[r], P);
        if (u) s = fma4(f4(u[3 * e + k]), P, s);
        d[k] += sum4(mul4(ww, P));
      }
    };
    term(v, W1.w, W1.u);
    if constexpr (kSecond) {
      if (v2) term(v2, W2.w, W2.u);
    }
    // the head's second channel sits 32 lanes up
    s.x += __shfl_xor(s.x, 32, kWave);
    s.y += __shfl_xor(s.y, 32, kWave);
    s.z += __shfl_xor(s.z, 32, kWave);
    s.w += __shfl_xor(s.w, 32, kWave);
    if (lane < 32) st4(dw + e * kTH + h4, s);
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      d[k] = dpp_row_sum16(d[k]);
      d[k] += __shfl_xor(d[k], 16, kWave);
      d[k] += __shfl_xor(d[k], 32, kWave);
    }
    if (lane < 3) du[3 * e + lane] = lane == 0 ? d[0] : lane == 1 ? d[1] : d[2];
  }
}

// ---------------------------------------------------------------------------
// Attention weights of the segmented softmax (e2former.py:327-364), per query row and head:
//   a = gate qk, m = max a, E = exp(a - m) p, s = sum E, rho = 1 / (s + 1e-3), alpha = E ih rho.
// A workgroup per row: lane (g, q) holds heads 4 q .. 4 q + 3 for the edges g, g + 8, ...; the row statistics are
// added over the eight groups in LDS in order.  Every pass recomputes E from gate, qk and the kept m, so that a
// pass reads each [E, 128] operand from HBM once (again from L2 for the second walk over the row).
//
// Gradient for G = dL/d alpha, with B = G ih and D = sum B E over the row:
//   d ih = G E rho,  dE = rho (B - rho D),  dp = sum_h dE exp(a - m),
//   da = dE E (+ the maximum's share -1e-3 rho^2 D / ties on the edges that attain it; the sum over the row of
//   dE E is what the maximum's own gradient has to cancel),  d gate = da qk,  d qk = da gate.
//
// Second order, for cotangents cg, cq, ci, cp of (d gate, d qk, d ih, dp): with kappa = cg qk + cq gate,
// lambda = exp(a - m) (p kappa + cp) and the row sums L = sum lambda, t = sum over ties of kappa / ties,
// X = sum B lambda + ci G E, the scalar being differentiated is sum over rows of rho X - rho^2 D (L + 1e-3 t), so with
//   delta = rho^2 (L + 1e-3 t),  zeta = rho^2 D,  sigma = -rho^2 (X - 2 rho D (L + 1e-3 t)):
//   f_B = rho lambda - delta E,     f_G = f_B ih + rho ci E,    f_ih = f_B G,
//   f_lambda = rho B - zeta,        f_E = rho ci G - delta B + sigma,
//   f_kappa = f_lambda E (- 1e-3 zeta / ties on ties),  f_p = sum_h f_lambda exp(a - m) kappa + f_E exp(a - m),
//   f_a = f_lambda lambda + f_E E (- its row sum / ties on ties),
//   f_gate = f_kappa cq + f_a qk,   f_qk = f_kappa cg + f_a gate,
// where the row sum of f_a is rho X - zeta L - delta D + sigma s.
// 128 k edges, one layer: the gradient 122 us, where the composition passed some twenty times over [E, 128]
// tensors of 65 MB (16 us each).
constexpr float kAwEps = 1e-3f;
constexpr int kAwGroups = 8;

__device__ __forceinline__ float aw_logit(float gate, float qk) {
#pragma clang fp contract(off)
  return gate * qk;   // rounded on its own: the maximum is matched bitwise
}
__device__ __forceinline__ float at(const float4& v, int i) { return i == 0 ? v.x : i == 1 ? v.y : i == 2 ? v.z : v.w; }

struct AwIn {
  const float* gate;
  const float* ih;
  int64_t ld_gate, ld_ih;
  const float* qk;      // [E, 128]
  const float* p;       // [E]
};

// Sum over the groups of each quad, returned to every lane.  red: [kAwGroups][32] float4.
__device__ __forceinline__ float4 aw_sum(float4 (*red)[32], float4 v, int g, int q) {
  __syncthreads();
  red[g][q] = v;
  __syncthreads();
  float4 s = red[0][q];
#pragma unroll
  for (int u = 1; u < kAwGroups; ++u) s = add4(s, red[u][q]);
  return s;
}
// Sum over the 32 lanes of a group and their four heads.
__device__ __forceinline__ float aw_heads(float v) {
  v = dpp_row_sum16(v);
  return v + __shfl_xor(v, 16, kWave);
}

__global__ __launch_bounds__(256) void k_aw_fwd(const int32_t* __restrict__ row_ptr, int n, AwIn I,
                                                float* __restrict__ alpha, float* __restrict__ mrow,
                                                float* __restrict__ srow, float* __restrict__ ties) {
  __shared__ float4 rm[kAwGroups][32], rs[kAwGroups][32], rc[kAwGroups][32];
  const int i = xcd_row(blockIdx.x, n);
  if (i >= n) return;
  const int q = threadIdx.x & 31, g = threadIdx.x >> 5;
  const int64_t e0 = row_ptr[i], e1 = row_ptr[i + 1];
  float m[4], s[4], cn[4];
#pragma unroll
  for (int z = 0; z < 4; ++z) {
    m[z] = -INFINITY;
    s[z] = cn[z] = 0.f;
  }
  for (int64_t e = e0 + g; e < e1; e += kAwGroups) {
    const float4 ga = ld4(I.gate + e * I.ld_gate + 4 * q), qk = ld4(I.qk + e * kTH + 4 * q);
    const float p = I.p[e];
#pragma unroll
    for (int z = 0; z < 4; ++z) {
      const float a = aw_logit(at(ga, z), at(qk, z));
      if (a > m[z]) {
        s[z] = s[z] * expf(m[z] - a) + p;
        m[z] = a;
        cn[z] = 1.f;
      } else {
        s[z] += (a == m[z] ? 1.f : expf(a - m[z])) * p;     // (a = m = -inf: worth 0 once a larger one comes)
        cn[z] += a == m[z] ? 1.f : 0.f;
      }
    }
  }
  rm[g][q] = make_float4(m[0], m[1], m[2], m[3]);
  rs[g][q] = make_float4(s[0], s[1], s[2], s[3]);
  rc[g][q] = make_float4(cn[0], cn[1], cn[2], cn[3]);
  __syncthreads();
  float M[4], rho[4], S[4], Cn[4];
#pragma unroll
  for (int z = 0; z < 4; ++z) {
    M[z] = -INFINITY;
#pragma unroll
    for (int u = 0; u < kAwGroups; ++u) M[z] = fmaxf(M[z], at(rm[u][q], z));
    S[z] = Cn[z] = 0.f;
#pragma unroll
    for (int u = 0; u < kAwGroups; ++u) {
      const float mu = at(rm[u][q], z);
      S[z] += at(rs[u][q], z) * (mu > -INFINITY ? expf(mu - M[z]) : 0.f);   // (a group of NaN alone: its sum is NaN)
      if (mu == M[z]) Cn[z] += at(rc[u][q], z);
    }
    if (M[z] == INFINITY) S[z] = NAN;         // inf - inf on the edge that attains it
    rho[z] = 1.f / (S[z] + kAwEps);
  }
  if (g == 0) {
    const size_t o = (size_t)i * kTH + 4 * q;
    st4(mrow + o, make_float4(M[0], M[1], M[2], M[3]));
    st4(srow + o, make_float4(S[0], S[1], S[2], S[3]));
    st4(ties + o, make_float4(fmaxf(Cn[0], 1.f), fmaxf(Cn[1], 1.f), fmaxf(Cn[2], 1.f), fmaxf(Cn[3], 1.f)));
  }
  for (int64_t e = e0 + g; e < e1; e += kAwGroups) {
    const float4 ga = ld4(I.gate + e * I.ld_gate + 4 * q), qk = ld4(I.qk + e * kTH + 4 * q);
    const float4 ih = ld4(I.ih + e * I.ld_ih + 4 * q);
    const float p = I.p[e];
    float o[4];
#pragma unroll
    for (int z = 0; z < 4; ++z)
      o[z] = expf(aw_logit(at(ga, z), at(qk, z)) - M[z]) * p * at(ih, z) * rho[z];
    st4(alpha + e * kTH + 4 * q, make_float4(o[0], o[1], o[2], o[3]));
  }
}

__global__ __launch_bounds__(256) void k_aw_bwd(const int32_t* __restrict__ row_ptr, int n, AwIn I,
                                                const float* __restrict__ mrow, const float* __restrict__ srow,
                                                const float* __restrict__ ties, const float* __restrict__ G,
                                                float* __restrict__ dgate, float* __restrict__ dih, int64_t ld_dgate,
                                                int64_t ld_dih, float* __restrict__ dqk, float* __restrict__ dp) {
  __shared__ float4 red[kAwGroups][32];
  const int i = xcd_row(blockIdx.x, n);
  if (i >= n) return;
  const int q = threadIdx.x & 31, g = threadIdx.x >> 5;
  const int64_t e0 = row_ptr[i], e1 = row_ptr[i + 1];
  const float4 M = ld4(mrow + (size_t)i * kTH + 4 * q), S = ld4(srow + (size_t)i * kTH + 4 * q);
  const float4 cn = ld4(ties + (size_t)i * kTH + 4 * q);
  float4 Da = f4(0.f);
  for (int64_t e = e0 + g; e < e1; e += kAwGroups) {
    const float4 ga = ld4(I.gate + e * I.ld_gate + 4 * q), qk = ld4(I.qk + e * kTH + 4 * q);
    const float4 ih = ld4(I.ih + e * I.ld_ih + 4 * q), gr = ld4(G + e * kTH + 4 * q);
    const float p = I.p[e];
    float d[4];
#pragma unroll
    for (int z = 0; z < 4; ++z) d[z] = at(gr, z) * at(ih, z) * (expf(aw_logit(at(ga, z), at(qk, z)) - at(M, z)) * p);
    Da = add4(Da, make_float4(d[0], d[1], d[2], d[3]));
  }
  const float4 D = aw_sum(red, Da, g, q);
  float rho[4], dmc[4];
#pragma unroll
  for (int z = 0; z < 4; ++z) {
    rho[z] = 1.f / (at(S, z) + kAwEps);
    dmc[z] = -kAwEps * rho[z] * rho[z] * at(D, z) / at(cn, z);
  }
  for (int64_t e = e0 + g; e < e1; e += kAwGroups) {
    const float4 ga = ld4(I.gate + e * I.ld_gate + 4 * q), qk = ld4(I.qk + e * kTH + 4 * q);
    const float4 ih = ld4(I.ih + e * I.ld_ih + 4 * q), gr = ld4(G + e * kTH + 4 * q);
    const float p = I.p[e];
    float og[4], oq[4], oi[4], sp = 0.f;
#pragma unroll
    for (int z = 0; z < 4; ++z) {
      const float a = aw_logit(at(ga, z), at(qk, z)), ex = expf(a - at(M, z)), Ez = ex * p;
      oi[z] = at(gr, z) * Ez * rho[z];
      const float dE = rho[z] * (at(gr, z) * at(ih, z) - rho[z] * at(D, z));
      const float da = dE * Ez + (a == at(M, z) ? dmc[z] : 0.f);
      sp = fmaf(dE, ex, sp);
      og[z] = da * at(qk, z);
      oq[z] = da * at(ga, z);
    }
    st4(dgate + e * ld_dgate + 4 * q, make_float4(og[0], og[1], og[2], og[3]));
    st4(dih + e * ld_dih + 4 * q, make_float4(oi[0], oi[1], oi[2], oi[3]));
    st4(dqk + e * kTH + 4 * q, make_float4(oq[0], oq[1], oq[2], oq[3]));
    sp = aw_heads(sp);
    if (q == 0) dp[e] = sp;
  }
}

struct AwCot {          // cotangents (NULL: zero)
  const float* gate;
  const float* ih;
  int64_t ld_gate, ld_ih;
  const float* qk;
  const float* p;
};
struct AwOut2 {
  float* G;
  float* gate;
  float* ih;
  int64_t ld_gate, ld_ih;
  float* qk;
  float* p;
};

__global__ __launch_bounds__(256) void k_aw_bwd2(const int32_t* __restrict__ row_ptr, int n, AwIn I,
                                                 const float* __restrict__ mrow, const float* __restrict__ srow,
                                                 const float* __restrict__ ties, const float* __restrict__ G, AwCot Q,
                                                 AwOut2 O) {
  __shared__ float4 red[kAwGroups][32];
  const int i = xcd_row(blockIdx.x, n);
  if (i >= n) return;
  const int q = threadIdx.x & 31, g = threadIdx.x >> 5;
  const int64_t e0 = row_ptr[i], e1 = row_ptr[i + 1];
  const float4 M = ld4(mrow + (size_t)i * kTH + 4 * q), S = ld4(srow + (size_t)i * kTH + 4 * q);
  const float4 cn = ld4(ties + (size_t)i * kTH + 4 * q);
  struct In {
    float4 ga, qk, ih, gr, cg, cq, ci;
    float p, cp;
  };
  auto load = [&](int64_t e) {
    In x;
    x.ga = ld4(I.gate + e * I.ld_gate + 4 * q);
    x.qk = ld4(I.qk + e * kTH + 4 * q);
    x.ih = ld4(I.ih + e * I.ld_ih + 4 * q);
    x.gr = ld4(G + e * kTH + 4 * q);
    x.cg = Q.gate ? ld4(Q.gate + e * Q.ld_gate + 4 * q) : f4(0.f);
    x.ci = Q.ih ? ld4(Q.ih + e * Q.ld_ih + 4 * q) : f4(0.f);
    x.cq = Q.qk ? ld4(Q.qk + e * kTH + 4 * q) : f4(0.f);
    x.p = I.p[e];
    x.cp = Q.p ? Q.p[e] : 0.f;
    return x;
  };
  float D[4] = {0.f, 0.f, 0.f, 0.f}, X[4] = {0.f, 0.f, 0.f, 0.f}, L[4] = {0.f, 0.f, 0.f, 0.f};
  float T[4] = {0.f, 0.f, 0.f, 0.f};
  for (int64_t e = e0 + g; e < e1; e += kAwGroups) {
    const In x = load(e);
#pragma unroll
    for (int z = 0; z < 4; ++z) {
      const float a = aw_logit(at(x.ga, z), at(x.qk, z)), ex = expf(a - at(M, z)), Ez = ex * x.p;
      const float B = at(x.gr, z) * at(x.ih, z), kap = at(x.cg, z) * at(x.qk, z) + at(x.cq, z) * at(x.ga, z);
      const float lam = ex * (x.p * kap + x.cp);
      D[z] = fmaf(B, Ez, D[z]);
      X[z] += B * lam + at(x.ci, z) * at(x.gr, z) * Ez;
      L[z] += lam;
      if (a == at(M, z)) T[z] += kap;
    }
  }
  const float4 D4 = aw_sum(red, make_float4(D[0], D[1], D[2], D[3]), g, q);
  const float4 X4 = aw_sum(red, make_float4(X[0], X[1], X[2], X[3]), g, q);
  const float4 L4 = aw_sum(red, make_float4(L[0], L[1], L[2], L[3]), g, q);
  const float4 T4 = aw_sum(red, make_float4(T[0], T[1], T[2], T[3]), g, q);
  float rho[4], del[4], zet[4], sig[4], tie_k[4], tie_a[4];
#pragma unroll
  for (int z = 0; z < 4; ++z) {
    const float r = 1.f / (at(S, z) + kAwEps), d = at(D4, z), lt = at(L4, z) + kAwEps * at(T4, z) / at(cn, z);
    rho[z] = r;
    del[z] = r * r * lt;
    zet[z] = r * r * d;
    sig[z] = -r * r * (at(X4, z) - 2.f * r * d * lt);
    tie_k[z] = -kAwEps * zet[z] / at(cn, z);
    tie_a[z] = -(r * at(X4, z) - zet[z] * at(L4, z) - del[z] * d + sig[z] * at(S, z)) / at(cn, z);
  }
  for (int64_t e = e0 + g; e < e1; e += kAwGroups) {
    const In x = load(e);
    float oG[4], og[4], oi[4], oq[4], sp = 0.f;
#pragma unroll
    for (int z = 0; z < 4; ++z) {
      const float a = aw_logit(at(x.ga, z), at(x.qk, z)), ex = expf(a - at(M, z)), Ez = ex * x.p;
      const float B = at(x.gr, z) * at(x.ih, z), kap = at(x.cg, z) * at(x.qk, z) + at(x.cq, z) * at(x.ga, z);
      const float lam = ex * (x.p * kap + x.cp);
      const float fB = rho[z] * lam - del[z] * Ez, fl = rho[z] * B - zet[z];
      const float fE = rho[z] * at(x.ci, z) * at(x.gr, z) - del[z] * B + sig[z];
      const bool tie = a == at(M, z);
      const float fk = fl * Ez + (tie ? tie_k[z] : 0.f);
      const float fa = fl * lam + fE * Ez + (tie ? tie_a[z] : 0.f);
      oG[z] = fB * at(x.ih, z) + rho[z] * at(x.ci, z) * Ez;
      oi[z] = fB * at(x.gr, z);
      sp += ex * (fl * kap + fE);
      og[z] = fk * at(x.cq, z) + fa * at(x.qk, z);
      oq[z] = fk * at(x.cg, z) + fa * at(x.ga, z);
    }
    // kappa = cg qk + cq gate: its derivative by gate is cq, by qk is cg
    st4(O.G + e * kTH + 4 * q, make_float4(oG[0], oG[1], oG[2], oG[3]));
    st4(O.gate + e * O.ld_gate + 4 * q, make_float4(og[0], og[1], og[2], og[3]));
    st4(O.ih + e * O.ld_ih + 4 * q, make_float4(oi[0], oi[1], oi[2], oi[3]));
    st4(O.qk + e * kTH + 4 * q, make_float4(oq[0], oq[1], oq[2], oq[3]));
    sp = aw_heads(sp);
    if (q == 0) O.p[e] = sp;
  }
}

// out[e, :] = (y[e, :] +) A[ia[e], :] + B[ib[e], :], rows of K floats (K % 4 == 0), y NULL: no such term
constexpr int kAgU = 4;
__global__ __launch_bounds__(256) void k_add_gather2(const float* __restrict__ y, const float* __restrict__ A,
                                                     const int32_t* __restrict__ ia, const float* __restrict__ B,
                                                     const int32_t* __restrict__ ib, int64_t n, int K,
                                                     float* __restrict__ out) {
  const int kq = K / 4, ng = 256 / kq, q = (int)threadIdx.x % kq, g = (int)threadIdx.x / kq;
  if (g >= ng) return;
  const int64_t e0 = (int64_t)blockIdx.x * ng * kAgU + g;
  float4 a[kAgU], b[kAgU], v[kAgU];
#pragma unroll
  for (int u = 0; u < kAgU; ++u) {
    const int64_t e = min(e0 + (int64_t)u * ng, n - 1);
    a[u] = ld4(A + (int64_t)ia[e] * K + 4 * q);
    b[u] = ld4(B + (int64_t)ib[e] * K + 4 * q);
    v[u] = y ? ld4(y + e * K + 4 * q) : f4(0.f);
  }
#pragma unroll
  for (int u = 0; u < kAgU; ++u) {
    const int64_t e = e0 + (int64_t)u * ng;
    if (e < n) st4(out + e * K + 4 * q, add4(add4(v[u], a[u]), b[u]));
  }
}

bool al16(const void* p) { return ((uintptr_t)p & 15) == 0; }

int check_lists(const e2v2_train_edges* L, const char* who) {
  E2V2_REQUIRE(L && L->n_rows >= 0 && L->n_edges >= 0, "%s: null or negative edge list", who);
  E2V2_REQUIRE(L->n_rows == 0 || (L->row_ptr && L->key_ptr), "%s: null row or column pointers", who);
  E2V2_REQUIRE(L->n_edges == 0 || (L->col && L->edge_row && L->key_eid), "%s: null edge arrays", who);
  return 0;
}
// The m-contraction of SO3_Linear2Scalar (module_utils.py:2241-2266) on separate operands a, b [9][n][hid]:
// h[i][l hid + c] = the sum over the rows m of degree l of a[m][i][c] b[m][i][c], and its adjoint
// y[m][i][c] = h[i][l hid + c] b[m][i][c].  Each is the other's derivative, so two passes over the operands serve
// every order; composed (product, splits, sums, concatenation, expansions) a layer's double backward took some
// fifty.  Bound by memory: the expansion takes 6.2 us at 1500 nodes
// of 512 (55 MB, mostly in the Infinity Cache).
__global__ __launch_bounds__(256) void k_mdot(const float* __restrict__ a, const float* __restrict__ b, int n, int hid,
                                              float* __restrict__ h) {
  const int q = hid / 4;
  const int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (t >= (int64_t)n * q) return;
  const int64_t i = t / q, c = 4 * (t % q), step = (int64_t)n * hid, o = i * hid + c;
#pragma unroll
  for (int l = 0; l < 3; ++l) {
    float4 s = mul4(ld4(a + l * l * step + o), ld4(b + l * l * step + o));
#pragma unroll
    for (int m = l * l + 1; m < (l + 1) * (l + 1); ++m) s = fma4(ld4(a + m * step + o), ld4(b + m * step + o), s);
    st4(h + (i * 3 + l) * hid + c, s);
  }
}
__global__ __launch_bounds__(256) void k_mexpand(const float* __restrict__ h, const float* __restrict__ b, int n,
                                                 int hid, float* __restrict__ y) {
  const int q = hid / 4;
  const int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (t >= (int64_t)n * q) return;
  const int64_t i = t / q, c = 4 * (t % q), step = (int64_t)n * hid, o = i * hid + c;
#pragma unroll
  for (int l = 0; l < 3; ++l) {
    const float4 w = ld4(h + (i * 3 + l) * hid + c);
#pragma unroll
    for (int m = l * l; m < (l + 1) * (l + 1); ++m) st4(y + m * step + o, mul4(w, ld4(b + m * step + o)));
  }
}

}  // namespace
}  // namespace e2v2

using namespace e2v2;

E2V2_API int e2v2_so2_agg(const e2v2_train_edges* L, const float* w1, const float* u1, const float* w2,
                          const float* u2, const float* v, const float* w3, const float* u3, const float* v2,
                          float* out, hipStream_t s) {
  if (int rc = check_lists(L, "so2_agg")) return rc;
  if (L->n_rows == 0) return 0;
  E2V2_REQUIRE(v && out && (!w1 || u1) && (!w2 || u2) && (!v2 || (w3 && u3)), "so2_agg: null operand");
  E2V2_REQUIRE(al16(w1) && al16(w2) && al16(v) && al16(w3) && al16(v2) && al16(out), "so2_agg: 16-byte alignment");
  const dim3 grid(xcd_grid(L->n_rows)), blk(kTThreads);
  if (w2 || v2)
    hipLaunchKernelGGL(k_so2_agg<true>, grid, blk, 0, s, L->row_ptr, L->col, L->n_rows, EdgeW{w1, u1}, EdgeW{w2, u2}, v,
                       EdgeW{w3, u3}, v2, out);
  else
    hipLaunchKernelGGL(k_so2_agg<false>, grid, blk, 0, s, L->row_ptr, L->col, L->n_rows, EdgeW{w1, u1},
                       EdgeW{nullptr, nullptr}, v, EdgeW{nullptr, nullptr}, nullptr, out);
  E2V2_LAUNCHED("k_so2_agg");
  return 0;
}

E2V2_API int e2v2_so2_agg_dv(const e2v2_train_edges* L, const float* w1, const float* u1, const float* w2,
                             const float* u2, const float* g, float* dv, hipStream_t s) {
  if (int rc = check_lists(L, "so2_agg_dv")) return rc;
  if (L->n_rows == 0) return 0;
  E2V2_REQUIRE(g && dv && (!w1 || u1) && (!w2 || u2), "so2_agg_dv: null operand");
  E2V2_REQUIRE(al16(w1) && al16(w2) && al16(g) && al16(dv), "so2_agg_dv: 16-byte alignment");
  const dim3 grid(xcd_grid(L->n_rows)), blk(kTThreads);
  if (w2)
    hipLaunchKernelGGL(k_so2_dv<true>, grid, blk, 0, s, L->key_ptr, L->key_eid, L->edge_row, L->n_rows, EdgeW{w1, u1},
                       EdgeW{w2, u2}, g, dv);
  else
    hipLaunchKernelGGL(k_so2_dv<false>, grid, blk, 0, s, L->key_ptr, L->key_eid, L->edge_row, L->n_rows, EdgeW{w1, u1},
                       EdgeW{nullptr, nullptr}, g, dv);
  E2V2_LAUNCHED("k_so2_dv");
  return 0;
}

E2V2_API int e2v2_so2_agg_dw(const e2v2_train_edges* L, const float* w1, const float* u1, const float* v,
                             const float* w2, const float* u2, const float* v2, const float* g, float* dw, float* du,
                             hipStream_t s) {
  if (int rc = check_lists(L, "so2_agg_dw")) return rc;
  if (L->n_rows == 0 || L->n_edges == 0) return 0;
  E2V2_REQUIRE(v && g && dw && du, "so2_agg_dw: null operand");
  E2V2_REQUIRE(al16(w1) && al16(w2) && al16(v) && al16(v2) && al16(g) && al16(dw), "so2_agg_dw: 16-byte alignment");
  const dim3 grid(xcd_grid(L->n_rows)), blk(kTThreads);
  if (v2)
    hipLaunchKernelGGL(k_so2_dw<true>, grid, blk, 0, s, L->row_ptr, L->col, L->n_rows, EdgeW{w1, u1}, v, EdgeW{w2, u2},
                       v2, g, dw, du);
  else
    hipLaunchKernelGGL(k_so2_dw<false>, grid, blk, 0, s, L->row_ptr, L->col, L->n_rows, EdgeW{w1, u1}, v,
                       EdgeW{nullptr, nullptr}, nullptr, g, dw, du);
  E2V2_LAUNCHED("k_so2_dw");
  return 0;
}

static int check_aw(const e2v2_train_edges* L, const float* gate, int64_t ld_gate, const float* ih, int64_t ld_ih,
                    const float* qk, const float* p, const char* who) {
  if (int rc = check_lists(L, who)) return rc;
  E2V2_REQUIRE(L->n_edges == 0 || (gate && ih && qk && p && ld_gate >= kTH && ld_ih >= kTH && ld_gate % 4 == 0 &&
                                   ld_ih % 4 == 0 && al16(gate) && al16(ih) && al16(qk)),
               "%s: the edge operands need 128 heads per row on 16-byte rows", who);
  return 0;
}

E2V2_API int e2v2_attn_weights_fwd(const e2v2_train_edges* L, const float* gate, int64_t ld_gate, const float* ih,
                                   int64_t ld_ih, const float* qk, const float* p, float* alpha, float* mrow,
                                   float* srow, float* ties, hipStream_t s) {
  if (int rc = check_aw(L, gate, ld_gate, ih, ld_ih, qk, p, "attn_weights_fwd")) return rc;
  if (L->n_rows == 0) return 0;
  E2V2_REQUIRE(mrow && srow && ties && (alpha || L->n_edges == 0), "attn_weights_fwd: null output");
  hipLaunchKernelGGL(k_aw_fwd, dim3(xcd_grid(L->n_rows)), dim3(256), 0, s, L->row_ptr, L->n_rows,
                     AwIn{gate, ih, ld_gate, ld_ih, qk, p}, alpha, mrow, srow, ties);
  E2V2_LAUNCHED("k_aw_fwd");
  return 0;
}

E2V2_API int e2v2_attn_weights_bwd(const e2v2_train_edges* L, const float* gate, int64_t ld_gate, const float* ih,
                                   int64_t ld_ih, const float* qk, const float* p, const float* mrow,
                                   const float* srow, const float* ties, const float* grad, float* dgate,
                                   int64_t ld_dgate, float* dih, int64_t ld_dih, float* dqk, float* dp,
                                   hipStream_t s) {
  if (int rc = check_aw(L, gate, ld_gate, ih, ld_ih, qk, p, "attn_weights_bwd")) return rc;
  if (L->n_rows == 0 || L->n_edges == 0) return 0;
  E2V2_REQUIRE(mrow && srow && ties && grad && dgate && dih && dqk && dp && ld_dgate % 4 == 0 && ld_dih % 4 == 0 &&
                   al16(grad) && al16(dgate) && al16(dih) && al16(dqk),
               "attn_weights_bwd: null or unaligned operand");
  hipLaunchKernelGGL(k_aw_bwd, dim3(xcd_grid(L->n_rows)), dim3(256), 0, s, L->row_ptr, L->n_rows,
                     AwIn{gate, ih, ld_gate, ld_ih, qk, p}, mrow, srow, ties, grad, dgate, dih, ld_dgate, ld_dih, dqk,
                     dp);
  E2V2_LAUNCHED("k_aw_bwd");
  return 0;
}

E2V2_API int e2v2_attn_weights_bwd2(const e2v2_train_edges* L, const float* gate, int64_t ld_gate, const float* ih,
                                    int64_t ld_ih, const float* qk, const float* p, const float* mrow,
                                    const float* srow, const float* ties, const float* grad, const float* cgate,
                                    int64_t ld_cgate, const float* cih, int64_t ld_cih, const float* cqk,
                                    const float* cp, float* fgrad, float* fgate, int64_t ld_fgate, float* fih,
                                    int64_t ld_fih, float* fqk, float* fp, hipStream_t s) {
  if (int rc = check_aw(L, gate, ld_gate, ih, ld_ih, qk, p, "attn_weights_bwd2")) return rc;
  if (L->n_rows == 0 || L->n_edges == 0) return 0;
  E2V2_REQUIRE(mrow && srow && ties && grad && fgrad && fgate && fih && fqk && fp && ld_cgate % 4 == 0 &&
                   ld_cih % 4 == 0 && ld_fgate % 4 == 0 && ld_fih % 4 == 0 && al16(grad) && al16(cgate) &&
                   al16(cih) && al16(cqk) && al16(fgrad) && al16(fgate) && al16(fih) && al16(fqk),
               "attn_weights_bwd2: null or unaligned operand");
  hipLaunchKernelGGL(k_aw_bwd2, dim3(xcd_grid(L->n_rows)), dim3(256), 0, s, L->row_ptr, L->n_rows,
                     AwIn{gate, ih, ld_gate, ld_ih, qk, p}, mrow, srow, ties, grad,
                     AwCot{cgate, cih, ld_cgate, ld_cih, cqk, cp}, AwOut2{fgrad, fgate, fih, ld_fgate, ld_fih, fqk, fp});
  E2V2_LAUNCHED("k_aw_bwd2");
  return 0;
}

E2V2_API int e2v2_add_gather2(const float* y, const float* a, const int32_t* ia, const float* b, const int32_t* ib,
                              int64_t n, int K, float* out, hipStream_t s) {
  E2V2_REQUIRE(n >= 0 && K >= 4 && K % 4 == 0 && K <= 1024, "add_gather2: n %lld, K %d (a multiple of 4 up to 1024)",
               (long long)n, K);
  if (n == 0) return 0;
  E2V2_REQUIRE(a && ia && b && ib && out && al16(y) && al16(a) && al16(b) && al16(out),
               "add_gather2: null or unaligned operand");
  const int per = 256 / (K / 4) * kAgU;
  hipLaunchKernelGGL(k_add_gather2, dim3((unsigned)((n + per - 1) / per)), dim3(256), 0, s, y, a, ia, b, ib, n, K, out);
  E2V2_LAUNCHED("k_add_gather2");
  return 0;
}

static int check_mdot(const void* x, const void* y, const void* z, int n, int hid, const char* who) {
  E2V2_REQUIRE(n > 0 && hid > 0 && hid % 4 == 0 && (int64_t)n * hid < (1LL << 36), "%s: n %d, hid %d", who, n, hid);
  E2V2_REQUIRE(x && y && z && ((uintptr_t)x | (uintptr_t)y | (uintptr_t)z) % 16 == 0,
               "%s: operands must be 16-byte aligned", who);
  return 0;
}

E2V2_API int e2v2_mdot(const float* a, const float* b, int n, int hid, float* h, hipStream_t s) {
  if (int rc = check_mdot(a, b, h, n, hid, "mdot")) return rc;
  const int64_t t = (int64_t)n * (hid / 4);
  hipLaunchKernelGGL(k_mdot, dim3((uint32_t)((t + 255) / 256)), dim3(256), 0, s, a, b, n, hid, h);
  E2V2_LAUNCHED("k_mdot");
  return 0;
}

E2V2_API int e2v2_mexpand(const float* h, const float* b, int n, int hid, float* y, hipStream_t s) {
  if (int rc = check_mdot(h, b, y, n, hid, "mexpand")) return rc;
  const int64_t t = (int64_t)n * (hid / 4);
  hipLaunchKernelGGL(k_mexpand, dim3((uint32_t)((t + 255) / 256)), dim3(256), 0, s, h, b, n, hid, y);
  E2V2_LAUNCHED("k_mexpand");
  return 0;
}
