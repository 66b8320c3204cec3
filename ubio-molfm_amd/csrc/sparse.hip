// Segment (CSR) kernels behind the reference's op-level sparse edge functions
// (src/molfm/models/e2former/triton_dr/): edge-indexed dot products, their
// grouped reductions (the QK logits, the value aggregation and both of their
// gradients), the segmented alpha sum, row gathers and the edge-degree outer
// product with its gradient.  A segment layout is the reference's
// (row_ptr [R+1], col_index, alpha_index): slot p of row r carries edge
// alpha_index[p] and its partner row col_index[p].  Every row is summed in a
// fixed order by one workgroup (deterministic, no atomics).  Tensors are fp32
// with explicit element strides, so [R, H, D] and [M, C, H] operands share
// the kernels.  Slots whose partner row or edge id is out of range are skipped
// and row bounds are clamped to the slot arrays, so malformed metadata cannot
// make a kernel read or write outside its operands.  The attention and degree
// paths of the model run fused in attn.hip and deg.hip; these serve callers of
// the reference's op-level interfaces.
#include <algorithm>
#include <type_traits>

#include "common.h"
#include "../../include/e2v2.h"

namespace e2v2 {

constexpr int kSegThreads = 256;
constexpr int kSegMaxD = 16;   // d per thread of the h-fast segmented reduction
constexpr int kSegMaxA = 24;   // d of a segmented dot held in registers

struct SegRow {
  int p0, p1;
};

__device__ __forceinline__ SegRow seg_row(const e2v2_segments& S, int r) {
  const int64_t n = S.n_slots;
  int64_t a = S.row_ptr[r], b = S.row_ptr[r + 1];
  a = a < 0 ? 0 : (a > n ? n : a);
  b = b < a ? a : (b > n ? n : b);
  return {(int)a, (int)b};
}

__device__ __forceinline__ bool slot_ok(const e2v2_segments& S, int c, int e) {
  return c >= 0 && c < S.n_cols && e >= 0 && (int64_t)e < S.n_edges;
}

// Slots of one row staged in LDS (edge id and partner row, -1 for a skipped slot) when the row has at most
// kSegStage of them; longer rows read the slot arrays directly.
constexpr int kSegStage = 512;

__device__ __forceinline__ bool stage_row(const e2v2_segments& S, const SegRow& R, bool with_col, int* se, int* sc) {
  const int np = R.p1 - R.p0;
  if (np > kSegStage) return false;
  for (int t = threadIdx.x; t < np; t += kSegThreads) {
    const int p = R.p0 + t;
    const int e = S.alpha_index[p], c = with_col ? S.col_index[p] : 0;
    const bool ok = e >= 0 && (int64_t)e < S.n_edges && (!with_col || (c >= 0 && c < S.n_cols));
    se[t] = ok ? e : -1;
    sc[t] = ok ? c : 0;
  }
  __syncthreads();
  return true;
}

// out[alpha_index[p], h] = sum_d A[r, h, d] B[col_index[p], h, d] for the slots p of row r
__global__ __launch_bounds__(kSegThreads) void k_seg_dot(e2v2_segments S, const float* __restrict__ A, int64_t sa_r,
                                                         int64_t sa_h, int64_t sa_d, const float* __restrict__ B,
                                                         int64_t sb_r, int64_t sb_h, int64_t sb_d, int H, int D,
                                                         float* __restrict__ out, int64_t so_e, int64_t so_h) {
  __shared__ int se[kSegStage], sc[kSegStage];
  const int r = blockIdx.x;
  const SegRow R = seg_row(S, r);
  const bool staged = stage_row(S, R, true, se, sc);
  const unsigned n = (unsigned)(R.p1 - R.p0) * (unsigned)H;
  const float* a = A + (int64_t)r * sa_r;
  // H dividing the block: thread t keeps head t % H for every slot it takes (t / H, + 256 / H, ...), so its
  // A row stays in registers; each slot's B row is loaded whole before the products (summed in d order)
  if (kSegThreads % H == 0 && D <= kSegMaxA) {
    const int h = (int)threadIdx.x % H, ks = kSegThreads / H, np = R.p1 - R.p0;
    const float* ah = a + (int64_t)h * sa_h;
    float ar[kSegMaxA];
#pragma unroll
    for (int j = 0; j < kSegMaxA; ++j) ar[j] = j < D ? ah[(int64_t)j * sa_d] : 0.f;
    for (int k = (int)threadIdx.x / H; k < np; k += ks) {
      int c, e;
      if (staged) {
        e = se[k];
        c = sc[k];
        if (e < 0) continue;
      } else {
        const int p = R.p0 + k;
        c = S.col_index[p];
        e = S.alpha_index[p];
        if (!slot_ok(S, c, e)) continue;
      }
      const float* b = B + (int64_t)c * sb_r + (int64_t)h * sb_h;
      float y[kSegMaxA];
#pragma unroll
      for (int j = 0; j < kSegMaxA; ++j) y[j] = j < D ? b[(int64_t)j * sb_d] : 0.f;
      float s = 0.f;
#pragma unroll
      for (int j = 0; j < kSegMaxA; ++j)
        if (j < D) s = fmaf(ar[j], y[j], s);
      out[(int64_t)e * so_e + (int64_t)h * so_h] = s;
    }
    return;
  }
  // unit-stride rows of 16-byte aligned groups of four: float4 loads (the same products, summed in d order)
  const bool v4 = sa_d == 1 && sb_d == 1 && (D & 3) == 0 && ((sa_r | sa_h | sb_r | sb_h) & 3) == 0 &&
                  (((uintptr_t)A | (uintptr_t)B) & 15) == 0;
  for (unsigned idx = threadIdx.x; idx < n; idx += kSegThreads) {
    const int k = (int)(idx / (unsigned)H), h = (int)(idx % (unsigned)H);
    int c, e;
    if (staged) {
      e = se[k];
      c = sc[k];
      if (e < 0) continue;
    } else {
      const int p = R.p0 + k;
      c = S.col_index[p];
      e = S.alpha_index[p];
      if (!slot_ok(S, c, e)) continue;
    }
    const float* b = B + (int64_t)c * sb_r + (int64_t)h * sb_h;
    const float* ah = a + (int64_t)h * sa_h;
    float s = 0.f;
    if (v4) {
      for (int d = 0; d < D; d += 4) {
        const float4 x = *reinterpret_cast<const float4*>(ah + d), y = *reinterpret_cast<const float4*>(b + d);
        s = fmaf(x.x, y.x, s);
        s = fmaf(x.y, y.y, s);
        s = fmaf(x.z, y.z, s);
        s = fmaf(x.w, y.w, s);
      }
    } else {
      // four d steps' loads issued before their products (the same order of the sum)
      int d = 0;
      for (; d + 4 <= D; d += 4) {
        float x[4], y[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          x[u] = ah[(int64_t)(d + u) * sa_d];
          y[u] = b[(int64_t)(d + u) * sb_d];
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) s = fmaf(x[u], y[u], s);
      }
      for (; d < D; ++d) s = fmaf(ah[(int64_t)d * sa_d], b[(int64_t)d * sb_d], s);
    }
    out[(int64_t)e * so_e + (int64_t)h * so_h] = s;
  }
}

// out[r, h, d] = sum_{p in row r} W[alpha_index[p], h] X[col_index[p], h, d]; X NULL: the plain
// sum of W (D = 1).  Threads walk (h, d) with the operand's unit-stride index fastest.
__global__ __launch_bounds__(kSegThreads) void k_seg_reduce(e2v2_segments S, const float* __restrict__ W,
                                                            int64_t sw_e, int64_t sw_h, const float* __restrict__ X,
                                                            int64_t sx_r, int64_t sx_h, int64_t sx_d, int H, int D,
                                                            bool h_fast, float* __restrict__ out, int64_t so_r,
                                                            int64_t so_h, int64_t so_d) {
  __shared__ int se[kSegStage], sc[kSegStage];
  const int r = blockIdx.x;
  const SegRow R = seg_row(S, r);
  const bool staged = stage_row(S, R, X != nullptr, se, sc);
  const int np = R.p1 - R.p0;
  // h-fast X with H dividing the block: thread (g, h) = (t / H, t % H) owns d = g, g + G, ... (G = 256 / H,
  // at most kSegMaxD of them) and loads W[e, h] once per slot for all of them; the sums keep slot order
  const int G = (X && h_fast && kSegThreads % H == 0) ? kSegThreads / H : 0;
  if (staged && G > 0 && (D + G - 1) / G <= kSegMaxD) {
    const int t = threadIdx.x, h = t % H, g = t / H;
    const int nd = g < D ? (D - g + G - 1) / G : 0;
    const float* wh = W + (int64_t)h * sw_h;
    const float* xh = X + (int64_t)h * sx_h + (int64_t)g * sx_d;
    const int64_t xs = (int64_t)G * sx_d;
    float acc[kSegMaxD];
#pragma unroll
    for (int j = 0; j < kSegMaxD; ++j) acc[j] = 0.f;
    int k = 0;
    for (; k + 2 <= np; k += 2) {   // two slots' loads in flight
      float w[2], x[2][kSegMaxD];
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        const int e = se[k + u];
        w[u] = e >= 0 ? wh[(int64_t)e * sw_e] : 0.f;
        const float* xr = xh + (int64_t)sc[k + u] * sx_r;
#pragma unroll
        for (int j = 0; j < kSegMaxD; ++j) x[u][j] = (e >= 0 && j < nd) ? xr[j * xs] : 0.f;
      }
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        if (se[k + u] < 0) continue;
#pragma unroll
        for (int j = 0; j < kSegMaxD; ++j)
          if (j < nd) acc[j] = fmaf(w[u], x[u][j], acc[j]);
      }
    }
    if (k < np && se[k] >= 0) {
      const float w = wh[(int64_t)se[k] * sw_e];
      const float* xr = xh + (int64_t)sc[k] * sx_r;
#pragma unroll
      for (int j = 0; j < kSegMaxD; ++j)
        if (j < nd) acc[j] = fmaf(w, xr[j * xs], acc[j]);
    }
#pragma unroll
    for (int j = 0; j < kSegMaxD; ++j)
      if (j < nd) out[(int64_t)r * so_r + (int64_t)h * so_h + (int64_t)(g + j * G) * so_d] = acc[j];
    return;
  }
  for (int idx = threadIdx.x; idx < H * D; idx += kSegThreads) {
    const int h = h_fast ? idx % H : idx / D, d = h_fast ? idx / H : idx % D;
    const float* wh = W + (int64_t)h * sw_h;
    const float* xh = X ? X + (int64_t)h * sx_h + (int64_t)d * sx_d : nullptr;
    float s = 0.f;
    if (staged) {
      // four slots' loads in flight at a time (a skipped slot loads nothing and adds nothing); the sum keeps
      // slot order
      int k = 0;
      for (; k + 4 <= np; k += 4) {
        int e[4];
        float w[4], x[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          e[u] = se[k + u];
          w[u] = e[u] >= 0 ? wh[(int64_t)e[u] * sw_e] : 0.f;
          x[u] = (xh && e[u] >= 0) ? xh[(int64_t)sc[k + u] * sx_r] : 1.f;
        }
#pragma unroll
        for (int u = 0; u < 4; ++u)
          if (e[u] >= 0) s = xh ? fmaf(w[u], x[u], s) : s + w[u];
      }
      for (; k < np; ++k) {
        const int e = se[k];
        if (e < 0) continue;
        const float w = wh[(int64_t)e * sw_e];
        s = xh ? fmaf(w, xh[(int64_t)sc[k] * sx_r], s) : s + w;
      }
    } else {
      for (int p = R.p0; p < R.p1; ++p) {
        const int e = S.alpha_index[p];
        if (e < 0 || (int64_t)e >= S.n_edges) continue;
        const float w = wh[(int64_t)e * sw_e];
        if (X) {
          const int c = S.col_index[p];
          if (c < 0 || c >= S.n_cols) continue;
          s = fmaf(w, xh[(int64_t)c * sx_r], s);
        } else {
          s += w;
        }
      }
    }
    out[(int64_t)r * so_r + (int64_t)h * so_h + (int64_t)d * so_d] = s;
  }
}

// out[e, k] = in[index[e], k] (rows of K contiguous floats; an index outside [0, n_in) gives a zero row)
__global__ void k_gather_rows(const float* __restrict__ in, int64_t n_in, const int32_t* __restrict__ index,
                              int64_t n, int K, float* __restrict__ out) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= n * K) return;
  const int64_t e = t / K;
  const int64_t i = index[e];
  out[t] = (i >= 0 && i < n_in) ? in[i * K + t % K] : 0.f;
}

// The same in 16-byte pieces: K / 4 lanes per row, kGatherU rows of a lane group in flight (127,610 rows of 128:
// 46.5 -> 15.3 us, most of it the output's write).
constexpr int kGatherU = 4;
__global__ __launch_bounds__(kSegThreads) void k_gather_rows_v(const float* __restrict__ in, int64_t n_in,
                                                               const int32_t* __restrict__ index, int64_t n, int K,
                                                               float* __restrict__ out) {
  const int kq = K / 4, ng = kSegThreads / kq, q = (int)threadIdx.x % kq, g = (int)threadIdx.x / kq;
  if (g >= ng) return;
  const int64_t e0 = (int64_t)blockIdx.x * ng * kGatherU + g;
  float4 v[kGatherU];
#pragma unroll
  for (int u = 0; u < kGatherU; ++u) {
    const int64_t e = e0 + (int64_t)u * ng;
    const int64_t i = e < n ? index[e] : -1;
    v[u] = make_float4(0.f, 0.f, 0.f, 0.f);
    if (i >= 0 && i < n_in) v[u] = *reinterpret_cast<const float4*>(in + i * K + 4 * q);
  }
#pragma unroll
  for (int u = 0; u < kGatherU; ++u) {
    const int64_t e = e0 + (int64_t)u * ng;
    if (e < n) *reinterpret_cast<float4*>(out + e * K + 4 * q) = v[u];
  }
}

// out[r, l, h] = sum_{p in row r} sh[e, l] fea[e, h], e = alpha_index[p]
__global__ __launch_bounds__(kSegThreads) void k_outer_reduce(e2v2_segments S, const float* __restrict__ sh,
                                                              const float* __restrict__ fea, int L, int H,
                                                              float* __restrict__ out) {
  const int r = blockIdx.x;
  const SegRow R = seg_row(S, r);
  for (int idx = threadIdx.x; idx < L * H; idx += kSegThreads) {
    const int l = idx / H, h = idx % H;
    float s = 0.f;
    for (int p = R.p0; p < R.p1; ++p) {
      const int64_t e = S.alpha_index[p];
      if (e < 0 || e >= S.n_edges) continue;
      s = fmaf(sh[e * L + l], fea[e * H + h], s);
    }
    out[(int64_t)r * L * H + idx] = s;
  }
}

// dsh[e, l] = sum_h g[q[e], l, h] fea[e, h]  (q[e] outside [0, n_rows): 0)
__global__ void k_outer_dsh(const float* __restrict__ g, int n_rows, const float* __restrict__ fea,
                            const int32_t* __restrict__ qidx, int64_t n_edges, int L, int H, float* __restrict__ dsh) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= n_edges * L) return;
  const int64_t e = t / L;
  const int l = (int)(t % L);
  const int q = qidx[e];
  float s = 0.f;
  if (q >= 0 && q < n_rows) {
    const float* gr = g + ((int64_t)q * L + l) * H;
    const float* f = fea + e * H;
    for (int h = 0; h < H; ++h) s = fmaf(gr[h], f[h], s);
  }
  dsh[t] = s;
}

constexpr int kOuterL = 9;   // rows l of the vector forms

// dfea[e, h] = sum_l g[q[e], l, h] sh[e, l]  (q[e] outside [0, n_rows): 0)
__global__ void k_outer_dfea(const float* __restrict__ g, int n_rows, const float* __restrict__ sh,
                             const int32_t* __restrict__ qidx, int64_t n_edges, int L, int H,
                             float* __restrict__ dfea) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= n_edges * H) return;
  const int64_t e = t / H;
  const int h = (int)(t % H);
  const int q = qidx[e];
  float s = 0.f;
  if (q >= 0 && q < n_rows) {
    const float* gr = g + (int64_t)q * L * H + h;
    const float* s_e = sh + e * L;
    for (int l = 0; l < L; ++l) s = fmaf(gr[(int64_t)l * H], s_e[l], s);
  }
  dfea[t] = s;
}

// ---------------------------------------------------------------------------
// Vector forms (16-byte loads) of the segment kernels, for operands whose unit stride runs over the heads
// ("h-fast", [M, C, H]) or over d ("d-fast", [R, H, D]) in aligned groups of four.  What bounds them is the gather
// of the partner rows from L2 (18 rows of 128 heads: 9 KB an edge), so: four values per lane and several slots'
// rows in flight, every operand row read once per row (the A row of a dot stays in registers), and the rows of an
// XCD contiguous (xcd_row), so that the partner rows of spatially ordered atoms are found in its own L2.  Slots
// are staged in LDS in chunks of kSegStage.  1,500 rows of 85 edges, 128 heads: dot over 18 rows 69 us and over 8 d
// 40 us (one value per lane: 521 us together), reduction of 18 rows 94 us, of 8 d 49 us, plain sum 13 us (two, two
// and one of them: 602 us before).
template <typename F>
__device__ __forceinline__ void for_staged(const e2v2_segments& S, const SegRow& R, bool with_col, int* se, int* sc,
                                           F&& f) {
  for (int p0 = R.p0; p0 < R.p1; p0 += kSegStage) {
    const SegRow C{p0, min(R.p1, p0 + kSegStage)};
    __syncthreads();                     // the previous chunk has been read
    stage_row(S, C, with_col, se, sc);
    f(C.p1 - C.p0);
  }
}

struct SegOp {
  const float* p;
  int64_t r, h, d;                       // strides of the row, the head and d
};

__device__ __forceinline__ float4 ld4(const float* p) { return *reinterpret_cast<const float4*>(p); }
__device__ __forceinline__ float4 fma4(float4 a, float4 b, float4 c) {
  return make_float4(fmaf(a.x, b.x, c.x), fmaf(a.y, b.y, c.y), fmaf(a.z, b.z, c.z), fmaf(a.w, b.w, c.w));
}
__device__ __forceinline__ float4 zero4() { return make_float4(0.f, 0.f, 0.f, 0.f); }

// out[e, h] = sum_d A[r, h, d] B[c, h, d], h-fast operands: H / 4 lanes per slot, D <= kND (a missing d repeats
// the last row of B against a zero of A's).
template <int kND>
__global__ __launch_bounds__(kSegThreads) void k_seg_dot_h(e2v2_segments S, SegOp A, SegOp B, int H, int D,
                                                           float* __restrict__ out, int64_t so_e) {
  __shared__ int se[kSegStage], sc[kSegStage];
  const int r = xcd_row(blockIdx.x, S.n_rows);
  if (r >= S.n_rows) return;
  const SegRow R = seg_row(S, r);
  const int hq = H / 4, ng = kSegThreads / hq, q = (int)threadIdx.x % hq, g = (int)threadIdx.x / hq;
  float4 a[kND];
#pragma unroll
  for (int j = 0; j < kND; ++j) a[j] = j < D && g < ng ? ld4(A.p + (int64_t)r * A.r + 4 * q + j * A.d) : zero4();
  for_staged(S, R, true, se, sc, [&](int np) {
    if (g >= ng) return;
    for (int k = g; k < np; k += ng) {
      const int e = se[k];
      if (e < 0) continue;
      const float* b = B.p + (int64_t)sc[k] * B.r + 4 * q;
      float4 y[kND];
#pragma unroll
      for (int j = 0; j < kND; ++j) y[j] = ld4(b + min(j, D - 1) * B.d);
      float4 s = zero4();
#pragma unroll
      for (int j = 0; j < kND; ++j)
        if (j < D) s = fma4(a[j], y[j], s);
      *reinterpret_cast<float4*>(out + (int64_t)e * so_e + 4 * q) = s;
    }
  });
}

// d-fast operands, D = 4 kDQ: a lane per (slot, head), the A row of its head in registers.
template <int kDQ>
__global__ __launch_bounds__(kSegThreads) void k_seg_dot_d(e2v2_segments S, SegOp A, SegOp B, int H,
                                                           float* __restrict__ out, int64_t so_e, int64_t so_h) {
  __shared__ int se[kSegStage], sc[kSegStage];
  const int r = xcd_row(blockIdx.x, S.n_rows);
  if (r >= S.n_rows) return;
  const SegRow R = seg_row(S, r);
  const int ng = kSegThreads / H, h = (int)threadIdx.x % H, g = (int)threadIdx.x / H;
  float4 a[kDQ];
#pragma unroll
  for (int j = 0; j < kDQ; ++j) a[j] = ld4(A.p + (int64_t)r * A.r + (int64_t)h * A.h + 4 * j);
  for_staged(S, R, true, se, sc, [&](int np) {
    if (g >= ng) return;
    constexpr int kU = 4;                // slots in flight
    for (int k = g; k < np; k += kU * ng) {
      float4 y[kU][kDQ];
      int e[kU];
#pragma unroll
      for (int u = 0; u < kU; ++u) {
        const int ku = min(k + u * ng, np - 1);
        e[u] = k + u * ng < np ? se[ku] : -1;
        const float* b = B.p + (int64_t)sc[ku] * B.r + (int64_t)h * B.h;
#pragma unroll
        for (int j = 0; j < kDQ; ++j) y[u][j] = ld4(b + 4 * j);
      }
#pragma unroll
      for (int u = 0; u < kU; ++u) {
        float s = 0.f;
#pragma unroll
        for (int j = 0; j < kDQ; ++j) {
          s = fmaf(a[j].x, y[u][j].x, s);
          s = fmaf(a[j].y, y[u][j].y, s);
          s = fmaf(a[j].z, y[u][j].z, s);
          s = fmaf(a[j].w, y[u][j].w, s);
        }
        if (e[u] >= 0) out[(int64_t)e[u] * so_e + (int64_t)h * so_h] = s;
      }
    }
  });
}

// out[r, h, d] = sum over the row's slots of W[e, h] X[c, h, d] (kForm 0: h-fast, 1: d-fast; 2: no X, the plain
// sum of W).  A row's sums are held as quads of four values (n_quad of them: of heads, or of d); lane (gs, gd, q)
// owns quad q of the h-fast rows d = gd, gd + Gd, ... (at most kND) and the slots gs, gs + Gs, ...: what the row
// has no quads for is spent on the slots, whose Gs partial sums are added in LDS in order.
template <int kND, int kForm>
__global__ __launch_bounds__(kSegThreads) void k_seg_reduce_v(e2v2_segments S, const float* __restrict__ W,
                                                              int64_t sw_e, SegOp X, int H, int D, int n_quad, int Gd,
                                                              int Gs, float* __restrict__ out, int64_t so_r,
                                                              int64_t so_h, int64_t so_d) {
  __shared__ int se[kSegStage], sc[kSegStage];
  __shared__ float4 red[kSegThreads];
  const int r = xcd_row(blockIdx.x, S.n_rows);
  if (r >= S.n_rows) return;
  const SegRow R = seg_row(S, r);
  const int t = threadIdx.x, q = t % n_quad, g = t / n_quad, gd = g % Gd, gs = g / Gd;
  const int quad = q + (int)blockIdx.y * n_quad;       // (d-fast rows of more than 256 quads: one part per y)
  const bool on = gs < Gs && (kForm != 1 || quad < H * D / 4);
  const int h = kForm == 1 ? quad / (D / 4) : 4 * quad, d4 = kForm == 1 ? 4 * (quad % (D / 4)) : 0;
  const int nd = kForm == 0 ? (D - gd + Gd - 1) / Gd : 1;
  const float* wh = W + h;
  const float* xh = kForm == 2 ? nullptr : kForm == 1 ? X.p + (int64_t)h * X.h + d4 : X.p + h + (int64_t)gd * X.d;
  const int64_t xs = (int64_t)Gd * X.d;
  float4 acc[kND];
#pragma unroll
  for (int j = 0; j < kND; ++j) acc[j] = zero4();
  for_staged(S, R, kForm != 2, se, sc, [&](int np) {
    if (!on) return;
    constexpr int kU = kND <= 2 ? 8 : kND <= 4 ? 4 : 2;  // slots in flight
    for (int k = gs; k < np; k += kU * Gs) {
      float4 w[kU], x[kU][kND];
#pragma unroll
      for (int u = 0; u < kU; ++u) {
        const int ku = min(k + u * Gs, np - 1), e = se[ku];
        const bool ok = k + u * Gs < np && e >= 0;
        const int64_t wo = (int64_t)max(e, 0) * sw_e;
        if constexpr (kForm == 1) {
          const float v = wh[wo];
          w[u] = ok ? make_float4(v, v, v, v) : zero4();
        } else {
          const float4 v = ld4(wh + wo);
          w[u] = ok ? v : zero4();
        }
        if constexpr (kForm != 2) {
          const float* xr = xh + (int64_t)sc[ku] * X.r;
#pragma unroll
          for (int j = 0; j < kND; ++j) {
            const float4 v = ld4(xr + (kForm == 0 ? min(j, nd - 1) * xs : 0));
            x[u][j] = ok ? v : zero4();     // (a skipped slot adds nothing, whatever its partner row holds)
          }
        }
      }
#pragma unroll
      for (int u = 0; u < kU; ++u)
#pragma unroll
        for (int j = 0; j < kND; ++j) {
          if constexpr (kForm == 2)
            acc[j] = make_float4(acc[j].x + w[u].x, acc[j].y + w[u].y, acc[j].z + w[u].z, acc[j].w + w[u].w);
          else
            acc[j] = fma4(w[u], x[u][j], acc[j]);
        }
    }
  });
  auto put = [&](int j, float4 v) {
    float* o = out + (int64_t)r * so_r + (int64_t)h * so_h + (int64_t)(kForm == 1 ? d4 : gd + j * Gd) * so_d;
    const int64_t st = kForm == 1 ? so_d : so_h;
    o[0] = v.x;
    o[st] = v.y;
    o[2 * st] = v.z;
    o[3 * st] = v.w;
  };
  if (Gs == 1) {
#pragma unroll
    for (int j = 0; j < kND; ++j)
      if (on && j < nd) put(j, acc[j]);
    return;
  }
  // (Gs > 1 only with one d per lane)
  red[t] = acc[0];
  __syncthreads();
  if (gs == 0 && on) {
    float4 v = acc[0];
    for (int u = 1; u < Gs; ++u) {
      const float4 x = red[t + u * Gd * n_quad];
      v = make_float4(v.x + x.x, v.y + x.y, v.z + x.z, v.w + x.w);
    }
    put(0, v);
  }
}

// Degree outer product, out[r, l, h] = sum over the row's slots of sh[e, l] fea[e, h] for L <= kL: lane (gs, q)
// owns channels 4 q .. +3 of all L rows for the slots gs, gs + Gs, ... (fea is read once, four slots in flight);
// the Gs partial sums are added in LDS in order.  1,500 rows of 85 edges, L 5, H 256: 309 -> 29 us (before: one pass
// over fea per l).
template <int kL>
__global__ __launch_bounds__(kSegThreads) void k_outer_reduce_v(e2v2_segments S, const float* __restrict__ sh,
                                                                const float* __restrict__ fea, int L, int H, int Gs,
                                                                float* __restrict__ out) {
  __shared__ int se[kSegStage], sc[kSegStage];
  __shared__ float4 red[kSegThreads];
  const int r = xcd_row(blockIdx.x, S.n_rows);
  if (r >= S.n_rows) return;
  const SegRow R = seg_row(S, r);
  const int t = threadIdx.x, hq = H / 4, q = t % hq, gs = t / hq;
  const bool on = gs < Gs;
  float4 acc[kL];
#pragma unroll
  for (int l = 0; l < kL; ++l) acc[l] = zero4();
  for_staged(S, R, false, se, sc, [&](int np) {
    if (!on) return;
    constexpr int kU = 4;
    for (int k = gs; k < np; k += kU * Gs) {
      float4 f[kU];
      float y[kU][kL];
#pragma unroll
      for (int u = 0; u < kU; ++u) {
        const int ku = min(k + u * Gs, np - 1), e = se[ku];
        const bool ok = k + u * Gs < np && e >= 0;
        const int64_t eo = max(e, 0);
        const float4 v = ld4(fea + eo * H + 4 * q);
        f[u] = ok ? v : zero4();
#pragma unroll
        for (int l = 0; l < kL; ++l) {
          const float z = sh[eo * L + min(l, L - 1)];
          y[u][l] = ok ? z : 0.f;
        }
      }
#pragma unroll
      for (int u = 0; u < kU; ++u)
#pragma unroll
        for (int l = 0; l < kL; ++l) {
          const float z = y[u][l];
          acc[l] = fma4(make_float4(z, z, z, z), f[u], acc[l]);
        }
    }
  });
#pragma unroll
  for (int l = 0; l < kL; ++l) {
    if (l >= L) break;
    float4 v = acc[l];
    if (Gs > 1) {
      __syncthreads();
      red[t] = v;
      __syncthreads();
      if (gs == 0)
        for (int u = 1; u < Gs; ++u) {
          const float4 x = red[t + u * hq];
          v = make_float4(v.x + x.x, v.y + x.y, v.z + x.z, v.w + x.w);
        }
    }
    if (gs == 0 && on) *reinterpret_cast<float4*>(out + ((int64_t)r * L + l) * H + 4 * q) = v;
  }
}

// Its gradient in one pass: dsh[e, l] = <g[q_e, l], fea[e]>, dfea[e] = sum_l sh[e, l] g[q_e, l].  kLanes lanes per
// edge (H / 4 of them hold channels), a run of kOuterRun consecutive edges per lane group, whose L gradient rows
// stay in registers while the query row does (edges of a row are consecutive in sorted lists); fea is read and
// dfea written once.  Either result may be left out.  1,500 rows of 85 edges, L 5, H 256: 203 (two kernels) -> 55 us,
// the time a copy of fea takes.
constexpr int kOuterRun = 8;
template <int kL, int kLanes>
__global__ __launch_bounds__(kSegThreads) void k_outer_bwd_v(const float* __restrict__ g, int n_rows,
                                                             const float* __restrict__ sh,
                                                             const float* __restrict__ fea,
                                                             const int32_t* __restrict__ qidx, int64_t n_edges, int L,
                                                             int H, float* __restrict__ dsh,
                                                             float* __restrict__ dfea) {
  const int64_t run = (int64_t)blockIdx.x * (kSegThreads / kLanes) + threadIdx.x / kLanes;
  const int lane = threadIdx.x % kLanes, c = 4 * lane;
  const bool in = c < H;
  const int64_t e0 = run * kOuterRun, e1 = min(n_edges, e0 + kOuterRun);
  float4 gr[kL];
  int have = -1;                          // the query row held in gr (-1: none, zero)
#pragma unroll
  for (int l = 0; l < kL; ++l) gr[l] = zero4();
  constexpr int kU = 2;
  for (int64_t e = e0; e < e1; e += kU) {
    float4 f[kU];
    float y[kU][kL];
    int qr[kU];
#pragma unroll
    for (int u = 0; u < kU; ++u) {
      const int64_t eu = min(e + u, e1 - 1);
      const int q = qidx[eu];
      qr[u] = q >= 0 && q < n_rows ? q : -1;
      f[u] = dsh && in ? ld4(fea + eu * H + c) : zero4();
#pragma unroll
      for (int l = 0; l < kL; ++l) y[u][l] = dfea ? sh[eu * L + min(l, L - 1)] : 0.f;
    }
#pragma unroll
    for (int u = 0; u < kU; ++u) {
      if (e + u >= e1) break;
      if (qr[u] != have) {
        have = qr[u];
#pragma unroll
        for (int l = 0; l < kL; ++l)
          gr[l] = have >= 0 && in ? ld4(g + ((int64_t)have * L + min(l, L - 1)) * H + c) : zero4();
      }
      if (dfea && in) {
        float4 v = zero4();
        if (have >= 0) {
#pragma unroll
          for (int l = 0; l < kL; ++l) {
            const float z = y[u][l];
            if (l < L) v = fma4(make_float4(z, z, z, z), gr[l], v);
          }
        }
        *reinterpret_cast<float4*>(dfea + (e + u) * H + c) = v;
      }
      if (dsh) {
#pragma unroll
        for (int l = 0; l < kL; ++l) {
          if (l >= L) break;
          float v = gr[l].x * f[u].x;
          v = fmaf(gr[l].y, f[u].y, v);
          v = fmaf(gr[l].z, f[u].z, v);
          v = fmaf(gr[l].w, f[u].w, v);
          if (have < 0) v = 0.f;
          if constexpr (kLanes >= 16) {
            v = dpp_row_sum16(v);
#pragma unroll
            for (int o = 16; o < kLanes; o <<= 1) v += __shfl_xor(v, o, kWave);
          } else {
#pragma unroll
            for (int o = 1; o < kLanes; o <<= 1) v += __shfl_xor(v, o, kWave);
          }
          if (lane == 0) dsh[(e + u) * L + l] = v;
        }
      }
    }
  }
}

static inline unsigned blocks_of(int64_t n, int per) { return (unsigned)((n + per - 1) / per); }

static inline bool aligned16(const void* p) { return ((uintptr_t)p & 15) == 0; }
// 16-byte groups of four heads (h-fast) or of four d (d-fast) in every row of the operand
static bool quads_h(const SegOp& x, int H, int D) {
  return x.h == 1 && H % 4 == 0 && x.r % 4 == 0 && (x.d % 4 == 0 || D == 1) && aligned16(x.p);
}
static bool quads_d(const SegOp& x, int D) {
  return x.d == 1 && D % 4 == 0 && x.r % 4 == 0 && x.h % 4 == 0 && aligned16(x.p);
}

static int check_segments(const e2v2_segments* S, bool need_col, const char* what) {
  E2V2_REQUIRE(S != nullptr, "%s: null segment layout", what);
  E2V2_REQUIRE(S->n_rows >= 0 && S->n_slots >= 0 && S->n_edges >= 0 && S->n_cols >= 0,
               "%s: negative size (rows %d, cols %d, slots %lld, edges %lld)", what, S->n_rows, S->n_cols,
               (long long)S->n_slots, (long long)S->n_edges);
  E2V2_REQUIRE(S->n_slots < (1ll << 31), "%s: %lld slots exceed the 32-bit slot index", what,
               (long long)S->n_slots);
  E2V2_REQUIRE(S->n_rows == 0 || S->row_ptr, "%s: null row_ptr", what);
  E2V2_REQUIRE(S->n_slots == 0 || (S->alpha_index && (!need_col || S->col_index)),
               "%s: null col_index / alpha_index", what);
  return 0;
}

// Per-edge contraction of a query node's irreps with the edge's spherical
// harmonics, l by l: x0[e][l][c] = sum_{m in l} Y[e][m] xn[m][row(e)][c] (the
// x_0_extra of the QKdot_alpha / QKdotS_alpha gates, e2former.py:271-277 and
// 288-296), for lmax = 2 (9 m-rows, 3 l-blocks) and C <= 256 channels.  One
// wavefront per query row (edges of a row contiguous, CSR row_ptr), lanes over
// channels (up to four each), the row's node values held in registers.  The
// backward of the same row forms dxn[m][i][c] = sum_e Y[e][m] g[e][l(m)][c]
// in registers (no atomics) and dY[e][m] = sum_c g[e][l(m)][c] xn[m][i][c] by a
// fixed-order butterfly over the lanes.
constexpr int kShWaves = 4, kShPer = 4;

__device__ __forceinline__ int sh_l(int m) { return m == 0 ? 0 : (m < 4 ? 1 : 2); }

__global__ __launch_bounds__(64 * kShWaves) void k_sh_contract(const float* __restrict__ Y,
                                                               const float* __restrict__ xn,
                                                               const int32_t* __restrict__ row_ptr, int32_t n_rows,
                                                               int32_t C, float* __restrict__ x0) {
  const int i = blockIdx.x * kShWaves + (threadIdx.x >> 6);
  if (i >= n_rows) return;
  const int lane = threadIdx.x & 63;
  const size_t ms = (size_t)n_rows * C;
  float xr[kShPer][9];
#pragma unroll
  for (int q = 0; q < kShPer; ++q) {
    const int c = lane + 64 * q;
#pragma unroll
    for (int m = 0; m < 9; ++m) xr[q][m] = c < C ? xn[m * ms + (size_t)i * C + c] : 0.f;
  }
  const int b = row_ptr[i], n = row_ptr[i + 1] - b;
  for (int k = 0; k < n; ++k) {
    const int64_t e = (int64_t)b + k;
    float y[9];
#pragma unroll
    for (int m = 0; m < 9; ++m) y[m] = Y[e * 9 + m];
#pragma unroll
    for (int q = 0; q < kShPer; ++q) {
      const int c = lane + 64 * q;
      if (c < C) {
        float* o = x0 + (size_t)e * 3 * C + c;
        o[0] = y[0] * xr[q][0];
        o[C] = fmaf(y[3], xr[q][3], fmaf(y[2], xr[q][2], y[1] * xr[q][1]));
        o[2 * C] = fmaf(y[8], xr[q][8], fmaf(y[7], xr[q][7], fmaf(y[6], xr[q][6], fmaf(y[5], xr[q][5],
                   y[4] * xr[q][4]))));
      }
    }
  }
}

__global__ __launch_bounds__(64 * kShWaves) void k_sh_contract_bwd(const float* __restrict__ Y,
                                                                   const float* __restrict__ xn,
                                                                   const int32_t* __restrict__ row_ptr,
                                                                   int32_t n_rows, int32_t C,
                                                                   const float* __restrict__ g,
                                                                   float* __restrict__ dY, float* __restrict__ dxn) {
  const int i = blockIdx.x * kShWaves + (threadIdx.x >> 6);
  if (i >= n_rows) return;
  const int lane = threadIdx.x & 63;
  const size_t ms = (size_t)n_rows * C;
  float xr[kShPer][9], dx[kShPer][9];
#pragma unroll
  for (int q = 0; q < kShPer; ++q) {
    const int c = lane + 64 * q;
#pragma unroll
    for (int m = 0; m < 9; ++m) {
      xr[q][m] = c < C ? xn[m * ms + (size_t)i * C + c] : 0.f;
      dx[q][m] = 0.f;
    }
  }
  const int b = row_ptr[i], n = row_ptr[i + 1] - b;
  for (int k = 0; k < n; ++k) {
    const int64_t e = (int64_t)b + k;
    float y[9], p[9];
#pragma unroll
    for (int m = 0; m < 9; ++m) {
      y[m] = Y[e * 9 + m];
      p[m] = 0.f;
    }
#pragma unroll
    for (int q = 0; q < kShPer; ++q) {
      const int c = lane + 64 * q;
      const float* gp = g + (size_t)e * 3 * C + c;
      const float gl[3] = {c < C ? gp[0] : 0.f, c < C ? gp[C] : 0.f, c < C ? gp[2 * C] : 0.f};
#pragma unroll
      for (int m = 0; m < 9; ++m) {
        dx[q][m] = fmaf(y[m], gl[sh_l(m)], dx[q][m]);
        p[m] = fmaf(gl[sh_l(m)], xr[q][m], p[m]);
      }
    }
#pragma unroll
    for (int m = 0; m < 9; ++m) {
#pragma unroll
      for (int o = 32; o >= 1; o >>= 1) p[m] += __shfl_xor(p[m], o, kWave);
    }
    if (lane < 9) {
      float v = p[0];
#pragma unroll
      for (int m = 1; m < 9; ++m) v = lane == m ? p[m] : v;
      dY[e * 9 + lane] = v;
    }
  }
#pragma unroll
  for (int q = 0; q < kShPer; ++q) {
    const int c = lane + 64 * q;
    if (c < C) {
#pragma unroll
      for (int m = 0; m < 9; ++m) dxn[m * ms + (size_t)i * C + c] = dx[q][m];
    }
  }
}

}  // namespace e2v2

using namespace e2v2;

E2V2_API int e2v2_seg_dot(const e2v2_segments* S, const float* A, const int64_t* a_strides, const float* B,
                          const int64_t* b_strides, int H, int D, float* out, const int64_t* out_strides,
                          hipStream_t s) {
  if (int rc = check_segments(S, true, "seg_dot")) return rc;
  E2V2_REQUIRE(H >= 1 && D >= 1 && a_strides && b_strides && out_strides, "seg_dot: bad sizes (H %d, D %d)", H, D);
  if (S->n_rows == 0 || S->n_slots == 0) return 0;
  E2V2_REQUIRE(A && B && out, "seg_dot: null operand");
  E2V2_REQUIRE((int64_t)S->n_slots * H < (1ll << 32), "seg_dot: rows of up to 2^32 / H slots");
  // the vector forms where the operands allow them (both at 16-byte granularity), else one value per lane
  const SegOp a{A, a_strides[0], a_strides[1], a_strides[2]}, b{B, b_strides[0], b_strides[1], b_strides[2]};
  const dim3 grid(xcd_grid(S->n_rows)), blk(kSegThreads);
  const bool some = S->n_cols > 0 && S->n_edges > 0;     // (a skipped slot reads row 0 and edge 0)
  if (some && quads_h(a, H, D) && quads_h(b, H, D) && D <= 24 && H <= 4 * kSegThreads && out_strides[1] == 1 &&
      out_strides[0] % 4 == 0 && aligned16(out)) {
    auto go = [&](auto nd) {
      hipLaunchKernelGGL((k_seg_dot_h<decltype(nd)::value>), grid, blk, 0, s, *S, a, b, H, D, out, out_strides[0]);
    };
    if (D <= 4) go(std::integral_constant<int, 4>{});
    else if (D <= 9) go(std::integral_constant<int, 9>{});
    else if (D <= 18) go(std::integral_constant<int, 18>{});
    else go(std::integral_constant<int, 24>{});
    E2V2_LAUNCHED("k_seg_dot_h");
    return 0;
  }
  if (some && quads_d(a, D) && quads_d(b, D) && H <= kSegThreads && (D == 4 || D == 8 || D == 16 || D == 32)) {
    auto go = [&](auto dq) {
      hipLaunchKernelGGL((k_seg_dot_d<decltype(dq)::value>), grid, blk, 0, s, *S, a, b, H, out, out_strides[0],
                         out_strides[1]);
    };
    if (D == 4) go(std::integral_constant<int, 1>{});
    else if (D == 8) go(std::integral_constant<int, 2>{});
    else if (D == 16) go(std::integral_constant<int, 4>{});
    else go(std::integral_constant<int, 8>{});
    E2V2_LAUNCHED("k_seg_dot_d");
    return 0;
  }
  hipLaunchKernelGGL(k_seg_dot, dim3(S->n_rows), dim3(kSegThreads), 0, s, *S, A, a_strides[0], a_strides[1],
                     a_strides[2], B, b_strides[0], b_strides[1], b_strides[2], H, D, out, out_strides[0],
                     out_strides[1]);
  E2V2_LAUNCHED("k_seg_dot");
  return 0;
}

E2V2_API int e2v2_seg_reduce(const e2v2_segments* S, const float* W, const int64_t* w_strides, const float* X,
                             const int64_t* x_strides, int H, int D, float* out, const int64_t* out_strides,
                             hipStream_t s) {
  if (int rc = check_segments(S, X != nullptr, "seg_reduce")) return rc;
  E2V2_REQUIRE(H >= 1 && D >= 1 && (int64_t)H * D < (1ll << 31) && w_strides && out_strides &&
                   (X == nullptr || x_strides),
               "seg_reduce: bad sizes (H %d, D %d)", H, D);
  E2V2_REQUIRE(X != nullptr || D == 1, "seg_reduce: a plain sum (X NULL) has D = 1");
  if (S->n_rows == 0) return 0;
  E2V2_REQUIRE(W && out, "seg_reduce: null operand");
  const SegOp x{X, X ? x_strides[0] : 0, X ? x_strides[1] : 0, X ? x_strides[2] : 0};
  const bool w4 = w_strides[1] == 1 && w_strides[0] % 4 == 0 && aligned16(W) && H % 4 == 0;
  const bool w1 = w_strides[1] == 1, some = S->n_edges > 0 && (X == nullptr || S->n_cols > 0);
  if (some && H <= 4 * kSegThreads && w4 && (X == nullptr || quads_h(x, H, D))) {
    const int nq = H / 4, ng = kSegThreads / nq, gd = X ? std::min(D, ng) : 1, gs = ng / gd, nd = (D + gd - 1) / gd;
    auto go = [&](auto k, auto form) {
      hipLaunchKernelGGL((k_seg_reduce_v<decltype(k)::value, decltype(form)::value>), dim3(xcd_grid(S->n_rows)),
                         dim3(kSegThreads), 0, s, *S, W, w_strides[0], x, H, D, nq, gd, nd == 1 ? gs : 1, out,
                         out_strides[0], out_strides[1], out_strides[2]);
    };
    using F0 = std::integral_constant<int, 0>;
    if (nd <= 12) {
      if (!X) go(std::integral_constant<int, 1>{}, std::integral_constant<int, 2>{});
      else if (nd == 1) go(std::integral_constant<int, 1>{}, F0{});
      else if (nd <= 3) go(std::integral_constant<int, 3>{}, F0{});
      else if (nd <= 6) go(std::integral_constant<int, 6>{}, F0{});
      else go(std::integral_constant<int, 12>{}, F0{});
      E2V2_LAUNCHED("k_seg_reduce_v");
      return 0;
    }
  }
  if (some && X && w1 && quads_d(x, D) && (int64_t)H * D / 4 <= 65535 * (int64_t)kSegThreads) {
    const int quads = H * D / 4, nq = std::min(quads, kSegThreads), gs = kSegThreads / nq;
    hipLaunchKernelGGL((k_seg_reduce_v<1, 1>), dim3(xcd_grid(S->n_rows), (quads + nq - 1) / nq), dim3(kSegThreads), 0,
                       s, *S, W, w_strides[0], x, H, D, nq, 1, gs, out, out_strides[0], out_strides[1],
                       out_strides[2]);
    E2V2_LAUNCHED("k_seg_reduce_v");
    return 0;
  }
  const int64_t z = 0;
  const bool h_fast = X ? (x_strides[1] <= x_strides[2]) : true;
  hipLaunchKernelGGL(k_seg_reduce, dim3(S->n_rows), dim3(kSegThreads), 0, s, *S, W, w_strides[0], w_strides[1], X,
                     X ? x_strides[0] : z, X ? x_strides[1] : z, X ? x_strides[2] : z, H, D, h_fast, out,
                     out_strides[0], out_strides[1], out_strides[2]);
  E2V2_LAUNCHED("k_seg_reduce");
  return 0;
}

E2V2_API int e2v2_gather_rows(const float* in, int64_t n_in, const int32_t* index, int64_t n, int K, float* out,
                              hipStream_t s) {
  E2V2_REQUIRE(n >= 0 && n_in >= 0 && K >= 1, "gather_rows: bad sizes (n %lld, K %d)", (long long)n, K);
  if (n == 0) return 0;
  E2V2_REQUIRE(in && index && out, "gather_rows: null pointer");
  if (K % 4 == 0 && K <= 4 * kSegThreads && aligned16(in) && aligned16(out)) {
    hipLaunchKernelGGL(k_gather_rows_v, dim3(blocks_of(n, kSegThreads / (K / 4) * kGatherU)), dim3(kSegThreads), 0, s, in,
                       n_in, index, n, K, out);
    E2V2_LAUNCHED("k_gather_rows_v");
    return 0;
  }
  hipLaunchKernelGGL(k_gather_rows, dim3(blocks_of(n * K, 256)), dim3(256), 0, s, in, n_in, index, n, K, out);
  E2V2_LAUNCHED("k_gather_rows");
  return 0;
}

E2V2_API int e2v2_outer_reduce(const e2v2_segments* S, const float* sh, const float* fea, int L, int H, float* out,
                               hipStream_t s) {
  if (int rc = check_segments(S, false, "outer_reduce")) return rc;
  E2V2_REQUIRE(L >= 1 && H >= 1 && (int64_t)L * H < (1ll << 31), "outer_reduce: bad sizes (L %d, H %d)", L, H);
  if (S->n_rows == 0) return 0;
  E2V2_REQUIRE(sh && fea && out, "outer_reduce: null operand");
  if (S->n_edges > 0 && L <= kOuterL && H % 4 == 0 && H <= 4 * kSegThreads && aligned16(fea) && aligned16(out)) {
    const int gs = kSegThreads / (H / 4);
    const auto go = [&](auto l) {
      hipLaunchKernelGGL((k_outer_reduce_v<decltype(l)::value>), dim3(xcd_grid(S->n_rows)), dim3(kSegThreads), 0, s, *S,
                         sh, fea, L, H, gs, out);
    };
    if (L == 1) go(std::integral_constant<int, 1>{});
    else if (L <= 3) go(std::integral_constant<int, 3>{});
    else if (L <= 5) go(std::integral_constant<int, 5>{});
    else go(std::integral_constant<int, 9>{});
    E2V2_LAUNCHED("k_outer_reduce_v");
    return 0;
  }
  hipLaunchKernelGGL(k_outer_reduce, dim3(S->n_rows), dim3(kSegThreads), 0, s, *S, sh, fea, L, H, out);
  E2V2_LAUNCHED("k_outer_reduce");
  return 0;
}

E2V2_API int e2v2_outer_bwd(const float* grad, int n_rows, const float* sh, const float* fea,
                            const int32_t* query_index, int64_t n_edges, int L, int H, float* dsh, float* dfea,
                            hipStream_t s) {
  E2V2_REQUIRE(n_rows >= 0 && n_edges >= 0 && L >= 1 && H >= 1, "outer_bwd: bad sizes (E %lld, L %d, H %d)",
               (long long)n_edges, L, H);
  if (n_edges == 0) return 0;
  E2V2_REQUIRE(grad && query_index && (dsh == nullptr || fea) && (dfea == nullptr || sh),
               "outer_bwd: null operand");
  if (!dsh && !dfea) return 0;
  if (H <= 256 && H % 4 == 0 && L <= kOuterL && aligned16(grad) && (!dsh || aligned16(fea)) &&
      (!dfea || aligned16(dfea))) {
    const auto lanes = [&](auto l, auto n) {
      constexpr int kLanes = decltype(n)::value;
      const unsigned grid = blocks_of(blocks_of(n_edges, kOuterRun), kSegThreads / kLanes);
      hipLaunchKernelGGL((k_outer_bwd_v<decltype(l)::value, kLanes>), dim3(grid), dim3(kSegThreads), 0, s, grad, n_rows,
                         sh, fea, query_index, n_edges, L, H, dsh, dfea);
    };
    const auto go = [&](auto l) {
      if (H <= 32) lanes(l, std::integral_constant<int, 8>{});
      else if (H <= 64) lanes(l, std::integral_constant<int, 16>{});
      else if (H <= 128) lanes(l, std::integral_constant<int, 32>{});
      else lanes(l, std::integral_constant<int, 64>{});
    };
    if (L == 1) go(std::integral_constant<int, 1>{});
    else if (L <= 3) go(std::integral_constant<int, 3>{});
    else if (L <= 5) go(std::integral_constant<int, 5>{});
    else go(std::integral_constant<int, 9>{});
    E2V2_LAUNCHED("k_outer_bwd_v");
    return 0;
  }
  if (dsh) {
    hipLaunchKernelGGL(k_outer_dsh, dim3(blocks_of(n_edges * L, 256)), dim3(256), 0, s, grad, n_rows, fea, query_index,
                       n_edges, L, H, dsh);
    E2V2_LAUNCHED("k_outer_dsh");
  }
  if (dfea) {
    hipLaunchKernelGGL(k_outer_dfea, dim3(blocks_of(n_edges * H, 256)), dim3(256), 0, s, grad, n_rows, sh,
                       query_index, n_edges, L, H, dfea);
    E2V2_LAUNCHED("k_outer_dfea");
  }
  return 0;
}

// Raw real spherical-harmonic polynomials l <= 2 of each vector v [n][3] (y the polar axis), or with `unit` those of
// v / |v| times sqrt(2 l + 1) / sqrt(4 pi), and the vectors' gradient.  As tensor operations these were some ninety
// launches of 3 us per evaluation (each a pass over [n] columns of [n][9]); a vector per thread is two launches.
constexpr float kS3 = 1.7320508075688772f;
__device__ __constant__ const float kShInt[3] = {0.28209479177387814f, 0.4886025119029199f, 0.6307831305050401f};

__global__ __launch_bounds__(256) void k_edge_sh(const float* __restrict__ v, int64_t n, int unit, float* __restrict__ Y) {
  const int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (e >= n) return;
  float x = v[3 * e], y = v[3 * e + 1], z = v[3 * e + 2];
  float c0 = 1.f, c1 = 1.f, c2 = 1.f;
  if (unit) {
    const float d = sqrtf(x * x + y * y + z * z);
    x /= d; y /= d; z /= d;
    c0 = kShInt[0]; c1 = kShInt[1]; c2 = kShInt[2];
  }
  float* o = Y + 9 * e;
  o[0] = c0;
  o[1] = c1 * x;
  o[2] = c1 * y;
  o[3] = c1 * z;
  o[4] = c2 * (kS3 * x * z);
  o[5] = c2 * (kS3 * x * y);
  o[6] = c2 * (y * y - 0.5f * (x * x + z * z));
  o[7] = c2 * (kS3 * y * z);
  o[8] = c2 * (0.5f * kS3 * (z * z - x * x));
}

__global__ __launch_bounds__(256) void k_edge_sh_bwd(const float* __restrict__ v, const float* __restrict__ g, int64_t n,
                                                     int unit, float* __restrict__ gv) {
  const int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (e >= n) return;
  float x = v[3 * e], y = v[3 * e + 1], z = v[3 * e + 2], d = 1.f, c1 = 1.f, c2 = 1.f;
  if (unit) {
    d = sqrtf(x * x + y * y + z * z);
    x /= d; y /= d; z /= d;
    c1 = kShInt[1]; c2 = kShInt[2];
  }
  const float* G = g + 9 * e;
  const float g4 = c2 * G[4], g5 = c2 * G[5], g6 = c2 * G[6], g7 = c2 * G[7], g8 = c2 * G[8];
  float a = c1 * G[1] + kS3 * (z * g4 + y * g5) - x * g6 - kS3 * x * g8;
  float b = c1 * G[2] + kS3 * (x * g5 + z * g7) + 2.f * y * g6;
  float c = c1 * G[3] + kS3 * (x * g4 + y * g7) - z * g6 + kS3 * z * g8;
  if (unit) {
    const float r = a * x + b * y + c * z;
    a = (a - r * x) / d;
    b = (b - r * y) / d;
    c = (c - r * z) / d;
  }
  gv[3 * e] = a;
  gv[3 * e + 1] = b;
  gv[3 * e + 2] = c;
}

E2V2_API int e2v2_edge_sh(const float* v, int64_t n, int unit, float* Y, hipStream_t s) {
  E2V2_REQUIRE(n >= 0 && n < (1LL << 38) && (n == 0 || (v && Y)), "edge_sh: n %lld, null pointer", (long long)n);
  if (n == 0) return 0;
  hipLaunchKernelGGL(k_edge_sh, dim3((uint32_t)((n + 255) / 256)), dim3(256), 0, s, v, n, unit, Y);
  E2V2_LAUNCHED("k_edge_sh");
  return 0;
}

E2V2_API int e2v2_edge_sh_bwd(const float* v, const float* g, int64_t n, int unit, float* gv, hipStream_t s) {
  E2V2_REQUIRE(n >= 0 && n < (1LL << 38) && (n == 0 || (v && g && gv)), "edge_sh_bwd: n %lld, null pointer",
               (long long)n);
  if (n == 0) return 0;
  hipLaunchKernelGGL(k_edge_sh_bwd, dim3((uint32_t)((n + 255) / 256)), dim3(256), 0, s, v, g, n, unit, gv);
  E2V2_LAUNCHED("k_edge_sh_bwd");
  return 0;
}

E2V2_API int e2v2_sh_contract(const float* Y, const float* xn, const int32_t* row_ptr, int32_t n_rows, int32_t C,
                              float* x0, hipStream_t s) {
  E2V2_REQUIRE(n_rows >= 0 && C >= 1 && C <= 64 * kShPer && (n_rows == 0 || (Y && xn && row_ptr && x0)),
               "sh_contract: bad arguments (n_rows %d, C %d; C must be 1..%d)", n_rows, C, 64 * kShPer);
  if (n_rows == 0) return 0;
  hipLaunchKernelGGL(k_sh_contract, dim3((unsigned)((n_rows + kShWaves - 1) / kShWaves)), dim3(64 * kShWaves), 0, s,
                     Y, xn, row_ptr, n_rows, C, x0);
  E2V2_LAUNCHED("k_sh_contract");
  return 0;
}

E2V2_API int e2v2_sh_contract_bwd(const float* Y, const float* xn, const int32_t* row_ptr, int32_t n_rows, int32_t C,
                                  const float* g, float* dY, float* dxn, hipStream_t s) {
  E2V2_REQUIRE(n_rows >= 0 && C >= 1 && C <= 64 * kShPer &&
                   (n_rows == 0 || (Y && xn && row_ptr && g && dY && dxn)),
               "sh_contract_bwd: bad arguments (n_rows %d, C %d; C must be 1..%d)", n_rows, C, 64 * kShPer);
  if (n_rows == 0) return 0;
  hipLaunchKernelGGL(k_sh_contract_bwd, dim3((unsigned)((n_rows + kShWaves - 1) / kShWaves)), dim3(64 * kShWaves), 0,
                     s, Y, xn, row_ptr, n_rows, C, g, dY, dxn);
  E2V2_LAUNCHED("k_sh_contract_bwd");
  return 0;
}
