// Weight gradients of the training path: dW_g [m][k] = sum over the batches b of group g and the rows r of
// A[b][r][:]^T B[b][r][:] (SO3_Linear_e2former's per-degree weight: 9 m-rows of N nodes in three groups), and the
// sums of the per-block partial rows that the norms' parameter gradients leave.
//
// fp32 throughout (v_mfma_f32_32x32x2_f32).  The contraction runs over the rows, so both operands are read as they
// lie, a row's 64 columns by the 32 lanes of a half wavefront (two columns per lane: the tile's even and odd columns
// are its two 32 x 32 MFMA tiles), straight into registers with four 8-row groups in flight: no LDS, no barrier in
// the loop.  A workgroup owns a 64 x 64 tile of dW over one chunk of one batch's rows, its four wavefronts a quarter
// of them each; they meet in LDS once and the chunks' partial tiles are added in order by a second kernel.
// Bound: the fp32 MFMA rate (four MFMAs of 64 cycles per 1 KB read).  The library product per m-row and its scatter over
// the degrees took 62 us of kernels at 412 nodes and 47 us at 1500 (mean of 256 x 256 and 512 x 256), this 19 and
// 36 us.
#include <algorithm>

#include "gemm_ks.h"
#include "../../include/e2v2.h"

namespace e2v2 {
namespace {

constexpr int kWgT = 64;           // tile of dW
constexpr int kWgRing = 4;         // 8-row groups in flight
constexpr int kWgTarget = 768;     // workgroups to aim at (three per CU)

struct WgArgs {
  const float* a; int64_t lda, a_bs;
  const float* b; int64_t ldb, b_bs;
  float* out;
  int n, rows, cpb, m, k;          // rows per chunk (a multiple of 32), chunks per batch
};

__device__ __forceinline__ __amdgpu_buffer_rsrc_t cols_rsrc(const float* base, int64_t ld, int row0, int n, int col0,
                                                            int width) {
  // rows row0 .. n-1 of columns col0 ..: reads past row n - 1 return zero
  const uint32_t bytes = row0 < n ? ((uint32_t)(n - 1 - row0) * (uint32_t)ld + (uint32_t)(width - col0)) * 4u : 0u;
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(base + (int64_t)row0 * ld + col0), (short)0, (int)bytes,
                                           0x00020000);
}

typedef float wg_f2 __attribute__((ext_vector_type(2)));

__global__ __launch_bounds__(kKsThreads, 2) void k_wgrad(WgArgs P, int n_wg) {
  __shared__ float red[kKsW * 32 * 64];
  const int wg = xcd_row(blockIdx.x, n_wg);
  if (wg >= n_wg) return;
  const int t = threadIdx.x, lane = t & 63, wv = __builtin_amdgcn_readfirstlane(t >> 6), h = lane >> 5;
  const int n_j = P.k / kWgT, tiles = (P.m / kWgT) * n_j;      // the tiles of a chunk are neighbours: they share its rows
  const int tile = wg % tiles, ch = wg / tiles, bi = ch / P.cpb;
  const int i0 = (tile / n_j) * kWgT, j0 = (tile % n_j) * kWgT;
  const int per = P.rows / kKsW, row0 = (ch % P.cpb) * P.rows + wv * per;
  const int ng = row0 < P.n ? (min(per, P.n - row0) + 7) / 8 : 0;
  const __amdgpu_buffer_rsrc_t ar = cols_rsrc(P.a + (int64_t)bi * P.a_bs, P.lda, row0, P.n, i0, P.m);
  const __amdgpu_buffer_rsrc_t br = cols_rsrc(P.b + (int64_t)bi * P.b_bs, P.ldb, row0, P.n, j0, P.k);
  const uint32_t sa = (uint32_t)P.lda * 4u, sb = (uint32_t)P.ldb * 4u;
  const uint32_t ao = (uint32_t)h * sa + 8u * (lane & 31), bo = (uint32_t)h * sb + 8u * (lane & 31);
  wg_f2 ra[kWgRing][4], rb[kWgRing][4];
  floatx16 acc[2][2];
  ks_zero(acc);
  auto load = [&](int g, int sl) {
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      ra[sl][s] = __builtin_bit_cast(wg_f2, __builtin_amdgcn_raw_buffer_load_b64(ar, ao + (uint32_t)(8 * g + 2 * s) * sa, 0, 0));
      rb[sl][s] = __builtin_bit_cast(wg_f2, __builtin_amdgcn_raw_buffer_load_b64(br, bo + (uint32_t)(8 * g + 2 * s) * sb, 0, 0));
    }
  };
#pragma unroll
  for (int sl = 0; sl < kWgRing; ++sl)
    if (sl < ng) load(sl, sl);
  for (int g = 0; g < ng; g += kWgRing) {
#pragma unroll
    for (int sl = 0; sl < kWgRing; ++sl) {
      if (g + sl < ng) {
#pragma unroll
        for (int s = 0; s < 4; ++s)
#pragma unroll
          for (int ta = 0; ta < 2; ++ta)
#pragma unroll
            for (int tb = 0; tb < 2; ++tb)
              acc[ta][tb] = __builtin_amdgcn_mfma_f32_32x32x2f32(ra[sl][s][ta], rb[sl][s][tb], acc[ta][tb], 0, 0, 0);
        if (g + sl + kWgRing < ng) load(g + sl + kWgRing, sl);
      }
    }
  }
  float* o = P.out + (int64_t)ch * P.m * P.k;
#pragma unroll
  for (int ta = 0; ta < 2; ++ta) {
    float part[32], sum[8];
#pragma unroll
    for (int q = 0; q < 32; ++q) part[q] = acc[ta][q / 16][q % 16];
    if (ta) __syncthreads();
    ks_reduce<32, kKsW>(red, part, wv, lane, [](int w, int i) { return 16 * (i & 1) + 4 * w + (i >> 1); }, sum);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int row = i0 + 2 * acc_row(4 * wv + i, lane) + ta, col = j0 + 2 * (lane & 31);
      *reinterpret_cast<float2*>(o + (int64_t)row * P.k + col) = make_float2(sum[2 * i], sum[2 * i + 1]);
    }
  }
}

struct PartBounds {
  int p[E2V2_MAX_PART_GROUPS + 1];
};

// out[g][w] = the sum of the rows p[g] .. p[g + 1] - 1 of part [.][w]: kL lanes take every kL-th row, then a tree.
// kL 128 with 32 columns per workgroup for the long narrow sums of the norms (2048 rows of 128 twice:
// 4.5 us, as two torch sums 25 us), kL 4 with 256 columns for the weight tiles.
template <int kL, int kCols>
__global__ __launch_bounds__(kL * kCols / 4) void k_sum_parts(const float* __restrict__ part, PartBounds B, int w,
                                                              float* __restrict__ out) {
  constexpr int kQ = kCols / 4;
  __shared__ float4 red[kL][kQ];
  const int c = threadIdx.x % kQ, r = threadIdx.x / kQ, col = blockIdx.x * kCols + 4 * c, g = blockIdx.y;
  float4 s = make_float4(0.f, 0.f, 0.f, 0.f);
  if (col < w) {
#pragma unroll 4
    for (int p = B.p[g] + r; p < B.p[g + 1]; p += kL) {
      const float4 v = *reinterpret_cast<const float4*>(part + (int64_t)p * w + col);
      s.x += v.x; s.y += v.y; s.z += v.z; s.w += v.w;
    }
  }
  red[r][c] = s;
  __syncthreads();
#pragma unroll
  for (int d = kL / 2; d > 0; d /= 2) {
    if (r < d) {
      const float4 v = red[r + d][c];
      s.x += v.x; s.y += v.y; s.z += v.z; s.w += v.w;
      red[r][c] = s;
    }
    __syncthreads();
  }
  if (r == 0 && col < w) *reinterpret_cast<float4*>(out + (int64_t)g * w + col) = s;
}

int sum_parts(const float* part, const PartBounds& B, int groups, int w, float* out, hipStream_t s) {
  int most = 0;
  for (int g = 0; g < groups; ++g) most = std::max(most, B.p[g + 1] - B.p[g]);
  if (most > 64)
    hipLaunchKernelGGL((k_sum_parts<128, 32>), dim3((w + 31) / 32, groups), dim3(1024), 0, s, part, B, w, out);
  else
    hipLaunchKernelGGL((k_sum_parts<4, 256>), dim3((w + 255) / 256, groups), dim3(256), 0, s, part, B, w, out);
  E2V2_LAUNCHED("k_sum_parts");
  return 0;
}

}  // namespace
}  // namespace e2v2

using namespace e2v2;

// Chunks of each batch's n rows: enough workgroups to fill the chip, at least 64 rows each.
E2V2_API int e2v2_wgrad_chunks(int n, int batches, int m, int k) {
  if (n <= 0 || batches <= 0 || m < kWgT || k < kWgT) return 1;
  const int64_t wgs = (int64_t)batches * (m / kWgT) * (k / kWgT);
  return (int)std::max<int64_t>(1, std::min<int64_t>((kWgTarget + wgs / 2) / wgs, (n + 63) / 64));
}

E2V2_API int e2v2_wgrad(const float* a, int64_t lda, int64_t a_bs, const float* b, int64_t ldb, int64_t b_bs, int n,
                        int batches, int m, int k, const int32_t* bounds, int groups, float* part, float* out,
                        hipStream_t s) {
  E2V2_REQUIRE(n > 0 && batches > 0 && m > 0 && k > 0 && m % kWgT == 0 && k % kWgT == 0,
               "wgrad: n %d, %d batches, %d x %d (multiples of %d)", n, batches, m, k, kWgT);
  E2V2_REQUIRE(groups > 0 && groups <= E2V2_MAX_PART_GROUPS && bounds && bounds[0] == 0 && bounds[groups] == batches,
               "wgrad: %d groups", groups);
  E2V2_REQUIRE(a && b && out && part, "wgrad: null operand");
  E2V2_REQUIRE(lda >= m && ldb >= k && lda % 2 == 0 && ldb % 2 == 0 && a_bs % 2 == 0 && b_bs % 2 == 0 &&
                   ((uintptr_t)a | (uintptr_t)b) % 8 == 0 && ((uintptr_t)out | (uintptr_t)part) % 16 == 0,
               "wgrad: operands need 8-byte aligned rows");
  E2V2_REQUIRE(((int64_t)n + 64) * std::max(lda, ldb) * 4 < (1LL << 31), "wgrad: %d rows exceed the 2 GiB offsets", n);
  PartBounds B{};
  WgArgs P{a, lda, a_bs, b, ldb, b_bs, part, n, 0, e2v2_wgrad_chunks(n, batches, m, k), m, k};
  P.rows = ((n + P.cpb - 1) / P.cpb + 31) / 32 * 32;
  for (int g = 0; g <= groups; ++g) {
    E2V2_REQUIRE(g == 0 || bounds[g] > bounds[g - 1], "wgrad: empty group %d", g - 1);
    B.p[g] = bounds[g] * P.cpb;
  }
  const bool direct = batches * P.cpb == groups;
  if (direct) P.out = out;
  const int64_t n_wg = (int64_t)batches * P.cpb * (m / kWgT) * (k / kWgT);
  E2V2_REQUIRE(n_wg < (1LL << 30), "wgrad: too many tiles");
  hipLaunchKernelGGL(k_wgrad, dim3((uint32_t)((n_wg + kXcd - 1) / kXcd * kXcd)), dim3(kKsThreads), 0, s, P, (int)n_wg);
  E2V2_LAUNCHED("k_wgrad");
  return direct ? 0 : sum_parts(part, B, groups, m * k, out, s);
}

E2V2_API int e2v2_sum_parts(const float* part, int groups, int rows, int w, float* out, hipStream_t s) {
  E2V2_REQUIRE(groups > 0 && groups <= E2V2_MAX_PART_GROUPS && rows > 0 && w > 0 && w % 4 == 0 &&
                   (int64_t)groups * rows < (1LL << 31),
               "sum_parts: %d groups of %d rows of %d", groups, rows, w);
  E2V2_REQUIRE(part && out && ((uintptr_t)part | (uintptr_t)out) % 16 == 0, "sum_parts: 16-byte aligned operands");
  PartBounds B{};
  for (int g = 0; g <= groups; ++g) B.p[g] = g * rows;
  return sum_parts(part, B, groups, w, out, s);
}
