// Tiles of the split-bf16 GEMMs for matrices of few rows (gemm.hip): K split over the wavefronts for three operand
// pieces, in one order for one piece.
//
// A 128 x 128 tile of gemm_core.h walks K in stages of 16 one after another, a barrier and the latency of its
// two-stages-ahead loads per stage: about 2 us a stage when the operands come from the Infinity Cache, 33 us
// for K = 256 however few rows there are, and a matrix of few rows has few such tiles (9 m-rows x 256 columns
// of 24 atoms: 18 tiles on 256 CUs).  Here a tile is 32 kR rows x 32 kJ columns and the four wavefronts of its
// workgroup split K (wavefront w the contiguous stages [w nks / 4, (w + 1) nks / 4)): each loads its fragments
// of both operands from memory straight into registers, kD stages ahead, with no LDS and no barrier in the
// loop; the four partial tiles meet once in LDS, where wavefront w adds a quarter of the tile's registers in
// wavefront order.  The packed weight is read as it lies (a 32-column subtile of a piece is 1 KB contiguous).
// The products, their pieces and the order inside a wavefront are those of kloop; the sum over K is the sum
// of four shorter ones in fixed order.  With one piece the wavefronts take a column subtile each and all of K, so
// that the sum is kloop's bit by bit.
#pragma once
#include "gemm_core.h"

namespace e2v2 {
namespace {

constexpr int kKsW = 4;                       // wavefronts per workgroup = parts of K
constexpr int kKsThreads = 64 * kKsW;

// Byte offset, within one packed piece of a stage, of this lane's granule (column lane % 32 of the 32-column
// subtile q, k 8 (lane / 32) .. +7).
__device__ __forceinline__ uint32_t ks_b_offset(int q, int lane) {
  return 16u * (uint32_t)b_slot(32 * q + (lane & 31), lane >> 5);
}
__device__ __forceinline__ bf16x8 ks_load_b(__amdgpu_buffer_rsrc_t r, uint32_t off) {
  return __builtin_bit_cast(bf16x8, __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, 0));
}
__device__ __forceinline__ floatx4 ks_load4(__amdgpu_buffer_rsrc_t r, uint32_t off) {
  return __builtin_bit_cast(floatx4, __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, 0));
}

template <int kR, int kJ>
__device__ __forceinline__ void ks_zero(floatx16 (&acc)[kR][kJ]) {
#pragma unroll
  for (int i = 0; i < kR; ++i)
#pragma unroll
    for (int j = 0; j < kJ; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;
}

template <int kP>
__device__ __forceinline__ void ks_mfma(const bf16x8 (&a)[kP], const bf16x8 (&b)[kP], floatx16& acc) {
  if constexpr (kP == 3) {
    constexpr int kPa[6] = {0, 1, 2, 0, 1, 0}, kPb[6] = {0, 0, 0, 1, 1, 2};
#pragma unroll
    for (int q = 0; q < 6; ++q) acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[kPa[q]], b[kPb[q]], acc, 0, 0, 0);
  } else {
    acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[0], b[0], acc, 0, 0, 0);
  }
}

// acc[i][j] += the sum over stages [ks0, ks1) of the row tile i (32 rows) times the column subtile j.  Raw: one row
// tile's A registers of a stage, loaded by load_a(ks, i, raw) and turned into pieces by split(ks, i, raw, a).
// boff[j]: the lane's byte offset of subtile j in a piece of stage 0.  A ring of kD stages' registers, each
// slot refilled as soon as it is consumed; no load past ks1 is issued.
template <int kP, int kR, int kJ, int kD, typename Raw, typename LoadA, typename Split>
__device__ __forceinline__ void ks_loop(__amdgpu_buffer_rsrc_t br, const uint32_t (&boff)[kJ], int ks0, int ks1,
                                        LoadA&& load_a_, Split&& split, floatx16 (&acc)[kR][kJ]) {
  Raw ra[kD][kR];
  bf16x8 rb[kD][kJ][kP];
  auto load = [&](int ks, auto slot) {
    constexpr int sl = decltype(slot)::value;
#pragma unroll
    for (int i = 0; i < kR; ++i) load_a_(ks, i, ra[sl][i]);
    const uint32_t st = (uint32_t)ks * (b_stage_granules(kP) * 16u);
#pragma unroll
    for (int j = 0; j < kJ; ++j)
#pragma unroll
      for (int p = 0; p < kP; ++p) rb[sl][j][p] = ks_load_b(br, st + (uint32_t)p * (kGBg * 16u) + boff[j]);
  };
  auto use = [&](int ks, auto slot) {
    constexpr int sl = decltype(slot)::value;
#pragma unroll
    for (int i = 0; i < kR; ++i) {
      bf16x8 a[kP];
      split(ks, i, ra[sl][i], a);
#pragma unroll
      for (int j = 0; j < kJ; ++j) ks_mfma<kP>(a, rb[sl][j], acc[i][j]);
    }
  };
  auto each = [&](auto&& f) {
    f(std::integral_constant<int, 0>{});
    if constexpr (kD > 1) f(std::integral_constant<int, 1>{});
    if constexpr (kD > 2) f(std::integral_constant<int, 2>{});
    if constexpr (kD > 3) f(std::integral_constant<int, 3>{});
    if constexpr (kD > 4) f(std::integral_constant<int, 4>{});
    if constexpr (kD > 5) f(std::integral_constant<int, 5>{});
    if constexpr (kD > 6) f(std::integral_constant<int, 6>{});
    if constexpr (kD > 7) f(std::integral_constant<int, 7>{});
    static_assert(kD >= 1 && kD <= 8, "ring of one to eight stages");
  };
  each([&](auto s) {
    if (ks0 + s.value < ks1) load(ks0 + s.value, s);
  });
  for (int ks = ks0; ks < ks1; ks += kD) {
    each([&](auto s) {
      if (ks + s.value < ks1) {
        use(ks + s.value, s);
        if (ks + s.value + kD < ks1) load(ks + s.value + kD, s);
      }
    });
  }
}

// Adds the kW wavefronts' partial tiles: every wavefront stores its registers in LDS, then wavefront w returns
// the sums (in wavefront order) of its share of the kN registers (register 16 (kJ i + j) + r of the flattened
// accumulator): part(w, i), i < kN / kW, names them.  red: kW * kN * 64 floats.
template <int kN, int kW, typename Part>
__device__ __forceinline__ void ks_reduce(float* red, const float (&part)[kN], int wv, int lane, Part&& reg,
                                          float (&sum)[kN / kW]) {
#pragma unroll
  for (int i = 0; i < kN; ++i) red[(wv * kN + i) * 64 + lane] = part[i];
  __syncthreads();
#pragma unroll
  for (int i = 0; i < kN / kW; ++i) {
    const int q = reg(wv, i);
    float s = red[q * 64 + lane];
#pragma unroll
    for (int w = 1; w < kW; ++w) s += red[(w * kN + q) * 64 + lane];
    sum[i] = s;
  }
}
template <int kR, int kJ>
__device__ __forceinline__ void ks_flat(const floatx16 (&acc)[kR][kJ], float (&part)[16 * kR * kJ]) {
#pragma unroll
  for (int i = 0; i < kR; ++i)
#pragma unroll
    for (int j = 0; j < kJ; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) part[16 * (kJ * i + j) + r] = acc[i][j][r];
}

}  // namespace
}  // namespace e2v2
