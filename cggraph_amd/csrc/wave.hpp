// Sums, minima and prefix sums over a wavefront's 64 lanes, every lane active,
// in DPP moves within the register file: a shuffle goes through LDS (about 60
// cycles each, and each step of these waits for the one before), which a
// kernel of a few microseconds cannot hide.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>
#include <type_traits>

namespace cg {

// x of the lane that step S of a prefix operation reads, `none` where there is
// none: 0 to 3 lanes 1, 2, 4, 8 below within the row of 16, 4 the last lane of
// the row before (rows 1, 3), 5 the last lane of the lower half (rows 2, 3).
template <int S>
__device__ __forceinline__ uint32_t wave_below(uint32_t x, uint32_t none) {
  constexpr int kCtl[6] = {0x111, 0x112, 0x114, 0x118, 0x142, 0x143};
  constexpr int kRows[6] = {0xf, 0xf, 0xf, 0xf, 0xa, 0xc};
  return (uint32_t)__builtin_amdgcn_update_dpp((int)none, (int)x, kCtl[S], kRows[S], 0xf, false);
}

__device__ __forceinline__ uint32_t lane_value(uint32_t x, uint32_t l) {  // l wave-uniform
  return (uint32_t)__builtin_amdgcn_readlane((int)x, (int)l);
}

// Inclusive prefix sum.
__device__ __forceinline__ uint32_t wave_scan(uint32_t x) {
  x += wave_below<0>(x, 0u);
  x += wave_below<1>(x, 0u);
  x += wave_below<2>(x, 0u);
  x += wave_below<3>(x, 0u);
  x += wave_below<4>(x, 0u);
  x += wave_below<5>(x, 0u);
  return x;
}

__device__ __forceinline__ uint32_t wave_excl_scan(uint32_t x, uint32_t* total) {
  const uint32_t v = wave_scan(x);
  *total = lane_value(v, 63);
  return v - x;
}

__device__ __forceinline__ uint32_t wave_sum_u32(uint32_t x) { return lane_value(wave_scan(x), 63); }

__device__ __forceinline__ uint64_t wave_sum_u64(uint64_t x) {
  auto below = [&](auto s) {
    constexpr int S = decltype(s)::value;
    return (uint64_t)wave_below<S>((uint32_t)(x >> 32), 0u) << 32 | wave_below<S>((uint32_t)x, 0u);
  };
  x += below(std::integral_constant<int, 0>{});
  x += below(std::integral_constant<int, 1>{});
  x += below(std::integral_constant<int, 2>{});
  x += below(std::integral_constant<int, 3>{});
  x += below(std::integral_constant<int, 4>{});
  x += below(std::integral_constant<int, 5>{});
  return (uint64_t)lane_value((uint32_t)(x >> 32), 63) << 32 | lane_value((uint32_t)x, 63);
}

__device__ __forceinline__ uint32_t wave_min_u32(uint32_t x) {
  constexpr uint32_t kNone = 0xFFFFFFFFu;
  auto low = [](uint32_t a, uint32_t b) { return b < a ? b : a; };
  x = low(x, wave_below<0>(x, kNone));
  x = low(x, wave_below<1>(x, kNone));
  x = low(x, wave_below<2>(x, kNone));
  x = low(x, wave_below<3>(x, kNone));
  x = low(x, wave_below<4>(x, kNone));
  x = low(x, wave_below<5>(x, kNone));
  return lane_value(x, 63);
}

}  // namespace cg
