// Reductions and scans over the lanes of a wavefront by lane moves of the vector ALU (DPP). A shuffle through LDS
// has about ten times their latency, which is all that the short integer kernels of the preparation and the
// backward's work list are made of. All lanes of the groups or the wavefront have to be active.
#pragma once

#include <hip/hip_runtime.h>

#include <type_traits>

namespace ct {

#define CT_LANES __device__ __forceinline__

// v over the aligned group of `lanes` lanes (a power of two) that the lane belongs to, for all of them.
template <class T, class F>
CT_LANES T over_lanes(T v, int lanes, F f) {
  static_assert(sizeof(T) == 4, "lane moves carry 32 bits");
  const auto step = [&](auto control) { v = f(v, (T)__builtin_amdgcn_mov_dpp((int)v, control.value, 0xf, 0xf, true)); };
  if (lanes >= 2) step(std::integral_constant<int, 0xb1>{});    // quad_perm 1, 0, 3, 2
  if (lanes >= 4) step(std::integral_constant<int, 0x4e>{});    // quad_perm 2, 3, 0, 1
  if (lanes >= 8) step(std::integral_constant<int, 0x141>{});   // the other four of eight, mirrored
  if (lanes >= 16) step(std::integral_constant<int, 0x140>{});  // the other eight of sixteen
  if (lanes >= 32) v = f(v, (T)__shfl_xor((int)v, 16, 64));
  if (lanes >= 64) v = f(v, (T)__shfl_xor((int)v, 32, 64));
  return v;
}
CT_LANES int min_over(int v, int lanes) {
  return over_lanes(v, lanes, [](int a, int b) { return a < b ? a : b; });
}
CT_LANES int max_over(int v, int lanes) {
  return over_lanes(v, lanes, [](int a, int b) { return a > b ? a : b; });
}
CT_LANES int sum_over(int v, int lanes) {
  return over_lanes(v, lanes, [](int a, int b) { return a + b; });
}

// Inclusive scan over the wavefront (values are not negative: 0 is neutral for sums and maxima).
template <bool MAX = false>
CT_LANES int wave_scan(int v) {
  const auto add = [&](int moved) { v = !MAX ? v + moved : v > moved ? v : moved; };
  add(__builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, false));  // from 1, 2, 4, 8 lanes below in a row of 16
  add(__builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, false));
  add(__builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, false));
  add(__builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, false));
  add(__builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false));  // lane 15 to the second row, 47 to the fourth
  add(__builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, false));  // lane 31 to the upper half
  return v;
}
// The value of the lane below, `first` for lane 0; lane k's value, as a scalar.
CT_LANES int lane_below(int v, int first) { return __builtin_amdgcn_update_dpp(first, v, 0x138, 0xf, 0xf, false); }
CT_LANES int lane_value(int v, int k) { return __builtin_amdgcn_readlane(v, k); }

#undef CT_LANES

}  // namespace ct
