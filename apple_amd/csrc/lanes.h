// Lane exchanges of a wave in the VALU (no LDS round trip as with
// ds_bpermute, which a shuffle compiles to).
#pragma once

#include <hip/hip_runtime.h>

namespace apl {

// Moves by DPP.
// Lanes whose DPP source does not exist read 0: at a row's start by the bound
// control, in rows that the row mask leaves out from `old` (which takes an
// instruction to clear, so bound control wherever no row is left out).
template <int CTRL, int ROW_MASK = 0xF>
__device__ __forceinline__ float dpp_f32(float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, ROW_MASK, 0xF, ROW_MASK == 0xF));
}
template <int CTRL, int ROW_MASK = 0xF>
__device__ __forceinline__ double dpp_f64(double v) {
  const long long b = __builtin_bit_cast(long long, v);
  const int lo = __builtin_amdgcn_update_dpp(0, (int)(b & 0xffffffffll), CTRL, ROW_MASK, 0xF, ROW_MASK == 0xF);
  const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), CTRL, ROW_MASK, 0xF, ROW_MASK == 0xF);
  return __builtin_bit_cast(double, ((long long)hi << 32) | (unsigned int)lo);
}
template <class T, int CTRL, int ROW_MASK = 0xF>
__device__ __forceinline__ T dpp(T v) {
  if constexpr (sizeof(T) == 4)
    return dpp_f32<CTRL, ROW_MASK>(v);
  else
    return dpp_f64<CTRL, ROW_MASK>(v);
}
// gfx9 DPP controls
constexpr int DPP_QUAD_XOR1 = 0xB1;  // quad_perm [1,0,3,2]: the partner lane ^ 1
constexpr int DPP_QUAD_XOR2 = 0x4E;  // quad_perm [2,3,0,1]: the partner lane ^ 2
constexpr int DPP_ROW_SHR1 = 0x111, DPP_ROW_SHR2 = 0x112, DPP_ROW_SHR4 = 0x114, DPP_ROW_SHR8 = 0x118;
constexpr int DPP_ROW_BCAST15 = 0x142, DPP_ROW_BCAST31 = 0x143;

constexpr int DPP_ROW_ROR8 = 0x128;        // within 16 lanes: the partner lane ^ 8
constexpr int DPP_ROW_HALF_MIRROR = 0x141;  // within 8 lanes: 7 - lane
constexpr int DPP_QUAD_REVERSE = 0x1B;      // quad_perm [3,2,1,0]

__device__ __forceinline__ double from_halves(unsigned lo, unsigned hi) {
  return __builtin_bit_cast(double, ((unsigned long long)hi << 32) | lo);
}
// a + b after the upper half of every OFF * 2 lanes of `a` has changed places
// with the lower half of `b` (OFF = 32, 16): each lane keeps one of its two
// values and adds its partner's copy of that one
template <int OFF>
__device__ __forceinline__ double swap_add(double a, double b) {
  const unsigned long long x = __builtin_bit_cast(unsigned long long, a), y = __builtin_bit_cast(unsigned long long, b);
  if constexpr (OFF == 32) {
    const auto lo = __builtin_amdgcn_permlane32_swap((unsigned)x, (unsigned)y, false, false);
    const auto hi = __builtin_amdgcn_permlane32_swap((unsigned)(x >> 32), (unsigned)(y >> 32), false, false);
    return from_halves(lo[0], hi[0]) + from_halves(lo[1], hi[1]);
  } else {
    const auto lo = __builtin_amdgcn_permlane16_swap((unsigned)x, (unsigned)y, false, false);
    const auto hi = __builtin_amdgcn_permlane16_swap((unsigned)(x >> 32), (unsigned)(y >> 32), false, false);
    return from_halves(lo[0], hi[0]) + from_halves(lo[1], hi[1]);
  }
}
// The value of lane ^ OFF.
template <int OFF>
__device__ __forceinline__ double xor_lane(double v) {
  if constexpr (OFF == 1) return dpp_f64<DPP_QUAD_XOR1>(v);
  if constexpr (OFF == 2) return dpp_f64<DPP_QUAD_XOR2>(v);
  if constexpr (OFF == 4) return dpp_f64<DPP_QUAD_REVERSE>(dpp_f64<DPP_ROW_HALF_MIRROR>(v));  // (lane ^ 7) ^ 3
  if constexpr (OFF == 8) return dpp_f64<DPP_ROW_ROR8>(v);
}
// v + (the value of lane ^ OFF)
template <int OFF>
__device__ __forceinline__ double add_xor(double v) {
  if constexpr (OFF >= 16)
    return swap_add<OFF>(v, v);
  else
    return v + xor_lane<OFF>(v);
}

// Sum over the 64 lanes of a wave by a fixed DPP tree: prefix sums within
// each row of 16 lanes, then row 0's total into row 1 and row 2's into
// row 3, then lane 31's into rows 2-3.  The total is in lane 63.
__device__ inline double wave_sum(double v) {
  v += dpp_f64<DPP_ROW_SHR1>(v);
  v += dpp_f64<DPP_ROW_SHR2>(v);
  v += dpp_f64<DPP_ROW_SHR4>(v);
  v += dpp_f64<DPP_ROW_SHR8>(v);
  v += dpp_f64<DPP_ROW_BCAST15, 0xA>(v);
  v += dpp_f64<DPP_ROW_BCAST31, 0xC>(v);
  return v;
}

}  // namespace apl
