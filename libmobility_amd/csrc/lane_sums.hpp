// Sums over the lanes of a wave in a fixed order, by lane swaps and rotations
// inside the rows of 16 (no LDS).
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>

namespace lm {

// a' = {a's lanes 0-31, b's lanes 0-31}, b' = {a's lanes 32-63, b's 32-63};
// returns a' + b': lane l < 32 holds a(l) + a(l + 32), lane l >= 32 the same of b.
__device__ inline double fold32(double a, double b) {
  const uint64_t x = __builtin_bit_cast(uint64_t, a), y = __builtin_bit_cast(uint64_t, b);
  const auto lo = __builtin_amdgcn_permlane32_swap((uint32_t)x, (uint32_t)y, false, false);
  const auto hi =
      __builtin_amdgcn_permlane32_swap((uint32_t)(x >> 32), (uint32_t)(y >> 32), false, false);
  return __builtin_bit_cast(double, ((uint64_t)hi[0] << 32) | lo[0]) +
         __builtin_bit_cast(double, ((uint64_t)hi[1] << 32) | lo[1]);
}
// The same between the even and the odd rows of 16 lanes: even rows hold a's
// sums, odd rows b's.
__device__ inline double fold16(double a, double b) {
  const uint64_t x = __builtin_bit_cast(uint64_t, a), y = __builtin_bit_cast(uint64_t, b);
  const auto lo = __builtin_amdgcn_permlane16_swap((uint32_t)x, (uint32_t)y, false, false);
  const auto hi =
      __builtin_amdgcn_permlane16_swap((uint32_t)(x >> 32), (uint32_t)(y >> 32), false, false);
  return __builtin_bit_cast(double, ((uint64_t)hi[0] << 32) | lo[0]) +
         __builtin_bit_cast(double, ((uint64_t)hi[1] << 32) | lo[1]);
}
// Every lane gets v of the lane N places on in its row of 16 (cyclic).
template <int N>
__device__ inline double row_ror(double v) {
  const uint64_t b = __builtin_bit_cast(uint64_t, v);
  const uint32_t lo = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)b, 0x120 + N, 0xf,
                                                            0xf, true);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)(b >> 32),
                                                            0x120 + N, 0xf, 0xf, true);
  return __builtin_bit_cast(double, ((uint64_t)hi << 32) | lo);
}
__device__ inline double row_sum(double v) {
  v += row_ror<8>(v);
  v += row_ror<4>(v);
  v += row_ror<2>(v);
  return v + row_ror<1>(v);
}

// The sum over the 64 lanes, in every lane.  Adds the same pairs as the
// butterfly v += shfl_xor(v, o), o = 32, 16, 8, 4, 2, 1: after the first three
// steps a lane's value depends on its number modulo 8 only, and so on, so the
// rotations pair what the exclusive-or does.
__device__ inline double wave_sum(double v) { return row_sum(fold16(fold32(v, v), fold32(v, v))); }

}  // namespace lm
