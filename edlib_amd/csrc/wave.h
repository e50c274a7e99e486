// Exchanges between the lanes of a wavefront on the register file.
#pragma once

#include <hip/hip_runtime.h>

namespace edh {

// x of lane (lane xor 8, 4, 2, 1) within its row of sixteen, for values that
// repeat with period 2 S: a row rotation by S reaches the same value.
template <int S>
__device__ __forceinline__ double row_rotate(double x) {
  const long long b = __double_as_longlong(x);
  const int lo = __builtin_amdgcn_update_dpp(0, (int)b, 0x120 + S, 0xf, 0xf, false);
  const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), 0x120 + S, 0xf, 0xf, false);
  return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}

// Sum over the wavefront, on every lane: the halving tree (lane distances 32,
// 16, 8, 4, 2, 1) on the register file's own exchanges, about 150 cycles where
// the six shuffles through LDS took about 800.
__device__ __forceinline__ double wave_sum(double x) {
  const long long b = __double_as_longlong(x);
  const auto l5 = __builtin_amdgcn_permlane32_swap((unsigned)b, (unsigned)b, false, false);
  const auto h5 = __builtin_amdgcn_permlane32_swap((unsigned)(b >> 32), (unsigned)(b >> 32), false, false);
  x = __longlong_as_double(((long long)h5[0] << 32) | l5[0]) + __longlong_as_double(((long long)h5[1] << 32) | l5[1]);
  const long long c = __double_as_longlong(x);
  const auto l4 = __builtin_amdgcn_permlane16_swap((unsigned)c, (unsigned)c, false, false);
  const auto h4 = __builtin_amdgcn_permlane16_swap((unsigned)(c >> 32), (unsigned)(c >> 32), false, false);
  x = __longlong_as_double(((long long)h4[0] << 32) | l4[0]) + __longlong_as_double(((long long)h4[1] << 32) | l4[1]);
  x += row_rotate<8>(x);
  x += row_rotate<4>(x);
  x += row_rotate<2>(x);
  x += row_rotate<1>(x);
  return x;
}

}  // namespace edh
