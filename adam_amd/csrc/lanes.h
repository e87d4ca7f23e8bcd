// Sums and maxima over the lanes of a wave, in the vector unit.
//
// Step for step what __shfl_xor with 32, 16, 8, 4, 2, 1 adds up, bit for bit: an addition does not mind which side comes first,
// and behind the step of 8 the values repeat every 8 lanes, so that a rotation by 4 stands in for lane ^ 4.  __shfl_xor goes
// through LDS, and six of them wait for one another.  ms, the library with it in this place and so, the same words: 24 + 8 tokens of the
// Llama 8B shape 17.73 and 17.25, 21 + 16 of the 4096-wide mixers 9.87 and 9.60, 40 + 16 steps of the expert design 6.39 and 6.18, 17 + 16
// of the Gemma 1B shape 15.46 and 15.14 (runs of one side differ by 0.1 to 1.4 %).  All 64 lanes take part, or none.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace adamah {

typedef uint32_t u2x_t __attribute__((ext_vector_type(2)));
#define LANE_DPP(v, ctrl) __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), ctrl, 0xF, 0xF, false))
#define LANE_X1(v) LANE_DPP(v, 0xB1)
#define LANE_X2(v) LANE_DPP(v, 0x4E)
#define LANE_ROR4(v) LANE_DPP(v, 0x124)      // lane ^ 4 of values that repeat every 8 lanes
#define LANE_X8(v) LANE_DPP(v, 0x128)
__device__ __forceinline__ float lane_x4(float v) {
  const int up = __builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x12C, 0xF, 0x5, false);       // lanes 0 .. 3 and 8 .. 11 of 16
  return __int_as_float(__builtin_amdgcn_update_dpp(up, __float_as_int(v), 0x124, 0xF, 0xA, false));
}
__device__ __forceinline__ u2x_t lanes_x16(float v) { return __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false); }
__device__ __forceinline__ u2x_t lanes_x32(float v) { return __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false); }
__device__ __forceinline__ float add_x16(float v) { const u2x_t a = lanes_x16(v); return __uint_as_float(a.x) + __uint_as_float(a.y); }
__device__ __forceinline__ float add_x32(float v) { const u2x_t a = lanes_x32(v); return __uint_as_float(a.x) + __uint_as_float(a.y); }
__device__ __forceinline__ float max_x16(float v) { const u2x_t a = lanes_x16(v); return fmaxf(__uint_as_float(a.x), __uint_as_float(a.y)); }
__device__ __forceinline__ float max_x32(float v) { const u2x_t a = lanes_x32(v); return fmaxf(__uint_as_float(a.x), __uint_as_float(a.y)); }
__device__ __forceinline__ float wave_add(float v) {
  v = add_x16(add_x32(v));
  v += LANE_X8(v); v += LANE_ROR4(v); v += LANE_X2(v); v += LANE_X1(v);
  return v;
}
__device__ __forceinline__ float wave_max(float v) {
  v = max_x16(max_x32(v));
  v = fmaxf(v, LANE_X8(v)); v = fmaxf(v, LANE_ROR4(v)); v = fmaxf(v, LANE_X2(v)); v = fmaxf(v, LANE_X1(v));
  return v;
}

}  // namespace adamah
