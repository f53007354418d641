// Floor to int32, and reductions over the 64 lanes of a wave, on the VALU (DPP row shifts and row
// broadcasts: one instruction a step, where a shuffle is an LDS round trip).
#pragma once

#include <hip/hip_runtime.h>

namespace ilc {

// floor(f) as int32, saturated, 0 for a NaN: what v_cvt_flr_i32_f32 does (a
// C++ cast says nothing of what lies outside the range)
__device__ inline int32_t floor_to_int(float f) {
  int32_t i;
  asm("v_cvt_flr_i32_f32 %0, %1" : "=v"(i) : "v"(f));
  return i;
}

// x of the lane that DPP control CTRL names, `id` where there is none (lanes
// of rows outside ROWS keep `id`)
template <int CTRL, int ROWS>
__device__ inline int dpp_from(int id, int x) {
  return __builtin_amdgcn_update_dpp(id, x, CTRL, ROWS, 0xf, false);
}

// The reduction of v over the wave with the associative op, whose identity is
// id; the result is wave-uniform.  row_shr 1, 2, 4, 8 leave each row of 16's
// result in its last lane, row_bcast 15 and 31 carry it over the rows to lane 63.
template <class Op>
__device__ inline int wave_reduce(int v, int id, Op&& op) {
  v = op(v, dpp_from<0x111, 0xf>(id, v));
  v = op(v, dpp_from<0x112, 0xf>(id, v));
  v = op(v, dpp_from<0x114, 0xf>(id, v));
  v = op(v, dpp_from<0x118, 0xf>(id, v));
  v = op(v, dpp_from<0x142, 0xa>(id, v));
  v = op(v, dpp_from<0x143, 0xc>(id, v));
  return __builtin_amdgcn_readlane(v, 63);
}

__device__ inline int wave_mini(int v) {
  return wave_reduce(v, INT32_MAX, [](int a, int b) { return min(a, b); });
}
__device__ inline int wave_maxi(int v) {
  return wave_reduce(v, INT32_MIN, [](int a, int b) { return max(a, b); });
}
__device__ inline float wave_minf(float v) {
  return __int_as_float(wave_reduce(__float_as_int(v), __float_as_int(INFINITY), [](int a, int b) {
    return __float_as_int(fminf(__int_as_float(a), __int_as_float(b)));
  }));
}
__device__ inline float wave_maxf(float v) {
  return __int_as_float(wave_reduce(__float_as_int(v), __float_as_int(-INFINITY), [](int a, int b) {
    return __float_as_int(fmaxf(__int_as_float(a), __int_as_float(b)));
  }));
}

// the inclusive sum of v over the lanes up to this one
__device__ inline uint32_t wave_scan(uint32_t v) {
  int s = int(v);
  s += dpp_from<0x111, 0xf>(0, s);
  s += dpp_from<0x112, 0xf>(0, s);
  s += dpp_from<0x114, 0xf>(0, s);
  s += dpp_from<0x118, 0xf>(0, s);
  s += dpp_from<0x142, 0xa>(0, s);
  s += dpp_from<0x143, 0xc>(0, s);
  return uint32_t(s);
}

}  // namespace ilc
