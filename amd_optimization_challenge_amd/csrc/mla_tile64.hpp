// Pieces shared by the kernels that run 32x32x64 MFMAs on pairs of 32-token
// tiles of fp8 rows (decode_h128.hip, decode_rows.hip): the swizzled LDS row
// layout, and lane helpers of their softmax.
#pragma once

#include "mla_common.hpp"

namespace mla {

constexpr int kRowSt = 608;  // LDS row stride: 576 bytes + 32 of padding (38 chunk positions of 16 bytes)

// 16-byte chunks of row r are XOR-swizzled by (r >> 2) & 7, which keeps the K
// fragment reads (ds_read_b128) and the V^T transpose reads
// (ds_read_b64_tr_b8) near their bank-conflict floor.
__device__ __forceinline__ int g128_key(int r) { return (r >> 2) & 7; }
// LDS chunk position (0..35) of logical chunk c of row r; an involution
__device__ __forceinline__ int g128_pos(int r, int c) {
  const int x = g128_key(r);
  return c < 32 ? (c ^ x) : 32 + ((c - 32) ^ (x & 3));
}

// v_permlane32_swap of x with itself: each lane ends with its own value and
// its partner's (lane +- 32)
__device__ __forceinline__ float xhalf_max(float x) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float xhalf_sum(float x) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
// {hi, lo}: hi = e4m3(x), lo = e4m3(x - hi) of four values in [0, 448)
__device__ __forceinline__ int2 split4(float a, float b, float c, float d) {
  const uint32_t h = pack4_fp8(a, b, c, d);
  const v2f h01 = __builtin_amdgcn_cvt_pk_f32_fp8((int)h, false);
  const v2f h23 = __builtin_amdgcn_cvt_pk_f32_fp8((int)h, true);
  return make_int2((int)h, (int)pack4_fp8(a - h01[0], b - h01[1], c - h23[0], d - h23[1]));
}

}  // namespace mla
