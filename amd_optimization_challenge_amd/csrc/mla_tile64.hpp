// Pieces shared by the kernels that run 32x32x64 MFMAs on pairs of 32-token
// tiles of fp8 rows (decode_h128.hip, decode_rows.hip): the swizzled LDS row
// layout, and lane helpers of their softmax.
#pragma once

#include "mla_common.hpp"

namespace mla {

constexpr int kRowSt = 576;           // LDS row stride: rows are not padded
constexpr int kRowCh = kRowSt / 16;  // 16-byte chunks of a row
// Chunk c of row r lies at position c ^ row_key(r) of the row.  The 144-dword
// stride moves a row 16 banks, so the four rows r & 3 and the four keys cover
// the 64 banks: neither the K fragment reads (ds_read_b128, 16 rows at one chunk)
// nor the V^T transpose reads (ds_read_b64_tr_b8) conflict, no DMA lane is spent
// on padding, and a fragment's address is one register plus constants (the key
// moves only the chunk's low two bits, and rows 16 apart share it).
__device__ __forceinline__ int row_key(int r) { return (r >> 2) & 3; }

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
