// Shared by the banded-attention kernels: 16-byte accesses, bf16 pairs, rotary embedding (gfx950).
#pragma once

#include "dh_common.h"

namespace {

typedef __attribute__((__vector_size__(8 * sizeof(short)))) short bf16x8;
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float f32x4;

__device__ __forceinline__ uint4 ld16(const void* p) { return *reinterpret_cast<const uint4*>(p); }
__device__ __forceinline__ uint2 ld8(const void* p) { return *reinterpret_cast<const uint2*>(p); }
__device__ __forceinline__ float lo_f(uint32_t w) { return __uint_as_float(w << 16); }
__device__ __forceinline__ float hi_f(uint32_t w) { return __uint_as_float(w & 0xffff0000u); }
// bf16 rounding through the compiler's conversion (v_cvt_pk_bf16_f32: round to nearest even, the
// rounding torch's bf16 ops use); a pair packs in one instruction
typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
__device__ __forceinline__ float rnd(float x) { return (float)(__bf16)x; }
__device__ __forceinline__ uint32_t pack2(float lo, float hi) {
  bf16x2_t v;
  v.x = (__bf16)lo;
  v.y = (__bf16)hi;
  return __builtin_bit_cast(uint32_t, v);
}

// rope of 8 consecutive elements (4 interleaved pairs) with their 4 cos / sin values; every product
// and sum rounded to bf16 on its own (torch evaluates them as separate bf16 tensor ops)
__device__ __forceinline__ uint4 rope8(const uint4& x, const uint2& c, const uint2& s) {
  const uint32_t xw[4] = {x.x, x.y, x.z, x.w};
  const float cv[4] = {lo_f(c.x), hi_f(c.x), lo_f(c.y), hi_f(c.y)};
  const float sv[4] = {lo_f(s.x), hi_f(s.x), lo_f(s.y), hi_f(s.y)};
  uint32_t o[4];
#pragma unroll
  for (int p = 0; p < 4; ++p) {
    const float e = lo_f(xw[p]), d = hi_f(xw[p]);
    float r0, r1;
    {
#pragma clang fp contract(off)
      r0 = rnd(rnd(e * cv[p]) - rnd(d * sv[p]));
      r1 = rnd(rnd(e * sv[p]) + rnd(d * cv[p]));
    }
    o[p] = pack2(r0, r1);
  }
  return make_uint4(o[0], o[1], o[2], o[3]);
}

__device__ __forceinline__ bf16x8 as_bf16x8(const uint4& v) {
  bf16x8 r;
  __builtin_memcpy(&r, &v, 16);
  return r;
}

}  // namespace
