// How K/V rows become byte codes (per-row INT8, per-tensor fp8): the arithmetic the append kernels (kv_int8.hip) and the byte-code
// decode kernel with its append (swa_decode_i8.hip) share, so that both store and attend to the same codes.
#pragma once
#include "common.h"

namespace sb {

constexpr float kScaleMin = 1e-5f, kScaleMax = 1e4f;

// eight 16-bit elements as floats, and back
template <int DT>
__device__ __forceinline__ void unpack8(const uint4 &w, float (&x)[8]) {
  const uint32_t ws[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    if constexpr (DT == SB_BF16) {
      x[2 * i] = bf16_lo(ws[i]);
      x[2 * i + 1] = bf16_hi(ws[i]);
    } else {
      typedef _Float16 h2 __attribute__((ext_vector_type(2)));
      const h2 h = __builtin_bit_cast(h2, ws[i]);
      x[2 * i] = (float)h.x;
      x[2 * i + 1] = (float)h.y;
    }
  }
}
template <int DT>
__device__ __forceinline__ uint4 pack8(const float (&x)[8]) {
  if constexpr (DT == SB_BF16) {
    return make_uint4(pack_bf16(x[0], x[1]), pack_bf16(x[2], x[3]), pack_bf16(x[4], x[5]), pack_bf16(x[6], x[7]));
  } else {
    typedef _Float16 h2 __attribute__((ext_vector_type(2)));
    uint32_t w[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const h2 h = {(_Float16)x[2 * i], (_Float16)x[2 * i + 1]};
      w[i] = __builtin_bit_cast(uint32_t, h);
    }
    return make_uint4(w[0], w[1], w[2], w[3]);
  }
}

// INT8: the scale of a row whose largest magnitude is amax, and its codes (as floats, whole numbers)
__device__ __forceinline__ float int8_scale(float amax) { return fminf(fmaxf(amax / 127.f, kScaleMin), kScaleMax); }
__device__ __forceinline__ float max_abs8(const float (&x)[8], float amax) {
#pragma unroll
  for (int i = 0; i < 8; ++i) amax = fmaxf(amax, fabsf(x[i]));
  return amax;
}
__device__ __forceinline__ void int8_codes(const float (&x)[8], float scale, float (&code)[8]) {
#pragma unroll
  for (int i = 0; i < 8; ++i) code[i] = fminf(fmaxf(rintf(x[i] / scale), -128.f), 127.f);
}
__device__ __forceinline__ uint2 int8_bytes(const float (&code)[8]) {
  uint32_t lo = 0, hi = 0;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    lo |= ((uint32_t)(int)code[i] & 0xffu) << (8 * i);
    hi |= ((uint32_t)(int)code[4 + i] & 0xffu) << (8 * i);
  }
  return make_uint2(lo, hi);
}

// ---- fp8 (OCP e4m3fn) K/V with per-tensor scales ---------------------------------------------------
// code = e4m3fn(clamp(x / scale, -448, 448)), round to nearest even: what the kv_cache_dtype="fp8"
// branch of reshape_and_cache_flash stores (vllm_hymeta/attention/meta_attention.py:790-799 with
// layer._k_scale / layer._v_scale). gfx950's v_cvt_pk_fp8_f32 is that rounding; it does not saturate,
// hence the clamp. NaN stays NaN.
__device__ __forceinline__ uint32_t to_fp8x4(float a, float b, float c, float d) {
  auto q = [&](float x) { return fminf(fmaxf(x, -448.f), 448.f); };  // fminf/fmaxf would drop a NaN: kept below
  const float qa = a != a ? a : q(a), qb = b != b ? b : q(b), qc = c != c ? c : q(c), qd = d != d ? d : q(d);
  int r = __builtin_amdgcn_cvt_pk_fp8_f32(qa, qb, 0, false);
  r = __builtin_amdgcn_cvt_pk_fp8_f32(qc, qd, r, true);
  return (uint32_t)r;
}
// (a quotient by a power of two, which the usual scale of 1 is, is the product with its reciprocal to the bit, and a tenth of
// the instructions: the queries' round trip of every decode workgroup took 2 us in divisions)
__device__ __forceinline__ uint2 fp8_bytes(const float (&x)[8], float s) {
  float y[8];
  if ((__float_as_uint(s) & 0x7fffffu) == 0 && s >= 0x1p-126f && s <= 0x1p126f) {
    const float inv = 1.f / s;
#pragma unroll
    for (int i = 0; i < 8; ++i) y[i] = x[i] * inv;
  } else {
#pragma unroll
    for (int i = 0; i < 8; ++i) y[i] = x[i] / s;
  }
  return make_uint2(to_fp8x4(y[0], y[1], y[2], y[3]), to_fp8x4(y[4], y[5], y[6], y[7]));
}
__device__ __forceinline__ void fp8_values(const uint2 &w, float s, float (&y)[8]) {
  y[0] = __builtin_amdgcn_cvt_f32_fp8((int)w.x, 0) * s; y[1] = __builtin_amdgcn_cvt_f32_fp8((int)w.x, 1) * s;
  y[2] = __builtin_amdgcn_cvt_f32_fp8((int)w.x, 2) * s; y[3] = __builtin_amdgcn_cvt_f32_fp8((int)w.x, 3) * s;
  y[4] = __builtin_amdgcn_cvt_f32_fp8((int)w.y, 0) * s; y[5] = __builtin_amdgcn_cvt_f32_fp8((int)w.y, 1) * s;
  y[6] = __builtin_amdgcn_cvt_f32_fp8((int)w.y, 2) * s; y[7] = __builtin_amdgcn_cvt_f32_fp8((int)w.y, 3) * s;
}

}  // namespace sb
