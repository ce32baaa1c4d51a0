// One value's quantization in the reference's own arithmetic (src/innerq/quant.py):
// every op of the reference is an fp32 op rounded to the activation dtype
// (fp16, or bf16 with bf), the clamp keeps NaN, the rounding is half-to-even
// and a NaN code is INT32_MIN in dense outputs, 0 (asym) or the offset (sym)
// in packed fields.  The prompt quantizers (iq_quantize.h) use these forms for
// groups that hold NaN or infinity, the lane-per-value quantizers of
// iq_quant.hip (the window append, short calls of values) for every group.
#pragma once
#include "iq_common.h"
#include "iq_device.h"

namespace iq {

constexpr int32_t I32_MIN = (int32_t)0x80000000u;

// What a quantize call writes: the packed store (or null) and the dense
// reference-format outputs (each or null).
struct QuantOut {
  uint32_t* codes;     // packed store codes (or null)
  uint16_t* meta;      // packed store meta
  int64_t cap_units;   // K: t_cap/64 blocks, V: t_cap/G groups
  int64_t t_off;       // first token written in the store
  int32_t* codes_i32;  // dense outputs (optional)
  uint16_t* scale16;
  uint16_t* zero16;
  uint16_t* signs16;
};

__device__ __forceinline__ bool is_nan(float v) { return v != v; }

// clamp(y, 0, L) keeping NaN, then half-to-even round.  Returns the dense
// int32 code (INT32_MIN for NaN, as torch's float->int32 on x86).
__device__ __forceinline__ int32_t code_of(float y, float L) {
  if (is_nan(y)) return I32_MIN;
  y = fminf(fmaxf(y, 0.0f), L);
  return (int32_t)rintf(y);
}

// Group statistics and per-element codes of the two quantizers, one rounding
// to the activation dtype (fp16, or bf16 with bf) per reference op (runtime
// bit width; the templates below pass a constant).
// asym (quant.py:66-71): scale of b-bit codes from the group's min and max
__device__ __forceinline__ float asym_scale_b(float mn, float mx, int bits, bool bf = false) {
  return round_act(round_act(mx - mn, bf) / float((1 << bits) - 1), bf);    // quant.py:68
}
__device__ __forceinline__ int32_t asym_code_b(float x, float mn, float s, int bits, bool bf = false) {
  return code_of(round_act(round_act(x - mn, bf) / s, bf), float((1 << bits) - 1));  // quant.py:69-71
}
// sym (quant.py:104-109): scale of b-bit codes (one bit is the sign)
__device__ __forceinline__ float sym_scale_b(float mx, int bits, bool bf = false) {
  return round_act(mx / float((1 << (bits - 1)) - 1), bf);              // quant.py:107
}
__device__ __forceinline__ int32_t sym_code_b(float x, float s, int bits, bool bf = false) {
  return code_of(round_act(fabsf(x) / s, bf), float((1 << (bits - 1)) - 1));  // quant.py:108-109
}
__device__ __forceinline__ float sign_of(float x) { return x > 0.f ? 1.f : (x < 0.f ? -1.f : 0.f); }  // torch.sign
// stored fields: the asym code (0 for NaN); sym sign*magnitude + 2^(b-1)
__device__ __forceinline__ uint32_t asym_field_b(int32_t c, int bits) {
  return (c == I32_MIN) ? 0u : (uint32_t(c) & ((1u << bits) - 1u));
}
__device__ __forceinline__ uint32_t sym_field_b(int32_t c, float sg, int bits) {
  const int32_t sc = (c == I32_MIN) ? 0 : (sg > 0.f ? c : (sg < 0.f ? -c : 0));
  return uint32_t(sc + (1 << (bits - 1))) & ((1u << bits) - 1u);  // offset binary
}


__device__ __forceinline__ uint32_t meta_word(float s, float z, bool bf = false) {
  return uint32_t(f2act(s, bf)) | (uint32_t(f2act(z, bf)) << 16);
}

}  // namespace iq
