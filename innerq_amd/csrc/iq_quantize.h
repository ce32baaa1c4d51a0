// Quantize-on-append (gfx950), shared by iq_quantize_k.hip and iq_quantize_v.h: iq_quantize_k (groups along head_dim) and
// iq_quantize_v (groups along tokens), to packed stores and / or quant.py's
// dense outputs, from fp16 or bf16 tokens.
//
// Bound: HBM.  A prompt's quantization reads 2 B and writes b/8 + m/G B per
// value (m = 2 or 4); at 4-bit and G = 32 that is 2.6 B against ~7 VALU
// instructions per two values.  Three things keep the arithmetic below the
// stream (iq_qcodes.h has the reference's own per-value forms, ~25
// instructions each, which these replace for every finite group):
//
//  * fp16 values stay packed: x - min is one v_pk_add_f16 for two values (the
//    reference's fp16 subtraction, exactly), the clamp and the rounding too.
//  * No divide per value.  The code is rint(RN16(d / s)); it equals
//    rint(RN16(RN32(d r))) for every pair of finite fp16 operands d >= 0,
//    s > 0 with r within one fp32 ulp of 1/s (what v_rcp_f32 gives): the
//    quotient only has to fall on the right side of a half-integer, moved
//    by half an fp16 ulp, and d / s is never closer to such a point than
//    2^-23.  The same holds for bf16 operands with s in [2^-100, 2^100].  Both
//    are checked over all operand pairs (tests/test_quant_reciprocal.py).
//    The scale's division by L = 2^b - 1 likewise equals a multiplication by
//    RN32(1/L) for every operand.
//  * rint and the field come from one addition: y + 1024 (fp16) or y + 1.5 2^23
//    (fp32) leaves the half-to-even integer in the low mantissa bits, and
//    fields are packed by shifted adds of those bit patterns; the exponent
//    patterns' sum is a constant, subtracted once per word.
//
// A group whose scale is not finite (it holds a NaN or an infinity, or its
// range overflows), underflows to 0 or, in bf16, is extreme takes the
// per-value forms of iq_qcodes.h.  A constant group (scale 0: the reference divides 0 / 0 and
// packs code 0) comes out of the fast form with r = 0.
#pragma once
#include "iq_common.h"
#include "iq_device.h"
#include "iq_qcodes.h"

using namespace iq;

namespace {

typedef float f2_t __attribute__((ext_vector_type(2)));
typedef __bf16 b2_t __attribute__((ext_vector_type(2)));
typedef unsigned short u16x2_t __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4a_t __attribute__((ext_vector_type(4), aligned(4)));  // dword-aligned vector stores
typedef uint32_t u32x3a_t __attribute__((ext_vector_type(3), aligned(4)));
typedef uint32_t u32x2a_t __attribute__((ext_vector_type(2), aligned(4)));

__device__ __forceinline__ h2_t as_h2(uint32_t x) { return __builtin_bit_cast(h2_t, x); }
__device__ __forceinline__ uint32_t as_u32(h2_t x) { return __builtin_bit_cast(uint32_t, x); }
__device__ __forceinline__ float lo16(uint32_t w, bool bf) { return bf ? __uint_as_float(w << 16) : float(as_h2(w).x); }
__device__ __forceinline__ float hi16(uint32_t w, bool bf) {
  return bf ? __uint_as_float(w & 0xffff0000u) : float(as_h2(w).y);
}
__device__ __forceinline__ float lo_f(h2_t x) { return float(x.x); }
__device__ __forceinline__ float hi_f(h2_t x) { return float(x.y); }
// two fp32 values rounded to bf16, as one dword of bf16 halves
__device__ __forceinline__ uint32_t bf2_bits(float a, float b) {
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(f2_t{a, b}, b2_t));
}
__device__ __forceinline__ h2_t h2_of(float a, float b) { return __builtin_convertvector(f2_t{a, b}, h2_t); }
__device__ __forceinline__ h2_t h2_splat(float a) { return h2_t{_Float16(a), _Float16(a)}; }
__device__ __forceinline__ h2_t pk_min(h2_t a, h2_t b) { return __builtin_elementwise_minimum(a, b); }  // NaN propagates
__device__ __forceinline__ h2_t pk_max(h2_t a, h2_t b) { return __builtin_elementwise_maximum(a, b); }
__device__ __forceinline__ uint32_t pk_umax(uint32_t a, uint32_t b) {
  return __builtin_bit_cast(uint32_t, __builtin_elementwise_max(__builtin_bit_cast(u16x2_t, a),
                                                                 __builtin_bit_cast(u16x2_t, b)));
}

constexpr float L_of(int bits, bool sym) { return float((1 << (sym ? bits - 1 : bits)) - 1); }
// RN16 / RNbf of R / L (quant.py:68, 107): a multiplication by RN32(1/L)
// rounds alike for every R and L in {1, 3, 7, 15}
template <bool BF>
__device__ __forceinline__ float scale_of(float range, float L) { return round_act(__fmul_rn(range, 1.0f / L), BF); }

// r of the fast form (within one ulp of 1/s; 0 for a constant group) and
// whether the group takes the per-value forms: a scale that is not finite, or
// that underflowed to 0 over a range that is not
template <bool BF>
__device__ __forceinline__ bool group_rcp(float s, float range, float& r) {
  r = s > 0.f ? __builtin_amdgcn_rcpf(s) : 0.f;
  return !(s >= (BF ? 0x1p-100f : 0x1p-24f) && s <= (BF ? 0x1p100f : 65504.f)) && range != 0.f;
}

// fp32 form of the field's integer: y clamped and rounded, in the low bits of
// the result's pattern (RNE_BITS + field)
constexpr uint32_t RNE_BITS = 0x4b400000u;  // 1.5 * 2^23
constexpr float RNE_ONE = 12582912.f;       // its value
constexpr uint32_t H2_BITS = 0x64006400u;   // {1024, 1024} in fp16

// sum of shifted exponent patterns of N fields at bit step b
constexpr uint32_t shifted_sum(uint32_t pat, int n, int b) {
  uint32_t s = 0;
  for (int i = 0; i < n; ++i) s += pat << (b * i);
  return s;
}

// ---- one group's parameters -------------------------------------------------
struct GroupQ {
  float s, z;    // asym scale and minimum (hybrid: its (b-1)-bit asym half)
  float ss;      // sym scale (sym, hybrid)
  float r, rs;   // reciprocals of s and ss
  bool slow;     // per-value forms
};
template <int BITS, int MODE, bool BF>
__device__ __forceinline__ GroupQ group_params(float mn, float mx, float amx) {
  GroupQ g{};
  const float nan = __builtin_nanf("");  // a group with a NaN: the canonical one everywhere
  if constexpr (MODE != IQ_MODE_SYM) {
    if (is_nan(mn)) { mn = nan; mx = nan; }
    const float range = round_act(mx - mn, BF);
    g.s = scale_of<BF>(range, L_of(MODE == IQ_MODE_HYBRID ? BITS - 1 : BITS, false));
    g.z = mn;
    g.slow = group_rcp<BF>(g.s, range, g.r);
  }
  if constexpr (MODE != IQ_MODE_ASYM) {
    if (is_nan(amx)) amx = nan;
    g.ss = scale_of<BF>(amx, L_of(BITS, true));
    const bool sl = group_rcp<BF>(g.ss, amx, g.rs);
    g.slow = MODE == IQ_MODE_SYM ? sl : (g.slow || sl);
  }
  return g;
}

// the meta word of a group (sym: the scale alone, in the low half)
template <int MODE, bool BF>
__device__ __forceinline__ uint32_t meta_of(float s, float z, float ss, bool pick_sym) {
  if constexpr (MODE == IQ_MODE_SYM) return f2act(ss, BF);
  if constexpr (MODE == IQ_MODE_ASYM) return meta_word(s, z, BF);
  const uint32_t sh = f2act(pick_sym ? ss : s, BF);
  return pick_sym ? (sh | HYB_FLAG) : ((sh & 0x7fffu) | (uint32_t(f2act(z, BF)) << 16));
}

// the reference's dequantization errors of one value of a hybrid group
// (quant.py:133-151), per-value forms: fp32 differences
template <int BITS, bool BF>
__device__ __forceinline__ void slow_errors(float v, float z, float s, float ss, float& ea, float& es) {
  const float da = __fadd_rn(__fmul_rn(float(asym_code_b(v, z, s, BITS - 1, BF)), s), z);
  const float ds = __fmul_rn(__fmul_rn(float(sym_code_b(v, ss, BITS, BF)), ss), sign_of(v));
  ea = fabsf(__fsub_rn(da, v));
  es = fabsf(__fsub_rn(ds, v));
}
// per-value field and dense code
template <int BITS, int MODE, bool BF>
__device__ __forceinline__ uint32_t slow_field(float v, float z, float s, float ss, bool sym, int32_t& c) {
  if (sym) {
    c = sym_code_b(v, ss, BITS, BF);
    return sym_field_b(c, sign_of(v), BITS);
  }
  constexpr int AB = MODE == IQ_MODE_HYBRID ? BITS - 1 : BITS;
  c = asym_code_b(v, z, s, AB, BF);
  return asym_field_b(c, BITS);
}

// fp16 patterns {1024 + field} of two values (asym: x - min, sym: signed x)
template <int BITS>
__device__ __forceinline__ h2_t asym_y(h2_t x, h2_t mn, float r0, float r1) {
  const h2_t d = x - mn;  // quant.py:69, fp16
  const h2_t y = h2_of(__builtin_fmaf(lo_f(d), r0, 0.f), __builtin_fmaf(hi_f(d), r1, 0.f));  // :70
  return __builtin_elementwise_min(y, h2_splat(L_of(BITS, false))) + h2_splat(1024.f);   // :71
}
template <int BITS>
__device__ __forceinline__ h2_t sym_y(h2_t x, float r0, float r1) {
  const h2_t y = h2_of(__builtin_fmaf(lo_f(x), r0, 0.f), __builtin_fmaf(hi_f(x), r1, 0.f));  // quant.py:108, signed
  constexpr float L = L_of(BITS, true);
  return __builtin_elementwise_max(__builtin_elementwise_min(y, h2_splat(L)), h2_splat(-L)) +
         h2_splat(1024.f + float(1 << (BITS - 1)));  // :109, offset binary
}
// fp32 patterns RNE_BITS + field of one bf16 value
template <int BITS>
__device__ __forceinline__ float clamp_rne(float y, bool sym) {
  constexpr float LA = L_of(BITS, false), LS = L_of(BITS, true);
  const float c = sym ? __builtin_amdgcn_fmed3f(y, -LS, LS) : fminf(y, LA);
  return c + (sym ? RNE_ONE + float(1 << (BITS - 1)) : RNE_ONE);
}

// f.operator()<BITS, G, MODE>() for a store format (1-bit: asym only)
template <typename F>
int dispatch_format(int bits, int group, int mode, F&& f) {
  return dispatch_store_bits_group(bits, group, [&]<int BITS, int G>() {
    if constexpr (BITS > 1) {
      if (mode == IQ_MODE_SYM) return f.template operator()<BITS, G, IQ_MODE_SYM>();
      if (mode == IQ_MODE_HYBRID) return f.template operator()<BITS, G, IQ_MODE_HYBRID>();
    }
    return f.template operator()<BITS, G, IQ_MODE_ASYM>();
  });
}

}  // namespace
