// Quantization of keys, groups along head_dim (iq_quantize.h has the arithmetic).
#include "iq_quantize.h"

namespace {

// ============================================================================
// K: groups along head_dim
// ============================================================================
struct KArgs {
  const uint16_t* x;
  int64_t sxb, sxh, sxt;
  const uint16_t* norm;  // [B,H,D] key normalization factor, or null
  int H, n, D;
  int n_pad;             // rows written: n, or up to the block's end (the rest as zeros)
  int lpr, lpr_sh;       // lanes (8 values each) per row, and its log2 where it is a power of two <= 256, else -1
  int64_t tiles;         // workgroups per (batch, head)
};

// x / s rounded to fp16 for finite x and finite s > 0 (fp16 values), given
// r = RN32(1/s): q0 = RN32(x r), then one correction by the residual, which
// an fma gives exactly (Markstein's division step), so the fp32 result is
// RN32(x / s); checked over every such pair (tests/test_quant_division.py).
// (The residual is taken negated, q0 s - x, so that a zero keeps its sign.)
__device__ __forceinline__ float div_rcp(float x, float s, float r) {
  const float q0 = __fmul_rn(x, r);
  return __fmaf_rn(-__fmaf_rn(q0, s, -x), r, q0);
}

// the eight normalization factors of a lane's columns
struct NormRegs {
  float n[8], r[8];
  bool ok;  // every factor is in the fast form's range
};
template <bool BF>
__device__ __forceinline__ NormRegs load_norm(const uint16_t* p) {
  NormRegs q;
  q.ok = true;
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    q.n[i] = act2f(p[i], BF);
    q.ok = q.ok && (BF ? q.n[i] >= 0x1p-60f && q.n[i] <= 0x1p60f : q.n[i] > 0.f && q.n[i] < INFINITY);
    q.r[i] = BF ? __builtin_amdgcn_rcpf(q.n[i]) : __fdiv_rn(1.0f, q.n[i]);
  }
  return q;
}
// x / factor rounded to the activation type (cache.py:125), packed.  fp16:
// the exact division step.  bf16: an 8-bit quotient is never closer to a
// rounding boundary than 2^-17, so one multiplication (by a reciprocal within
// one ulp) rounds alike wherever the result is normal: every |x| is 0 or at least 2^-60 (else per value).
template <bool BF>
__device__ __forceinline__ void normalize(uint32_t (&w)[4], const NormRegs& q) {
  bool ok = q.ok;
  if constexpr (BF) {
    uint32_t lo = 0xffffffffu;  // smallest |x| bits - 1 (zero wraps to the top)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const u16x2_t t = __builtin_bit_cast(u16x2_t, w[j] & 0x7fff7fffu) - u16x2_t{1, 1};
      lo = __builtin_bit_cast(uint32_t, __builtin_elementwise_min(__builtin_bit_cast(u16x2_t, lo), t));
    }
    constexpr uint32_t T = ((127 - 60) << 7) - 1;
    ok = ok && (lo & 0xffffu) >= T && (lo >> 16) >= T;
  } else {  // an infinity has no residual
    const uint32_t m = pk_umax(pk_umax(w[0] & 0x7fff7fffu, w[1] & 0x7fff7fffu),
                               pk_umax(w[2] & 0x7fff7fffu, w[3] & 0x7fff7fffu));
    ok = ok && (m & 0xffffu) < 0x7c00u && (m >> 16) < 0x7c00u;
  }
  if (ok) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const float a = lo16(w[j], BF), b = hi16(w[j], BF);
      if constexpr (BF) {
        w[j] = bf2_bits(__fmul_rn(a, q.r[2 * j]), __fmul_rn(b, q.r[2 * j + 1]));
      } else {
        w[j] = as_u32(h2_of(div_rcp(a, q.n[2 * j], q.r[2 * j]), div_rcp(b, q.n[2 * j + 1], q.r[2 * j + 1])));
      }
    }
  } else {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const float a = lo16(w[j], BF) / q.n[2 * j], b = hi16(w[j], BF) / q.n[2 * j + 1];
      w[j] = uint32_t(f2act(a, BF)) | (uint32_t(f2act(b, BF)) << 16);
    }
  }
}

// op over the LPG lanes of a group (aligned lanes of one 16-lane row)
template <int LPG, typename T, typename F>
__device__ __forceinline__ T group_reduce(T x, F op) {
  static_assert(sizeof(T) == 4 && (LPG == 4 || LPG == 8 || LPG == 16));
  auto step = [&]<int CTRL>() {
    x = op(x, __builtin_bit_cast(T, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, x), CTRL, 0xf, 0xf, true)));
  };
  step.template operator()<0xb1>();                              // quad_perm [1,0,3,2]
  step.template operator()<0x4e>();                              // quad_perm [2,3,0,1]
  if constexpr (LPG >= 8) step.template operator()<0x141>();     // row_half_mirror
  if constexpr (LPG == 16) step.template operator()<0x140>();    // row_mirror
  return x;
}
template <int LPG>
__device__ __forceinline__ double group_sum(double x) {
  auto step = [&]<int CTRL>() {
    const int lo = __builtin_amdgcn_mov_dpp(__double2loint(x), CTRL, 0xf, 0xf, true);
    const int hi = __builtin_amdgcn_mov_dpp(__double2hiint(x), CTRL, 0xf, 0xf, true);
    x += __hiloint2double(hi, lo);
  };
  step.template operator()<0xb1>();
  step.template operator()<0x4e>();
  if constexpr (LPG >= 8) step.template operator()<0x141>();
  if constexpr (LPG == 16) step.template operator()<0x140>();
  return x;
}

// hybrid's choice (quant.py:144): the asym errors' sum exceeds the sym one's,
// both in fp64.  fp16 errors are multiples of 2^-24 below 2^18, so 128 of
// them add exactly in any order; bf16 errors may span more than fp64 holds
// and are added in element order, lane by lane.
template <int LPG, bool BF>
__device__ __forceinline__ bool hybrid_pick(const float (&ea)[8], const float (&es)[8]) {
  double a = 0.0, s = 0.0;
  if constexpr (!BF) {
#pragma unroll
    for (int i = 0; i < 8; ++i) { a += double(ea[i]); s += double(es[i]); }
    return group_sum<LPG>(a) > group_sum<LPG>(s);
  }
  const int base = int(threadIdx.x & 63) & ~(LPG - 1);
#pragma unroll 1
  for (int l = 0; l < LPG; ++l) {
#pragma unroll
    for (int i = 0; i < 8; ++i) { a += double(ea[i]); s += double(es[i]); }
    a = __hiloint2double(__shfl(__double2hiint(a), base + l, 64), __shfl(__double2loint(a), base + l, 64));
    s = __hiloint2double(__shfl(__double2hiint(s), base + l, 64), __shfl(__double2loint(s), base + l, 64));
  }
  return a > s;
}

// fields of a lane's 8 values, 8 * BITS bits in value order, from the fp16
// patterns {1024 + field}: the halves are regrouped as (0,4) (1,5) (2,6) (3,7)
// so that each half's four fields are one run of bits
template <int BITS>
__device__ __forceinline__ uint32_t pack8(const uint32_t (&y)[4]) {
  const uint32_t z[4] = {__builtin_amdgcn_perm(y[2], y[0], 0x05040100u), __builtin_amdgcn_perm(y[2], y[0], 0x07060302u),
                         __builtin_amdgcn_perm(y[3], y[1], 0x05040100u), __builtin_amdgcn_perm(y[3], y[1], 0x07060302u)};
  uint32_t acc = z[0] - shifted_sum(H2_BITS, 4, BITS);
#pragma unroll
  for (int i = 1; i < 4; ++i) acc += z[i] << (BITS * i);
  if constexpr (BITS == 4) return acc;
  if constexpr (BITS == 3) return (acc & 0xfffu) | ((acc >> 4) & 0xfff000u);
  if constexpr (BITS == 2) return (acc & 0xffu) | ((acc >> 8) & 0xff00u);
  return (acc & 0xfu) | ((acc >> 12) & 0xf0u);
}

// eight values of one K group: one lane.  LPG lanes hold a group; the group's
// extremes meet by DPP, its fields as words over lane quads.
template <int BITS, int G, int MODE, bool BF>
__device__ __forceinline__ void quant_k8(uint32_t (&w)[4], int j, const QuantOut& o, int64_t unit, int64_t el,
                                         int64_t red) {
  constexpr int LPG = G / 8;
  // --- the group's extremes (fp16: packed, NaN propagating)
  float mn = 0.f, mx = 0.f, amx = 0.f;
  if constexpr (MODE != IQ_MODE_SYM) {
    if constexpr (!BF) {
      h2_t lo = pk_min(pk_min(as_h2(w[0]), as_h2(w[1])), pk_min(as_h2(w[2]), as_h2(w[3])));
      h2_t hi = pk_max(pk_max(as_h2(w[0]), as_h2(w[1])), pk_max(as_h2(w[2]), as_h2(w[3])));
      lo = group_reduce<LPG>(lo, [](h2_t a, h2_t b) { return pk_min(a, b); });
      hi = group_reduce<LPG>(hi, [](h2_t a, h2_t b) { return pk_max(a, b); });
      mn = __builtin_elementwise_minimum(lo_f(lo), hi_f(lo));
      mx = __builtin_elementwise_maximum(lo_f(hi), hi_f(hi));
    } else {
      mn = lo16(w[0], true);
      mx = mn;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float a = lo16(w[i], true), b = hi16(w[i], true);
        mn = __builtin_elementwise_minimum(__builtin_elementwise_minimum(mn, a), b);
        mx = __builtin_elementwise_maximum(__builtin_elementwise_maximum(mx, a), b);
      }
      mn = group_reduce<LPG>(mn, [](float a, float b) { return __builtin_elementwise_minimum(a, b); });
      mx = group_reduce<LPG>(mx, [](float a, float b) { return __builtin_elementwise_maximum(a, b); });
    }
  }
  if constexpr (MODE != IQ_MODE_ASYM) {  // |x| orders like its bits; a NaN is above every number
    uint32_t m = 0u;
#pragma unroll
    for (int i = 0; i < 4; ++i) m = pk_umax(m, w[i] & 0x7fff7fffu);
    m = group_reduce<LPG>(m, [](uint32_t a, uint32_t b) { return pk_umax(a, b); });
    amx = act2f(uint16_t(max(m & 0xffffu, m >> 16)), BF);
  }
  const GroupQ g = group_params<BITS, MODE, BF>(mn, mx, amx);
  constexpr int AB = MODE == IQ_MODE_HYBRID ? BITS - 1 : BITS;  // bits of the asym form

  uint32_t bits = 0u;     // the lane's 8 fields
  bool pick = MODE == IQ_MODE_SYM;
  if (!g.slow) {
    if constexpr (!BF) {
      uint32_t ya[4], ys[4];
      const h2_t mn2 = h2_splat(mn);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        if constexpr (MODE != IQ_MODE_SYM) ya[i] = as_u32(asym_y<AB>(as_h2(w[i]), mn2, g.r, g.r));
        if constexpr (MODE != IQ_MODE_ASYM) ys[i] = as_u32(sym_y<BITS>(as_h2(w[i]), g.rs, g.rs));
      }
      if constexpr (MODE == IQ_MODE_HYBRID) {
        float ea[8], es[8];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const h2_t ca = as_h2(ya[i]) - h2_splat(1024.f);
          const h2_t cs = as_h2(ys[i]) - h2_splat(1024.f + float(1 << (BITS - 1)));
          const float x0 = lo16(w[i], false), x1 = hi16(w[i], false);
          ea[2 * i] = fabsf(__fmaf_rn(lo_f(ca), g.s, g.z) - x0);
          es[2 * i] = fabsf(__fmul_rn(lo_f(cs), g.ss) - x0);
          ea[2 * i + 1] = fabsf(__fmaf_rn(hi_f(ca), g.s, g.z) - x1);
          es[2 * i + 1] = fabsf(__fmul_rn(hi_f(cs), g.ss) - x1);
        }
        pick = hybrid_pick<LPG, BF>(ea, es);
#pragma unroll
        for (int i = 0; i < 4; ++i) ya[i] = pick ? ys[i] : ya[i];
      }
      if constexpr (MODE == IQ_MODE_SYM) bits = pack8<BITS>(ys);
      else bits = pack8<BITS>(ya);
    } else {
      uint32_t ba = 0u, bs = 0u;
      float ea[8], es[8];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float v[2] = {lo16(w[i], true), hi16(w[i], true)};
        float fa[2], fs[2];
        if constexpr (MODE != IQ_MODE_SYM) {
          const uint32_t d = bf2_bits(v[0] - mn, v[1] - mn);
          const uint32_t y = bf2_bits(__fmul_rn(lo16(d, true), g.r), __fmul_rn(hi16(d, true), g.r));
          fa[0] = clamp_rne<AB>(lo16(y, true), false);
          fa[1] = clamp_rne<AB>(hi16(y, true), false);
          ba += (__float_as_uint(fa[0]) << (BITS * 2 * i)) + (__float_as_uint(fa[1]) << (BITS * (2 * i + 1)));
        }
        if constexpr (MODE != IQ_MODE_ASYM) {
          const uint32_t y = bf2_bits(__fmul_rn(v[0], g.rs), __fmul_rn(v[1], g.rs));
          fs[0] = clamp_rne<BITS>(lo16(y, true), true);
          fs[1] = clamp_rne<BITS>(hi16(y, true), true);
          bs += (__float_as_uint(fs[0]) << (BITS * 2 * i)) + (__float_as_uint(fs[1]) << (BITS * (2 * i + 1)));
        }
        if constexpr (MODE == IQ_MODE_HYBRID) {
#pragma unroll
          for (int h = 0; h < 2; ++h) {
            ea[2 * i + h] = fabsf(__fmaf_rn(fa[h] - RNE_ONE, g.s, g.z) - v[h]);
            es[2 * i + h] = fabsf(__fmul_rn(fs[h] - (RNE_ONE + float(1 << (BITS - 1))), g.ss) - v[h]);
          }
        }
      }
      if constexpr (MODE == IQ_MODE_HYBRID) pick = hybrid_pick<LPG, BF>(ea, es);
      bits = (pick ? bs : ba) - shifted_sum(RNE_BITS, 8, BITS);
    }
  } else {  // NaN or infinity in the group (or an extreme bf16 scale): quant.py's arithmetic value by value
    if constexpr (MODE == IQ_MODE_HYBRID) {
      float ea[8], es[8];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        slow_errors<BITS, BF>(lo16(w[i], BF), g.z, g.s, g.ss, ea[2 * i], es[2 * i]);
        slow_errors<BITS, BF>(hi16(w[i], BF), g.z, g.s, g.ss, ea[2 * i + 1], es[2 * i + 1]);
      }
      pick = hybrid_pick<LPG, BF>(ea, es);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        int32_t c;
        const float v = h ? hi16(w[i], BF) : lo16(w[i], BF);
        bits |= slow_field<BITS, MODE, BF>(v, g.z, g.s, g.ss, pick, c) << (BITS * (2 * i + h));
        if (o.codes_i32) o.codes_i32[el + 2 * i + h] = c;
      }
    }
  }

  if (o.codes) {
    uint32_t* cp = o.codes + unit * (G * BITS / 32);
    const int q = j & 3;
    if constexpr (BITS == 4) {
      cp[j] = bits;
    } else if constexpr (BITS == 3) {  // four lanes' 24 bits are three words
      const uint32_t nx = uint32_t(__builtin_amdgcn_mov_dpp(int(bits), 0xf9, 0xf, 0xf, true));  // quad_perm [1,2,3,3]
      if (q < 3) cp[(j >> 2) * 3 + q] = (bits >> (8 * q)) | (nx << (24 - 8 * q));
    } else if constexpr (BITS == 2) {
      const uint32_t nx = uint32_t(__builtin_amdgcn_mov_dpp(int(bits), 0xf5, 0xf, 0xf, true));  // quad_perm [1,1,3,3]
      if (!(j & 1)) cp[j >> 1] = bits | (nx << 16);
    } else {
      const uint32_t word = group_reduce<4>(bits << (8 * q), [](uint32_t a, uint32_t b) { return a | b; });
      if (q == 0) cp[j >> 2] = word;
    }
    if (j == 0) {
      const uint32_t mw = meta_of<MODE, BF>(g.s, g.z, g.ss, pick);
      if constexpr (MODE == IQ_MODE_SYM) o.meta[unit] = uint16_t(mw);
      else reinterpret_cast<uint32_t*>(o.meta)[unit] = mw;
    }
  }
  if constexpr (MODE != IQ_MODE_HYBRID) {  // the reference-format outputs (quant.py API)
    if (o.codes_i32 && !g.slow) {
      const bool flat = (MODE == IQ_MODE_SYM ? g.ss : g.s) == 0.f;  // 0 / 0: INT32_MIN
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        int32_t c = int32_t((bits >> (BITS * i)) & ((1u << BITS) - 1u));
        if constexpr (MODE == IQ_MODE_SYM) c = abs(c - (1 << (BITS - 1)));
        o.codes_i32[el + i] = flat ? I32_MIN : c;
      }
    }
    if (o.signs16) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        o.signs16[el + 2 * i] = f2act(sign_of(lo16(w[i], BF)), BF);
        o.signs16[el + 2 * i + 1] = f2act(sign_of(hi16(w[i], BF)), BF);
      }
    }
    if (j == 0) {
      if (o.scale16) o.scale16[red] = f2act(MODE == IQ_MODE_SYM ? g.ss : g.s, BF);
      if (o.zero16) o.zero16[red] = f2act(g.z, BF);
    }
  }
}

// One lane per 8 consecutive values of a row: a wave loads whole rows (16 B
// per lane), KU such loads in flight per lane.  A lane's columns are the
// same in all of them where a row's lanes divide the workgroup, so a
// normalization factor's reciprocals are made once.
// A thread per group, the form before, read 64 B per lane at a 64 B stride and
// spent ~25 instructions a value.  8 x 8 heads x 32768 tokens, 4-bit asym G =
// 32 (537 MB read, 168 MB written), both traced on one box: kernel 174 -> 137
// us (5.2 TB/s).  PackedStore.append of them, untraced: 180 -> 161 us a call,
// 134 once it no longer clears the whole new store first.
//
// Four rows per lane, or one up to K_FEW lanes, where the device is not full
// and a call is one lane's chain.  8 heads x 128-d tokens, fp16, us a launch in
// a graph with one / four rows (before this kernel: a lane per value, later a
// thread per group): 128 tokens 4-bit asym 2.4 / 4.3 (3.4), with a factor 2.9 /
// 5.3 (3.6), 2-bit hybrid 2.7 / 5.4 (8.2); 4096 tokens (K_FEW) 4.4 / 5.1, 6.1 /
// 6.2, 5.9 / 6.9; 8192 tokens 6.5 / 7.0, 9.7 / 9.0, 9.2 / 10.1; 32768 tokens
// 19.4 / 19.4, 31.8 / 25.5, 30.1 / 30.0.  bf16 lies alike.
constexpr int KROWS = 4;
constexpr int64_t K_FEW = 1 << 19;
template <int BITS, int G, int MODE, bool BF, int KU>
__global__ __launch_bounds__(256) void quant_k_kernel(KArgs a, QuantOut o) {
  constexpr int LPG = G / 8;
  const int64_t bh = int64_t(blockIdx.x) / a.tiles, tile = int64_t(blockIdx.x) % a.tiles;
  const uint16_t* xb = a.x + (bh / a.H) * a.sxb + (bh % a.H) * a.sxh;
  const bool fixed = a.lpr_sh >= 0;
  int64_t row[KU];
  int c8[KU];
  uint32_t w[KU][4];
#pragma unroll
  for (int u = 0; u < KU; ++u) {
    const int64_t e = (tile * KU + u) * 256 + threadIdx.x;
    row[u] = fixed ? e >> a.lpr_sh : e / a.lpr;
    c8[u] = fixed ? int(threadIdx.x) & (a.lpr - 1) : int(e - row[u] * a.lpr);
    if (row[u] < a.n) {
      const uint4 v = *reinterpret_cast<const uint4*>(xb + row[u] * a.sxt + c8[u] * 8);
      w[u][0] = v.x; w[u][1] = v.y; w[u][2] = v.z; w[u][3] = v.w;
    }
  }
  NormRegs nr;
  if (a.norm && fixed) nr = load_norm<BF>(a.norm + bh * a.D + c8[0] * 8);
  const int ng = a.D / G;
#pragma unroll
  for (int u = 0; u < KU; ++u) {
    if (row[u] >= a.n_pad) break;  // whole groups of lanes
    const int g = c8[u] / LPG, j = c8[u] % LPG;
    const int64_t tt = o.t_off + row[u];
    const int64_t unit = ((bh * o.cap_units + tt / TOKEN_BLOCK) * ng + g) * TOKEN_BLOCK + tt % TOKEN_BLOCK;
    if (row[u] >= a.n) {  // the block's rows past the tokens
      constexpr int W = G * BITS / 32;
      if (j < W) o.codes[unit * W + j] = 0u;
      if (j == 0) {
        if constexpr (MODE == IQ_MODE_SYM) o.meta[unit] = 0;
        else reinterpret_cast<uint32_t*>(o.meta)[unit] = 0u;
      }
      continue;
    }
    if (a.norm) {
      if (!fixed) nr = load_norm<BF>(a.norm + bh * a.D + c8[u] * 8);
      normalize<BF>(w[u], nr);
    }
    const int64_t r = bh * a.n + row[u];
    quant_k8<BITS, G, MODE, BF>(w[u], j, o, unit, r * a.D + c8[u] * 8, r * ng + g);
  }
}

template <int BITS, int G, int MODE, bool BF>
int launch_k(KArgs a, const QuantOut& o, int64_t heads, hipStream_t st) {
  const int64_t lanes = int64_t(a.n_pad) * a.lpr;
  const bool few = heads * lanes <= K_FEW;
  a.tiles = ceil_div(lanes, 256 * (few ? 1 : KROWS));
  auto* kern = few ? quant_k_kernel<BITS, G, MODE, BF, 1> : quant_k_kernel<BITS, G, MODE, BF, KROWS>;
  kern<<<dim3(unsigned(heads * a.tiles)), 256, 0, st>>>(a, o);
  return launch_status();
}
}  // namespace

extern "C" {

int iq_quantize_k(const void* x, int64_t sx_b, int64_t sx_h, int64_t sx_t, const void* norm, int B, int H,
                  int n, int D, int group, int bits, int mode, uint32_t* k_codes, uint16_t* k_meta,
                  int64_t t_cap, int64_t t_off, int32_t* codes_i32, void* scale16, void* zero16, void* signs16,
                  void* stream) {
  IQ_CHECK(x, IQ_ERR_NULL);
  const bool bf = act_bf16(mode), zero_tail = (mode & IQ_MODE_ZERO_TAIL) != 0;
  mode = base_mode(mode) & ~int(IQ_MODE_ZERO_TAIL);
  if (int e = check_store(bits, group, mode)) return e;
  IQ_CHECK(B >= 0 && H >= 0 && n >= 0 && D > 0, IQ_ERR_SHAPE);
  IQ_CHECK(D % group == 0, IQ_ERR_GROUP);
  IQ_CHECK(aligned(x, 16) && sx_b % 8 == 0 && sx_h % 8 == 0 && sx_t % 8 == 0, IQ_ERR_ALIGN);
  IQ_CHECK((k_codes == nullptr) == (k_meta == nullptr), IQ_ERR_NULL);
  if (k_codes) {
    IQ_CHECK(t_cap % TOKEN_BLOCK == 0 && t_off >= 0, IQ_ERR_ALIGN);
    IQ_CHECK(t_off + n <= t_cap, IQ_ERR_RANGE);
    IQ_CHECK(aligned(k_codes, 4) && aligned(k_meta, 4), IQ_ERR_ALIGN);
  }
  IQ_CHECK(!(mode == IQ_MODE_SYM && zero16), IQ_ERR_MODE);
  IQ_CHECK(!(mode == IQ_MODE_ASYM && signs16), IQ_ERR_MODE);
  const bool dense = codes_i32 || scale16 || zero16 || signs16;
  IQ_CHECK(mode != IQ_MODE_HYBRID || (k_codes && !dense), IQ_ERR_MODE);
  if (int64_t(B) * H * n == 0) return IQ_OK;
  QuantOut o{k_codes, k_meta, t_cap / TOKEN_BLOCK, t_off, codes_i32, (uint16_t*)scale16, (uint16_t*)zero16,
             (uint16_t*)signs16};
  const int lpr = D / 8;
  const bool pow2 = (lpr & (lpr - 1)) == 0 && lpr <= 256;
  const int pad = zero_tail && k_codes ? int((TOKEN_BLOCK - (t_off + n) % TOKEN_BLOCK) % TOKEN_BLOCK) : 0;
  KArgs a{(const uint16_t*)x, sx_b, sx_h, sx_t, (const uint16_t*)norm, H, n, D, n + pad, lpr,
          pow2 ? __builtin_ctz(unsigned(lpr)) : -1, 0};
  return dispatch_format(bits, group, mode, [&]<int BITS, int G, int MODE>() {
    return bf ? launch_k<BITS, G, MODE, true>(a, o, int64_t(B) * H, (hipStream_t)stream)
              : launch_k<BITS, G, MODE, false>(a, o, int64_t(B) * H, (hipStream_t)stream);
  });
}

}  // extern "C"
