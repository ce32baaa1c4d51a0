// Quantization of values, groups along tokens (iq_quantize.h has the
// arithmetic).  The kernels and their launch for one activation type;
// iq_quantize_v.hip (fp16, and the entry point) and iq_quantize_v_bf.hip
// instantiate them, so that they compile in parallel.
#pragma once
#include "iq_quantize.h"

namespace iq::detail {

struct VArgs {
  const uint16_t* x;
  int64_t sxb, sxh, sxt;
  int H, n, D;
  int dp;          // column pairs per row, ceil(D / 2)
  int pairs_ok;    // rows of dword-aligned column pairs (D even, base and strides)
  int64_t items;   // B * H * (n / G) * dp
};
int quantize_v_f16(const VArgs& a, const QuantOut& o, int group, int bits, int mode, bool dense, hipStream_t st);
int quantize_v_bf16(const VArgs& a, const QuantOut& o, int group, int bits, int mode, bool dense, hipStream_t st);
// the same by a lane per value (iq_quant.hip): groups of 32 or 64, asym or sym
int quantize_v_lanes(const VArgs& a, const QuantOut& o, int64_t heads, int group, int bits, int mode, bool bf,
                     hipStream_t st);

}  // namespace iq::detail

namespace {

using detail::VArgs;

// one column of a group, value by value from memory
template <int BITS, int G, int MODE, bool BF>
__device__ __noinline__ void slow_v_column(const uint16_t* xp, int64_t sxt, float mn, float mx, float amx,
                                           QuantOut o, int64_t unit, int64_t el, int64_t el_step, int64_t red) {
  const GroupQ g = group_params<BITS, MODE, BF>(mn, mx, amx);
  bool pick = MODE == IQ_MODE_SYM;
  if constexpr (MODE == IQ_MODE_HYBRID) {
    double ea = 0.0, es = 0.0;
#pragma unroll 1
    for (int i = 0; i < G; ++i) {
      float fa, fs;
      slow_errors<BITS, BF>(act2f(xp[i * sxt], BF), g.z, g.s, g.ss, fa, fs);
      ea += double(fa);
      es += double(fs);
    }
    pick = ea > es;
  }
  uint64_t acc = 0;
  int pos = 0, wj = 0;
#pragma unroll 1
  for (int i = 0; i < G; ++i) {
    int32_t c;
    const float v = act2f(xp[i * sxt], BF);
    acc |= uint64_t(slow_field<BITS, MODE, BF>(v, g.z, g.s, g.ss, pick, c)) << pos;
    if (o.codes_i32) o.codes_i32[el + i * el_step] = c;
    if (o.signs16) o.signs16[el + i * el_step] = f2act(sign_of(v), BF);
    pos += BITS;
    if (pos >= 32) {
      if (o.codes) o.codes[unit * (G * BITS / 32) + wj] = uint32_t(acc);
      ++wj;
      acc >>= 32;
      pos -= 32;
    }
  }
  if (o.codes) {
    const uint32_t mw = meta_of<MODE, BF>(g.s, g.z, g.ss, pick);
    if constexpr (MODE == IQ_MODE_SYM) o.meta[unit] = uint16_t(mw);
    else reinterpret_cast<uint32_t*>(o.meta)[unit] = mw;
  }
  if (o.scale16) o.scale16[red] = f2act(MODE == IQ_MODE_SYM ? g.ss : g.s, BF);
  if (o.zero16) o.zero16[red] = f2act(g.z, BF);
}

// The words of two columns' next 32 fields (BITS words each), from patterns
// added token by token.  fp16 tokens: one dword of two {1024 + field} halves
// per token; a half holds CH = floor(16 / b) fields, so CH tokens are one
// chunk of 16 (3-bit: 15) bits per column.
template <int BITS>
struct PairWords {
  static constexpr int CH = 16 / BITS, NC = (32 + CH - 1) / CH;
  uint32_t c[NC];
  template <int I>
  __device__ __forceinline__ void add(uint32_t y) {
    constexpr int k = I / CH, p = I % CH, last = (k + 1) * CH <= 32 ? CH : 32 - k * CH;
    if constexpr (p == 0) c[k] = y - shifted_sum(H2_BITS, last, BITS);
    else c[k] += y << (BITS * p);
  }
  __device__ __forceinline__ void words(uint32_t* w0, uint32_t* w1) const {
    if constexpr (BITS != 3) {
#pragma unroll
      for (int j = 0; j < BITS; ++j) {
        w0[j] = __builtin_amdgcn_perm(c[2 * j + 1], c[2 * j], 0x05040100u);
        w1[j] = __builtin_amdgcn_perm(c[2 * j + 1], c[2 * j], 0x07060302u);
      }
    } else {
#pragma unroll
      for (int j = 0; j < BITS; ++j) w0[j] = w1[j] = 0u;
#pragma unroll
      for (int k = 0; k < NC; ++k) {  // chunk k: bits [15k, 15k + 15) of a column
        const uint32_t a = c[k] & 0xffffu, b = c[k] >> 16;
        const int wi = (15 * k) >> 5, sh = (15 * k) & 31;
        w0[wi] |= a << sh;
        w1[wi] |= b << sh;
        if (sh > 17 && wi + 1 < BITS) {
          w0[wi + 1] |= a >> (32 - sh);
          w1[wi + 1] |= b >> (32 - sh);
        }
      }
    }
  }
};
// bf16 tokens: one {RNE_BITS + field} dword per column and token
template <int BITS>
struct ColWords {
  static constexpr int CH = 32 / BITS, NC = (32 + CH - 1) / CH;
  uint32_t c[NC];
  template <int I>
  __device__ __forceinline__ void add(float y) {
    constexpr int k = I / CH, p = I % CH, last = (k + 1) * CH <= 32 ? CH : 32 - k * CH;
    if constexpr (p == 0) c[k] = __float_as_uint(y) - shifted_sum(RNE_BITS, last, BITS);
    else c[k] += __float_as_uint(y) << (BITS * p);
  }
  __device__ __forceinline__ void words(uint32_t* w) const {
    if constexpr (BITS != 3) {
#pragma unroll
      for (int j = 0; j < BITS; ++j) w[j] = c[j];
    } else {
#pragma unroll
      for (int j = 0; j < BITS; ++j) w[j] = 0u;
#pragma unroll
      for (int k = 0; k < NC; ++k) {  // chunk k: bits [30k, 30k + 30)
        const int wi = (30 * k) >> 5, sh = (30 * k) & 31;
        w[wi] |= c[k] << sh;
        if (sh > 2 && wi + 1 < BITS) w[wi + 1] |= c[k] >> (32 - sh);
      }
    }
  }
};

template <int N, typename F, int I = 0>
__device__ __forceinline__ void static_for(F&& f) {
  if constexpr (I < N) {
    f.template operator()<I>();
    static_for<N, F, I + 1>(static_cast<F&&>(f));
  }
}

template <int N>
__device__ __forceinline__ void store_words(uint32_t* p, const uint32_t (&w)[N]) {
#pragma unroll
  for (int c = 0; c + 4 <= N; c += 4)
    *reinterpret_cast<u32x4a_t*>(p + c) = u32x4a_t{w[c], w[c + 1], w[c + 2], w[c + 3]};
  constexpr int R = N % 4, C = N - R;
  if constexpr (R == 3) *reinterpret_cast<u32x3a_t*>(p + C) = u32x3a_t{w[C], w[C + 1], w[C + 2]};
  if constexpr (R == 2) *reinterpret_cast<u32x2a_t*>(p + C) = u32x2a_t{w[C], w[C + 1]};
  if constexpr (R == 1) p[C] = w[C];
}

// extremes of the two columns: min / max (asym, hybrid; fp16 packed) and max
// |x| (sym, hybrid; as bit patterns, a NaN above every number)
template <int MODE, bool BF>
struct Extremes {
  h2_t lo, hi;
  float fl[2], fh[2];
  uint32_t m = 0u;
  bool first = true;
  __device__ __forceinline__ void add(uint32_t w) {
    if constexpr (MODE != IQ_MODE_SYM) {
      if constexpr (!BF) {
        lo = first ? as_h2(w) : pk_min(lo, as_h2(w));
        hi = first ? as_h2(w) : pk_max(hi, as_h2(w));
      } else {
        const float x[2] = {lo16(w, true), hi16(w, true)};
#pragma unroll
        for (int c = 0; c < 2; ++c) {
          fl[c] = first ? x[c] : __builtin_elementwise_minimum(fl[c], x[c]);
          fh[c] = first ? x[c] : __builtin_elementwise_maximum(fh[c], x[c]);
        }
      }
      first = false;
    }
    if constexpr (MODE != IQ_MODE_ASYM) m = pk_umax(m, w & 0x7fff7fffu);
  }
  __device__ __forceinline__ void get(float (&mn)[2], float (&mx)[2], float (&amx)[2]) const {
    if constexpr (MODE != IQ_MODE_SYM) {
      mn[0] = BF ? fl[0] : lo_f(lo); mn[1] = BF ? fl[1] : hi_f(lo);
      mx[0] = BF ? fh[0] : lo_f(hi); mx[1] = BF ? fh[1] : hi_f(hi);
    }
    if constexpr (MODE != IQ_MODE_ASYM) {
      amx[0] = act2f(uint16_t(m & 0xffffu), BF);
      amx[1] = act2f(uint16_t(m >> 16), BF);
    }
  }
};

// 32 tokens of both columns in the fast form: words of the asym form wa and /
// or the sym form ws (column c's at [c]), hybrid's error sums, and each
// token's dense codes to `dense`
template <int BITS, int MODE, bool BF, typename F>
__device__ __forceinline__ void chunk32(const uint32_t (&v)[32], const GroupQ (&g)[2], uint32_t (&wa)[2][BITS],
                                        uint32_t (&ws)[2][BITS], double (&ea)[2], double (&es)[2], F&& dense) {
  constexpr int AB = MODE == IQ_MODE_HYBRID ? BITS - 1 : BITS;
  constexpr float OFS = float(1 << (BITS - 1));  // sym offset
  if constexpr (!BF) {
    PairWords<BITS> pa, ps;
    const h2_t mn2 = h2_t{_Float16(g[0].z), _Float16(g[1].z)};
    static_for<32>([&]<int I>() {
      const h2_t x = as_h2(v[I]);
      h2_t ya, ys;
      if constexpr (MODE != IQ_MODE_SYM) {
        ya = asym_y<AB>(x, mn2, g[0].r, g[1].r);
        pa.template add<I>(as_u32(ya));
      }
      if constexpr (MODE != IQ_MODE_ASYM) {
        ys = sym_y<BITS>(x, g[0].rs, g[1].rs);
        ps.template add<I>(as_u32(ys));
      }
      if constexpr (MODE == IQ_MODE_HYBRID) {
        const h2_t ca = ya - h2_splat(1024.f), cs = ys - h2_splat(1024.f + OFS);
        ea[0] += double(fabsf(__fmaf_rn(lo_f(ca), g[0].s, g[0].z) - lo_f(x)));
        ea[1] += double(fabsf(__fmaf_rn(hi_f(ca), g[1].s, g[1].z) - hi_f(x)));
        es[0] += double(fabsf(__fmul_rn(lo_f(cs), g[0].ss) - lo_f(x)));
        es[1] += double(fabsf(__fmul_rn(hi_f(cs), g[1].ss) - hi_f(x)));
      } else {
        const uint32_t yb = as_u32(MODE == IQ_MODE_SYM ? ys : ya) & 0x03ff03ffu;
        constexpr int Z = MODE == IQ_MODE_SYM ? int(OFS) : 0;
        dense(I, int(yb & 0xffffu) - Z, int(yb >> 16) - Z);
      }
    });
    if constexpr (MODE != IQ_MODE_SYM) pa.words(wa[0], wa[1]);
    if constexpr (MODE != IQ_MODE_ASYM) ps.words(ws[0], ws[1]);
  } else {
    ColWords<BITS> pa[2], ps[2];
    static_for<32>([&]<int I>() {
      const float x[2] = {lo16(v[I], true), hi16(v[I], true)};
      float fa[2], fs[2];
      if constexpr (MODE != IQ_MODE_SYM) {
        const uint32_t d = bf2_bits(x[0] - g[0].z, x[1] - g[1].z);
        const uint32_t y = bf2_bits(__fmul_rn(lo16(d, true), g[0].r), __fmul_rn(hi16(d, true), g[1].r));
        fa[0] = clamp_rne<AB>(lo16(y, true), false);
        fa[1] = clamp_rne<AB>(hi16(y, true), false);
        pa[0].template add<I>(fa[0]);
        pa[1].template add<I>(fa[1]);
      }
      if constexpr (MODE != IQ_MODE_ASYM) {
        const uint32_t y = bf2_bits(__fmul_rn(x[0], g[0].rs), __fmul_rn(x[1], g[1].rs));
        fs[0] = clamp_rne<BITS>(lo16(y, true), true);
        fs[1] = clamp_rne<BITS>(hi16(y, true), true);
        ps[0].template add<I>(fs[0]);
        ps[1].template add<I>(fs[1]);
      }
      if constexpr (MODE == IQ_MODE_HYBRID) {
#pragma unroll
        for (int c = 0; c < 2; ++c) {
          ea[c] += double(fabsf(__fmaf_rn(fa[c] - RNE_ONE, g[c].s, g[c].z) - x[c]));
          es[c] += double(fabsf(__fmul_rn(fs[c] - (RNE_ONE + OFS), g[c].ss) - x[c]));
        }
      } else {
        constexpr int Z = MODE == IQ_MODE_SYM ? int(OFS) : 0;
        const float* f = MODE == IQ_MODE_SYM ? fs : fa;
        dense(I, int(__float_as_uint(f[0]) - RNE_BITS) - Z, int(__float_as_uint(f[1]) - RNE_BITS) - Z);
      }
    });
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      if constexpr (MODE != IQ_MODE_SYM) pa[c].words(wa[c]);
      if constexpr (MODE != IQ_MODE_ASYM) ps[c].words(ws[c]);
    }
  }
}

// One thread per two adjacent columns of one token group: the loads of a wave
// are whole row pieces (256 B), every fp16 op covers both columns, a column's
// words leave in one store.  Groups of 32 and 64 tokens stay in registers
// (one or two chunks of 32); a group of 128 is read again chunk by chunk once
// its extremes are known (and, hybrid, its errors), from L2.  DENSE 1: quant.py's
// outputs as well, those that are asked for; 2: all of them, the signs of a
// column pair as one dword, with no branch per store (8 heads x 512 tokens,
// 3-bit sym fp16: 7.0 -> 5.4 us a launch, a thread per column before 5.5;
// 32768 tokens 45 us, 47 before).  A bf16 prompt's prefill (innerq_base, 4 x 8 heads x 8190
// tokens, K and V): 558 -> 166 us with this kernel and quant_k_kernel; one
// lane or one thread per value or group took 239 (K) and 214 us (V) of it.
template <int BITS, int G, int MODE, bool BF, int DENSE>
__global__ __launch_bounds__(256) void quant_v_kernel(VArgs a, QuantOut o) {
  constexpr int W = G * BITS / 32, NCH = G / 32;
  constexpr bool HELD = NCH <= 2;
  const int64_t e = int64_t(blockIdx.x) * 256 + threadIdx.x;
  if (e >= a.items) return;
  const int ngn = a.n / G;
  const int64_t r = e / a.dp;  // bh * ngn + gi
  const int d = int(e - r * a.dp) * 2;
  const int64_t bh = r / ngn;
  const int gi = int(r - bh * ngn);
  const uint16_t* xp = a.x + (bh / a.H) * a.sxb + (bh % a.H) * a.sxh + int64_t(gi) * G * a.sxt + d;
  const bool two = d + 1 < a.D;  // a last single column of an odd D is read as a pair of itself
  auto load = [&](int k, uint32_t (&v)[32]) {
    const uint16_t* p = xp + int64_t(k) * 32 * a.sxt;
    if (a.pairs_ok) {
#pragma unroll
      for (int i = 0; i < 32; ++i) v[i] = *reinterpret_cast<const uint32_t*>(p + i * a.sxt);
    } else {
#pragma unroll
      for (int i = 0; i < 32; ++i) v[i] = uint32_t(p[i * a.sxt]) | (uint32_t(p[i * a.sxt + (two ? 1 : 0)]) << 16);
    }
  };

  uint32_t v[HELD ? NCH : 1][32];
  Extremes<MODE, BF> ex;
  if constexpr (HELD) {
#pragma unroll
    for (int k = 0; k < NCH; ++k) load(k, v[k]);
#pragma unroll
    for (int k = 0; k < NCH; ++k)
#pragma unroll
      for (int i = 0; i < 32; ++i) ex.add(v[k][i]);
  } else {
    load(0, v[0]);
#pragma unroll
    for (int i = 0; i < 32; ++i) ex.add(v[0][i]);
#pragma unroll 1
    for (int k = 1; k < NCH; ++k) {
      load(k, v[0]);
#pragma unroll
      for (int i = 0; i < 32; ++i) ex.add(v[0][i]);
    }
  }
  float mn[2] = {0.f, 0.f}, mx[2] = {0.f, 0.f}, amx[2] = {0.f, 0.f};
  ex.get(mn, mx, amx);
  const GroupQ g[2] = {group_params<BITS, MODE, BF>(mn[0], mx[0], amx[0]),
                       group_params<BITS, MODE, BF>(mn[1], mx[1], amx[1])};
  const int64_t unit = (bh * o.cap_units + o.t_off / G + gi) * a.D + d;
  const int64_t red = r * a.D + d;
  const int64_t el = (bh * a.n + int64_t(gi) * G) * a.D + d;

  if (g[0].slow || g[1].slow) {  // quant.py's arithmetic value by value, for both columns
#pragma unroll 1
    for (int c = 0; c < (two ? 2 : 1); ++c)
      slow_v_column<BITS, G, MODE, BF>(xp + c, a.sxt, c ? mn[1] : mn[0], c ? mx[1] : mx[0], c ? amx[1] : amx[0], o,
                                       unit + c, el + c, a.D, red + c);
    return;
  }

  bool pick[2] = {MODE == IQ_MODE_SYM, MODE == IQ_MODE_SYM};
  double ea[2] = {0.0, 0.0}, es[2] = {0.0, 0.0};
  const int next = two ? 1 : 0;  // a single last column is a pair of itself: the same value twice, and no branch per store
  auto dense = [&](int k, int i, int32_t c0, int32_t c1) {
    if constexpr (DENSE) {
      const int64_t at = el + int64_t(32 * k + i) * a.D;
      const uint32_t w = v[HELD ? k : 0][i];
      if constexpr (MODE == IQ_MODE_SYM) { c0 = abs(c0); c1 = abs(c1); }
      if (DENSE == 2 || o.codes_i32) {  // a constant group's codes: 0 / 0
        o.codes_i32[at] = (MODE == IQ_MODE_SYM ? g[0].ss : g[0].s) == 0.f ? I32_MIN : c0;
        o.codes_i32[at + next] = (MODE == IQ_MODE_SYM ? g[1].ss : g[1].s) == 0.f ? I32_MIN : c1;
      }
      if (MODE != IQ_MODE_ASYM && (DENSE == 2 || o.signs16)) {
        const uint32_t s0 = f2act(sign_of(lo16(w, BF)), BF), s1 = f2act(sign_of(hi16(w, BF)), BF);
        if constexpr (DENSE == 2) {
          *reinterpret_cast<uint32_t*>(o.signs16 + at) = s0 | (s1 << 16);
        } else {
          o.signs16[at] = uint16_t(s0);
          o.signs16[at + next] = uint16_t(s1);
        }
      }
    }
  };
  uint32_t* cp = o.codes + unit * W;
  if constexpr (HELD) {
    uint32_t wa[NCH][2][BITS], ws[NCH][2][BITS];
#pragma unroll
    for (int k = 0; k < NCH; ++k)
      chunk32<BITS, MODE, BF>(v[k], g, wa[k], ws[k], ea, es,
                              [&](int i, int32_t c0, int32_t c1) { dense(k, i, c0, c1); });
    if constexpr (MODE == IQ_MODE_HYBRID) {
      pick[0] = ea[0] > es[0];
      pick[1] = ea[1] > es[1];
    }
    if (o.codes) {
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        uint32_t w[W];
#pragma unroll
        for (int i = 0; i < W; ++i) {
          const int k = i / BITS, j = i % BITS;
          if constexpr (MODE == IQ_MODE_ASYM) w[i] = wa[k][c][j];
          else if constexpr (MODE == IQ_MODE_SYM) w[i] = ws[k][c][j];
          else w[i] = pick[c] ? ws[k][c][j] : wa[k][c][j];
        }
        if (c == 0 || two) store_words(cp + c * W, w);
      }
    }
  } else {
    if constexpr (MODE == IQ_MODE_HYBRID) {
#pragma unroll 1
      for (int k = 0; k < NCH; ++k) {
        uint32_t wa[2][BITS], ws[2][BITS];
        load(k, v[0]);
        chunk32<BITS, MODE, BF>(v[0], g, wa, ws, ea, es, [](int, int32_t, int32_t) {});
      }
      pick[0] = ea[0] > es[0];
      pick[1] = ea[1] > es[1];
    }
#pragma unroll 1
    for (int k = 0; k < NCH; ++k) {
      uint32_t wa[2][BITS], ws[2][BITS];
      load(k, v[0]);
      chunk32<BITS, MODE, BF>(v[0], g, wa, ws, ea, es, [&](int i, int32_t c0, int32_t c1) { dense(k, i, c0, c1); });
      if (o.codes) {
#pragma unroll
        for (int c = 0; c < 2; ++c) {
          uint32_t w[BITS];
#pragma unroll
          for (int j = 0; j < BITS; ++j) {
            if constexpr (MODE == IQ_MODE_ASYM) w[j] = wa[c][j];
            else if constexpr (MODE == IQ_MODE_SYM) w[j] = ws[c][j];
            else w[j] = pick[c] ? ws[c][j] : wa[c][j];
          }
          if (c == 0 || two) store_words(cp + c * W + k * BITS, w);
        }
      }
    }
  }

  if (o.codes) {
    const uint32_t m0 = meta_of<MODE, BF>(g[0].s, g[0].z, g[0].ss, pick[0]);
    const uint32_t m1 = meta_of<MODE, BF>(g[1].s, g[1].z, g[1].ss, pick[1]);
    if constexpr (MODE == IQ_MODE_SYM) {
      o.meta[unit] = uint16_t(m0);
      if (two) o.meta[unit + 1] = uint16_t(m1);
    } else {
      uint32_t* mp = reinterpret_cast<uint32_t*>(o.meta) + unit;
      if (two) *reinterpret_cast<u32x2a_t*>(mp) = u32x2a_t{m0, m1};
      else mp[0] = m0;
    }
  }
  if constexpr (DENSE) {
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      if (c && !two) break;
      if (o.scale16) o.scale16[red + c] = f2act(MODE == IQ_MODE_SYM ? g[c].ss : g[c].s, BF);
      if (o.zero16) o.zero16[red + c] = f2act(g[c].z, BF);
    }
  }
}

template <bool BF>
int launch_quant_v(const VArgs& a, const QuantOut& o, int group, int bits, int mode, bool dense, hipStream_t st) {
  const dim3 grid(unsigned(ceil_div(a.items, 256)));
  return dispatch_format(bits, group, mode, [&]<int BITS, int G, int MODE>() {
    if constexpr (MODE != IQ_MODE_HYBRID) {
      if (dense) {
        const bool pairs = o.signs16 && a.D % 2 == 0 && aligned(o.signs16, 4);
        auto* kern = o.codes_i32 && (MODE == IQ_MODE_ASYM || pairs) ? quant_v_kernel<BITS, G, MODE, BF, 2>
                                                                    : quant_v_kernel<BITS, G, MODE, BF, 1>;
        kern<<<grid, 256, 0, st>>>(a, o);
        return launch_status();
      }
    }
    quant_v_kernel<BITS, G, MODE, BF, 0><<<grid, 256, 0, st>>>(a, o);
    return launch_status();
  });
}

}  // namespace
