// Dense values of packed stores (gfx950): iq_dequant_k (groups along head_dim)
// and iq_dequant_v (groups along tokens), the reads of the reference's dense
// path (cache.py:235-281).
//
// value = fp32(c * s + z) with c * s exact (quant.py:83-93, 121-131; hybrid
// groups as their flag says, quant.py:153-176), times the key normalization
// factor in fp32 (cache.py:132), rounded once to the output's type.
//
// Bound: HBM, and by its writes (2 B out against b/8 + m/G B in per value), so
// the split follows the output: a lane writes 16 bytes of a row (K) or 8 (V)
// and a wave writes whole rows.  (A thread per group, the form before, wrote
// single halves, of keys 2 G bytes apart: 393 us for 3-bit keys with a factor
// of 4 x 8 heads x 16256 tokens, D = 128, and 42 us for 2-bit values; with this
// split 42 and 33 us, and 28 and 26 with the stores of put.)  Fields become
// fp16 integers two at a time: one shift and one and-or with an exponent
// pattern, one packed subtraction.
#include "iq_common.h"
#include "iq_device.h"

using namespace iq;

namespace {

typedef float f2_t __attribute__((ext_vector_type(2)));
typedef float f4_t __attribute__((ext_vector_type(4)));
typedef __bf16 b2_t __attribute__((ext_vector_type(2)));
typedef uint32_t u2_t __attribute__((ext_vector_type(2)));
typedef uint32_t u4_t __attribute__((ext_vector_type(4)));

// NT: the values leave with the non-temporal policy, where a launch writes
// more than NT_BYTES.  Up to there the 256 MB Infinity Cache still holds a
// layer's K and V when the model's attention reads them, and plain stores are
// ahead over both; past it they run into its evictions.  K and V of 4 x 8
// heads read and then reduced once, us a layer, plain / non-temporal: 64 MB
// per tensor 70 / 76, 96 MB 91 / 99, 112 MB 119 / 113, 128 MB 150 / 134, 256
// MB 287 / 263 (the read alone at 128 MB: 76 / 53, 6.1 TB/s).  The quantizers'
// stores, a quarter of what they read, measure the same either way.
constexpr int64_t NT_BYTES = int64_t(104) << 20;
template <bool NT, typename V>
__device__ __forceinline__ void put(void* p, V v) {
  if constexpr (NT) __builtin_nontemporal_store(v, reinterpret_cast<V*>(p));
  else *reinterpret_cast<V*>(p) = v;
}

struct DeqOut {
  uint16_t* out16;  // in the activation dtype
  float* out32;
  int64_t sob, soh, sot;
  int vec16, vec32;  // rows take 16-byte (K) / 8-byte (V) stores of out16, 16-byte stores of out32
};

// Dense rows copied beside the packed ones (iq_read_dense): the first ns and
// last nr tokens of every (batch, head), by the workgroups from blocks0 on,
// one lane per 8 values.
struct CopyRows {
  int64_t blocks0;
  const uint16_t *sink, *recent;
  int64_t ss_b, ss_h, ss_t, sr_b, sr_h, sr_t;
  uint16_t* out;        // the output's first row
  int ns, nq, nr;       // sink, packed and recent rows
  int H, lpr, vec;      // vec: every row takes 16-byte loads and stores
  uint32_t items;       // B * H * (ns + nr) * lpr
};
__device__ __forceinline__ void copy_rows(const CopyRows& c, const DeqOut& o) {
  const uint32_t e = uint32_t(int64_t(blockIdx.x) - c.blocks0) * 256u + threadIdx.x;
  if (e >= c.items) return;
  const uint32_t r = e / uint32_t(c.lpr), col = (e - r * uint32_t(c.lpr)) * 8u, per = uint32_t(c.ns + c.nr);
  const uint32_t bh = r / per, b = bh / uint32_t(c.H), h = bh - b * uint32_t(c.H);
  const int t = int(r - bh * per);
  const uint16_t* src = t < c.ns ? c.sink + b * c.ss_b + h * c.ss_h + t * c.ss_t
                                 : c.recent + b * c.sr_b + h * c.sr_h + int64_t(t - c.ns) * c.sr_t;
  uint16_t* dst = c.out + b * o.sob + h * o.soh + int64_t(t < c.ns ? t : t + c.nq) * o.sot;
  if (c.vec) {
    *reinterpret_cast<uint4*>(dst + col) = *reinterpret_cast<const uint4*>(src + col);
  } else {
#pragma unroll
    for (int i = 0; i < 8; ++i) dst[col + i] = src[col + i];
  }
}

// {scale, zero} of a unit and the integer subtracted from its fields:
// value = (field - off) * s + z
template <bool BF>
__device__ __forceinline__ void unit_params(const uint16_t* meta, int64_t unit, int mode, int bits, float& s, float& z,
                                            int& off) {
  if (mode == IQ_MODE_SYM) {
    s = act2f(meta[unit], BF);
    z = 0.f;
    off = 1 << (bits - 1);
    return;
  }
  const uint32_t mw = reinterpret_cast<const uint32_t*>(meta)[unit];
  const bool sym = mode == IQ_MODE_HYBRID && hyb_sym(mw);
  s = mode == IQ_MODE_HYBRID ? hyb_scale(mw, BF) : act2f(uint16_t(mw & 0xffffu), BF);
  z = sym ? 0.f : act2f(uint16_t(mw >> 16), BF);
  off = sym ? 1 << (bits - 1) : 0;
}

// fields at bit p of both halves of y as fp16 integers less off2
__device__ __forceinline__ h2_t pair_at(uint32_t y, int p, uint32_t mask, h2_t bias) {
  return __builtin_bit_cast(h2_t, ((y >> p) & mask) | 0x64006400u) - bias;
}
__device__ __forceinline__ h2_t bias_of(int off0, int off1) {  // {1024 + off} halves
  return __builtin_bit_cast(h2_t, 0x64006400u + uint32_t(off0) + (uint32_t(off1) << 16));
}

template <bool BF>
__device__ __forceinline__ uint32_t out_pair(float a, float b) {
  if constexpr (BF) return uint32_t(f2bf(a)) | (uint32_t(f2bf(b)) << 16);
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(f2_t{a, b}, h2_t));
}
// the same for values known to be numbers (v_cvt_pk_bf16_f32 keeps a NaN's sign and payload, f2bf does not)
template <bool BF>
__device__ __forceinline__ uint32_t out_pair_num(float a, float b) {
  if constexpr (BF) return __builtin_bit_cast(uint32_t, __builtin_convertvector(f2_t{a, b}, b2_t));
  return out_pair<BF>(a, b);
}
__device__ __forceinline__ bool tame(float s, float z) { return fabsf(s) < 0x1p100f && fabsf(z) < 0x1p100f; }

// ---- K: one lane per 8 values of a row, four rows in flight per lane --------
struct KDeq {
  const uint32_t* codes;
  const uint16_t* meta;
  const uint16_t* norm;
  int64_t cap_blocks;
  int H, t0, T, D, mode;
  int lpr, lpr_sh;  // lanes per row, log2 where it is a power of two <= 256, else -1
  int64_t tiles;    // workgroups per (batch, head)
};
constexpr int KU = 4;

template <int BITS, int G, bool BF, bool NT>
__global__ __launch_bounds__(256) void dequant_k_kernel(KDeq a, DeqOut o, CopyRows cr) {
  constexpr int LPG = G / 8, W = G * BITS / 32;
  if (int64_t(blockIdx.x) >= cr.blocks0) {
    copy_rows(cr, o);
    return;
  }
  const int64_t bh = int64_t(blockIdx.x) / a.tiles, tile = int64_t(blockIdx.x) % a.tiles;
  const int ng = a.D / G;
  const bool fixed = a.lpr_sh >= 0;
  int row[KU], c8[KU];
  uint32_t w[KU];
  float s[KU], z[KU];
  int off[KU];
#pragma unroll
  for (int u = 0; u < KU; ++u) {
    const int64_t e = (tile * KU + u) * 256 + threadIdx.x;
    const int64_t r64 = fixed ? e >> a.lpr_sh : e / a.lpr;
    row[u] = r64 < a.T ? int(r64) : a.T;  // a.T: past the end
    c8[u] = fixed ? int(threadIdx.x) & (a.lpr - 1) : int(e - r64 * a.lpr);
    if (row[u] < a.T) {
      const int g = c8[u] / LPG, j = c8[u] % LPG, q = j & 3;
      const int64_t tt = int64_t(a.t0) + row[u];
      const int64_t unit = ((bh * a.cap_blocks + tt / TOKEN_BLOCK) * ng + g) * TOKEN_BLOCK + tt % TOKEN_BLOCK;
      const int wi = BITS == 4 ? j : BITS == 3 ? (j >> 2) * 3 + (q < 3 ? q : 2) : BITS == 2 ? j >> 1 : j >> 2;
      w[u] = a.codes[unit * W + wi];
      unit_params<BF>(a.meta, unit, a.mode, BITS, s[u], z[u], off[u]);
    }
  }
  float nf[8];
  bool nt = true;
  auto load_norm = [&](int c) {
    const uint16_t* p = a.norm + bh * a.D + c * 8;
    nt = true;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      nf[i] = act2f(p[i], BF);
      nt = nt && tame(nf[i], 0.f);
    }
  };
  if (a.norm && fixed) load_norm(c8[0]);
#pragma unroll
  for (int u = 0; u < KU; ++u) {
    if (row[u] >= a.T) break;  // whole rows of lanes
    const int j = c8[u] % LPG, q = j & 3;
    // the lane's 8 fields: two runs of four, in the halves of y
    uint32_t y;
    if constexpr (BITS == 4) {
      y = w[u];
    } else if constexpr (BITS == 3) {  // 24 bits at 24 q of the quad's three words
      const uint32_t pv = uint32_t(__builtin_amdgcn_mov_dpp(int(w[u]), 0x90, 0xf, 0xf, true));  // quad_perm [0,0,1,2]
      const uint32_t b = __builtin_amdgcn_alignbit(w[u], pv, (32 - 8 * q) & 31);
      y = (b & 0xfffu) | ((b << 4) & 0x0fff0000u);
    } else if constexpr (BITS == 2) {
      const uint32_t b = w[u] >> (16 * (j & 1));
      y = (b & 0xffu) | ((b << 8) & 0x00ff0000u);
    } else {
      const uint32_t b = w[u] >> (8 * q);
      y = (b & 0xfu) | ((b << 12) & 0x000f0000u);
    }
    const h2_t bias = bias_of(off[u], off[u]);
    float v[8];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const h2_t c = pair_at(y, BITS * i, ((1u << BITS) - 1u) * 0x10001u, bias);
      v[i] = __builtin_fmaf(float(c.x), s[u], z[u]);  // quant.py:84-85 (c*s exact)
      v[i + 4] = __builtin_fmaf(float(c.y), s[u], z[u]);
    }
    if (a.norm) {  // cache.py:132
      if (!fixed) load_norm(c8[u]);
#pragma unroll
      for (int i = 0; i < 8; ++i) v[i] = __fmul_rn(v[i], nf[i]);
    }
    const int64_t at = (bh / a.H) * o.sob + (bh % a.H) * o.soh + int64_t(row[u]) * o.sot + c8[u] * 8;
    if (o.out16) {
      uint32_t p[4];
      if (nt && tame(s[u], z[u])) {
#pragma unroll
        for (int i = 0; i < 4; ++i) p[i] = out_pair_num<BF>(v[2 * i], v[2 * i + 1]);
      } else {
#pragma unroll
        for (int i = 0; i < 4; ++i) p[i] = out_pair<BF>(v[2 * i], v[2 * i + 1]);
      }
      if (o.vec16) {
        put<NT>(o.out16 + at, u4_t{p[0], p[1], p[2], p[3]});
      } else {
#pragma unroll
        for (int i = 0; i < 8; ++i) o.out16[at + i] = uint16_t(p[i / 2] >> (16 * (i & 1)));
      }
    }
    if (o.out32) {
      if (o.vec32) {
        put<NT>(o.out32 + at, f4_t{v[0], v[1], v[2], v[3]});
        put<NT>(o.out32 + at + 4, f4_t{v[4], v[5], v[6], v[7]});
      } else {
#pragma unroll
        for (int i = 0; i < 8; ++i) o.out32[at + i] = v[i];
      }
    }
  }
}

// ---- V: one thread per 4 columns of 32 tokens --------------------------------
struct VDeq {
  const uint32_t* codes;
  const uint16_t* meta;
  int64_t cap_groups;
  int H, g0, D, mode;
  int nch;        // 32-token chunks read
  int dq;         // column quads per row, ceil(D / 4)
  int64_t items;  // B * H * nch * dq
};

// nd <= 4 columns of one token: v to element `at`
template <bool BF, bool NT>
__device__ __forceinline__ void put_cols(const DeqOut& o, int64_t at, int nd, bool num, const float (&v)[4]) {
  if (o.out16) {
    uint32_t p0, p1;
    if (num) { p0 = out_pair_num<BF>(v[0], v[1]); p1 = out_pair_num<BF>(v[2], v[3]); }
    else { p0 = out_pair<BF>(v[0], v[1]); p1 = out_pair<BF>(v[2], v[3]); }
    if (o.vec16) {
      put<NT>(o.out16 + at, u2_t{p0, p1});
    } else {
#pragma unroll
      for (int c = 0; c < 4; ++c)
        if (c < nd) o.out16[at + c] = uint16_t((c < 2 ? p0 : p1) >> (16 * (c & 1)));
    }
  }
  if (o.out32) {
    if (o.vec32) {
      put<NT>(o.out32 + at, f4_t{v[0], v[1], v[2], v[3]});
    } else {
#pragma unroll
      for (int c = 0; c < 4; ++c)
        if (c < nd) o.out32[at + c] = v[c];
    }
  }
}

template <int BITS, int G, bool BF, bool NT>
__global__ __launch_bounds__(256) void dequant_v_kernel(VDeq a, DeqOut o, CopyRows cr) {
  constexpr int W = G * BITS / 32, CPG = G / 32;  // chunks per group
  constexpr int CH = 16 / BITS;                   // fields per half
  if (int64_t(blockIdx.x) >= cr.blocks0) {
    copy_rows(cr, o);
    return;
  }
  const int64_t e = int64_t(blockIdx.x) * 256 + threadIdx.x;
  if (e >= a.items) return;
  const int64_t r = e / a.dq;
  const int d = int(e - r * a.dq) * 4;
  const int64_t bh = r / a.nch;
  const int k = int(r - bh * a.nch);
  const int nd = min(4, a.D - d);
  uint32_t w[4][BITS];
  float s[4], z[4];
  int off[4];
  bool num = true;
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    const int64_t unit = (bh * a.cap_groups + a.g0 + k / CPG) * a.D + d + (c < nd ? c : 0);
#pragma unroll
    for (int i = 0; i < BITS; ++i) w[c][i] = a.codes[unit * W + (k % CPG) * BITS + i];
    unit_params<BF>(a.meta, unit, a.mode, BITS, s[c], z[c], off[c]);
    num = num && tame(s[c], z[c]);
  }
  const h2_t b01 = bias_of(off[0], off[1]), b23 = bias_of(off[2], off[3]);
  const int64_t at = (bh / a.H) * o.sob + (bh % a.H) * o.soh + int64_t(k) * 32 * o.sot + d;
  // fields of tokens [CH x, CH x + CH) of two columns, in the halves of a dword
  auto halves = [](const uint32_t* p, const uint32_t* q, int x) {
    if constexpr (BITS != 3) {
      return __builtin_amdgcn_perm(q[x / 2], p[x / 2], x & 1 ? 0x07060302u : 0x05040100u);
    } else {  // 15 bits at 15 x
      const int wi = (15 * x) >> 5, sh = (15 * x) & 31;
      uint32_t u = p[wi] >> sh, v = q[wi] >> sh;
      if (sh > 17 && wi + 1 < BITS) {
        u |= p[wi + 1] << (32 - sh);
        v |= q[wi + 1] << (32 - sh);
      }
      return (u & 0x7fffu) | (v << 16);
    }
  };
  constexpr uint32_t M = ((1u << BITS) - 1u) * 0x10001u;
#pragma unroll
  for (int x = 0; x * CH < 32; ++x) {
    const uint32_t y01 = halves(w[0], w[1], x), y23 = halves(w[2], w[3], x);
#pragma unroll
    for (int i = 0; i < CH; ++i) {
      const int t = x * CH + i;
      if (t >= 32) break;
      const h2_t c01 = pair_at(y01, BITS * i, M, b01), c23 = pair_at(y23, BITS * i, M, b23);
      const float v[4] = {__builtin_fmaf(float(c01.x), s[0], z[0]), __builtin_fmaf(float(c01.y), s[1], z[1]),
                          __builtin_fmaf(float(c23.x), s[2], z[2]), __builtin_fmaf(float(c23.y), s[3], z[3])};
      put_cols<BF, NT>(o, at + int64_t(t) * o.sot, nd, num, v);
    }
  }
}

// The same for launches of at most V_FEW of those threads: four threads per
// chunk and four columns, 8 tokens each.  Such a launch does not fill the
// device and is bound by a thread's chain (its words, then 32 rows of stores),
// which this cuts to 8 rows with 32-bit indices; past the line the words read
// four times over cost more.  2-bit hybrid / 3-bit sym / 4-bit asym values, G =
// 32, D = 128, us a launch with a thread per group and column (the first form),
// with 32 tokens per thread, with 8: 1024 threads of 32 tokens 3.9 / 3.9 / 4.1,
// 4.9 / 4.7 / 5.1, 3.2 / 3.0 / 3.2; 16384 4.6 / 4.6 / 4.8, 6.0 / 5.6 / 6.2, 3.8 /
// 3.7 / 3.7; 49152 6.4 / 6.4 / 6.6, 7.0 / 6.4 / 7.0, 6.3 / 6.1 / 6.3; 53248 7.1 /
// 7.1 / 7.2, 7.0 / 6.5 / 7.4, 7.1 / 6.9 / 7.1; 131072 11.0 / 11.0 / 11.3, 9.8 /
// 9.5 / 10.7, 12.0 / 11.2 / 12.4.
constexpr int64_t V_FEW = 49152;
template <int BITS, int G, bool BF>
__global__ __launch_bounds__(256) void dequant_v_few_kernel(VDeq a, DeqOut o, CopyRows cr) {
  constexpr int W = G * BITS / 32, CPG = G / 32;
  if (int64_t(blockIdx.x) >= cr.blocks0) {
    copy_rows(cr, o);
    return;
  }
  const uint32_t e = blockIdx.x * 256u + threadIdx.x;  // 4 a.items <= 4 V_FEW of them
  if (e >= 4u * uint32_t(a.items)) return;
  const uint32_t rq = e / uint32_t(a.dq), r = rq >> 2, b = r / uint32_t(a.nch);
  const int d = int(e - rq * uint32_t(a.dq)) * 4, q = int(rq & 3u), k = int(r - b * uint32_t(a.nch));
  const int64_t bh = b;
  const int nd = min(4, a.D - d);
  // the 8 fields: 8 BITS bits at 8 BITS q of the column's BITS words
  constexpr int FB = 8 * BITS;
  const int wi = FB * q >> 5, sh = FB * q & 31;
  uint32_t y[4];
  float s[4], z[4];
  int off[4];
  bool num = true;
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    const int64_t unit = (bh * a.cap_groups + a.g0 + k / CPG) * a.D + d + (c < nd ? c : 0);
    const uint32_t* w = a.codes + unit * W + (k % CPG) * BITS;
    y[c] = w[wi] >> sh;
    if constexpr (BITS == 3)  // q = 1, 2: the rest is in the next word
      y[c] |= w[min(wi + 1, BITS - 1)] << ((32 - sh) & 31) & (sh > 8 ? ~0u : 0u);
    unit_params<BF>(a.meta, unit, a.mode, BITS, s[c], z[c], off[c]);
    num = num && tame(s[c], z[c]);
  }
  const h2_t b01 = bias_of(off[0], off[1]), b23 = bias_of(off[2], off[3]);
  const int64_t at = (bh / a.H) * o.sob + (bh % a.H) * o.soh + (int64_t(k) * 32 + 8 * q) * o.sot + d;
  constexpr uint32_t M = ((1u << BITS) - 1u) * 0x10001u, M4 = (1u << (4 * BITS)) - 1u;
#pragma unroll
  for (int x = 0; x < 2; ++x) {  // four tokens of two columns in the halves of a dword
    const uint32_t y01 = (y[0] >> (4 * BITS * x) & M4) | (y[1] >> (4 * BITS * x) & M4) << 16;
    const uint32_t y23 = (y[2] >> (4 * BITS * x) & M4) | (y[3] >> (4 * BITS * x) & M4) << 16;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const h2_t c01 = pair_at(y01, BITS * i, M, b01), c23 = pair_at(y23, BITS * i, M, b23);
      const float v[4] = {__builtin_fmaf(float(c01.x), s[0], z[0]), __builtin_fmaf(float(c01.y), s[1], z[1]),
                          __builtin_fmaf(float(c23.x), s[2], z[2]), __builtin_fmaf(float(c23.y), s[3], z[3])};
      put_cols<BF, false>(o, at + int64_t(4 * x + i) * o.sot, nd, num, v);
    }
  }
}

bool streams(int64_t B, int64_t H, int64_t T, int64_t D, const DeqOut& o) {
  return B * H * T * D * ((o.out16 ? 2 : 0) + (o.out32 ? 4 : 0)) > NT_BYTES;
}
int launch_k(const uint32_t* codes, const uint16_t* meta, int64_t t_cap, const void* norm, int B, int H, int t0, int T,
             int D, int group, int bits, int mode, bool bf, const DeqOut& o, CopyRows cr, int64_t copy_blocks,
             hipStream_t st) {
  const int lpr = D / 8;
  const bool pow2 = (lpr & (lpr - 1)) == 0 && lpr <= 256;
  const KDeq a{codes, meta, (const uint16_t*)norm, t_cap / TOKEN_BLOCK, H, t0, T, D, mode, lpr,
               pow2 ? __builtin_ctz(unsigned(lpr)) : -1, ceil_div(int64_t(T) * lpr, 256 * KU)};
  cr.blocks0 = int64_t(B) * H * a.tiles;
  const bool nt = streams(B, H, T, D, o);
  const dim3 grid(unsigned(cr.blocks0 + copy_blocks));
  return dispatch_store_bits_group(bits, group, [&]<int BITS, int G>() {
    auto* kern = bf   ? (nt ? dequant_k_kernel<BITS, G, true, true> : dequant_k_kernel<BITS, G, true, false>)
                 : nt ? dequant_k_kernel<BITS, G, false, true>
                      : dequant_k_kernel<BITS, G, false, false>;
    kern<<<grid, 256, 0, st>>>(a, o, cr);
    return launch_status();
  });
}
int launch_v(const uint32_t* codes, const uint16_t* meta, int64_t t_cap, int B, int H, int t0, int T, int D, int group,
             int bits, int mode, bool bf, const DeqOut& o, CopyRows cr, int64_t copy_blocks, hipStream_t st) {
  const int nch = T / 32, dq = (D + 3) / 4;
  const VDeq a{codes, meta, t_cap / group, H, t0 / group, D, mode, nch, dq, int64_t(B) * H * nch * dq};
  const bool few = a.items <= V_FEW;
  cr.blocks0 = ceil_div(few ? 4 * a.items : a.items, 256);
  const bool nt = streams(B, H, T, D, o);
  const dim3 grid(unsigned(cr.blocks0 + copy_blocks));
  return dispatch_store_bits_group(bits, group, [&]<int BITS, int G>() {
    auto* kern = few ? (bf ? dequant_v_few_kernel<BITS, G, true> : dequant_v_few_kernel<BITS, G, false>)
                 : bf ? (nt ? dequant_v_kernel<BITS, G, true, true> : dequant_v_kernel<BITS, G, true, false>)
                 : nt ? dequant_v_kernel<BITS, G, false, true>
                      : dequant_v_kernel<BITS, G, false, false>;
    kern<<<grid, 256, 0, st>>>(a, o, cr);
    return launch_status();
  });
}
bool strides_of(int64_t m, int64_t b, int64_t h, int64_t t) { return b % m == 0 && h % m == 0 && t % m == 0; }

}  // namespace

extern "C" {

int iq_dequant_k(const uint32_t* k_codes, const uint16_t* k_meta, int64_t t_cap, const void* norm, int B, int H,
                 int t0, int T, int D, int group, int bits, int mode, void* out16, float* out32, int64_t so_b,
                 int64_t so_h, int64_t so_t, void* stream) {
  IQ_CHECK(k_codes && k_meta, IQ_ERR_NULL);
  IQ_CHECK(out16 || out32, IQ_ERR_NULL);
  const bool bf = act_bf16(mode);
  mode = base_mode(mode);
  if (int e = check_store(bits, group, mode)) return e;
  IQ_CHECK(B >= 0 && H >= 0 && T >= 0 && t0 >= 0 && D > 0, IQ_ERR_SHAPE);
  IQ_CHECK(D % group == 0, IQ_ERR_GROUP);
  IQ_CHECK(t_cap % TOKEN_BLOCK == 0, IQ_ERR_ALIGN);
  IQ_CHECK(int64_t(t0) + T <= t_cap, IQ_ERR_RANGE);
  if (int64_t(B) * H * T == 0) return IQ_OK;
  const DeqOut o{(uint16_t*)out16, out32, so_b, so_h, so_t, aligned(out16, 16) && strides_of(8, so_b, so_h, so_t),
                 aligned(out32, 16) && strides_of(4, so_b, so_h, so_t)};
  return launch_k(k_codes, k_meta, t_cap, norm, B, H, t0, T, D, group, bits, mode, bf, o, CopyRows{}, 0,
                  (hipStream_t)stream);
}

int iq_dequant_v(const uint32_t* v_codes, const uint16_t* v_meta, int64_t t_cap, int B, int H, int t0, int T,
                 int D, int group, int bits, int mode, void* out16, float* out32, int64_t so_b, int64_t so_h,
                 int64_t so_t, void* stream) {
  IQ_CHECK(v_codes && v_meta, IQ_ERR_NULL);
  IQ_CHECK(out16 || out32, IQ_ERR_NULL);
  const bool bf = act_bf16(mode);
  mode = base_mode(mode);
  if (int e = check_store(bits, group, mode)) return e;
  IQ_CHECK(B >= 0 && H >= 0 && T >= 0 && t0 >= 0 && D > 0, IQ_ERR_SHAPE);
  IQ_CHECK(T % group == 0 && t0 % group == 0 && t_cap % group == 0, IQ_ERR_GROUP);
  IQ_CHECK(int64_t(t0) + T <= t_cap, IQ_ERR_RANGE);
  if (int64_t(B) * H * T == 0) return IQ_OK;
  const bool s4 = D % 4 == 0 && strides_of(4, so_b, so_h, so_t);
  const DeqOut o{(uint16_t*)out16, out32, so_b, so_h, so_t, aligned(out16, 8) && s4, aligned(out32, 16) && s4};
  return launch_v(v_codes, v_meta, t_cap, B, H, t0, T, D, group, bits, mode, bf, o, CopyRows{}, 0, (hipStream_t)stream);
}

int iq_read_dense(const iq_segment* s, int axis, const void* norm, int B, int H, int D, void* out16, int64_t so_b,
                  int64_t so_h, int64_t so_t, void* stream) {
  IQ_CHECK(s && out16, IQ_ERR_NULL);
  IQ_CHECK(B >= 0 && H >= 0 && D > 0 && D % 8 == 0 && (axis == 0 || axis == 1), IQ_ERR_SHAPE);
  const iq_segment &k = s[1], &a0 = s[0], &a2 = s[2];
  IQ_CHECK(a0.n >= 0 && k.n > 0 && a2.n >= 0, IQ_ERR_SHAPE);
  IQ_CHECK((a0.n == 0 || a0.dense) && (a2.n == 0 || a2.dense) && k.codes && k.meta, IQ_ERR_NULL);
  const bool bf = act_bf16(k.mode);
  const int mode = base_mode(k.mode);
  for (const iq_segment* d : {&a0, &a2}) IQ_CHECK(d->n == 0 || d->mode == (bf ? int(IQ_MODE_BF16) : 0), IQ_ERR_MODE);
  if (int e = check_store(k.bits, k.group, mode)) return e;
  IQ_CHECK(k.t0 >= 0 && int64_t(k.t0) + k.n <= k.t_cap, IQ_ERR_RANGE);
  if (axis == 0) {
    IQ_CHECK(D % k.group == 0, IQ_ERR_GROUP);
    IQ_CHECK(k.t_cap % TOKEN_BLOCK == 0, IQ_ERR_ALIGN);
  } else {
    IQ_CHECK(!norm, IQ_ERR_SHAPE);
    IQ_CHECK(k.n % k.group == 0 && k.t0 % k.group == 0 && k.t_cap % k.group == 0, IQ_ERR_GROUP);
  }
  const int64_t items = int64_t(B) * H * (int64_t(a0.n) + a2.n) * (D / 8);
  IQ_CHECK(items < (int64_t(1) << 31) && int64_t(a0.n) + k.n + a2.n < (int64_t(1) << 31), IQ_ERR_SHAPE);
  if (int64_t(B) * H == 0) return IQ_OK;
  uint16_t* out = (uint16_t*)out16;
  uint16_t* mid = out + int64_t(a0.n) * so_t;
  const bool s8 = strides_of(8, so_b, so_h, so_t), s4 = D % 4 == 0 && strides_of(4, so_b, so_h, so_t);
  const DeqOut o{mid, nullptr, so_b, so_h, so_t, axis == 0 ? aligned(mid, 16) && s8 : aligned(mid, 8) && s4, 0};
  auto rows16 = [](const iq_segment& d) { return d.n == 0 || (aligned(d.dense, 16) && strides_of(8, d.s_b, d.s_h, d.s_t)); };
  CopyRows c{0, (const uint16_t*)a0.dense, (const uint16_t*)a2.dense, a0.s_b, a0.s_h, a0.s_t, a2.s_b, a2.s_h, a2.s_t,
             out, a0.n, k.n, a2.n, H, D / 8, aligned(out, 16) && s8 && rows16(a0) && rows16(a2), uint32_t(items)};
  const int64_t blocks = ceil_div(items, 256);
  return axis == 0 ? launch_k(k.codes, k.meta, k.t_cap, norm, B, H, k.t0, k.n, D, k.group, k.bits, mode, bf, o, c, blocks,
                              (hipStream_t)stream)
                   : launch_v(k.codes, k.meta, k.t_cap, B, H, k.t0, k.n, D, k.group, k.bits, mode, bf, o, c, blocks,
                              (hipStream_t)stream);
}

}  // extern "C"
