// Quantization of fp16 values, groups along tokens, and the entry point.
#include "iq_quantize_v.h"

int iq::detail::quantize_v_f16(const VArgs& a, const QuantOut& o, int group, int bits, int mode, bool dense,
                               hipStream_t st) {
  return launch_quant_v<false>(a, o, group, bits, mode, dense, st);
}

namespace {

// Values up to which a call goes by a lane per value (groups of 32 or 64, asym
// or sym): a thread's chain over its 32 tokens and two columns bounds a short
// call, whose lanes are few.  8 heads x 128 columns, us a launch in a graph,
// lanes / threads: 128 tokens (2^17) bf16 to a store 3.3 / 3.9 (G = 32 asym), 3.2
// / 3.5 (sym), 3.9 / 5.2 (G = 64), fp16 3.2 / 3.2, 3.1 / 3.3, 3.8 / 4.0; 256
// tokens bf16 4.1 / 4.0, 3.9 / 3.6, 4.8 / 5.3, fp16 3.9 / 3.3, 3.8 / 3.3, 4.6 /
// 4.0.  With quant.py's outputs the threads store more: 256 tokens bf16 4.4 /
// 4.7, 4.7 / 5.9, 5.6 / 6.8, fp16 4.2 / 4.5, 4.7 / 5.2, 5.5 / 6.4; 512 tokens
// 6.3 / 4.9, 6.7 / 6.0, 8.1 / 6.9, fp16 6.0 / 4.6, 6.4 / 5.4, 7.9 / 6.5.
int64_t lane_values(int group, bool bf, bool dense) { return dense || (bf && group == 64) ? 1 << 18 : 1 << 17; }

}  // namespace

extern "C" {

int iq_quantize_v(const void* x, int64_t sx_b, int64_t sx_h, int64_t sx_t, int B, int H, int n, int D,
                  int group, int bits, int mode, uint32_t* v_codes, uint16_t* v_meta, int64_t t_cap,
                  int64_t t_off, int32_t* codes_i32, void* scale16, void* zero16, void* signs16, void* stream) {
  IQ_CHECK(x, IQ_ERR_NULL);
  const bool bf = act_bf16(mode);
  mode = base_mode(mode);
  if (int e = check_store(bits, group, mode)) return e;
  IQ_CHECK(B >= 0 && H >= 0 && n >= 0 && D > 0, IQ_ERR_SHAPE);
  IQ_CHECK(n % group == 0, IQ_ERR_GROUP);
  IQ_CHECK(aligned(x, 2), IQ_ERR_ALIGN);
  IQ_CHECK((v_codes == nullptr) == (v_meta == nullptr), IQ_ERR_NULL);
  if (v_codes) {
    IQ_CHECK(t_cap % group == 0 && t_off % group == 0 && t_off >= 0, IQ_ERR_ALIGN);
    IQ_CHECK(t_off + n <= t_cap, IQ_ERR_RANGE);
    IQ_CHECK(aligned(v_codes, 4) && aligned(v_meta, 4), IQ_ERR_ALIGN);
  }
  IQ_CHECK(!(mode == IQ_MODE_SYM && zero16), IQ_ERR_MODE);
  IQ_CHECK(!(mode == IQ_MODE_ASYM && signs16), IQ_ERR_MODE);
  const bool dense = codes_i32 || scale16 || zero16 || signs16;
  IQ_CHECK(mode != IQ_MODE_HYBRID || (v_codes && !dense), IQ_ERR_MODE);
  if (int64_t(B) * H * (n / group) * D == 0) return IQ_OK;
  QuantOut o{v_codes, v_meta, t_cap / group, t_off, codes_i32, (uint16_t*)scale16, (uint16_t*)zero16,
             (uint16_t*)signs16};
  const int dp = (D + 1) / 2;
  const detail::VArgs a{(const uint16_t*)x, sx_b, sx_h, sx_t, H, n, D, dp,
          D % 2 == 0 && aligned(x, 4) && sx_b % 2 == 0 && sx_h % 2 == 0 && sx_t % 2 == 0,
          int64_t(B) * H * (n / group) * dp};
  if (group <= 64 && mode != IQ_MODE_HYBRID && int64_t(B) * H * n * D <= lane_values(group, bf, dense))
    return detail::quantize_v_lanes(a, o, int64_t(B) * H, group, bits, mode, bf, (hipStream_t)stream);
  return bf ? detail::quantize_v_bf16(a, o, group, bits, mode, dense, (hipStream_t)stream)
            : detail::quantize_v_f16(a, o, group, bits, mode, dense, (hipStream_t)stream);
}

}  // extern "C"
