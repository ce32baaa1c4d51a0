// Quantization of bf16 values, groups along tokens.
#include "iq_quantize_v.h"

int iq::detail::quantize_v_bf16(const VArgs& a, const QuantOut& o, int group, int bits, int mode, bool dense,
                                hipStream_t st) {
  return launch_quant_v<true>(a, o, group, bits, mode, dense, st);
}
