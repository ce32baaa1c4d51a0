// Instantiations of the fused flash-decoding kernel for 2-bit K and a V store of
// another group size (every V bit width, head_dim and query heads per KV head).
#include "iq_flash.h"

namespace iq::detail {

int flash_fused_launch_mg_k2(const FusedArgs& a, int vbits, int group, int D, int nrep, bool norm, int* grid,
                             hipStream_t stream, bool launch) {
  return fused_launch_mixed<2>(a, vbits, group, D, nrep, norm, grid, stream, launch);
}

}  // namespace iq::detail
