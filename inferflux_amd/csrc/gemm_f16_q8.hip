// gemm_f16_q8.hip -- the Q8_0 instances of the prefill GEMM (gemm_f16.h).
#include "gemm_f16.h"

namespace ifx {

hipError_t launch_gemm_f16_q8(int tile, bool ah, const F16Args &g, int grid, hipStream_t s) {
  return ah ? launch_by_tile<kTypeQ8_0, true>(tile, g, grid, s)
            : launch_by_tile<kTypeQ8_0, false>(tile, g, grid, s);
}

}  // namespace ifx
