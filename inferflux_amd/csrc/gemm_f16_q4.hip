// gemm_f16_q4.hip -- the Q4_K instances of the prefill GEMM (gemm_f16.h).
#include "gemm_f16.h"

namespace ifx {

hipError_t launch_gemm_f16_q4(int tile, bool ah, const F16Args &g, int grid, hipStream_t s) {
  return ah ? launch_by_tile<kTypeQ4_K, true>(tile, g, grid, s)
            : launch_by_tile<kTypeQ4_K, false>(tile, g, grid, s);
}

}  // namespace ifx
