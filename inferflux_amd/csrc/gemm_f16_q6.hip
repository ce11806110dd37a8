// gemm_f16_q6.hip -- the Q6_K instances of the prefill GEMM (gemm_f16.h).
#include "gemm_f16.h"

namespace ifx {

hipError_t launch_gemm_f16_q6(int tile, bool ah, const F16Args &g, int grid, hipStream_t s) {
  return ah ? launch_by_tile<kTypeQ6_K, true>(tile, g, grid, s)
            : launch_by_tile<kTypeQ6_K, false>(tile, g, grid, s);
}

}  // namespace ifx
