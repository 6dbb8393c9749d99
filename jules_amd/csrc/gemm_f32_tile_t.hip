// gemm_f32_tile_t.hip - the fp32 MFMA GEMM tiles with a transposed operand.
#include "gemm_f32_kernel.hpp"

namespace jh {

void launch_f32_tile_trans(int plan, int v, const F32Gemm& g, int splits, int kc, int chunk, float* part, hipStream_t s) {
    if (!g.tb) launch_f32_tile<true, false>(plan, v, g, splits, kc, chunk, part, s);
    else if (!g.ta) launch_f32_tile<false, true>(plan, v, g, splits, kc, chunk, part, s);
    else launch_f32_tile<true, true>(plan, v, g, splits, kc, chunk, part, s);
}

}  // namespace jh
