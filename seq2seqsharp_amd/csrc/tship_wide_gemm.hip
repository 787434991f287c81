// The other widths of the 256-row prefill GEMM tile (big_gemm3_f16_kernel with 128, 192 and 320 columns) in a translation unit
// of their own: it compiles beside tship_gpt.hip instead of behind it.
#include "tship_gpt_kernels.h"

namespace tship {

template <int NJ>
static WideGemm wide_gemm_of(int epi) {
    const BigKernel k = epi == BEPI_F32_BIAS ? big_gemm3_f16_kernel<BEPI_F32_BIAS, NJ> : epi == BEPI_RESID ? big_gemm3_f16_kernel<BEPI_RESID, NJ> : big_gemm3_f16_kernel<BEPI_ACT16, NJ>;
    return {k, 2 * NJ, BigShape<NJ>::SHM};
}
WideGemm wide_gemm(int tile, int epi) {
    if (tile == 42) return wide_gemm_of<2>(epi);
    if (tile == 43) return wide_gemm_of<3>(epi);
    if (tile == 45) return wide_gemm_of<5>(epi);
    throw Error("internal: no such width of the 256-row tile");
}

}  // namespace tship
