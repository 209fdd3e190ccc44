// The many-row integer products with the GELU in their store (gemm_kernels.h).
#include "gemm_kernels.h"

namespace trit {
void gemm_gelu(const Layer& L, const GemvArgs& a, const GemmScratch& sc, hipStream_t s) {
    launch_product<true>(L, a, sc, s);
}
}  // namespace trit
