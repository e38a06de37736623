// sc_ctx.hip -- k_mlp_context for one output mode and tile size (built with
// -DSC_CTX_MODE=0: int8 logits, 1: int32 CDF tables; -DSC_CTX_RT=1..4: tiles
// of 32 * SC_CTX_RT rows).
#include "sc_kernels.h"

#if !defined(SC_CTX_MODE) || !defined(SC_CTX_RT)
#error "build with -DSC_CTX_MODE=0 or 1 and -DSC_CTX_RT=1..4"
#endif

namespace sc {

template <>
void launch_mlp_context<SC_CTX_MODE, SC_CTX_RT>(const ModelDev &M, unsigned grid, hipStream_t s, const int64_t *ctx,
                                                int64_t rows, int8_t *logits, int32_t *cdf, int32_t *status) {
    auto *kern = M.pipe == CORE_PIPE_UNI ? k_mlp_context<SC_CTX_MODE, CORE_PIPE_UNI, SC_CTX_RT>
                 : M.pipe == CORE_PIPE   ? k_mlp_context<SC_CTX_MODE, CORE_PIPE, SC_CTX_RT>
                                         : k_mlp_context<SC_CTX_MODE, CORE_PLAIN, SC_CTX_RT>;
    hipLaunchKernelGGL(kern, dim3(grid), dim3(THREADS), 0, s, M, ctx, rows, logits, cdf, status);
}

}  // namespace sc
