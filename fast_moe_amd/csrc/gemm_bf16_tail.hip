// bf16 ring kernels for contraction lengths that are no whole number of K-slice pairs.
#include "gemm_kernel.h"

namespace fmoe {

template <int EPI>
static int launch(const GemmParams& p, hipStream_t stream) {
    if (p.b_sn == 1 && p.b_sk != 1)
        return launch_ring_cfg<TileRing5W, false, EPI, true, false, false, false, true>(p, stream);
    return launch_ring_bf16<TileRing5W, EPI, true>(p, stream);
}

int run_ring_tail_bf16(const GemmParams& p, int epilogue, hipStream_t stream) {
    switch (epilogue) {
        case FMOE_EPI_NONE: return launch<FMOE_EPI_NONE>(p, stream);
        case FMOE_EPI_SILU: return launch<FMOE_EPI_SILU>(p, stream);
        case FMOE_EPI_SWIGLU: return launch<FMOE_EPI_SWIGLU>(p, stream);
        case FMOE_EPI_GATED: return launch<FMOE_EPI_GATED>(p, stream);
    }
    return fail(FMOE_ERR_ARGUMENT, "fmoe_grouped_gemm: unknown epilogue %d", epilogue);
}

}  // namespace fmoe
