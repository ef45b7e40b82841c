// e4m3 ring kernels on 64-row tiles: experts with a handful of rows.
#include "gemm_kernel.h"

namespace fmoe {

template <int EPI, bool KTAIL>
static int launch(const GemmParams& p, hipStream_t stream) {
    if (p.scale_pow2) return launch_ring_cfg<TileRingS, true, EPI, false, false, false, true, KTAIL>(p, stream);
    return launch_ring_cfg<TileRingS, true, EPI, false, false, false, false, KTAIL>(p, stream);
}

template <int EPI>
static int launch(const GemmParams& p, hipStream_t stream) {
    return p.K % 128 ? launch<EPI, true>(p, stream) : launch<EPI, false>(p, stream);
}

int run_ring_short_fp8(const GemmParams& p, int epilogue, hipStream_t stream) {
    switch (epilogue) {
        case FMOE_EPI_NONE: return launch<FMOE_EPI_NONE>(p, stream);
        case FMOE_EPI_SILU: return launch<FMOE_EPI_SILU>(p, stream);
        case FMOE_EPI_SWIGLU: return launch<FMOE_EPI_SWIGLU>(p, stream);
    }
    return fail(FMOE_ERR_ARGUMENT, "fmoe_grouped_gemm: unknown epilogue %d", epilogue);
}

}  // namespace fmoe
