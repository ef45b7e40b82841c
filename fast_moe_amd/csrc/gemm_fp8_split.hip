// e4m3 ring kernels that cut the tiles of a part-filled last round along K.
#include "gemm_kernel.h"

namespace fmoe {

// Whole pairs of slices and up to 64 experts (split_takes): the other instantiations keep more than the registers hold (17 to 24 spilled).
template <int EPI, bool MSC>
static int launch(const GemmParams& p, hipStream_t stream) {
    return launch_ring_cfg<RingSplitCfg<1>, true, EPI, false, false, false, MSC>(p, stream);
}

template <int EPI>
static int launch(const GemmParams& p, hipStream_t stream) {
    return p.scale_pow2 ? launch<EPI, true>(p, stream) : launch<EPI, false>(p, stream);
}

int run_ring_split_fp8(const GemmParams& p, int epilogue, hipStream_t stream) {
    switch (epilogue) {
        case FMOE_EPI_NONE: return launch<FMOE_EPI_NONE>(p, stream);
        case FMOE_EPI_SILU: return launch<FMOE_EPI_SILU>(p, stream);
        case FMOE_EPI_SWIGLU: return launch<FMOE_EPI_SWIGLU>(p, stream);
    }
    return fail(FMOE_ERR_ARGUMENT, "fmoe_grouped_gemm: unknown epilogue %d", epilogue);
}

}  // namespace fmoe
