// bf16 ring kernels that cut the tiles of a part-filled last round along K.
#include "gemm_kernel.h"

namespace fmoe {

template <int EPI, bool WTR>
static int launch(const GemmParams& p, hipStream_t stream) {
    const bool tail = p.K % 64 || p.E > TileRing5::kMaxExperts;
    if constexpr (WTR) {
        if (tail) return launch_ring_cfg<RingSplitCfg<4>, false, EPI, true, false, false, false, true>(p, stream);
        return launch_ring_cfg<RingSplitCfg<1>, false, EPI, true>(p, stream);
    }
    return tail ? launch_ring_bf16<RingSplitCfg<4>, EPI, true>(p, stream) : launch_ring_bf16<RingSplitCfg<1>, EPI>(p, stream);
}

template <int EPI>
static int launch(const GemmParams& p, hipStream_t stream) {
    return p.b_sn == 1 && p.b_sk != 1 ? launch<EPI, true>(p, stream) : launch<EPI, false>(p, stream);
}

int run_ring_split_bf16(const GemmParams& p, int epilogue, hipStream_t stream) {
    switch (epilogue) {
        case FMOE_EPI_NONE: return launch<FMOE_EPI_NONE>(p, stream);
        case FMOE_EPI_SILU: return launch<FMOE_EPI_SILU>(p, stream);
        case FMOE_EPI_SWIGLU: return launch<FMOE_EPI_SWIGLU>(p, stream);
    }
    return fail(FMOE_ERR_ARGUMENT, "fmoe_grouped_gemm: unknown epilogue %d", epilogue);
}

}  // namespace fmoe
