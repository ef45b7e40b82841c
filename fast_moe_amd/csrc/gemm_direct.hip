// Streaming kernels for a handful of rows per expert (bf16, e4m3, fp32).
#include "gemm_direct.h"
#include "gemm_kernel.h"

namespace fmoe {

// Eight waves to a tile up to one tile per CU: fewer pieces of K one after the other.  Four beyond: blocks that share a CU, and two
// pieces on their way per wave, stream better (us, 8 / 4: 4 rows, 6 experts, 1640 -> 2 x 1280 fp32 15.7 / 20.3, bf16 8.8 / 9.3;
// 512 rows, 128 experts, 1536 -> 4096 fp32 630 / 571).
template <int DT, int EPI, bool A_SILU, int NW>
static int launch(GemmParams p, hipStream_t stream) {
    typedef DirectCfg<DT, NW> CF;
    auto kern = grouped_gemm_direct_kernel<CF, DT, EPI, A_SILU>;
    static bool attr_done = false;
    if (int rc = reserve_lds(kern, CF::LDS_BYTES, attr_done)) return rc;
    const int64_t tiles = most_row_tiles(p.total_rows, p.E, CF::BM) * p.n_tiles;
    kern<<<(unsigned)((tiles + kNumXcd - 1) / kNumXcd * kNumXcd), CF::NT, CF::LDS_BYTES, stream>>>(p);
    return check_launch("fmoe_grouped_gemm");
}

template <int DT, int EPI, bool A_SILU>
static int launch(GemmParams p, hipStream_t stream) {
    p.n_tiles = direct_columns(p.N, EPI == FMOE_EPI_SWIGLU);
    if (most_row_tiles(p.total_rows, p.E, 64) * p.n_tiles <= compute_units()) return launch<DT, EPI, A_SILU, 8>(p, stream);
    return launch<DT, EPI, A_SILU, 4>(p, stream);
}

template <int DT>
static int launch(const GemmParams& p, int epilogue, bool a_silu, hipStream_t stream) {
    switch (epilogue) {
        case FMOE_EPI_NONE:
            if constexpr (DT != kDtE4m3) {
                if (a_silu) return launch<DT, FMOE_EPI_NONE, true>(p, stream);
            }
            return launch<DT, FMOE_EPI_NONE, false>(p, stream);
        case FMOE_EPI_SILU: return launch<DT, FMOE_EPI_SILU, false>(p, stream);
        case FMOE_EPI_SWIGLU: return launch<DT, FMOE_EPI_SWIGLU, false>(p, stream);
    }
    return fail(FMOE_ERR_ARGUMENT, "fmoe_grouped_gemm: unknown epilogue %d", epilogue);
}

int run_gemm_direct(const GemmParams& p, int dtype, int epilogue, bool a_silu, hipStream_t stream) {
    if (dtype == kDtBf16) return launch<kDtBf16>(p, epilogue, a_silu, stream);
    if (dtype == kDtE4m3) return launch<kDtE4m3>(p, epilogue, a_silu, stream);
    return launch<kDtF32>(p, epilogue, a_silu, stream);
}

}  // namespace fmoe
