// fp32 instantiations of the jagged GEMM (v_mfma_f32_32x32x2_f32: fp32 operands, bias and
// output).  Serves the fp32 cases of the reference's operator tests and fp32 FastMoELayer.
#include "gemm_kernel.h"

namespace fmoe {

namespace {

// An fp32 MFMA runs 64 cycles on operands of two LDS reads, so LDS and L2 bandwidth leave room for small tiles, and small
// tiles are what fills the chip: a launch is bound by the last round of tiles over 256 CUs (4096 rows, 8 experts,
// 4096 -> 1024 columns: 80 tiles of 256 x 256).  Several blocks share a CU and hide each other's barriers and epilogues.
// us per GEMM, tiles of 256 x 256 / 128 x 128 / 64 x 128 / 64 x 64:
//   4096 rows,  8 experts, 1024 -> 4096      554 /  391 /  339 /  335      (k contiguous)
//   4096 rows,  8 experts, 4096 -> 1024     1005 /  545 /  421 /  390
//   9189 rows, 12 experts, 2600 -> 1000      673 /  541 /  461 /  484
//  16384 rows,  8 experts, 1024 -> 4096     1371 / 1171 / 1172 / 1235
//     64 rows,  8 experts, 1024 -> 2048      254 /   81 /   50 /   33
typedef TileCfg<64, 128, 2, 2> TileF32Wide;     // 4 waves, wave tile 32 x 64
typedef TileCfg<64, 64, 2, 2> TileF32;          // 4 waves, wave tile 32 x 32

// From four wide tiles per CU on, the remainder of the last round is a small share and the 25 % fewer operand bytes of the
// wide tile count for more (1172 against 1235 us above); below, the finer tile fills the chip better (390 against 421).
// With n-contiguous weights, whose parking costs four LDS writes a chunk, the small tile was faster at every size (four to
// seven blocks per CU instead of three): 398 / 350, 527 / 413, 1425 / 1299 us for the first, second and fourth line.
// SwiGLU needs gate and up fragments in one wave: always wide.
template <int EPI, int LOADS, bool A_SILU>
int pick_tile(const GemmParams& p, hipStream_t stream) {
    if constexpr (EPI != FMOE_EPI_SWIGLU) {
        const int64_t wide = (p.total_rows / TileF32Wide::BM + p.E) * ((p.N + TileF32Wide::BN - 1) / TileF32Wide::BN);
        if (LOADS == kLoadChunksN || wide < 4 * (int64_t)compute_units())
            return launch_gemm<TileF32, kDtF32, EPI, LOADS, A_SILU>(p, stream);
    }
    if constexpr (EPI == FMOE_EPI_SWIGLU || LOADS != kLoadChunksN)
        return launch_gemm<TileF32Wide, kDtF32, EPI, LOADS, A_SILU>(p, stream);
}

template <int EPI, bool A_SILU>
int dispatch(const GemmParams& p, int sel, hipStream_t stream) {
    if (sel == kSelGeneric) return launch_gemm<TileSmall, kDtF32, EPI, kLoadElements, A_SILU>(p, stream);
    if (p.b_sk != 1) return pick_tile<EPI, kLoadChunksN, A_SILU>(p, stream);
    return pick_tile<EPI, kLoadChunks, A_SILU>(p, stream);
}

}  // namespace

int run_gemm_f32(GemmParams& p, int epilogue, bool a_silu, int sel, hipStream_t stream) {
    if (a_silu) {
        if (epilogue != FMOE_EPI_NONE)
            return fail(FMOE_ERR_UNSUPPORTED, "fmoe_grouped_gemm: a_silu is only built for the plain epilogue");
        return dispatch<FMOE_EPI_NONE, true>(p, sel, stream);
    }
    switch (epilogue) {
        case FMOE_EPI_NONE: return dispatch<FMOE_EPI_NONE, false>(p, sel, stream);
        case FMOE_EPI_SILU: return dispatch<FMOE_EPI_SILU, false>(p, sel, stream);
        case FMOE_EPI_SWIGLU: return dispatch<FMOE_EPI_SWIGLU, false>(p, sel, stream);
    }
    return fail(FMOE_ERR_ARGUMENT, "fmoe_grouped_gemm: unknown epilogue %d", epilogue);
}

}  // namespace fmoe
