// fp32 instantiations of the jagged GEMM (fp32 operands, bias and output).  Serves the fp32 cases of the reference's operator tests
// and fp32 FastMoELayer: on the bf16 matrix cores with every value in three parts (gemm_f32x3.h), and, where K is short or the
// strides allow no 16-byte loads, with v_mfma_f32_32x32x2_f32 on the register-staged kernel.
#include "gemm_f32x3.h"
#include "gemm_kernel.h"

namespace fmoe {

namespace {

// The tiles of v_mfma_f32_32x32x2_f32 (their figures are from before longer K went to the other kernel).
// It runs 64 cycles on operands of two LDS reads, so LDS and L2 bandwidth leave room for small tiles, and small
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
// wide tile count for more (1172 against 1235 us above); below, the finer tile fills the chip better (390 against 421).  With
// SiLU on load, which every column of tiles repeats, from one per CU on: 375 rows, 16 experts, 860 -> 3320 columns 91 / 107 us,
// 300 rows, 8 experts, 1024 -> 1024 80 / 61.
// With n-contiguous weights, whose parking costs four LDS writes a chunk, the small tile was faster at every size (four to
// seven blocks per CU instead of three): 398 / 350, 527 / 413, 1425 / 1299 us for the first, second and fourth line.
// SwiGLU needs gate and up fragments in one wave: wide, or 64 x 256 where that is one round of tiles (two blocks per CU) and
// wide more than one (three): 2000 rows, 200 experts, 256 -> 2 x 256 51.0 / 45.2 us.
//
// Whole rounds of 256 x 256 tiles, one block per CU, are faster still: a quarter of the operand reads and of the SiLU.  us,
// 256 x 256 / 64 x 128: 4096 rows, 1 expert, 4096 -> 4096 (one round) 1037 / 1123, SiLU on load 1241 / 1479; 8192 rows, 2048 -> 4096
// 1053 / 1123; but with 1056 tiles (65536 rows, 8 experts, 512 -> 1024: a fifth round of 32) 750 / 614.  The bound on the row
// tiles holds however the experts share the rows; 6 % (15 % with SiLU on load) is what an unfilled remainder may cost.
template <int EPI, int LOADS, bool A_SILU>
int pick_tile(const GemmParams& p, hipStream_t stream) {
    constexpr int out_cols = EPI == FMOE_EPI_SWIGLU ? 2 : 1;    // tile columns per output column
    const int64_t cus = compute_units();
    auto tiles = [&](int bm, int bn) { return (p.total_rows / bm + p.E) * ((p.N + bn / out_cols - 1) / (bn / out_cols)); };
    if constexpr (LOADS == kLoadChunks) {
        const int64_t most = (p.total_rows + 255 * (int64_t)p.E) / 256 * ((p.N + 256 / out_cols - 1) / (256 / out_cols));
        const double rounds = (double)((most + cus - 1) / cus * cus) * (256 * 256 / out_cols);
        if (rounds <= (A_SILU ? 1.15 : 1.06) * (double)p.total_rows * p.N)
            return launch_gemm<TileBig, kDtF32, EPI, LOADS, A_SILU>(p, stream);
        if constexpr (EPI == FMOE_EPI_SWIGLU) {
            if (tiles(TileF32Wide::BM, TileF32Wide::BN) > 3 * cus && tiles(TileSmall::BM, TileSmall::BN) <= 2 * cus)
                return launch_gemm<TileSmall, kDtF32, EPI, LOADS, A_SILU>(p, stream);
        }
    }
    if constexpr (EPI != FMOE_EPI_SWIGLU) {
        if (LOADS == kLoadChunksN || tiles(TileF32Wide::BM, TileF32Wide::BN) < (A_SILU ? 1 : 4) * cus)
            return launch_gemm<TileF32, kDtF32, EPI, LOADS, A_SILU>(p, stream);
    }
    if constexpr (EPI == FMOE_EPI_SWIGLU || LOADS != kLoadChunksN)
        return launch_gemm<TileF32Wide, kDtF32, EPI, LOADS, A_SILU>(p, stream);
}

template <typename TL, int EPI, bool NCONT, bool A_SILU>
int launch_f32x3(GemmParams p, hipStream_t stream) {
    constexpr int bn_out = EPI == FMOE_EPI_SWIGLU ? TL::BN / 2 : TL::BN;
    p.n_tiles = (p.N + bn_out - 1) / bn_out;
    auto kern = grouped_gemm_f32x3_kernel<TL, EPI, NCONT, A_SILU>;
    static bool attr_done = false;
    return launch_tiles<TL>(kern, p, attr_done, stream);
}

// From three slices on; up to two (K = 64) there is hardly a loop to be faster in (4096 rows, 8 experts, 512 columns, K = 72: 10.2 us on
// v_mfma_f32_32x32x2_f32, 9.6 here; SwiGLU, K = 68: 15.2 / 13.7).
//
// us per GEMM, v_mfma_f32_32x32x2_f32 on its best tile / three parts on 64 x 64 / 64 x 128 / 128 x 128:
//   4096 rows,  8 experts, 1024 -> 4096 columns  291 / 274 / 252 / 225        16384 rows  1130 / 1051 / 960 / 865
//   4096 rows,  8 experts, 4096 -> 1024          305 / 272 / 238 / 256        6000 rows, 10 experts, 1024 -> 1024  138 / 116 / 127 / 97
//   1000 rows, 32 experts,  512 -> 1024           26 /  24 /  27 /  38        2048 rows, 64 experts,  256 -> 1024   26 /  24 /  21 / 30
//   1600 rows, 32 experts,  512 -> 512             - /  19 /  26 /  39        512 rows, 8 experts, 128 -> 256      8.3 / 8.3 / 10.6 / 15.4
//   SwiGLU (not on 64 x 64): 4096 rows, 8 experts, 1024 -> 4096  577 / 507 / 446; 600 rows, 16 experts, 512 -> 2048  47 / 38 / 57
// 16384 rows are 159 TFLOP/s, 1270 of bf16 products: what the chip's power allows.
//   * 128 x 128 reads the least from LDS for a product: where the rows fill five such tiles for every four CUs.
//   * 64 x 64: up to four per CU however the rows fall (two with SiLU on load, which every column of tiles repeats).
template <int EPI, bool NCONT, bool A_SILU>
int pick_f32x3(const GemmParams& p, hipStream_t stream) {
    constexpr bool swiglu = EPI == FMOE_EPI_SWIGLU;     // its gate and up fragments share a wave
    typedef TileF32x3<128, 128, 2, 2> Large;            // wave tile 64 x 64
    typedef TileF32x3<64, 128, swiglu ? 2 : 1, swiglu ? 2 : 4> Mid;
    typedef TileF32x3<64, 64, 2, 2> Small;
    const int64_t cus = compute_units();
    auto columns = [&](int bn) { return (p.N * (swiglu ? 2 : 1) + bn - 1) / bn; };
    if (p.total_rows / 128 * columns(128) * 4 >= 5 * cus) return launch_f32x3<Large, EPI, NCONT, A_SILU>(p, stream);
    if constexpr (!swiglu) {
        if ((p.total_rows / 64 + p.E) * columns(64) <= (A_SILU ? 2 : 4) * cus) return launch_f32x3<Small, EPI, NCONT, A_SILU>(p, stream);
    }
    return launch_f32x3<Mid, EPI, NCONT, A_SILU>(p, stream);
}

template <int EPI, bool A_SILU>
int dispatch(const GemmParams& p, int sel, hipStream_t stream) {
    if (sel == kSelGeneric) return launch_gemm<TileSmall, kDtF32, EPI, kLoadElements, A_SILU>(p, stream);
    if (p.K > 2 * 32) return p.b_sk != 1 ? pick_f32x3<EPI, true, A_SILU>(p, stream) : pick_f32x3<EPI, false, A_SILU>(p, stream);
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
