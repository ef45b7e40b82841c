// fp32 instantiations of the jagged GEMM (fp32 operands, bias and output).  Serves the fp32 cases of the reference's operator tests
// and fp32 FastMoELayer: on the bf16 matrix cores with every value in three parts (gemm_f32x3.h), and, where K is short or the
// strides allow no 16-byte loads, with v_mfma_f32_32x32x2_f32 on the register-staged kernel.
#include "gemm_f32x3.h"
#include "gemm_kernel.h"

namespace fmoe {

namespace {

// The tiles of v_mfma_f32_32x32x2_f32, for K of up to 64: a tile is the latency of one or two slices and its stores.  us per GEMM at K = 32 (64),
// tiles of 64 x 64 / 64 x 128 / 64 x 256, and 256 x 256 for comparison:
//   1000 rows, 8 experts, 1024 columns    6.8 /  8.7 / 11.0   19.6    (7.7 / 10.1 / 13.4    27.3)
//   4096 rows, 8 experts, 1024           11.9 / 11.9 / 13.1   22.4   (14.3 / 14.5 / 15.9    30.3)
//   4096 rows, 1 expert,  4096           33.0 / 31.5 / 31.2   43.3   (42.0 / 40.1 / 39.9    52.1)
//   600 rows, 64 experts, 4096           29.7 / 28.7 / 22.8   57.3   (38.5 / 39.0 / 32.6    87.7)
//   65536 rows, 16 experts, 64           11.4 / 17.9 / 25.7   22.4   (13.9 / 22.1 / 34.3    31.1)
//   SwiGLU (gate and up fragments in one wave: not 64 x 64): 4096 rows, 8 experts, 256  - / 8.8 / 11.7, 1024 - / 19.4 / 17.2; 600 rows, 64 experts,
//   1024  - / 16.7 / 12.4; 2000 rows, 200 experts, 256  - / 20.6 / 14.4
// So small tiles up to four 64 x 128 ones to a CU (SwiGLU: those up to two to a CU), the wide ones beyond, where they are not half empty.  With
// SiLU on load the same.  With n-contiguous weights, whose parking costs four LDS writes a chunk, the small ones (four to seven blocks per CU).
typedef TileCfg<64, 128, 2, 2> TileF32Wide;     // 4 waves, wave tile 32 x 64
typedef TileCfg<64, 64, 2, 2> TileF32;          // 4 waves, wave tile 32 x 32

template <int EPI, int LOADS, bool A_SILU>
int pick_tile(const GemmParams& p, hipStream_t stream) {
    constexpr bool swiglu = EPI == FMOE_EPI_SWIGLU;
    if constexpr (LOADS == kLoadChunks) {
        constexpr int columns = swiglu ? TileF32Wide::BN / 2 : TileF32Wide::BN;
        const int64_t tiles = (p.total_rows / TileF32Wide::BM + p.E) * ((p.N + columns - 1) / columns);
        if (tiles > (swiglu ? 2 : 4) * (int64_t)compute_units() && p.N > 64)
            return launch_gemm<TileSmall, kDtF32, EPI, LOADS, A_SILU>(p, stream);
    }
    return launch_gemm<std::conditional_t<swiglu, TileF32Wide, TileF32>, kDtF32, EPI, LOADS, A_SILU>(p, stream);
}

template <typename TL, int EPI, bool NCONT, bool A_SILU>
int launch_f32x3(GemmParams p, hipStream_t stream) {
    constexpr int bn_out = EPI == FMOE_EPI_SWIGLU ? TL::BN / 2 : TL::BN;
    p.n_tiles = (p.N + bn_out - 1) / bn_out;
    auto kern = grouped_gemm_f32x3_kernel<TL, EPI, NCONT, A_SILU>;
    static bool attr_done = false;
    if (!TL::template kCut<EPI == FMOE_EPI_SWIGLU> || !p.split_ws) return launch_tiles<TL>(kern, p, attr_done, stream);
    if (int rc = reserve_lds(kern, TL::LDS_BYTES, attr_done)) return rc;
    const int64_t blocks = split_blocks(), rounds = most_row_tiles(p.total_rows, p.E, TL::BM) * p.n_tiles / blocks;
    p.split_slots = (int)blocks / kNumXcd;
    kern<<<(unsigned)((rounds + 2) * blocks), TL::NT, TL::LDS_BYTES, stream>>>(p);      // (up to two pieces to a CU)
    constexpr int waves = TL::BM * bn_out / 1024;                                       // of a cut tile
    f32x3_reduce_kernel<TL, EPI><<<(unsigned)((blocks * waves + 3) / 4), 256, 0, stream>>>(p);
    return check_launch("fmoe_grouped_gemm");
}

// Whether a call's last round is cut along K: the tiles of BM x 128 it leaves, halfway between the fewest and the most that the row count allows (which
// lie in one round of one per CU or the next), cost less as pieces by 8 us at least.
//   * not behind a single round: its tiles run one to a CU, at seven eighths of the rate of two, until the pieces join them.  4096 rows, 8 experts,
//     4096 -> 1024 (64 x 128 tiles instead) 320 / 341, 3000 rows, 5 experts, 2048 -> 2048 184 / 189; a few gain (4 experts, 1000 rows, 2048 -> 4096 162 / 155)
//   * less than a round, from 5/8 of one on, all of it as pieces, two or three to a CU: 3000 rows, 4 experts, 4096 -> 1024, hot 256 / 201; 1000 rows,
//     4 experts, 4096 -> 2560 206 / 196, 4096 -> 2 x 1280 207 / 193
//   * 64 x 128 tiles behind two whole rounds, the pieces as third blocks (behind one, three and four 12 calls, gate and Zipf loads, are level, 0.99 to
//     1.013: 5000 rows, 8 experts, 4096 -> 1280 379 / 384, 2300 rows, 10 experts, 1024 -> 2560 106 / 105).  An even load that leaves no tile pays for
//     the second launch, which takes 4 us to find that: 4096 rows, 8 experts, 4096 -> 1024 238 / 246, 1024 -> 4096 230 / 233
// From six pairs of slices on (K of 321): 8192 rows, 8 experts, 324 -> 1024 72.9 / 62.6, 384 76.1 / 64.9, 504 98.2 / 79.3; 16384 rows, 384 -> 1024 121 / 110;
// 24 experts, 8000 rows, 480 -> 1024 89.8 / 82.1; SwiGLU, 8192 rows, 416 -> 2 x 1024 129 / 120.
template <int BM>
bool f32x3_split_pays(const GemmParams& p, bool swiglu) {
    const int bn_out = swiglu ? 64 : 128, pairs = (p.K + 63) / 64;
    const int64_t blocks = split_blocks(), n_tiles = (p.N + bn_out - 1) / bn_out;
    const int64_t least = (p.total_rows + BM - 1) / BM * n_tiles, most = most_row_tiles(p.total_rows, p.E, BM) * n_tiles;
    if (blocks < kNumXcd || blocks > kSplitMost || pairs < 4 || least < kNumXcd || most >= ((int64_t)1 << 30) ||
        p.total_rows >= ((int64_t)1 << 31))
        return false;
    const int64_t middle = (least + most) / 2, rounds = middle / blocks;
    if (most / blocks > least / blocks + 1) return false;
    if (BM == 64 ? rounds != 2 || least < 2 * blocks : rounds == 1 || (rounds == 0 && (most > blocks || 8 * least < 5 * blocks))) return false;
    const int rest = (int)(middle % blocks);
    int cost;
    return rest && f32x3_split_pieces<BM>(rest, pairs, (int)blocks, &cost) > 1 && (BM == 128 ? 36 : 18) * pairs - cost >= 72;
}

// From three slices on.  Up to two (K = 64) it is level or ahead too (4096 rows, 8 experts, 4096 columns, K = 32 30.6 / 27.4), but a third behind
// where many experts have a few rows each (2000 rows, 200 experts, 4096 columns, K = 64 108 / 157, SwiGLU 218 / 342).
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
bool f32x3_takes_large(const GemmParams& p, bool swiglu) {
    return p.total_rows / 128 * ((p.N * (swiglu ? 2 : 1) + 127) / 128) * 4 >= 5 * compute_units();
}
bool f32x3_takes_small(const GemmParams& p, bool a_silu) { return (p.total_rows / 64 + p.E) * ((p.N + 63) / 64) <= (a_silu ? 2 : 4) * compute_units(); }
bool f32x3_takes_mid(const GemmParams& p, bool a_silu) { return !f32x3_takes_large(p, false) && !f32x3_takes_small(p, a_silu); }

template <int EPI, bool NCONT, bool A_SILU>
int pick_f32x3(const GemmParams& p, hipStream_t stream) {
    constexpr bool swiglu = EPI == FMOE_EPI_SWIGLU;
    typedef TileF32x3<64, 128, swiglu ? 2 : 1, swiglu ? 2 : 4> Mid;
    typedef TileF32x3<64, 64, 2, 2> Small;
    if (p.split_ws ? f32x3_split_pays<128>(p, swiglu) : f32x3_takes_large(p, swiglu)) return launch_f32x3<TileF32Large, EPI, NCONT, A_SILU>(p, stream);
    if constexpr (!swiglu) {
        if (!p.split_ws && f32x3_takes_small(p, A_SILU)) return launch_f32x3<Small, EPI, NCONT, A_SILU>(p, stream);
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

size_t gemm_f32_split_bytes(const GemmParams& p, int epilogue, bool a_silu, int sel) {
    if (sel == kSelGeneric || p.K <= 2 * 32 || p.k_window || epilogue == FMOE_EPI_GATED) return 0;
    const bool swiglu = epilogue == FMOE_EPI_SWIGLU;
    const int bm = f32x3_split_pays<128>(p, swiglu) ? 128 : !swiglu && f32x3_takes_mid(p, a_silu) && f32x3_split_pays<64>(p, false) ? 64 : 0;
    return bm ? kSplitHeaderBytes + (size_t)(2 * split_blocks()) * f32x3_piece_bytes(bm) : 0;
}

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
