// Host side of the grouped GEMM: tile configurations, kernel choice, launches.
#pragma once

#include "gemm_ring.h"
#include "gemm_staged.h"
#include "gemm_stream.h"

namespace fmoe {

// ------------------------------------------------------------------- host side
typedef TileCfg<256, 256, 2, 4> TileBig;        // 8 waves, wave tile 128 x 64
typedef TileCfg<64, 256, 1, 4> TileSmall;       // 4 waves, wave tile 64 x 64
typedef RingCfg<256, 256, 2, 4, 0> TileRing4;   // 8 waves, wave tile 128 x 64, 4-slot ring, LDS tables
typedef RingCfg<256, 256, 2, 4, 1> TileRing5;   // 5-slot ring, paired slices, E <= 64
// The plain forward calls take TileRing5F.  A build with -DFMOE_RING_NARROW gives them 256 x 128 tiles
// of 4 waves (one wave per SIMD, half the accumulator footprint per CU) instead: a measurement
// variant, kept so that the comparison can be repeated; 16-25 % slower than the 8-wave tile.
#ifdef FMOE_RING_NARROW
typedef RingCfg<256, 128, 2, 2, 1> TileRing5F;
#else
typedef TileRing5 TileRing5F;
#endif
typedef RingCfg<256, 256, 2, 4, 2> TileRing5M;  // 5-slot ring, paired slices, E <= 128 (the plain forward calls)
typedef RingCfg<256, 256, 2, 4, 4> TileRing5W;  // 5-slot ring, paired slices, E <= 256
typedef RingCfg<64, 256, 1, 4, 4, 3> TileRingS; // 4 waves, wave tile 64 x 64, 7 slots of 20 KB, E <= 256

enum GemmKernelSel { kSelRing = 0, kSelStagedBig = 1, kSelStagedSmall = 2, kSelGeneric = 3 };

template <typename Kern>
int reserve_lds(Kern kern, int bytes, bool& done) {
    if (done) return FMOE_OK;
    hipError_t err = hipFuncSetAttribute(reinterpret_cast<const void*>(kern),
                                         hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
    if (err != hipSuccess)
        return fail(FMOE_ERR_LAUNCH, "fmoe_grouped_gemm: cannot reserve %d B of LDS: %s", bytes,
                    hipGetErrorString(err));
    done = true;
    return FMOE_OK;
}

// one block per tile of TL, the grid an upper bound of their number
template <typename TL, typename Kern>
int launch_tiles(Kern kern, const GemmParams& p, bool& attr_done, hipStream_t stream) {
    if (int rc = reserve_lds(kern, TL::LDS_BYTES, attr_done)) return rc;
    const int64_t max_m_tiles = p.total_rows / TL::BM + p.E;
    const int64_t max_tiles = max_m_tiles * p.n_tiles;
    int64_t grid = (max_tiles + kNumXcd - 1) / kNumXcd * kNumXcd;
    if (p.k_window) {      // whole groups of kGroupM row tiles per XCD, round-robin
        const int64_t groups = (max_m_tiles + kGroupM - 1) / kGroupM;
        grid = (groups + kNumXcd - 1) / kNumXcd * kNumXcd * kGroupM * p.n_tiles;
    }
    if (grid >= ((int64_t)1 << 31)) return fail(FMOE_ERR_UNSUPPORTED, "fmoe_grouped_gemm: grid too large");
    kern<<<(unsigned)grid, TL::NT, TL::LDS_BYTES, stream>>>(p);
    return check_launch("fmoe_grouped_gemm");
}

template <typename TL, int DT, int EPI, int LOADS, bool A_SILU>
int launch_gemm(GemmParams p, hipStream_t stream) {
    constexpr int bn_out = EPI == FMOE_EPI_SWIGLU ? TL::BN / 2 : TL::BN;
    p.n_tiles = (p.N + bn_out - 1) / bn_out;
    auto kern = grouped_gemm_kernel<TL, DT, EPI, LOADS, A_SILU>;
    static bool attr_done = false;
    return launch_tiles<TL>(kern, p, attr_done, stream);
}

int compute_units();   // CUs of the current device (gemm_api.hip)
int lds_per_block();   // largest LDS allocation of one block on the current device (gemm_api.hip)

// the streaming kernel takes what the 64-row register-staged kernel takes with 16-byte loads, when
// the output can be stored 16 bytes at a time and no contraction window is set
inline bool stream_kernel_takes(const GemmParams& p) { return p.vec_store && !p.k_window && p.b_sk == 1; }

template <int DT, int EPI>
int launch_stream(GemmParams p, hipStream_t stream) {
    constexpr int bn_out = EPI == FMOE_EPI_SWIGLU ? 128 : 256;
    constexpr int lds_bytes = 2 * (64 + 256) * 128;
    p.n_tiles = (p.N + bn_out - 1) / bn_out;
    const int64_t max_tiles = (p.total_rows / 64 + p.E) * p.n_tiles;
    // two blocks per CU (80 KB of LDS each), a multiple of the XCD count; fewer when the launch is small
    int64_t grid = 2 * (int64_t)(compute_units() / kNumXcd * kNumXcd);
    if (grid < kNumXcd) grid = kNumXcd;
    const int64_t need = (max_tiles + kNumXcd - 1) / kNumXcd * kNumXcd;
    if (need < grid) grid = need;
    auto go = [&](auto kern, bool& attr_done) -> int {
        if (int rc = reserve_lds(kern, lds_bytes, attr_done)) return rc;
        kern<<<(unsigned)grid, 256, lds_bytes, stream>>>(p);
        return check_launch("fmoe_grouped_gemm");
    };
    if constexpr (DT == kDtE4m3) {
        if (p.scale_pow2) {
            static bool done_msc = false;
            return go(grouped_gemm_stream_kernel<DT, EPI, true>, done_msc);
        }
    }
    static bool done = false;
    return go(grouped_gemm_stream_kernel<DT, EPI, false>, done);
}

template <typename TL, bool FP8, int EPI, bool WTR = false, bool KWIN = false, bool XTR = false, bool MSC = false,
          bool KTAIL = false>
int launch_ring_cfg(GemmParams p, hipStream_t stream) {
    constexpr int bn_out = EPI == FMOE_EPI_SWIGLU ? TL::BN / 2 : TL::BN;
    p.n_tiles = (p.N + bn_out - 1) / bn_out;
    if (TL::PAIR) {
        // (tile numbers run up to the row tiles rounded up to a round of kNumXcd groups)
        if ((p.total_rows / TL::BM + p.E + (kNumXcd + 1) * kGroupM) * (int64_t)p.n_tiles >= ((int64_t)1 << 31))
            return fail(FMOE_ERR_UNSUPPORTED, "fmoe_grouped_gemm: more than 2^31 output tiles");
        magic_u31((int64_t)kGroupM * p.n_tiles, &p.group_magic, &p.group_magic_shift);
        // A tile that runs the shortened main loop gets ahead of the tiles of its group, which read
        // the same weights, by about 0.2 us per K-slice; a line lives about 10 us in an XCD's L2.
        // Up to 64 slices the group keeps sharing its fills and the shortened loop pays (forward
        // GEMMs of 64 experts -0.6 %, e4m3 at 128 experts -2.4 %); with 128 slices (K = 4096 in bf16,
        // 2048 rows per expert) the fills it breaks cost more than it saves (GEMM1 +1.8 %).
        // With two row tiles or fewer per expert on average there is little sharing to break, and the
        // second tile of most experts is a short one: the shortened loop stays on whatever K is.
        p.short_tile_rows = (p.K / (FP8 ? 64 : 32) <= 64 || p.total_rows / p.E <= 2 * TL::BM) ? TL::BM / 2 : 0;
    }
    auto kern = grouped_gemm_ring_kernel<TL, FP8, EPI, WTR, KWIN, XTR, MSC, KTAIL>;
    static bool attr_done = false;
    if (int rc = reserve_lds(kern, TL::LDS_BYTES, attr_done)) return rc;
    // persistent: one block per CU (the LDS footprint admits no second one), a multiple of
    // the XCD count so that every XCD owns the same number of blocks
    int grid = compute_units() / kNumXcd * kNumXcd;
    if (grid < kNumXcd) grid = kNumXcd;
    if (TL::BM < 256) {     // few rows: often fewer tiles than CUs
        const int64_t need = ((p.total_rows / TL::BM + p.E) * p.n_tiles + kNumXcd - 1) / kNumXcd * kNumXcd;
        if (need < grid) grid = (int)need;
    }
    kern<<<(unsigned)grid, TL::NT, TL::LDS_BYTES, stream>>>(p);
    if constexpr (TL::KSPLIT) split_reduce_kernel<FP8, EPI, MSC><<<8 * kSplitMost, 256, 0, stream>>>(p);
    return check_launch("fmoe_grouped_gemm");
}

// Ring kernels that cut the tiles of a part-filled last round along K (gemm_bf16_split.hip, gemm_fp8_split.hip).
int run_ring_split_bf16(const GemmParams& p, int epilogue, hipStream_t stream);
int run_ring_split_fp8(const GemmParams& p, int epilogue, hipStream_t stream);

// Ring kernels for K that is no whole number of K-slice pairs (gemm_bf16_tail.hip, gemm_fp8_tail.hip).
int run_ring_tail_bf16(const GemmParams& p, int epilogue, hipStream_t stream);
int run_ring_tail_fp8(const GemmParams& p, int epilogue, hipStream_t stream);

// What they take beyond the ring's own conditions: at least one pair of slices and a 16-byte chunk (8 bytes of e4m3).  On 9189 rows,
// 12 experts, 1000 <-> 2600 columns: weights with n contiguous 85 us per GEMM where the element-load kernel took 1368 and 1620;
// weights with k contiguous 94 us against 99 on the register-staged kernel.
constexpr int kRingTailChunk = 8;       // elements: 16 bytes of bf16, 8 of e4m3
inline bool ring_tail_takes(int esize, int64_t k, int num_experts, int64_t total_rows) {
    const int pair = 128 / esize, chunk = kRingTailChunk;
    return k > pair && k % pair != 0 && k % chunk == 0 && num_experts <= TileRing5W::kMaxExperts &&
           total_rows < ((int64_t)1 << 31) && lds_per_block() >= TileRing5W::LDS_BYTES;
}

// An odd number of whole slices is the 4-slot ring's as well, where it costs no half-empty pair but every slice comes as half
// lines.  us per GEMM, 4-slot ring / tail kernel, K in slices:
//   8192 rows, 8 experts, 1024 columns (one round of tiles)  bf16 3: 10.5 / 12.1   9: 14.5 / 15.1   17: 20.3 / 19.4
//                                                           e4m3 3: 11.7 / 12.9   9: 15.9 / 16.4   17: 21.1 / 20.8
//   16384 rows, 64 experts, 1408 columns (several)           bf16 3: 22.8 / 24.7   5: 26.9 / 27.4    7: 31.7 / 31.1
// Scales divided out in the epilogue (no powers of two) leave the e4m3 tail kernel short of registers:
//   one round  17: 21.3 / 21.6   21: 23.8 / 23.6        several  9: 39.7 / 39.8   17: 57.4 / 54.3
inline bool ring_tail_pays(const GemmParams& p, int esize, int epilogue) {
    const int slice = 64 / esize, bn_out = epilogue == FMOE_EPI_SWIGLU ? 128 : 256;
    if (p.K % slice || p.b_sk != 1) return true;
    const bool rounds = p.total_rows / 256 * ((p.N + bn_out - 1) / bn_out) > compute_units();   // however the rows fall
    return p.K / slice >= (esize == 1 && !p.scale_pow2 ? (rounds ? 17 : 21) : (rounds ? 7 : 17));
}

// The ring on 64-row tiles (gemm_bf16_short.hip, gemm_fp8_short.hip): experts with a handful of rows.
int run_ring_short_bf16(const GemmParams& p, int epilogue, hipStream_t stream);
int run_ring_short_fp8(const GemmParams& p, int epilogue, hipStream_t stream);

inline bool ring_short_takes(int esize, int64_t k, int num_experts, int64_t total_rows) {
    const int pair = 128 / esize, chunk = kRingTailChunk;
    return k > (TileRingS::AHEAD - 1) * pair && k % chunk == 0 && num_experts <= TileRingS::kMaxExperts &&
           total_rows < ((int64_t)1 << 31) && lds_per_block() >= TileRingS::LDS_BYTES;
}

// Where it is taken although another kernel takes the call as well (weights with k contiguous; with n contiguous the other is
// the element-load kernel and the ring always the faster one).  Only the row count is known here, not how the experts share
// it, so the rule goes by bounds that hold for every load.  us per GEMM, the streaming kernel / the ring (GATED: the
// register-staged kernel / the ring):
//   * no more tiles than CUs, however the rows fall: the ring keeps 120 KB per CU in flight where a lone streaming block has 40.
//     138 rows, 32 experts, 1728 -> 2 x 576 SwiGLU  30.2 / 22.5 (e4m3 19.5 / 16.6); 162 rows, 21 experts, 3648 -> 576
//     49.9 / 30.1 (GATED 63.8 / 31.0)
//   * beyond that one block per CU pays for a part-filled second round, where two blocks per CU hold it in the first:
//     512 rows, 128 experts, 4096 -> 1536: nine tenths of the rows in one expert 108 / 135, uniform 307 / 291; 9000 rows, 100
//     experts, 4096 -> 2 x 512 230 / 238; Zipf 243 / 258; 1000 rows, 63 experts, 1792 -> 2 x 640 52.4 / 61.4.  With twelve
//     rounds it depends on the load still (8000 rows, 128 experts, 4096 -> 2 x 1536: uniform 659 / 647, Zipf 725 / 735).
//   * GATED: 64 rows, 8 experts, 4096 -> 11008 142 / 154; 64 rows, 128 experts, 4096 -> 1536 125 / 148; 4096 rows, 128 experts,
//     4096 -> 1536 uniform 341 / 323, Zipf 309 / 317.  With more than two rounds of tiles even if one expert had all rows, and
//     whole pairs of K-slices, the ring is ahead by 3 to 11 % for every load: 8000 rows, 128 experts, 4096 -> 1536 uniform
//     402 / 367, Zipf 413 / 384, one hot expert 389 / 370 (5000 rows, 60 experts, 1000 -> 2600, K in part: 132 / 147).
inline bool ring_short_pays(const GemmParams& p, int esize, int epilogue) {
    const int bn_out = epilogue == FMOE_EPI_SWIGLU ? TileRingS::BN / 2 : TileRingS::BN;
    const int64_t cus = compute_units(), n_tiles = (p.N + bn_out - 1) / bn_out;
    const int64_t experts = p.E < p.total_rows ? p.E : p.total_rows;       // that can hold a row
    if ((p.total_rows / TileRingS::BM + experts) * n_tiles <= cus) return true;
    return epilogue == FMOE_EPI_GATED && p.K % (128 / esize) == 0 &&
           (p.total_rows + TileRingS::BM - 1) / TileRingS::BM * n_tiles > 2 * cus;
}

// rows per expert, on average, from which the tall tiles (256 rows) are the rule
constexpr int kTallRows = 96;

// The streaming kernels that take the weights straight into registers (gemm_direct.hip).
int run_gemm_direct(const GemmParams& p, int dtype, int epilogue, bool a_silu, hipStream_t stream);

// row tiles of a launch at most, however the experts share the rows
inline int64_t most_row_tiles(int64_t rows, int64_t num_experts, int bm) {
    const int64_t experts = num_experts < rows ? num_experts : rows;        // that can hold a row
    return (rows - experts) / bm + experts;
}
inline int direct_columns(int n, bool swiglu) { return swiglu ? (n + 31) / 32 : (n + 63) / 64; }

// Where they are taken (weights with k contiguous, 16-byte loads, no gate).  The host knows the row count and not how the experts share it, so
// the rule goes by the most tiles it allows.  us per GEMM on weights that are in no cache, the kernel that runs otherwise (the 64-row or the tall
// ring, the streaming or a register-staged kernel) / this one; even load, "hot" with nine tenths of the rows in one expert:
//   * no more tiles than CUs, whatever the rows (beyond 16 per expert on average from rows of K of 513 bytes on, from 96 per expert on of 2
//     KB): the tile that others walk alone (64 x 256 or 256 x 256, K serial) is a quarter as wide or less and its K is shared by eight
//     waves.  1 row, 8 experts, 1024 -> 4096 12.2 / 7.6 (e4m3 10.0 / 5.8, fp32 30.3 / 12.7); 3 rows, 64 experts, 2048 -> 2 x 1408 26.5 / 12.9
//     (14.2 / 8.7, 93 / 25); 24 rows, 10 experts, 2112 -> 408 27.9 / 12.6 (15.9 / 6.5, 70 / 22); 64 rows, 4 experts, 4096 -> 4096 54.2 / 30.4, hot
//     55.3 / 36.4; 160 rows, 10 experts, 1024 -> 1024 16.9 / 9.7, hot 16.6 / 12.3; 207 rows, 4 experts, 1088 -> 1152 13.4 / 11.8; 256 rows, 4
//     experts, 4096 -> 1024 46.8 / 33.1; 3000 rows, 4 experts, 1024 -> 320 23.1 / 12.2 (e4m3 16.9 / 9.3)
//   * up to two per CU: e4m3, and rows of K up to 1664 bytes, with up to 16 rows per expert on average.  98 rows, 11 experts, 2496 -> 2 x
//     832 e4m3 27.8 / 17.5, hot 26.9 / 14.5; 832 -> 2496 bf16 17.0 / 12.9, hot 15.8 / 16.6.  With more rows the 64-row ring is ahead where one
//     expert is hot (500 rows, 8 experts, 2048 -> 2 x 1024 bf16 32.6 / 22.7, hot 30.1 / 33.8; e4m3 19.0 / 16.0, 18.1 / 21.4) until the tall ring's
//     are the tiles, which then are a sixteenth as many: 1000 rows, 8 experts, 2048 -> 2 x 512 39.2 / 20.8, hot 44.9 / 33.4 (e4m3 26.1 / 14.7, 28.7 /
//     20.9); 1000 rows, 4 experts, 1024 -> 1024 23.0 / 13.0, hot 23.1 / 19.4.
//   * few rows per expert on average, where a hot expert has few as well, bf16 and up to six tiles per CU: two.  60 rows, 32 experts, 2048 -> 2048
//     65 / 71, hot 28.5 / 20.3; 64 rows, 2048 -> 3072 98 / 78, hot 40.0 / 32.7; 2 rows, 128 experts, 4096 -> 2 x 1536 47.0 / 21.2.  Eight: 128 rows, 64
//     experts, 1024 -> 2048 50.7 / 49.4, hot 23.1 / 19.9; e4m3 30.2 / 35.6.  Four rows: 256 rows 50.7 / 49.9, hot 24.8 / 31.3.
//   * K in part (no whole number of 128 bytes), which the other kernels mask or pad: four rows per expert and 13 tiles per CU; 160 rows, 40
//     experts, 2440 -> 2 x 1024 105 / 79, hot 67 / 39; 256 rows, 64 experts, 2440 -> 2048 126 / 126, hot 71 / 61, -> 3072 200 / 189, hot 101 / 88; e4m3
//     2448 -> 3072 113 / 101, hot 52 / 44.  Eight rows and seven tiles, rows of K of 2000 bytes: 768 rows, 96 experts, 1000 -> 768 46.5 / 35.8, hot
//     33.5 / 24.6; e4m3 2448 59 / 45, hot 40 / 31.  Sixteen, not taken: 620 rows, 40 experts, 3240 -> 2 x 1024 139 / 115, hot 127 / 116.
//   * beyond, an even load would gain (512 rows, 128 experts, 4096 -> 2 x 1536 526 / 513, e4m3 278 / 274), but an expert with many rows
//     has its weights read from L2 for every 64 of them and every 32 columns: hot 238 / 288, e4m3 124 / 156.
//   * fp32 streams half as much weight for a product and the other kernel is the slower one: up to 16 rows per expert whatever the tiles, from
//     K = 1024 on, up to two per CU or up to four rows (512 rows, 128 experts, 4096 -> 2 x 1536 1384 / 1075, hot 571 / 530; 512 rows, 64 experts, 512
//     -> 2048, not taken, level where one expert is hot), but not K of two slices (gemm_f32.hip).  With more rows the other kernel's tiles
//     hold more of them: K from 1024 on and one tile per CU (320 rows, 8 experts, 1024 -> 512 40.0 / 17.6), K from 128 on in whole lines and one for two CUs (587 rows,
//     16 experts, 960 -> 128 29.0 / 16.0; 644 rows, 4 experts, 128 -> 448 8.7 / 7.2; 306 rows, 8 experts, 640 -> 2 x 128 31.7 / 14.3: 26
//     such calls, 1.13 to 2.2 times as fast).  K in part and below 128 would gain as well (300 rows, 8 experts, 100 -> 128 8.3 / 6.2, 260 -> 128 11.9 / 7.7, 600
//     -> 128 19.7 / 10.2): not taken, the tests of the other kernel's edges and of this line are at such K.  Between them both ways: 164 tiles, 192 -> 256 10.7 / 14.6, 147 tiles, 960 -> 448 38.2 / 19.3; more tiles:
//     4000 rows, 8 experts, 4096 -> 512, four per CU, 143 / 180.
inline bool direct_pays(const GemmParams& p, int esize, bool swiglu) {
    const int64_t experts = p.E < p.total_rows ? p.E : p.total_rows, cus = compute_units();
    const int64_t tiles = most_row_tiles(p.total_rows, p.E, 64) * direct_columns(p.N, swiglu);
    const bool few = p.total_rows <= 16 * experts, tall = p.total_rows / p.E >= kTallRows;
    if (esize == 4) {
        if (!few) return p.K >= 1024 ? tiles <= cus : p.K >= 128 && p.K % 32 == 0 && tiles <= cus / 2;
        return p.K > 64 && (p.K >= 1024 || tiles <= 2 * cus || p.total_rows <= 4 * experts);
    }
    const int row = p.K * esize;
    const int64_t rows = p.total_rows, E = p.E;
    if (few && (row % 128 ? (rows <= 4 * E && tiles <= 13 * cus) || (rows <= 8 * E && row >= 2000 && tiles <= 7 * cus)
                          : rows <= 2 * E && esize == 2 && tiles <= 6 * cus))
        return true;
    if (few) return tiles <= cus || (tiles <= 2 * cus && (esize == 1 || row <= 1664));
    return tall ? row >= 2048 && tiles <= 2 * cus : row > 512 && tiles <= cus;
}

// Where the tall ring cuts its last round of tiles along K, for a caller that brings the workspace: K long enough and the round, however the
// experts share the rows, empty enough that the model of split_pieces gains 8 us at its fullest.  Only the row count is known here: the least
// and the most tiles it allows have to lie in the same round.  us, whole tiles / cut: 16384 rows, 8 experts, 4096 -> 1024 (256 tiles and up
// to 28) 171 / 135; 2000 rows, 8 experts, 4096 -> 1024 70.4 / 39.6; 4000, 4096 -> 512 70.4 / 38.3; 8000 70.6 / 49.9; 6540 rows, 5 experts, 3584
// -> 2 x 1216, Zipf 160 / 122; 33000 rows, 16 experts, 4096 -> 1024 290 / 260.  Launches that may have fewer tiles than XCDs stay whole.
inline bool split_pays(const GemmParams& p, int esize, int epilogue) {
    const int bn = epilogue == FMOE_EPI_SWIGLU ? 128 : 256, pairs = (p.K * esize + 127) / 128;
    const int64_t blocks = compute_units() / kNumXcd * kNumXcd, n_tiles = (p.N + bn - 1) / bn;
    const int64_t least = (p.total_rows + 255) / 256 * n_tiles, most = most_row_tiles(p.total_rows, p.E, 256) * n_tiles;
    if (blocks < kNumXcd || blocks > kSplitMost || pairs < 4 || most < kNumXcd || most >= ((int64_t)1 << 30)) return false;
    const int64_t rounds = least / blocks, rest = most - rounds * blocks;
    if (rest >= blocks || rest < 1) return false;
    int cost;
    return split_pieces((int)rest, pairs, (int)blocks, &cost) > 1 && 10 * pairs - cost >= 80;
}

// ... and where it does so with a call that the few-tiles kernel takes as well (96 rows per expert and more): bf16, beyond one of that kernel's
// 64 x 64 tiles per CU, and for K of more than 3584.  us, few-tiles kernel / cut; of 130 such calls the mean and the extremes of the ratio, even
// load / hot: more tiles than CUs 1.31 (0.68 to 1.84) / 1.47 (0.95 to 1.82), 2000 rows, 8 experts, 4096 -> 512 34.2 / 33.3, hot 60.4 / 33.1; up to
// one per CU, K of 3904 and 4096 1.08 (0.86 to 1.36) / 1.05 (0.86 to 1.19), 766 rows, 6 experts, 3904 -> 640 32.3 / 26.6; of 1536 to 3072 0.87 (0.65 to
// 1.12) / 0.84 (0.66 to 0.99).  e4m3, 30 calls, 0.75 (0.65 to 0.97).
inline bool split_before_direct(const GemmParams& p, int esize, int epilogue) {
    return esize == 2 &&
           (p.K > 3584 || most_row_tiles(p.total_rows, p.E, 64) * direct_columns(p.N, epilogue == FMOE_EPI_SWIGLU) > compute_units());
}

// bf16 tall ring with k contiguous: whether a launch, row tiles halfway between the fewest and the most that the row count allows, draws the chip's power
// cap in its main loops.  There the lower draw of 16 x 16 x 32 MFMAs is worth 1 to 4 %; below it their finer issue between the LDS reads costs up to
// 12 %, and a tile's end costs more (the exchange of lane groups).  us, 32 x 32 x 16 / 16 x 16 x 32 on two cards, 8 experts unless stated:
//   plain   4096 rows, 1024 -> 1024 24.3 / 26.5, 2048 -> 1024 39.5 / 43.7    16384, 1024 -> 3072 100.6 / 100.7, 106.2 / 109.1, -> 4096 126.6 / 125.3,
//           132.7 / 136.1    32768, 1024 -> 3072 184.5 / 181.7, 192.6 / 193.9, -> 5120 313 / 311, 323 / 318, 512 -> 3072 105.4 / 104.8, 113.6 / 113.9
//           8192, 2048 -> 3072 93.1 / 92.9, 98.3 / 96.2, 4096 -> 1024 74.9 / 80.3    12288, 4096 -> 1024 90.9 / 89.5, 95.3 / 92.3, 2048 -> 1024 51.1 / 51.7
//           16384, 2048 -> 1024 86.1 / 88.4, -> 2048 136.7 / 136.5, 143.3 / 140.6, 4096 -> 1024 125.8 / 122.8, 128.9 / 124.2
//           24 experts, Zipf, 8192, 2048 -> 2048 88.0 / 89.1    12 experts, 9189, 1000 -> 1024 32.5 / 33.3, 2600 -> 2600 135.7 / 131.1, 142.2 / 134.4
//   SwiGLU  16384, 1024 -> 2 x 2048 131.7 / 132.5, 140.6 / 146.5    32768, 1024 -> 2 x 1536 188.8 / 187.4, 200.8 / 206.6, -> 2 x 2560 309 / 305, 321 / 325
//           16384, 2048 -> 2 x 1536 190.3 / 190.1, 197.5 / 204.1, -> 2 x 2048 241 / 239, 250 / 252    32768, 2048 -> 2 x 2560 577 / 564, 589 / 579
//           16384, 4096 -> 2 x 512 127.2 / 124.5, 130.4 / 125.5    8192, 4096 -> 2 x 512 75.9 / 81.8    65536, 512 -> 2 x 2048 288.9 / 294.9
//   K in part (the loop of 32 x 32 x 16 masks behind its loads)    9189 rows, 12 experts, 2600 -> 1000 68.8 / 67.9, 1000 -> 2600 66.5 / 66.0, 1000 -> 1024
//           33.0 / 34.2, 4104 -> 1024 97.0 / 95.9    16384, 8 experts, 2600 -> 1000 101.5 / 98.6, 1000 -> 2600 102.7 / 101.3, 1000 -> 1024 57.8 / 59.0, 520 ->
//           3000 84.0 / 84.7    SwiGLU 2600 -> 2 x 1296 229 / 219, 1000 -> 2 x 1296 102.7 / 102.6, -> 2 x 2496 187 / 189, 520 -> 2 x 1496 82.5 / 87.1
// So by CUs' worths of K: 3072 from K of 2048 on (SwiGLU 4096), 6000 (8192) below; K in part 1600 from 2048 (plain 768) on.
inline bool mfma16_pays(const GemmParams& p, bool swiglu, bool in_part) {
    const int bn = swiglu ? 128 : 256;
    const int need = in_part && p.K >= (swiglu ? 2048 : 768) ? 1600 : p.K >= (swiglu ? 4096 : 2048) ? 3072 : swiglu ? 8192 : 6000;
    const int64_t n_tiles = (p.N + bn - 1) / bn, least = (p.total_rows + 255) / 256, most = most_row_tiles(p.total_rows, p.E, 256);
    return (least + most) * n_tiles >= 2 * (int64_t)need * compute_units() / p.K && (!swiglu || p.K >= 1024);
}
template <typename TL, int EPI, bool KTAIL = false>
int launch_ring_bf16(const GemmParams& p, hipStream_t stream) {
    if (mfma16_pays(p, EPI == FMOE_EPI_SWIGLU, p.K % 64 != 0)) return launch_ring_cfg<Mfma16<TL>, false, EPI, false, false, false, false, KTAIL>(p, stream);
    return launch_ring_cfg<TL, false, EPI, false, false, false, false, KTAIL>(p, stream);
}

// The 5-slot ring needs every byte of a 160 KB LDS, an even number of K-slices per tile,
// row numbers that fit 32 bits and few enough experts for the register tables.
template <bool FP8, int EPI>
int launch_ring(const GemmParams& p, hipStream_t stream) {
    const int slices = p.K / (FP8 ? 64 : 32);
    const bool pair_ok = slices % 2 == 0 && slices >= 4 && p.total_rows < ((int64_t)1 << 31) &&
                         lds_per_block() >= TileRing5::LDS_BYTES;
    // contraction windows: only the paired ring follows them, and only whole pairs of slices
    const int pair_elems = FP8 ? 128 : 64;
    const bool window_ok = !p.k_window || (p.k_window_multiple >= pair_elems && p.k_window_multiple % pair_elems == 0);
    if (p.a_sk != 1) {                     // both operands row-indexed (the caller checked the rest)
        if constexpr (!FP8 && EPI == FMOE_EPI_NONE) {
            if (p.E <= TileRing5::kMaxExperts) return launch_ring_cfg<TileRing5, FP8, EPI, true, true, true>(p, stream);
            return launch_ring_cfg<TileRing5W, FP8, EPI, true, true, true>(p, stream);
        }
        return fail(FMOE_ERR_UNSUPPORTED, "fmoe_grouped_gemm: row-indexed operands need bf16 and no epilogue");
    }
    if (!p.k_window && ring_tail_takes(FP8 ? 1 : 2, p.K, p.E, p.total_rows) && ring_tail_pays(p, FP8 ? 1 : 2, EPI))
        return FP8 ? run_ring_tail_fp8(p, EPI, stream) : run_ring_tail_bf16(p, EPI, stream);
    if (p.b_sn == 1 && p.b_sk != 1) {      // N-contiguous weights in place (the caller checked pair_ok's terms)
        if constexpr (!FP8) {
            if (p.E <= TileRing5::kMaxExperts) return launch_ring_cfg<TileRing5, FP8, EPI, true>(p, stream);
            return launch_ring_cfg<TileRing5W, FP8, EPI, true>(p, stream);
        }
        return fail(FMOE_ERR_UNSUPPORTED, "fmoe_grouped_gemm: no in-place path for these weights");
    }
    if (p.k_window) {                      // built for the weight gradient: bf16, no epilogue
        if constexpr (!FP8 && EPI == FMOE_EPI_NONE) {
            if (pair_ok && window_ok && p.E <= TileRing5::kMaxExperts)
                return launch_ring_cfg<Mfma16<TileRing5>, FP8, EPI, false, true>(p, stream);
            if (pair_ok && window_ok && p.E <= TileRing5W::kMaxExperts)
                return launch_ring_cfg<Mfma16<TileRing5W>, FP8, EPI, false, true>(p, stream);
        }
        return launch_gemm<TileBig, FP8 ? kDtE4m3 : kDtBf16, EPI, kLoadChunks, false>(p, stream);
    }
    if constexpr (FP8) {                   // power-of-two scales: applied by the MFMAs (row numbers fit 31 bits: pair_ok)
        if (p.scale_pow2 && pair_ok && p.E <= TileRing5::kMaxExperts)
            return launch_ring_cfg<TileRing5F, FP8, EPI, false, false, false, true>(p, stream);
        if (p.scale_pow2 && pair_ok && p.E <= TileRing5M::kMaxExperts)
            return launch_ring_cfg<TileRing5M, FP8, EPI, false, false, false, true>(p, stream);
        if (p.scale_pow2 && pair_ok && p.E <= TileRing5W::kMaxExperts)
            return launch_ring_cfg<TileRing5W, FP8, EPI, false, false, false, true>(p, stream);
    }
    auto go = [&](auto tile) {
        typedef decltype(tile) TL;
        if constexpr (FP8) return launch_ring_cfg<TL, true, EPI>(p, stream);
        else return launch_ring_bf16<TL, EPI>(p, stream);
    };
    if (pair_ok && p.E <= TileRing5::kMaxExperts) return go(TileRing5F{});
    if (pair_ok && p.E <= TileRing5M::kMaxExperts) return go(TileRing5M{});
    if (pair_ok && p.E <= TileRing5W::kMaxExperts) return go(TileRing5W{});
    return launch_ring_cfg<TileRing4, FP8, EPI>(p, stream);
}

template <int DT, int EPI, bool A_SILU>
int dispatch_tile(const GemmParams& p, int sel, hipStream_t stream) {
    static_assert(DT != kDtF32, "fp32 operands choose among tiles of their own (gemm_f32.hip)");
    switch (sel) {
        case kSelRing:
            if constexpr (!A_SILU) return launch_ring<DT == kDtE4m3, EPI>(p, stream);
            else return launch_gemm<TileBig, DT, EPI, kLoadChunks, A_SILU>(p, stream);
        case kSelStagedBig: return launch_gemm<TileBig, DT, EPI, kLoadChunks, A_SILU>(p, stream);
        case kSelStagedSmall:
            if constexpr (!A_SILU) {
                if (p.ring_short)
                    return DT == kDtE4m3 ? run_ring_short_fp8(p, EPI, stream) : run_ring_short_bf16(p, EPI, stream);
            }
            if constexpr (!A_SILU && EPI != FMOE_EPI_GATED) {
                if (stream_kernel_takes(p)) return launch_stream<DT, EPI>(p, stream);
            }
            return launch_gemm<TileSmall, DT, EPI, kLoadChunks, A_SILU>(p, stream);
        default: return launch_gemm<TileSmall, DT, EPI, kLoadElements, A_SILU>(p, stream);
    }
}

// Entry points of the translation units (one per operand type).
int run_gemm_bf16(GemmParams& p, int epilogue, bool a_silu, int sel, hipStream_t stream);
int run_gemm_fp8(GemmParams& p, int epilogue, int sel, hipStream_t stream);
int run_gemm_f32(GemmParams& p, int epilogue, bool a_silu, int sel, hipStream_t stream);
// workspace of a prepared fp32 call whose last round is cut along K, 0: none is
size_t gemm_f32_split_bytes(const GemmParams& p, int epilogue, bool a_silu, int sel);
inline int split_blocks() { return compute_units() / kNumXcd * kNumXcd; }

}  // namespace fmoe
