// fp32 grouped GEMM on the bf16 matrix cores: every operand value is cut into three bf16 values on its way into LDS.
#pragma once

#include "gemm_staged.h"

namespace fmoe {

// x = h + m + l with h, m, l the bf16 roundings of x and of what the ones before it leave: 8 + 8 + 8 bits and the signs of the
// remainders cover the 24 of an fp32 value, so the sum is exact.  A product of two such values is taken as eight of its nine partial
// products; ll, which is left out, is at most 2^-34 of it (|l| <= 2^-17 of the power of two below |x|), a thousandth of what rounding the
// product to fp32 costs.  hh, exact in fp32, has an accumulator of its own; the other seven, 2^-7 of it, share a second one, and the two
// are added once, behind the contraction.  So a product is not rounded before it meets the sum, as in a fused multiply-add: with six
// products in one accumulator a row of a single product had twice the error of one.
//
// Both operands are multiplied by 2^24 first (and the sums by 2^-48 last), so that l of the smallest normal fp32 value is still a
// normal bf16 value.  That, and the rounding of h, overflows for |x| near 2^104 and sums near 2^80; an infinity or a NaN in an
// operand makes a NaN of the partial products as well.  A wave that finds a sum that is not finite computes its part of the tile
// again with v_mfma_f32_32x32x2_f32, straight from global memory: what comes out for such operands is what that instruction gives.
constexpr float kF32x3Scale = 16777216.0f, kF32x3Unscale = 0x1p-48f;

// The partial products: the weight's and the activation's part of each (0: h, 1: m, 2: l).  The first has an accumulator of its own.
#define FMOE_F32X3_TERMS constexpr int W[8] = {0, 1, 0, 1, 2, 0, 2, 1}, X[8] = {0, 0, 1, 1, 0, 2, 1, 2}

template <int BM_, int BN_, int WGM_, int WGN_>
struct TileF32x3 {
    static constexpr int BM = BM_, BN = BN_, WGM = WGM_, WGN = WGN_;
    static constexpr int NT = kWave * WGM * WGN;
    static constexpr int TM = BM / WGM, TN = BN / WGN;
    static constexpr int FM = TM / 32, FN = TN / 32;
    static constexpr int BK = 32;                           // k per slice: 64-byte rows in each of the three planes
    static constexpr int A_PLANE = BM * 64, B_PLANE = BN * 64;
    static constexpr int LDS_BYTES = 3 * (A_PLANE + B_PLANE);
    static_assert(TM % 32 == 0 && TN % 32 == 0, "wave tile must hold whole 32x32 fragments");
    static_assert((BM * 4) % NT == 0 && (BN * 4) % NT == 0, "loader passes must be whole");
    // the tiles whose last round is cut along K
    template <bool SWIGLU>
    static constexpr bool kCut = BN == 128 && (BM == 128 || !SWIGLU);
};

// Last round cut along K, as the tall ring's (gemm_split.h).  Two 128 x 128 tiles on a CU take 1.75 times as long as one, so a launch ends
// with the CUs that have one tile more.  The tiles beyond whole rounds of one per CU go out as pieces of K behind them; each leaves its sums in the
// workspace, f32x3_reduce_kernel adds them in the order of K.  us, whole tiles / cut: 8000 rows, 24 experts, 2048 -> 1024 353 / 280; 16000 rows, 20
// experts, 1536 -> 1024 403 / 347; 9189 rows, 12 experts, 2600 -> 1000 429 / 345, 1000 -> 2600 396 / 370; 4096 rows, 8 experts, 1024 -> 4096 284 / 266; 2500
// rows, 10 experts, 768 -> 3072 137 / 115; 4096 rows, 4 experts, 3072 -> 2048, hot 542 / 377; SwiGLU, 8192 rows, 8 experts, 2048 -> 2 x 2048 935 / 879.
// 64 x 128 tiles: 1, 2 and 3 on a CU take 154, 255 and 342 us (K = 4096); 4096 rows, 8 experts, 4096 -> 1024 329 / 274, 2048 -> 1024 167 / 142, 1536 ->
// 1024 with SiLU 131 / 114; 2100 rows, 5 experts, 2048 -> 2048 170 / 148.  The error against 64 bits is no larger, fewer terms meet in one chain of
// roundings: 8192 rows, 324 -> 1024 relative 1.00e-7 (uncut 1.01e-7), 4096 rows, 4096 -> 1024 3.94e-7 (3.97e-7); rows of three values 2.67e-8 (2.65e-8).
//
// Pieces of each of `rest` tiles of BM rows: two pairs of slices to a piece at least, and the shortest of this model in us / 9: a pair of slices takes
// 4 us (BM = 64: 2) of a lone block, 1.75 times that (2) with more pieces than CUs, 64 KB of sums 0.025 us of everybody's bandwidth, the second
// launch 6.
// Integers: host and device agree.
typedef TileF32x3<128, 128, 2, 2> TileF32Large;         // wave tile 64 x 64
template <int BM>
__host__ __device__ inline int f32x3_split_pieces(int rest, int pairs, int blocks, int* cost = nullptr) {
    constexpr int pair = BM == 128 ? 36 : 18, two = BM == 128 ? 7 : 8;
    int best = 1, least = pair * pairs;
    for (int s = 2; s * rest <= 2 * blocks && 2 * s <= pairs; ++s) {
        const int loop = (pair * pairs + s - 1) / s;
        const int c = (s * rest > blocks ? loop * two / 4 : loop) + rest * s * (BM / 64) / 9 + 54;
        if (c < least) {
            least = c;
            best = s;
        }
    }
    if (cost) *cost = least;
    return best;
}
constexpr int f32x3_piece_bytes(int bm) { return bm * 128 * 4; }
// a 32 x 32 block of a piece's sums, [quad][lane]
template <typename TL>
__device__ __forceinline__ f32x4* f32x3_sums(SplitWorkspace* ws, int piece, int row_block, int col_block) {
    return reinterpret_cast<f32x4*>(reinterpret_cast<uint8_t*>(ws) + kSplitHeaderBytes + (int64_t)piece * f32x3_piece_bytes(TL::BM)) +
           (row_block * (TL::BN / 32) + col_block) * 4 * kWave;
}

// Wave: 32 x 32 outputs of a cut tile.
template <typename TL, int EPI>
__global__ __launch_bounds__(256) void f32x3_reduce_kernel(const GemmParams p) {
    constexpr bool SWIGLU = EPI == FMOE_EPI_SWIGLU;
    constexpr int PARTS = SWIGLU ? 2 : 1, COLS = TL::BN / 32 / PARTS, BLOCKS = TL::BM / 32 * COLS;
    const int lane = threadIdx.x & 63, w = blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int t = w / BLOCKS, rb = w % BLOCKS / COLS, cb = w % COLS;
    const int tiles = p.split_ws->tiles, pieces = p.split_ws->pieces;
    if (t >= tiles) return;
    const SplitTile tile = p.split_ws->tile[t];
    if (rb * 32 >= tile.rows_valid) return;
    f32x16 acc[PARTS][1];
#pragma unroll
    for (int i = 0; i < PARTS; ++i)
#pragma unroll
        for (int v = 0; v < 16; ++v) acc[i][0][v] = 0.0f;
#pragma unroll 4
    for (int s = 0; s < pieces; ++s)
#pragma unroll
        for (int i = 0; i < PARTS; ++i) {
            const f32x4* const src = f32x3_sums<TL>(p.split_ws, s * tiles + t, rb, i * COLS + cb) + lane;
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                const f32x4 v = src[g * kWave];
#pragma unroll
                for (int j = 0; j < 4; ++j) acc[i][0][4 * g + j] += v[j];
            }
        }
    gemm_epilogue_f32<1, PARTS, 32, 32 * PARTS, EPI>(p, acc, tile.expert, tile.nt * (TL::BN / PARTS), tile.row0, tile.rows_valid, rb, cb, lane);
}

// Written out with packed operations on two values: 11 VALU instructions, which a block does once per operand value and slice.
__device__ __forceinline__ void split3(float a, float b, uint32_t& h, uint32_t& m, uint32_t& l) {
    h = cvt_pk_bf16(a, b);
    a -= __uint_as_float(h << 16);
    b -= __uint_as_float(h & 0xffff0000u);
    m = cvt_pk_bf16(a, b);
    a -= __uint_as_float(m << 16);
    b -= __uint_as_float(m & 0xffff0000u);
    l = cvt_pk_bf16(a, b);
}

// Register-staged: the next slice is loaded while one is multiplied, then cut into parts and parked in the one LDS buffer (48 KB
// for 128 x 128; its two accumulators leave registers for two blocks to a CU, which multiply in each other's barriers).
//
// The error against 64 bits: 2 roundings of the large sum per 32 k where v_mfma_f32_32x32x2_f32 has 16.  Here / that instruction, 2-norm
// over standard normal operands: 8.9e-8 / 2.87e-7 at K = 256, 1.86e-7 / 5.73e-7 at 1024, 3.96e-7 / 1.15e-6 at 4096.  Rows of 1, 2, 4, 16 and 64
// non-zero values of 1024: 2.53e-8 / 2.53e-8, 2.56e-8 / 3.09e-8, 2.63e-8 / 3.98e-8, 3.37e-8 / 7.39e-8, 5.6e-8 / 1.45e-7; largest, of sum |a||b|:
// 5.99e-8 / 5.96e-8, 1.40e-7 / 1.14e-7, 1.72e-7 / 1.84e-7, 1.8e-7 / 3.2e-7, 1.7e-7 / 3.8e-7.
//
// NCONT: weights whose n is contiguous.  They are parked as they come, [32 k][128 n] per plane, and read with ds_read_b64_tr_b16.
template <typename TL, int EPI, bool NCONT, bool A_SILU>
__global__ __launch_bounds__(TL::NT, 2) void grouped_gemm_f32x3_kernel(const GemmParams p) {
    constexpr int BM = TL::BM, BN = TL::BN, NT = TL::NT, BK = TL::BK;
    constexpr int FM = TL::FM, FN = TL::FN, TM = TL::TM, TN = TL::TN;
    constexpr bool SWIGLU = EPI == FMOE_EPI_SWIGLU, CUT = TL::template kCut<SWIGLU>;
    constexpr int BN_OUT = SWIGLU ? BN / 2 : BN;
    constexpr int XP = BM * 4 / NT, WP = BN * 4 / NT;       // units of 8 values a thread brings in per slice
    static_assert(EPI != FMOE_EPI_SWIGLU || FN % 2 == 0, "gate and up fragments come in pairs");
    constexpr int NB = BN < 128 ? BN : 128;                 // NCONT: columns of a block of weights in LDS
    static_assert(!NCONT || BN == 64 || BN % 128 == 0, "n-contiguous weights are parked in blocks of 64 or 128 columns");

    extern __shared__ __align__(16) uint8_t smem[];
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave % TL::WGM, wn = wave / TL::WGM;
    const int khalf = lane >> 5;

    BlockTile tile;
    int piece = -1, first_slice = 0, slices = 0, cut_tiles = 1;
    const int pairs = (p.K + 2 * BK - 1) / (2 * BK);
    const bool here = CUT && p.split_ws ? tile.locate(p, BM, [&](int64_t total_tiles) -> int64_t {
        const SplitDeal deal((int)total_tiles, p.split_slots, blockIdx.x % kNumXcd, pairs,
                             [](int rest, int pairs, int blocks) { return f32x3_split_pieces<BM>(rest, pairs, blocks); });
        if (blockIdx.x == 0 && tid == 0) {      // (offsets that overlap name more tiles than the grid has blocks: nothing is added up then)
            p.split_ws->tiles = deal.pieces > 1 && deal.count * kNumXcd <= (int)gridDim.x ? deal.rest : 0;
            p.split_ws->pieces = deal.pieces;
        }
        const int j = blockIdx.x / kNumXcd;
        if (j >= deal.count) return -1;
        int part;
        const int number = deal.tile(j, piece, part);
        if (piece >= 0) deal.slices(part, pairs, first_slice, slices);
        cut_tiles = deal.rest;
        return number;
    }) : tile.locate(p, BM);
    if (!here) return;
    const int expert = __builtin_amdgcn_readfirstlane(tile.expert), nt = __builtin_amdgcn_readfirstlane(tile.nt);
    const int rows_valid = __builtin_amdgcn_readfirstlane(tile.rows_valid);
    const int64_t row0 = tile.row0;
    const int n0 = nt * BN_OUT;

    int Kdim = p.K;
    int64_t k_begin = 0;
    if (p.k_window) {
        k_begin = p.k_window[expert];
        const int64_t span = p.k_window[expert + 1] - k_begin;
        Kdim = (int)(span < 0 ? 0 : (span < p.K ? span : p.K));
    }
    if (CUT && piece >= 0) {
        k_begin = first_slice * BK;
        Kdim = p.K - (int)k_begin < slices * BK ? p.K - (int)k_begin : slices * BK;
    }

    const float* a_base = reinterpret_cast<const float*>(p.a) + (int64_t)expert * p.a_stride_e + k_begin;
    auto a_row = [&](int tile_row) -> const float* {
        return a_base + source_row(p, row0 + (tile_row < rows_valid ? tile_row : 0)) * p.a_stride_row;
    };
    // the matrix and the output column behind column c of the tile
    auto w_matrix = [&](int c) -> const float* {
        return reinterpret_cast<const float*>(SWIGLU && c >= BN / 2 ? p.b2 : p.b) + (int64_t)expert * p.b_se;
    };
    auto w_col = [&](int c) -> int { return n0 + (SWIGLU && c >= BN / 2 ? c - BN / 2 : c); };

    // ------------------------------------------------------------------- loaders
    const float* xptr[XP];
    const float* wptr[WP];
    int w_second[WP];           // NCONT: elements from the unit's first 16-byte chunk to its second
#pragma unroll
    for (int i = 0; i < XP; ++i) xptr[i] = a_row((tid + i * NT) >> 2) + (tid & 3) * 8;
#pragma unroll
    for (int i = 0; i < WP; ++i) {
        const int q = tid + i * NT;
        if constexpr (NCONT) {
            const int c = (q % (BN / 8)) * 8, k = q / (BN / 8);
            const int n = w_col(c), first = n + 4 <= p.N ? n : p.N - 4, second = n + 8 <= p.N ? n + 4 : p.N - 4;
            wptr[i] = w_matrix(c) + (k_begin + k) * p.b_sk + first;
            w_second[i] = second - first;
        } else {
            const int c = q >> 2, n = w_col(c);
            wptr[i] = w_matrix(c) + (int64_t)(n < p.N ? n : p.N - 1) * p.b_sn + k_begin + (q & 3) * 8;
            w_second[i] = 4;
        }
    }
    // NCONT: 16-byte chunk c of row k lies at position c ^ tr_swizzle(k): the four rows of a transposing read and the two groups
    // of 16 lanes served together fall into eight different groups of 32 bytes of the 64 banks
    auto tr_swizzle = [](int k) -> int { return NB == 64 ? 2 * (k & 2) : 4 * (k & 3); };
    u32x4 xr[XP][2], wr[WP][2];
    auto load_global = [&](int kt) {
        const bool whole = (kt + 1) * BK <= Kdim;           // uniform: no per-lane predicate inside K
        const int k0 = kt * BK;
        auto chunk = [&](const float* src, int k) { return whole || k < Kdim ? *reinterpret_cast<const u32x4*>(src) : u32x4{0, 0, 0, 0}; };
#pragma unroll
        for (int i = 0; i < XP; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j) xr[i][j] = chunk(xptr[i] + k0 + 4 * j, k0 + (tid & 3) * 8 + 4 * j);
#pragma unroll
        for (int i = 0; i < WP; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                if constexpr (NCONT) wr[i][j] = chunk(wptr[i] + (int64_t)k0 * p.b_sk + (j ? w_second[i] : 0), k0 + (tid + i * NT) / (BN / 8));
                else wr[i][j] = chunk(wptr[i] + k0 + 4 * j, k0 + (tid & 3) * 8 + 4 * j);
            }
    };
    auto park = [&](const u32x4 (&v)[2], uint8_t* dst, int plane) {
        u32x4 h, m, l;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            uint32_t ph, pm, pl;
            split3(__uint_as_float(v[j >> 1][2 * (j & 1)]) * kF32x3Scale, __uint_as_float(v[j >> 1][2 * (j & 1) + 1]) * kF32x3Scale, ph, pm, pl);
            h[j] = ph;
            m[j] = pm;
            l[j] = pl;
        }
        *reinterpret_cast<u32x4*>(dst) = h;
        *reinterpret_cast<u32x4*>(dst + plane) = m;
        *reinterpret_cast<u32x4*>(dst + 2 * plane) = l;
    };
    uint8_t* const sw = smem + 3 * TL::A_PLANE;
    auto store_lds = [&]() {
#pragma unroll
        for (int i = 0; i < XP; ++i) {
            if constexpr (A_SILU) {
                xr[i][0] = silu_f32x4(xr[i][0]);
                xr[i][1] = silu_f32x4(xr[i][1]);
            }
            const int q = tid + i * NT;
            park(xr[i], smem + lds_off64(q >> 2, q & 3), TL::A_PLANE);
        }
#pragma unroll
        for (int i = 0; i < WP; ++i) {
            const int q = tid + i * NT;
            if constexpr (NCONT) {
                const int c8 = q % (BN / 8), k = q / (BN / 8);
                park(wr[i], sw + c8 / (NB / 8) * (64 * NB) + k * (2 * NB) + (((c8 % (NB / 8)) ^ tr_swizzle(k)) << 4), TL::B_PLANE);
            } else {
                park(wr[i], sw + lds_off64(q >> 2, q & 3), TL::B_PLANE);
            }
        }
    };

    // ----------------------------------------------------------------- main loop
    f32x16 acc[FN][FM], low[FN][FM];
#pragma unroll
    for (int i = 0; i < FN; ++i)
#pragma unroll
        for (int j = 0; j < FM; ++j)
#pragma unroll
            for (int v = 0; v < 16; ++v) acc[i][j][v] = low[i][j][v] = 0.0f;

    // first tile column of weight fragment fn
    auto frag_col = [&](int fn) -> int {
        return SWIGLU ? (fn < FN / 2 ? 0 : BN / 2) + wn * (TN / 2) + (fn % (FN / 2)) * 32 : wn * TN + fn * 32;
    };
    auto read_w = [&](int fn, int plane, int sub) -> bf16x8 {
        const uint8_t* s = sw + plane * TL::B_PLANE;
        if constexpr (NCONT) {
            const int l16 = lane & 15, row = 8 * khalf + (l16 >> 2);
            const int col = frag_col(fn) % NB + 16 * ((lane >> 4) & 1) + 4 * (l16 & 3);
            return read_tr8<8 * NB>(s + frag_col(fn) / NB * (64 * NB) + row * (2 * NB) + (((col >> 3) ^ tr_swizzle(row)) << 4) + (col & 7) * 2 +
                                    sub * (32 * NB));
        } else {
            return *reinterpret_cast<const bf16x8*>(s + lds_off64(frag_col(fn) + (lane & 31), 2 * sub + khalf));
        }
    };
    auto read_x = [&](int fm, int plane, int sub) -> bf16x8 {
        return *reinterpret_cast<const bf16x8*>(smem + plane * TL::A_PLANE + lds_off64(wm * TM + fm * 32 + (lane & 31), 2 * sub + khalf));
    };
    auto barrier = [] { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); };

    const int KT = (Kdim + BK - 1) / BK;
    load_global(0);
    for (int kt = 0; kt < KT; ++kt) {
        if (kt) barrier();              // every wave has read the slice before
        store_lds();
        if (kt + 1 < KT) load_global(kt + 1);
        barrier();
#pragma unroll
        for (int sub = 0; sub < 2; ++sub) {
            bf16x8 wf[3][FN], xf[3][FM];
#pragma unroll
            for (int pl = 0; pl < 3; ++pl) {
#pragma unroll
                for (int fn = 0; fn < FN; ++fn) wf[pl][fn] = read_w(fn, pl, sub);
#pragma unroll
                for (int fm = 0; fm < FM; ++fm) xf[pl][fm] = read_x(fm, pl, sub);
            }
            FMOE_F32X3_TERMS;
#pragma unroll
            for (int t = 0; t < 8; ++t)
#pragma unroll
                for (int fn = 0; fn < FN; ++fn)
#pragma unroll
                    for (int fm = 0; fm < FM; ++fm) {
                        f32x16& sum = t ? low[fn][fm] : acc[fn][fm];
                        sum = __builtin_amdgcn_mfma_f32_32x32x16_bf16(wf[W[t]][fn], xf[X[t]][fm], sum, 0, 0, 0);
                    }
        }
    }

    float probe = 0.0f;                 // NaN as soon as one sum is not finite
#pragma unroll
    for (int fn = 0; fn < FN; ++fn)
#pragma unroll
        for (int fm = 0; fm < FM; ++fm)
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                acc[fn][fm][v] += low[fn][fm][v];
                probe = __builtin_fmaf(acc[fn][fm][v], 0.0f, probe);
                acc[fn][fm][v] *= kF32x3Unscale;
            }
    if (__builtin_expect(__any(probe != 0.0f), 0)) {
        // (k in groups of 8, the wave halves on 4 each, as the register-staged kernel steps)
        const float* xrow[FM];
        const float* wrow[FN];
#pragma unroll
        for (int fm = 0; fm < FM; ++fm) xrow[fm] = a_row(wm * TM + fm * 32 + (lane & 31));
#pragma unroll
        for (int fn = 0; fn < FN; ++fn) {
            const int c = frag_col(fn) + (lane & 31), n = w_col(c);
            wrow[fn] = w_matrix(c) + (int64_t)(n < p.N ? n : p.N - 1) * p.b_sn + k_begin * p.b_sk;
#pragma unroll
            for (int fm = 0; fm < FM; ++fm)
#pragma unroll
                for (int v = 0; v < 16; ++v) acc[fn][fm][v] = 0.0f;
        }
        for (int k0 = 0; k0 < Kdim; k0 += 8) {
            const int k = k0 + 4 * khalf;
            const bool in = k < Kdim;
            u32x4 xv[FM], wv[FN];
#pragma unroll
            for (int fm = 0; fm < FM; ++fm) {
                xv[fm] = in ? *reinterpret_cast<const u32x4*>(xrow[fm] + k) : u32x4{0, 0, 0, 0};
                if constexpr (A_SILU) xv[fm] = silu_f32x4(xv[fm]);
            }
#pragma unroll
            for (int fn = 0; fn < FN; ++fn) {
                if constexpr (NCONT) {
#pragma unroll
                    for (int j = 0; j < 4; ++j) wv[fn][j] = in ? __float_as_uint(wrow[fn][(int64_t)(k + j) * p.b_sk]) : 0u;
                } else {
                    wv[fn] = in ? *reinterpret_cast<const u32x4*>(wrow[fn] + k) : u32x4{0, 0, 0, 0};
                }
            }
#pragma unroll
            for (int j = 0; j < 4; ++j)
#pragma unroll
                for (int fn = 0; fn < FN; ++fn)
#pragma unroll
                    for (int fm = 0; fm < FM; ++fm)
                        acc[fn][fm] = __builtin_amdgcn_mfma_f32_32x32x2f32(__uint_as_float(wv[fn][j]), __uint_as_float(xv[fm][j]),
                                                                            acc[fn][fm], 0, 0, 0);
        }
    }
    if (CUT && piece >= 0) {
        if (first_slice == 0 && tid == 0) p.split_ws->tile[piece % cut_tiles] = SplitTile{expert, nt, (int)row0, rows_valid};
#pragma unroll
        for (int fm = 0; fm < FM; ++fm)
#pragma unroll
            for (int fn = 0; fn < FN; ++fn) {
                f32x4* const out = f32x3_sums<TL>(p.split_ws, piece, wm * FM + fm, frag_col(fn) / 32) + lane;
#pragma unroll
                for (int g = 0; g < 4; ++g)
                    out[g * kWave] = f32x4{acc[fn][fm][4 * g], acc[fn][fm][4 * g + 1], acc[fn][fm][4 * g + 2], acc[fn][fm][4 * g + 3]};
            }
        return;
    }
    gemm_epilogue_f32<FM, FN, TM, TN, EPI>(p, acc, expert, n0, row0, rows_valid, wm, wn, lane);
}

}  // namespace fmoe
