// Tiles cut along K: which of a launch's tiles the ring kernel's blocks share, where their sums meet, and the kernel that adds them.
#pragma once

#include "gemm_epilogue.h"

namespace fmoe {

constexpr int kSplitMost = 256;             // pieces of a launch: one per block

struct SplitTile { int expert, nt, row0, rows_valid; };
// Workspace of a launch: the header, then 256 KB for every piece
struct SplitWorkspace {
    int tiles, pieces;                      // tiles that were cut, pieces of each
    int pad[2];
    SplitTile tile[kSplitMost];
};
constexpr size_t kSplitHeaderBytes = 8192, kSplitPieceBytes = 256 * 256 * 4;
static_assert(sizeof(SplitWorkspace) <= kSplitHeaderBytes, "header");

// a wave's sums of a piece, [row block][column block][quad][lane]
__device__ __forceinline__ f32x4* split_sums(SplitWorkspace* ws, int piece, int wave) {
    return reinterpret_cast<f32x4*>(reinterpret_cast<uint8_t*>(ws) + kSplitHeaderBytes + piece * kSplitPieceBytes) + wave * 2048;
}

// Pieces of each of `rest` tiles (fewer than `blocks`) of `pairs` pairs of K-slices: no more pieces than blocks, two pairs to a
// piece at least, and the shortest of what the launch model gives: a pair of slices takes 1.1 us on a part-filled chip, a piece's sums 0.11 us
// of everybody's bandwidth (256 KB written and read at 4.7 TB/s), the second launch 5.  Integers: host and device agree.
__host__ __device__ inline int split_pieces(int rest, int pairs, int blocks, int* cost = nullptr) {
    int best = 1, least = 10 * pairs;
    for (int s = 2; s * rest <= blocks && 2 * s <= pairs; ++s) {
        const int c = (10 * pairs + s - 1) / s + rest * s + 50;
        if (c < least) {
            least = c;
            best = s;
        }
    }
    if (cost) *cost = least;
    return best;
}

// Rounds of whole tiles, one contiguous range per XCD and round-trip; the rest as pieces, the ones of the same part of K side by side (they share
// operands).
struct SplitDeal {
    int count;              // tiles and pieces of this XCD, in the order in which its blocks take them
    int rest, pieces;       // tiles left after the rounds, and what each is cut into
    int whole, base, first, xcd;

    __host__ __device__ __forceinline__ SplitDeal() : count(0), rest(0), pieces(1), whole(0), base(0), first(0), xcd(0) {}
    __host__ __device__ __forceinline__ SplitDeal(int total, int slots, int xcd_, int pairs)
        : SplitDeal(total, slots, xcd_, pairs, [](int rest, int pairs, int blocks) {
              return split_pieces(rest, pairs, blocks < kSplitMost ? blocks : kSplitMost);
          }) {}
    template <typename Pieces>
    __host__ __device__ __forceinline__ SplitDeal(int total, int slots, int xcd_, int pairs, Pieces&& pieces_of) : xcd(xcd_) {
        const int blocks = 8 * slots, rounds = total / blocks;
        whole = rounds * slots;
        base = rounds * blocks;
        rest = total - base;
        pieces = rest ? pieces_of(rest, pairs, blocks) : 1;
        const int all = rest * pieces, share = (all + 7) / 8;
        first = xcd * share;
        const int left = all - first;
        count = whole + (left < 0 ? 0 : left < share ? left : share);
    }
    // the XCD's j-th: a tile's number (piece -1), or piece number `piece`, which is part `part` of a tile
    __host__ __device__ __forceinline__ int tile(int j, int& piece, int& part) const {
        piece = -1;
        part = 0;
        if (j < whole) return xcd * whole + j;
        const int q = first + j - whole;
        if (pieces == 1) return base + q;
        piece = q;
        part = q / rest;
        return base + q - part * rest;
    }
    // K-slices of a part: first and number
    __host__ __device__ __forceinline__ void slices(int part, int pairs, int& first_slice, int& number) const {
        const int lo = (int)((int64_t)part * pairs / pieces), hi = (int)((int64_t)(part + 1) * pairs / pieces);
        first_slice = 2 * lo;
        number = 2 * (hi - lo);
    }
};

// Block: 32 rows of a cut tile, 4 waves of 64 columns as in the ring kernel.  The sums of a tile's pieces are added in the order of K.
template <bool FP8, int EPI, bool MSC>
__global__ __launch_bounds__(256) void split_reduce_kernel(const GemmParams p) {
    const int t = blockIdx.x >> 3, rb = blockIdx.x & 7;
    const int tiles = p.split_ws->tiles, pieces = p.split_ws->pieces;
    if (t >= tiles) return;
    const SplitTile tile = p.split_ws->tile[t];
    if (rb * 32 >= tile.rows_valid) return;
    const int lane = threadIdx.x & 63, wn = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wave = wn * 2 + (rb & 1);         // (the two wave rows hold the 32-row blocks alternately)
    f32x16 acc[2][1];
    for (int s = 0; s < pieces; ++s) {
        const f32x4* const src = split_sums(p.split_ws, s * tiles + t, wave) + (rb >> 1) * 8 * kWave + lane;
        f32x4 v[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) v[i] = src[i * kWave];
#pragma unroll
        for (int i = 0; i < 8; ++i)
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int at = 4 * (i & 3) + j;
                acc[i >> 2][0][at] = s ? acc[i >> 2][0][at] + v[i][j] : v[i][j];
            }
    }
    const int n0 = tile.nt * (EPI == FMOE_EPI_SWIGLU ? 128 : 256);
    __shared__ __align__(16) uint8_t stage[4 * kEpilogueStageBytes];
    gemm_epilogue<1, 2, 32, 64, FP8, EPI, true, true, false, false, NoAfterStores, MSC>(p, acc, tile.expert, n0, tile.row0, tile.rows_valid, rb, wn,
                                                                                       lane, stage + wn * kEpilogueStageBytes);
}

}  // namespace fmoe
