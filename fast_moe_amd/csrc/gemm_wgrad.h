// Weight gradients of experts with few rows: the contraction is short and the launch is a stream of stores.
#pragma once

#include "gemm_direct.h"
#include "gemm_epilogue.h"

namespace fmoe {

// out[e][m][n] = sum over the rows r of expert e's window of a[r][m] * b[r][n], bf16, both operands row-major: what XTR is for the ring
// kernel.  Tiles of 128 x 128 of an expert's matrix, 4 waves of 64 x 64; a block computes a strip of column tiles one after the other, several
// blocks to a CU, so that stores run under the chains of first loads (offsets -> window -> rows).  32 rows at a time travel through registers into LDS, in
// the layout the transposing reads of the ring kernel take ([32 k][128 columns], chunk c of row k in place c ^ 4*(k%4)); rows
// beyond the window are zeros in the registers already, so nothing behind it is read.
//
// What bounds it: the stores.  128 experts of 8 rows, 1536 x 4096: 1.6 GB in 279 us, 5.8 TB/s (the ring, one block per CU whose stores wait
// for the next tile's pipeline to fill: 421); one tile to a block 363, eight 316.  Three blocks to a CU: a fourth would spill the rows
// that are on their way under the epilogue (strips of four 302).
struct WgradTile {
    static constexpr int BM = 128, BN = 128, NT = 256, BK = 32;
    static constexpr int OPERAND_BYTES = BK * 256, LDS_BYTES = 2 * 2 * OPERAND_BYTES;     // two buffers of both operands
};

__global__ __launch_bounds__(WgradTile::NT, 3) void grouped_wgrad_kernel(const GemmParams p, int strip) {
    constexpr int BM = WgradTile::BM, BN = WgradTile::BN, BK = WgradTile::BK;
    extern __shared__ __align__(16) uint8_t smem[];
    BlockTile32 tile;
    if (!tile.locate<true>(p, BM)) return;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave & 1, wn = wave >> 1, khalf = lane >> 5, l16 = lane & 15;
    const int expert = __builtin_amdgcn_readfirstlane(tile.expert);
    const int64_t seg = clamp_i64(p.offsets[expert], 0, p.total_rows);
    const int m0 = (int)(tile.row0 - seg);
    int n0 = tile.nt * strip * BN;
    const int n_end = n0 + strip * BN < p.N ? n0 + strip * BN : p.N;
    const int64_t lo = clamp_i64(p.k_window[expert], 0, (int64_t)p.K), hi = clamp_i64(p.k_window[expert + 1], lo, (int64_t)p.K);
    const int rows = (int)(hi - lo);

    // this thread's 16-byte chunks: columns 8 * (tid % 16) .. of rows tid / 16 and 16 + tid / 16 of the 32
    const int c = tid & 15, r = tid >> 4;
    const bool m_ok = 8 * c < tile.rows_valid;
    const uint16_t* const a = reinterpret_cast<const uint16_t*>(p.a) + (lo + r) * p.a_sk + (m_ok ? m0 + 8 * c : 0);
    const uint16_t* const b = reinterpret_cast<const uint16_t*>(p.b) + (int64_t)expert * p.b_se + (lo + r) * p.b_sk + 8 * c;
    u32x4 av[2], bv[2];
    auto fetch = [&](int k) {
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const bool in = k + r + 16 * i < rows;
            av[i] = in && m_ok ? *reinterpret_cast<const u32x4*>(a + (int64_t)(k + 16 * i) * p.a_sk) : u32x4{0, 0, 0, 0};
            bv[i] = in && n0 + 8 * c < p.N ? *reinterpret_cast<const u32x4*>(b + (int64_t)(k + 16 * i) * p.b_sk + n0) : u32x4{0, 0, 0, 0};
        }
    };
    const int put = r * 256 + ((c ^ (4 * (r & 3))) << 4);       // (rows 16 apart: the same place in their group of 4)
    // this lane's first transposing read of the fragment of columns 32 * f .. 32 * f + 31
    auto place = [&](int f) -> int {
        const int col = 32 * f + 16 * ((lane >> 4) & 1) + 4 * (l16 & 3), row = 8 * khalf + (l16 >> 2);
        return row * 256 + (((col >> 3) ^ (4 * (l16 >> 2))) << 4) + (col & 7) * 2;
    };
    int at_a[2], at_b[2];
#pragma unroll
    for (int f = 0; f < 2; ++f) {
        at_a[f] = place(2 * wm + f);
        at_b[f] = place(2 * wn + f) + WgradTile::OPERAND_BYTES;
    }

    fetch(0);
    int buffer = 0;
    for (;;) {
        f32x16 acc[2][2];
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j)
#pragma unroll
                for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.0f;
        for (int k = 0; k < rows; k += BK) {
            uint8_t* const s = smem + buffer * 2 * WgradTile::OPERAND_BYTES;
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                *reinterpret_cast<u32x4*>(s + put + i * 4096) = av[i];
                *reinterpret_cast<u32x4*>(s + WgradTile::OPERAND_BYTES + put + i * 4096) = bv[i];
            }
            if (k + BK < rows) fetch(k + BK);
            __syncthreads();        // (a buffer is written again behind the barrier that follows its last reads)
#pragma unroll
            for (int sub = 0; sub < 2; ++sub) {
                bf16x8 xf[2], wf[2];
#pragma unroll
                for (int f = 0; f < 2; ++f) {
                    xf[f] = read_tr8<1024>(s + at_a[f] + sub * 4096);
                    wf[f] = read_tr8<1024>(s + at_b[f] + sub * 4096);
                }
#pragma unroll
                for (int fn = 0; fn < 2; ++fn)
#pragma unroll
                    for (int fm = 0; fm < 2; ++fm)
                        acc[fn][fm] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(wf[fn], xf[fm], acc[fn][fm], 0, 0, 0);
            }
            buffer ^= 1;
        }
        const int done = n0;
        n0 += BN;
        const bool more = n0 < n_end;
        if (more) fetch(0);     // the strip's next tile: its first rows arrive under this one's stores
        gemm_epilogue<2, 2, 64, 64, false, FMOE_EPI_NONE, true, true, true>(p, acc, expert, done, tile.row0, tile.rows_valid, wm, wn, lane);
        if (!more) break;
    }
}

}  // namespace fmoe
