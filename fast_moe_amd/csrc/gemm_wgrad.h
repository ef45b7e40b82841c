// Weight gradients of experts with few rows: the contraction is short and the launch is a stream of stores.
#pragma once

#include "gemm_epilogue.h"

namespace fmoe {

// out[e][m][n] = sum over the rows r of expert e's window of a[r][m] * b[r][n], both operands row-major (bf16 or fp32): what XTR is for
// the ring kernel.  Tiles of 128 x 128 of an expert's matrix, 4 waves of 64 x 64; a block computes a strip of column tiles one after the
// other, several blocks to a CU, so that stores run under the chains of first loads (window -> rows).  8 KB of an operand's rows (32, fp32
// 16) at a time travel through registers into LDS, two buffers; rows beyond the window are zeros in the registers already, so nothing
// behind it is read.  bf16 rows lie in LDS as the transposing reads of the ring kernel take them ([32 k][128 columns], chunk c of row k in
// place c ^ 4*(k%4)); an fp32 MFMA takes two rows of 32 columns as they are.
//
// What bounds it: the stores.  128 experts of 8 rows, 1536 x 4096: 1.6 GB in 279 us, 5.8 TB/s (the ring, one block per CU whose stores wait
// for the next tile's pipeline to fill: 421); one tile to a block 363, eight 316.  Three blocks to a CU: a fourth would spill the rows
// that are on their way under the epilogue (strips of four 302).  fp32 from about 40 rows per expert on its MFMAs.
struct WgradTile {
    static constexpr int BM = 128, BN = 128, NT = 256, OPERAND_BYTES = 8192, LDS_BYTES = 2 * 2 * OPERAND_BYTES;
    int m, row_tiles;           // rows of an expert's matrix and their tiles
    int strip, strips;          // column tiles of a block, blocks across a matrix
    int per_xcd;                // tiles of an expert on every XCD, or 0: matrices of fewer than eight are dealt as they come

    // every expert's tiles to all XCDs alike, a run of them to each: neighbours share rows, and a hot expert is everybody's
    __device__ __forceinline__ bool locate(int& expert, int& mt, int& st) const {
        const int tiles = row_tiles * strips, b = blockIdx.x;
        int at;
        if (per_xcd) {
            expert = (b >> 3) / per_xcd;
            at = (b & 7) * per_xcd + (b >> 3) - expert * per_xcd;
        } else {
            expert = b / tiles;
            at = b - expert * tiles;
        }
        st = at / row_tiles;
        mt = at - st * row_tiles;
        return at < tiles;
    }
};

template <bool F32>
__global__ __launch_bounds__(WgradTile::NT, 3) void grouped_wgrad_kernel(const GemmParams p, const WgradTile t) {
    constexpr int BM = WgradTile::BM, BN = WgradTile::BN, ESIZE = F32 ? 4 : 2;
    constexpr int CHUNKS = BN * ESIZE / 16, CE = 16 / ESIZE, STEP = WgradTile::NT / CHUNKS, BK = 2 * STEP;   // 16-byte chunks of a row, ...
    extern __shared__ __align__(16) uint8_t smem[];
    int expert, mt, st;
    if (!t.locate(expert, mt, st)) return;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave & 1, wn = wave >> 1, khalf = lane >> 5;
    const int m0 = mt * BM, rows_valid = t.m - m0 < BM ? t.m - m0 : BM;
    int n0 = st * t.strip * BN;
    const int n_end = n0 + t.strip * BN < p.N ? n0 + t.strip * BN : p.N;
    const int64_t lo = clamp_i64(p.k_window[expert], 0, (int64_t)p.K), hi = clamp_i64(p.k_window[expert + 1], lo, (int64_t)p.K);
    const int rows = (int)(hi - lo);

    // this thread's 16-byte chunks: columns CE * c .. of rows r and r + STEP of the BK
    const int c = tid % CHUNKS, r = tid / CHUNKS;
    const bool m_ok = CE * c < rows_valid;
    const uint8_t* const a = p.a + ((lo + r) * p.a_sk + (m_ok ? m0 + CE * c : 0)) * ESIZE;
    const uint8_t* const b = p.b + ((lo + r) * p.b_sk + CE * c) * ESIZE;
    u32x4 av[2], bv[2];
    auto fetch = [&](int k) {
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const bool in = k + r + STEP * i < rows;
            av[i] = in && m_ok ? *reinterpret_cast<const u32x4*>(a + (int64_t)(k + STEP * i) * p.a_sk * ESIZE) : u32x4{0, 0, 0, 0};
            bv[i] = in && n0 + CE * c < p.N ? *reinterpret_cast<const u32x4*>(b + ((int64_t)(k + STEP * i) * p.b_sk + n0) * ESIZE) : u32x4{0, 0, 0, 0};
        }
    };
    // (bf16: rows 16 apart have the same place in their group of 4)
    const int put = r * (BN * ESIZE) + ((F32 ? c : c ^ (4 * (r & 3))) << 4);
    // where this lane reads the fragment of columns 32 * f .. 32 * f + 31: its first transposing read; fp32: its column of row khalf
    auto place = [&](int f, int lane) -> int {
        const int khalf = lane >> 5, l16 = lane & 15;
        if constexpr (F32) return khalf * (BN * ESIZE) + (32 * f + (lane & 31)) * ESIZE;
        const int col = 32 * f + 16 * ((lane >> 4) & 1) + 4 * (l16 & 3), row = 8 * khalf + (l16 >> 2);
        return row * 256 + (((col >> 3) ^ (4 * (l16 >> 2))) << 4) + (col & 7) * 2;
    };
    fetch(0);
    int buffer = 0;
    for (;;) {
        // (found again for every tile: kept over the epilogue they are spilled, and the reload waits for the next tile's rows and this one's stores: 128
        // experts of 32 rows, 1536 x 4096 379 us, 303 so; 12 experts, 200 rows, 1000 x 2600 16.3 / 15.8)
        int at_a[2], at_b[2], l = lane;
        asm volatile("" : "+v"(l));
#pragma unroll
        for (int f = 0; f < 2; ++f) {
            at_a[f] = place(2 * wm + f, l);
            at_b[f] = place(2 * wn + f, l) + WgradTile::OPERAND_BYTES;
        }
        f32x16 acc[2][2];       // [column block][row block]
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
                *reinterpret_cast<u32x4*>(s + put + i * (STEP * BN * ESIZE)) = av[i];
                *reinterpret_cast<u32x4*>(s + WgradTile::OPERAND_BYTES + put + i * (STEP * BN * ESIZE)) = bv[i];
            }
            if (k + BK < rows) fetch(k + BK);
            __syncthreads();        // (a buffer is written again behind the barrier that follows its last reads)
            if constexpr (F32) {
                const int steps = (rows - k < BK ? rows - k + 1 : BK) / 2;
                for (int q = 0; q < steps; ++q) {
                    float xf[2], wf[2];
#pragma unroll
                    for (int f = 0; f < 2; ++f) {
                        xf[f] = *reinterpret_cast<const float*>(s + at_a[f] + q * (2 * BN * ESIZE));
                        wf[f] = *reinterpret_cast<const float*>(s + at_b[f] + q * (2 * BN * ESIZE));
                    }
#pragma unroll
                    for (int fn = 0; fn < 2; ++fn)
#pragma unroll
                        for (int fm = 0; fm < 2; ++fm)      // (rows of the result from the A port: a store writes 32 columns of a row)
                            acc[fn][fm] = __builtin_amdgcn_mfma_f32_32x32x2f32(xf[fm], wf[fn], acc[fn][fm], 0, 0, 0);
                }
            } else {
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
            }
            buffer ^= 1;
        }
        const int done = n0;
        n0 += BN;
        const bool more = n0 < n_end;
        if (more) fetch(0);     // the strip's next tile: its first rows arrive under this one's stores
        if constexpr (F32) {
#pragma unroll
            for (int fm = 0; fm < 2; ++fm) {
                const int block = m0 + wm * 64 + fm * 32;           // (the halves' rows are whole blocks)
                const bool upper = p.out2 && block >= p.out_half;
                float* const base = reinterpret_cast<float*>(upper ? p.out2 : p.out) +
                                    (p.out2 ? expert * p.out_half + block - (upper ? p.out_half : 0) : (int64_t)expert * t.m + block) * p.N;
#pragma unroll
                for (int fn = 0; fn < 2; ++fn) {
                    const int n = done + wn * 64 + fn * 32 + (lane & 31);
#pragma unroll
                    for (int v = 0; v < 16; ++v) {
                        const int row = 8 * (v >> 2) + 4 * khalf + (v & 3);
                        if (block + row < t.m && n < p.N) base[(int64_t)row * p.N + n] = acc[fn][fm][v];
                    }
                }
            }
        } else {
            // the output rows are staged in the buffer read last: behind this barrier by nobody any more, and filled again behind the next one
            __syncthreads();
            uint8_t* const stage = smem + (buffer ^ 1) * 2 * WgradTile::OPERAND_BYTES + (wm * 2 + wn) * kEpilogueStageBytes;
            static_assert(2 * WgradTile::OPERAND_BYTES >= 4 * kEpilogueStageBytes, "the epilogue's rows fit a buffer");
            gemm_epilogue<2, 2, 64, 64, false, FMOE_EPI_NONE, true, true, true>(p, acc, expert, done, (int64_t)expert * t.m + m0, rows_valid, wm,
                                                                                wn, lane, stage);
        }
        if (!more) break;
    }
}

}  // namespace fmoe
