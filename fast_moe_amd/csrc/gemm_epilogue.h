// The epilogue all grouped GEMM kernels share: scales, bias, SiLU / SwiGLU / gating, bf16 rounding,
// and the stores (through LDS, or between the lanes of a row, so that adjacent lanes write contiguous bytes).
#pragma once

#include "gemm_params.h"

namespace fmoe {

// ------------------------------------------------------------------------ epilogue
// acc[fn][fm][v]: fragment (fn, fm) of the wave tile, v = 4*g + j <-> output row
// (lane & 31) of fragment row block fm, output column 32*fn + 8*g + 4*(lane >> 5) + j.
// Rounding points follow the reference's bf16 path: GEMM result (+bias) rounded to bf16,
// SiLU rounded to bf16, product rounded to bf16; e4m3 operands: (acc / (s_a * s_w)) rounded,
// then the bias added in bf16.
// ALWAYS_VEC: the caller has checked p.vec_store (the ring kernel is only chosen with it), so
// the element-store path is not even compiled in.  ROWS32: total_rows < 2^31 (the paired ring's
// condition), so row numbers and row_index values fit 32 bits.
// OUT2: an expert's output rows are split in two halves that go to two tensors (p.out2; the
// weight gradients of two matrices from one GEMM); a 32-row block lies in one half.
// ROW_IL: the two wave rows share the tile's 32-row blocks alternately (block 2*fm + wm belongs to
// wave row wm) instead of owning one half of the tile each, so that a tile with few valid rows
// leaves both with the same number of blocks to compute.
// after_stores(): called at the very end, in the same straight-line code as the stores and the
// counted wait behind them, where the compiler's own count of what is still in flight is exact
// (behind the join of the epilogue's variants it is not: it has to assume the path that stored
// nothing).  The ring kernel converts the row indices it fetched before the epilogue there.
constexpr int kEpilogueStageBytes = 4096;      // LDS of a wave for the staged form (ALWAYS_VEC)
struct NoAfterStores {
    __device__ __forceinline__ void operator()() const {}
    __device__ __forceinline__ void block_done(int) const {}
};
// block_done(fm): called behind the stores of the wave's row block fm (straight-line code as well);
// the ring kernel issues the next tile's scale loads there, under the arithmetic of the blocks left.
template <typename BlockDone, typename AfterAll>
struct EpilogueHooks {
    BlockDone on_block;
    AfterAll on_end;
    __device__ __forceinline__ void operator()() const { on_end(); }
    __device__ __forceinline__ void block_done(int fm) const { on_block(fm); }
};
template <typename BlockDone, typename AfterAll>
__device__ __forceinline__ EpilogueHooks<BlockDone, AfterAll> make_hooks(BlockDone b, AfterAll a) {
    return EpilogueHooks<BlockDone, AfterAll>{b, a};
}

// E8M0 code (2^(code - 127)) of the reciprocal of a power-of-two fp32 scale: what the scale
// operands of v_mfma_scale_f32_32x32x64_f8f6f4 take.  2^127 (the quantiser's scale of an all-zero
// or non-finite row) gives code 0 = 2^-127.
__device__ __forceinline__ uint32_t e8m0_of_reciprocal(float scale) {
    return (254u - (__float_as_uint(scale) >> 23)) & 0xffu;
}
// one e4m3 MFMA whose products are scaled by 2^(byte OA of sa - 127) per weight row and
// 2^(byte OB of sb - 127) per activation row (lane l: row l % 32 of its fragment).
// Written as inline assembly with the accumulator tied to the destination: through the builtin the
// destination is a separate early-clobber operand, which costs the ring kernel (at 256 registers
// with 128 of them accumulators) about 50 spilled registers per lane around the tile boundary.
// The compiler therefore does not know that this is an MFMA and inserts none of the wait states
// the matrix pipe needs around VALU accesses to its registers.  VALU write -> MFMA read (the
// clears of a tile's accumulators, the packed scale codes): two idle issue cycles stand in front
// of every one of these instructions, inside the same statement (they pass while the pipe works
// on the MFMA before).  MFMA write -> VALU read (the epilogue): mfma_results_guard() behind the
// main loop.
template <int OA, int OB>
__device__ __forceinline__ void mfma_e4m3_scaled(const i32x8& a, const i32x8& b, f32x16& c, uint32_t sa, uint32_t sb) {
    asm volatile("s_nop 1\n\tv_mfma_scale_f32_32x32x64_f8f6f4 %0, %1, %2, %0, %3, %4 op_sel:[%5,%6,0] op_sel_hi:[%7,%8,0]"
                 : "+v"(c) : "v"(a), "v"(b), "v"(sa), "v"(sb), "n"(OA & 1), "n"(OB & 1), "n"(OA >> 1), "n"(OB >> 1));
}
// 32 idle issue cycles behind the last of those MFMAs (a 16-pass MFMA needs 18 before the VALU may
// read its result), and nothing that follows in the program may be scheduled in front of them.
__device__ __forceinline__ void mfma_results_guard() {
    asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
}
template <int I, int N, typename F>
__device__ __forceinline__ void static_for(F&& f) {
    if constexpr (I < N) {
        f(std::integral_constant<int, I>{});
        static_for<I + 1, N>(f);
    }
}

// The reciprocal scales of e4m3 operands that a lane's sums meet: of its rows, and of its columns, [fn][gp][q][j] <-> column nq + 8*q +
// 4*khalf + j with nq = first column of register-quad pair gp of fragment fn.
template <int FM, int FN, int TM, int TN, int EPI, bool ROWS32, bool ROW_IL>
__device__ __forceinline__ void fetch_reciprocal_scales(const GemmParams& p, float (&rsa)[FM], float (&rsw)[EPI == FMOE_EPI_SWIGLU ? FN / 2 : FN][2][2][4],
                                                        float (&rsw2)[EPI == FMOE_EPI_SWIGLU ? FN / 2 : FN][2][2][4], int expert, int n0, int64_t row0,
                                                        int rows_valid, int wm, int wn, int lane) {
    constexpr bool SWIGLU = EPI == FMOE_EPI_SWIGLU;
    constexpr int FN_OUT = SWIGLU ? FN / 2 : FN;
    asm volatile("" : "+v"(lane));      // (see gemm_epilogue)
    wm = __builtin_amdgcn_readfirstlane(wm);
    wn = __builtin_amdgcn_readfirstlane(wn);
    const int khalf = lane >> 5;
    auto frag_row = [&](int fm) -> int { return ROW_IL ? (fm * 2 + wm) * 32 : wm * TM + fm * 32; };
    const int col0 = n0 + (SWIGLU ? wn * (TN / 2) : wn * TN);
    bool row_ok[FM];
#pragma unroll
    for (int fm = 0; fm < FM; ++fm) row_ok[fm] = frag_row(fm) + (lane & 31) < rows_valid;
    // the activation scales of this lane's rows: all index loads, then all scale loads (two
    // memory latencies, not two per row block)
    typedef typename std::conditional<ROWS32, int32_t, int64_t>::type row_t;
    row_t src[FM];
#pragma unroll
    for (int fm = 0; fm < FM; ++fm)
        src[fm] = (row_t)(row0 + (row_ok[fm] ? frag_row(fm) + (lane & 31) : 0));
    if (p.row_index) {
#pragma unroll
        for (int fm = 0; fm < FM; ++fm) {
            if (ROWS32) src[fm] = reinterpret_cast<const int32_t*>(p.row_index)[2 * (int64_t)src[fm]];   // low half
            else src[fm] = (row_t)p.row_index[src[fm]];
        }
#pragma unroll
        for (int fm = 0; fm < FM; ++fm)
            if (ROWS32) src[fm] = (row_t)div_index32(p, (int32_t)src[fm]);
            else src[fm] = p.index_shift >= 0 ? (src[fm] >> p.index_shift) : src[fm] / (row_t)p.index_div;
    }
#pragma unroll
    for (int fm = 0; fm < FM; ++fm) {
        const row_t last = (row_t)(p.a_rows - 1);
        src[fm] = src[fm] < 0 ? 0 : (src[fm] > last ? last : src[fm]);
    }
#pragma unroll
    for (int fm = 0; fm < FM; ++fm) rsa[fm] = p.a_scale[src[fm]];
    // The weight-scale loads go out right behind the activation-scale loads, before anything
    // waits for either, so that the two round trips overlap (one memory latency per tile less;
    // the raw values wait in the registers their reciprocals end up in).
    constexpr int WCOLS = FN_OUT * 32;          // output columns of this wave
    if (p.scale_vec && col0 + WCOLS <= p.N) {
        // the wave's columns lie inside N: the 4 scales of a register quad in one 16-byte load
        // from a wave-uniform base plus the lane half's 16 bytes plus a constant
        const float* sb = p.b_scale + ((int64_t)expert * p.N + col0);
        const float* sb2 = SWIGLU ? p.b2_scale + ((int64_t)expert * p.N + col0) : sb;
        const int half4 = 4 * khalf;
        typedef __attribute__((ext_vector_type(4))) float f32x4;
#pragma unroll
        for (int fn = 0; fn < FN_OUT; ++fn)
#pragma unroll
            for (int gp = 0; gp < 2; ++gp)
#pragma unroll
                for (int q = 0; q < 2; ++q) {
                    const int c = fn * 32 + 16 * gp + 8 * q;
                    const f32x4 s1 = *reinterpret_cast<const f32x4*>(sb + half4 + c);
                    f32x4 s2 = s1;
                    if (SWIGLU) s2 = *reinterpret_cast<const f32x4*>(sb2 + half4 + c);
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        rsw[fn][gp][q][j] = s1[j];
                        if (SWIGLU) rsw2[fn][gp][q][j] = s2[j];
                    }
                }
    } else {
        // the last column tile, or scale tensors off a 16-byte boundary: one clamped load a column
#pragma unroll
        for (int fn = 0; fn < FN_OUT; ++fn)
#pragma unroll
            for (int gp = 0; gp < 2; ++gp)
#pragma unroll
                for (int q = 0; q < 2; ++q)
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        const int n = col0 + fn * 32 + 16 * gp + 8 * q + 4 * khalf + j;
                        const int nc = n < p.N ? n : p.N - 1;
                        rsw[fn][gp][q][j] = p.b_scale[(int64_t)expert * p.N + nc];
                        if (SWIGLU) rsw2[fn][gp][q][j] = p.b2_scale[(int64_t)expert * p.N + nc];
                    }
    }
    __builtin_amdgcn_sched_barrier(0);
    // (v_rcp_f32 is exact on the powers of two the reference's scales are)
#pragma unroll
    for (int fm = 0; fm < FM; ++fm) rsa[fm] = __builtin_amdgcn_rcpf(rsa[fm]);
#pragma unroll
    for (int fn = 0; fn < FN_OUT; ++fn)
#pragma unroll
        for (int gp = 0; gp < 2; ++gp)
#pragma unroll
            for (int q = 0; q < 2; ++q)
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    rsw[fn][gp][q][j] = __builtin_amdgcn_rcpf(rsw[fn][gp][q][j]);
                    if (SWIGLU) rsw2[fn][gp][q][j] = __builtin_amdgcn_rcpf(rsw2[fn][gp][q][j]);
                }
}

// Plain and SwiGLU: the sums divided by the scales in place, ahead of everything else an epilogue does.  The reciprocals of a SwiGLU wave's columns are
// 32 registers, and beside rows on their way through LDS the kernels spill 70 to 90, whose reloads lie in the tile loop.  us, scales multiplied at
// the sums' use / in place: 512 rows, 64 experts, 2048 -> 2 x 1408 90.2 / 73.5, plain 32.6 / 30.5; 8192 rows, 8 experts, 1024 -> 2 x 4096 89.2 /
// 86.4; 30000 rows, 200 experts, 1024 -> 2 x 512 79.1 / 76.0.  SiLU keeps them: with a bias 64.2 / 66.7, 8192 rows, 8 experts, 1024 -> 4096.
// whole: else the sums stay as they are (times one: a piece of a tile cut along K goes through here as well, as sums that two branches read
// are not scaled in their own registers).
constexpr bool divides_in_place(int epi) { return epi != FMOE_EPI_SILU; }
template <int FM, int FN, int TM, int TN, int EPI, bool ROWS32, bool ROW_IL>
__device__ __forceinline__ void divide_scales_out(const GemmParams& p, f32x16 (&acc)[FN][FM], int expert, int n0, int64_t row0, int rows_valid, int wm,
                                                  int wn, int lane, bool whole = true) {
    constexpr bool SWIGLU = EPI == FMOE_EPI_SWIGLU;
    constexpr int FN_OUT = SWIGLU ? FN / 2 : FN;
    float rsa[FM], rsw[FN_OUT][2][2][4], rsw2[FN_OUT][2][2][4];
    fetch_reciprocal_scales<FM, FN, TM, TN, EPI, ROWS32, ROW_IL>(p, rsa, rsw, rsw2, expert, n0, row0, rows_valid, wm, wn, lane);
    if (!whole) {
#pragma unroll
        for (int fm = 0; fm < FM; ++fm) rsa[fm] = 1.0f;
#pragma unroll
        for (int i = 0; i < FN_OUT * 16; ++i) {
            rsw[i / 16][i / 8 % 2][i / 4 % 2][i % 4] = 1.0f;
            if (SWIGLU) rsw2[i / 16][i / 8 % 2][i / 4 % 2][i % 4] = 1.0f;
        }
    }
#pragma unroll
    for (int fm = 0; fm < FM; ++fm)
#pragma unroll
        for (int fn = 0; fn < FN_OUT; ++fn)
#pragma unroll
            for (int g = 0; g < 4; ++g) {
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    acc[fn][fm][4 * g + j] *= rsa[fm] * rsw[fn][g / 2][g % 2][j];
                    if (SWIGLU) acc[fn + FN / 2][fm][4 * g + j] *= rsa[fm] * rsw2[fn][g / 2][g % 2][j];
                }
                __builtin_amdgcn_sched_barrier(0);      // (all products first is a register for each)
            }
}

// MSC (e4m3): the scales were applied by the MFMAs themselves (power-of-two scales as block scales of
// the instruction): acc already holds sum / (s_a * s_w) and the epilogue loads and multiplies nothing.
template <int FM, int FN, int TM, int TN, bool FP8, int EPI, bool ALWAYS_VEC = false, bool ROWS32 = false,
          bool OUT2 = false, bool ROW_IL = false, typename AfterStores = NoAfterStores, bool MSC = false>
__device__ __forceinline__ void gemm_epilogue(const GemmParams& p, f32x16 (&acc)[FN][FM], int expert,
                                              int n0, int64_t row0, int rows_valid, int wm, int wn,
                                              int lane, uint8_t* stage = nullptr, AfterStores after_stores = AfterStores(),
                                              uint64_t* ets = nullptr) {
    constexpr bool SWIGLU = EPI == FMOE_EPI_SWIGLU;
    constexpr bool GATED = EPI == FMOE_EPI_GATED;   // out = silu(gate from p.aux) * (acc + bias); bf16 operands
    static_assert(!(GATED && FP8), "the gated epilogue is built for bf16 operands");
    constexpr int FN_OUT = SWIGLU ? FN / 2 : FN;
    // (ring kernel: everything derived from the lane number below is recomputed per tile; as
    // tile-loop invariants the compiler keeps such values in registers across the main loop, or
    // spills them and reloads them here behind a wait that drains the LDS-DMA stream)
    if (ALWAYS_VEC) asm volatile("" : "+v"(lane));
    const int khalf = lane >> 5;
    const int64_t bias_row = (int64_t)expert * p.bias_se;
#ifdef FMOE_TRACE
#define FMOE_EPI_STAMP(i_) do { if (ets) ets[i_] = __builtin_amdgcn_s_memrealtime(); } while (0)
#else
#define FMOE_EPI_STAMP(i_) do {} while (0)
#endif
    // Output addresses are a wave-uniform 64-bit base (tile row block, column group: scalar
    // registers and scalar arithmetic) plus one 32-bit per-lane byte offset (the lane's row
    // inside the 32-row block and its 16-byte half): no per-row pointers to keep in vector
    // registers over an epilogue whose accumulators and column constants already fill them.
    wm = __builtin_amdgcn_readfirstlane(wm);
    wn = __builtin_amdgcn_readfirstlane(wn);
    row0 = (int64_t)(((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(row0 >> 32)) << 32) |
                     (uint32_t)__builtin_amdgcn_readfirstlane((int)row0));
    // (computed afresh at every store from a copy of the lane number the compiler cannot see
    // through: hoisted out of the loops it becomes a 64-bit offset that is spilled and reloaded,
    // with a full vmcnt(0) wait, before every single store)
    auto lane_offset = [&](int64_t stride) -> uint32_t {
        int l = lane;
        asm volatile("" : "+v"(l));
        return (uint32_t)(l & 31) * (uint32_t)stride * 2u + (uint32_t)(l >> 5) * 16u;
    };
    // first tile row of the wave's row block fm
    auto frag_row = [&](int fm) -> int { return ROW_IL ? (fm * 2 + wm) * 32 : wm * TM + fm * 32; };
    bool row_ok[FM];
#pragma unroll
    for (int fm = 0; fm < FM; ++fm) row_ok[fm] = frag_row(fm) + (lane & 31) < rows_valid;
    const int col0 = n0 + (SWIGLU ? wn * (TN / 2) : wn * TN);
    constexpr bool SCALE = FP8 && !MSC && !divides_in_place(EPI);       // times the reciprocal scales at their use
    float rsa[FM], rsw[FN_OUT][2][2][4], rsw2[FN_OUT][2][2][4];
    if constexpr (SCALE)
        fetch_reciprocal_scales<FM, FN, TM, TN, EPI, ROWS32, ROW_IL>(p, rsa, rsw, rsw2, expert, n0, row0, rows_valid, wm, wn, lane);
    else if constexpr (FP8 && !MSC)
        divide_scales_out<FM, FN, TM, TN, EPI, ROWS32, ROW_IL>(p, acc, expert, n0, row0, rows_valid, wm, wn, lane);
    // the bias-free form (FastMoE's SwiGLU experts, every fp8 call without bias) skips the adds
    auto run = [&](auto has_bias_c, auto has_aux_c) {
        constexpr bool HAS_BIAS = decltype(has_bias_c)::value;
        constexpr bool HAS_AUX = SWIGLU && decltype(has_aux_c)::value;   // keep the pre-activations (training)
        // per-column biases of this lane, indexed like rsw
        float bv[FN_OUT][2][2][4], bv2[FN_OUT][2][2][4];
        // with a bias, at least one of the two pointers is set: both loads go through a valid
        // pointer and a select drops the value of a missing one (a branch per load would make
        // every load wait for the one before).  Sums that were divided in place take a missing one as
        // -0, which changes no sum, instead of a branch at every pair of columns.
        constexpr bool SELECT = FP8 && !MSC && !SCALE;
        constexpr float NO_BIAS = SELECT ? -0.0f : 0.0f;
        const uint16_t* bias_a = p.bias ? p.bias : p.bias2;
        const uint16_t* bias_b = p.bias2 ? p.bias2 : p.bias;
#pragma unroll
        for (int fn = 0; fn < FN_OUT; ++fn)
#pragma unroll
            for (int gp = 0; gp < 2; ++gp)
#pragma unroll
                for (int q = 0; q < 2; ++q)
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        const int n = col0 + fn * 32 + 16 * gp + 8 * q + 4 * khalf + j;
                        const int nc = n < p.N ? n : p.N - 1;
                        bv[fn][gp][q][j] = bv2[fn][gp][q][j] = 0.0f;
                        if (HAS_BIAS) {
                            const float a = bf16_bits_to_f32(bias_a[bias_row + nc]);
                            bv[fn][gp][q][j] = p.bias ? a : NO_BIAS;
                        }
                        if (HAS_BIAS && SWIGLU) {
                            const float b = bf16_bits_to_f32(bias_b[bias_row + nc]);
                            bv2[fn][gp][q][j] = p.bias2 ? b : NO_BIAS;
                        }
                    }
        __builtin_amdgcn_sched_barrier(0);
        FMOE_EPI_STAMP(0);
        // Staged form.  The store unit merges what ADJACENT lanes write: a 128 KB tile drains in 1.3 us where neighbouring lanes write
        // neighbouring bytes and in 3.9 where a lane's neighbour in memory is 32 lanes away, as in the MFMA's layout.  So a row block
        // (two of them where the wave has 32 output columns) goes through the wave's own 4 KB of LDS: pieces of 4 columns in, whole rows of
        // 16-byte chunks out, which 8 (4) adjacent lanes store.  Rearranging the same rows in registers (lane swaps, transposes of
        // quads by DPP moves and selects) was 330 of an epilogue's 640 vector instructions, and the two waves of a SIMD are bound by those.
        // Chunk c of row r lies at position c ^ (r / 2) % 8 (c ^ (r / 4) % 4), its two halves swapped in rows 16..31 of each 32: the reads do not
        // meet in a bank, the writes, served 16 lanes and 128 bytes at a time, two by two (SQ_LDS_BANK_CONFLICT: 4 cycles a write, 2 to 9 % of a launch's
        // LDS cycles; c ^ r % 8, c ^ (r / 2) % 4 and halves swapped by r / 8 have none, and whole passes take the same time with them).  A
        // wave's LDS instructions execute in order, nothing has to be waited for in between.
        if constexpr (ALWAYS_VEC) {
            constexpr int CH = 4 * FN_OUT;                      // 16-byte chunks of a row
            constexpr int RB = FN_OUT == 2 || FM < 2 ? 1 : 2;   // row blocks at a time
            constexpr int RPI = kWave / CH;                     // rows of a store instruction
            constexpr int NI = 32 * RB / RPI;
            constexpr int KINDS = HAS_AUX ? 3 : 1;              // the result, the two pre-activations
            static_assert(32 * RB * CH * 16 <= kEpilogueStageBytes, "a wave's share of the staging rows");
            int l = lane;
            asm volatile("" : "+v"(l));
            const int wr = l & 31;
            const int put_at = wr * (16 * CH) + ((CH == 8 ? (wr >> 1) & 7 : (wr >> 2) & 3) << 4) + ((khalf ^ (wr >> 4)) << 3);
            const int sr = l / CH, sc = l % CH;
            const int take_at = sr * (16 * CH) + ((sc ^ (l >> 4)) << 4);
            // rows that this lane may store, counted from its row of a store instruction
            const int row_limit = col0 + 8 * sc + 7 < p.N ? rows_valid - sr : 0;
            auto put = [&](int b, int piece, uint32_t lo, uint32_t hi) {
                *reinterpret_cast<u32x2*>(stage + (b * 32 * 16 * CH) + (put_at ^ (piece << 4))) = u32x2{lo, hi};
            };
            u32x4 rows[NI];
            auto take = [&]() {
#pragma unroll
                for (int i = 0; i < NI; ++i) {
                    const u32x4 v = *reinterpret_cast<const u32x4*>(stage + i * 1024 + (CH == 8 && (i & 1) ? take_at ^ 64 : take_at));
                    const bool swapped = ((i * RPI) >> 4) & 1;
                    rows[i] = swapped ? u32x4{v[2], v[3], v[0], v[1]} : v;
                }
            };
            // GATED: a lane's gate values are the 16 bytes at the position its store i of a row block writes; the loads of
            // block fm + 1 go out before block fm's arithmetic, so that one memory latency per tile is waited for, not one per block.
            u32x4 gate_next[NI] = {}, gate_cur[NI] = {};
            auto fetch_gate = [&](int fm) {
#pragma unroll
                for (int i = 0; i < NI; ++i) {
                    const int col = col0 + 8 * sc;
                    const bool ok = frag_row(fm) + i * RPI < row_limit;
                    const uint16_t* src = p.aux + (row0 + (ok ? frag_row(fm) + i * RPI + sr : 0)) * p.aux_stride + (ok ? col : 0);
                    if (p.gate_vec16) {
                        gate_next[i] = *reinterpret_cast<const u32x4*>(src);
                    } else {
                        uint32_t e[8];
#pragma unroll
                        for (int j = 0; j < 8; ++j) e[j] = ok ? (uint32_t)src[j] : 0u;
                        gate_next[i] = u32x4{e[0] | (e[1] << 16), e[2] | (e[3] << 16), e[4] | (e[5] << 16), e[6] | (e[7] << 16)};
                    }
                }
            };
            // SwiGLU on 64-row tiles: the two lanes of a row trade the halves of 16 columns and store 32 bytes, in the midst of the arithmetic.  Such a
            // launch has a tile or two for a CU, and ends with them: rows through LDS leave only behind all of it.  us, LDS / this: 600 rows, 12
            // experts, 2368 -> 2 x 704 23.5 / 23.2, e4m3 16.2 / 15.6; 800 rows, 16 experts, 2048 -> 2 x 512 20.5 / 20.0, e4m3 14.6 / 14.1; many tiles are
            // level (4000 rows, 64 experts, 2048 -> 2 x 1408 189.5 / 189.1, with the pre-activations 197.6 / 198.7).
            constexpr bool DIRECT = SWIGLU && FM == 2;
            auto store_pair = [&](int fm, int kind, int nq, const uint32_t (&pk)[2][2]) {
                const int64_t stride = kind ? p.aux_stride : p.out_stride;
                const u32x2 s0 = __builtin_amdgcn_permlane32_swap(pk[0][0], pk[1][0], false, false);
                const u32x2 s1 = __builtin_amdgcn_permlane32_swap(pk[0][1], pk[1][1], false, false);
                uint16_t* const base = (kind == 0 ? p.out : kind == 1 ? p.aux : p.aux2) + (row0 + frag_row(fm)) * stride + nq;
                const bool ok = row_ok[fm] && nq + 8 * khalf + 7 < p.N;
                store16_uniform_base(base, ok ? lane_offset(stride) : kDropLane, u32x4{s0[0], s1[0], s0[1], s1[1]});
            };
            // what the lane contributes to piece 4 fn + 2 gp + q of row block fm, rounded to bf16
            auto emit = [&](int fm, int kind) {
#pragma unroll
                for (int fn = 0; fn < FN_OUT; ++fn)
#pragma unroll
                    for (int gp = 0; gp < 2; ++gp) {
                        uint32_t pk[2][2];
#pragma unroll
                        for (int q = 0; q < 2; ++q) {
#pragma unroll
                            for (int j = 0; j < 4; j += 2) {        // two columns at a time: one conversion instruction rounds a pair
                                const int v = 4 * (2 * gp + q) + j;
                                auto branch = [&](float a, float b, const float (&bias)[4], const void* given) -> uint32_t {
                                    if (SCALE) {        // (no SwiGLU: the first half's columns)
                                        a *= rsa[fm] * rsw[fn][gp][q][j];
                                        b *= rsa[fm] * rsw[fn][gp][q][j + 1];
                                    }
                                    if (HAS_BIAS && (!FP8 || SELECT || given)) {
                                        if (FP8) rbf2(a, b);
                                        a += bias[j];
                                        b += bias[j + 1];
                                    }
                                    return pack_bf16(a, b);
                                };
                                auto low = [](uint32_t u) { return __uint_as_float(u << 16); };
                                auto high = [](uint32_t u) { return __uint_as_float(u & 0xffff0000u); };
                                uint32_t y = kind == 2 ? 0u : branch(acc[fn][fm][v], acc[fn][fm][v + 1], bv[fn][gp][q], p.bias);
                                uint32_t u = 0;
                                if (SWIGLU && kind != 1)
                                    u = branch(acc[fn + FN / 2][fm][v], acc[fn + FN / 2][fm][v + 1], bv2[fn][gp][q], p.bias2);
                                if (kind == 2) y = u;
                                if (EPI == FMOE_EPI_SILU || (SWIGLU && kind == 0)) y = pack_bf16(fast_silu_f32(low(y)), fast_silu_f32(high(y)));
                                if (SWIGLU && kind == 0) y = pack_bf16(low(y) * low(u), high(y) * high(u));
                                pk[q][j / 2] = y;
                            }
                            if (!DIRECT) put(fm % RB, 4 * fn + 2 * gp + q, pk[q][0], pk[q][1]);
                        }
                        if (DIRECT) store_pair(fm, kind, col0 + 32 * fn + 16 * gp, pk);
                    }
            };
            auto store = [&](int fm0, int kind) {       // the rows taken last
                const int64_t stride = kind ? p.aux_stride : p.out_stride;
                const uint32_t lane_off = ((uint32_t)sr * (uint32_t)stride + (uint32_t)(8 * sc)) * 2u;
#pragma unroll
                for (int i = 0; i < NI; ++i) {
                    const int fm = fm0 + i * RPI / 32, in_block = i * RPI % 32;
                    const int64_t block_row = row0 + frag_row(fm);
                    uint16_t* obase = (kind == 0 ? p.out : kind == 1 ? p.aux : p.aux2) + block_row * stride;
                    if constexpr (OUT2) {
                        if (p.out2) {       // (scalar arithmetic: everything here is wave-uniform)
                            // (offsets that are not the promised e * 2h are not followed out of
                            // the two tensors: the block's row is forced into [0, 2h), whole blocks)
                            int64_t m = block_row - (int64_t)expert * (2 * p.out_half);
                            m = m < 0 ? 0 : (m > 2 * p.out_half - 32 ? 2 * p.out_half - 32 : m);
                            m &= ~(int64_t)31;
                            const bool upper = m >= p.out_half;
                            obase = (upper ? p.out2 : p.out) +
                                    ((int64_t)expert * p.out_half + (upper ? m - p.out_half : m)) * p.out_stride;
                        }
                    }
                    u32x4 v = rows[i];
                    if constexpr (GATED) {              // round(acc + bias) times the rounded SiLU of the gate
#pragma unroll
                        for (int d = 0; d < 4; ++d) {
                            float ga = __uint_as_float(gate_cur[i][d] << 16), gb = __uint_as_float(gate_cur[i][d] & 0xffff0000u);
                            ga = fast_silu_f32(ga);
                            gb = fast_silu_f32(gb);
                            rbf2(ga, gb);
                            v[d] = pack_bf16(ga * __uint_as_float(v[d] << 16), gb * __uint_as_float(v[d] & 0xffff0000u));
                        }
                    }
                    const bool ok = frag_row(fm) + in_block < row_limit;
                    store16_uniform_base(obase + in_block * stride + col0, ok ? lane_off : kDropLane, v);
                }
            };
            if constexpr (GATED) fetch_gate(0);
#pragma unroll
            for (int fm = 0; DIRECT && fm < FM; ++fm) {
#pragma unroll
                for (int kind = 0; kind < KINDS; ++kind) {
                    emit(fm, kind);
                    __builtin_amdgcn_sched_barrier(0);
                }
                after_stores.block_done(fm);
            }
            // a step's rows are stored behind the next step's arithmetic, by when they have arrived
#pragma unroll
            for (int step = 0; !DIRECT && step <= FM / RB * KINDS; ++step) {
                const int fm = step / KINDS * RB, kind = step % KINDS;
                if (step < FM / RB * KINDS) {
#pragma unroll
                    for (int b = 0; b < RB; ++b) emit(fm + b, kind);
                }
                if (step > 0) {
                    const int before = step - 1;
                    store(before / KINDS * RB, before % KINDS);
                    __builtin_amdgcn_sched_barrier(0);
                    if (before % KINDS == KINDS - 1) {
                        FMOE_EPI_STAMP(before / KINDS * RB);
                        after_stores.block_done(before / KINDS * RB);
                    }
                }
                if (step < FM / RB * KINDS) {
                    if constexpr (GATED) {
#pragma unroll
                        for (int i = 0; i < NI; ++i) gate_cur[i] = gate_next[i];
                        if (fm + 1 < FM) fetch_gate(fm + 1);
                    }
                    take();
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        // rows outermost: the stores that complete a row's 128-byte line follow each other
#pragma unroll
        for (int fm = 0; !ALWAYS_VEC && fm < FM; ++fm) {
            // GATED: the row block's gate values, all loads of the block issued together (one memory
            // latency per 32-row block; loaded where they are used, every group of 8 waits out its own)
            u32x2 graw[FN_OUT][2][2];
            if constexpr (GATED) {
                const int64_t grow = row0 + (row_ok[fm] ? frag_row(fm) + (lane & 31) : 0);
                const uint16_t* gp_row = p.aux + grow * p.aux_stride;
#pragma unroll
                for (int fn = 0; fn < FN_OUT; ++fn)
#pragma unroll
                    for (int gp = 0; gp < 2; ++gp)
#pragma unroll
                        for (int q = 0; q < 2; ++q) {
                            const int n = col0 + fn * 32 + 16 * gp + 8 * q + 4 * khalf;
                            if (p.gate_vec && n + 3 < p.N) {
                                graw[fn][gp][q] = *reinterpret_cast<const u32x2*>(gp_row + n);
                            } else {
                                uint32_t e[4];
#pragma unroll
                                for (int j = 0; j < 4; ++j) e[j] = n + j < p.N ? (uint32_t)gp_row[n + j] : 0u;
                                graw[fn][gp][q] = u32x2{e[0] | (e[1] << 16), e[2] | (e[3] << 16)};
                            }
                        }
            }
#pragma unroll
            for (int fn = 0; fn < FN_OUT; ++fn) {
#pragma unroll
                for (int gp = 0; gp < 2; ++gp) {
                    const int nq = col0 + fn * 32 + 16 * gp;
                    float o[2][4], pg[2][4], pu[2][4];
                    // GATED: this lane's 2 x 4 gate values (its row, columns nq + 8q + 4*khalf + 0..3)
                    float gate[2][4];
                    if constexpr (GATED) {
#pragma unroll
                        for (int q = 0; q < 2; ++q) {
                            const u32x2 g2 = graw[fn][gp][q];
                            gate[q][0] = __uint_as_float(g2[0] << 16);
                            gate[q][1] = __uint_as_float(g2[0] & 0xffff0000u);
                            gate[q][2] = __uint_as_float(g2[1] << 16);
                            gate[q][3] = __uint_as_float(g2[1] & 0xffff0000u);
                        }
                    }
                    // two columns at a time: one conversion instruction rounds a pair
#pragma unroll
                    for (int q = 0; q < 2; ++q)
#pragma unroll
                        for (int j = 0; j < 4; j += 2) {
                            const int v = 4 * (2 * gp + q) + j;
                            float ya = acc[fn][fm][v], yb = acc[fn][fm][v + 1];
                            float ua = SWIGLU ? acc[fn + FN / 2][fm][v] : 0.0f;
                            float ub = SWIGLU ? acc[fn + FN / 2][fm][v + 1] : 0.0f;
                            if (FP8) {
                                if (SCALE) {
                                    ya *= rsa[fm] * rsw[fn][gp][q][j];
                                    yb *= rsa[fm] * rsw[fn][gp][q][j + 1];
                                }
                                rbf2(ya, yb);
                                if (HAS_BIAS && p.bias) {
                                    ya += bv[fn][gp][q][j];
                                    yb += bv[fn][gp][q][j + 1];
                                    rbf2(ya, yb);
                                }
                                if (SWIGLU) {
                                    rbf2(ua, ub);
                                    if (HAS_BIAS && p.bias2) {
                                        ua += bv2[fn][gp][q][j];
                                        ub += bv2[fn][gp][q][j + 1];
                                        rbf2(ua, ub);
                                    }
                                }
                            } else {
                                if (HAS_BIAS) {
                                    ya += bv[fn][gp][q][j];
                                    yb += bv[fn][gp][q][j + 1];
                                }
                                rbf2(ya, yb);
                                if (SWIGLU) {
                                    if (HAS_BIAS) {
                                        ua += bv2[fn][gp][q][j];
                                        ub += bv2[fn][gp][q][j + 1];
                                    }
                                    rbf2(ua, ub);
                                }
                                if constexpr (GATED) {      // the product so far is the factor, the gate the argument
                                    ua = ya;
                                    ub = yb;
                                    ya = gate[q][j];
                                    yb = gate[q][j + 1];
                                }
                            }
                            pg[q][j] = ya;
                            pg[q][j + 1] = yb;
                            pu[q][j] = ua;
                            pu[q][j + 1] = ub;
                            if (EPI == FMOE_EPI_SILU) {
                                ya = fast_silu_f32(ya);
                                yb = fast_silu_f32(yb);
                            }
                            if (SWIGLU || GATED) {
                                ya = fast_silu_f32(ya);
                                yb = fast_silu_f32(yb);
                                rbf2(ya, yb);
                                ya *= ua;
                                yb *= ub;
                            }
                            o[q][j] = ya;
                            o[q][j + 1] = yb;
                        }
                    // base: first element of the 32-row block's first row (wave-uniform)
                    auto store = [&](const float (&val)[2][4], uint16_t* base, int64_t stride) {
                        if (p.vec_store) {
                            const uint32_t lane_off = lane_offset(stride);
                            // pair the quads of the two lane halves: low lanes end up with columns
                            // nq..nq+7, high lanes with nq+8..nq+15 of their row
                            const u32x2 s0 = __builtin_amdgcn_permlane32_swap(pack_bf16(val[0][0], val[0][1]),
                                                                              pack_bf16(val[1][0], val[1][1]), false, false);
                            const u32x2 s1 = __builtin_amdgcn_permlane32_swap(pack_bf16(val[0][2], val[0][3]),
                                                                              pack_bf16(val[1][2], val[1][3]), false, false);
                            const int nb = nq + 8 * khalf;
                            if (row_ok[fm] && nb + 7 < p.N)
                                *reinterpret_cast<u32x4*>(reinterpret_cast<uint8_t*>(base + nq) + lane_off) =
                                    u32x4{s0[0], s1[0], s0[1], s1[1]};
                        } else if (row_ok[fm]) {
                            uint16_t* dst = base + (int64_t)(lane & 31) * stride;
#pragma unroll
                            for (int q = 0; q < 2; ++q)
#pragma unroll
                                for (int j = 0; j < 4; ++j) {
                                    const int n = nq + 8 * q + 4 * khalf + j;
                                    if (n < p.N) dst[n] = (uint16_t)f32_to_bf16_bits(val[q][j]);
                                }
                        }
                    };
                    const int64_t block_row = row0 + frag_row(fm);
                    uint16_t* obase = p.out + block_row * p.out_stride;
                    store(o, obase, p.out_stride);
                    if (HAS_AUX) {
                        store(pg, p.aux + block_row * p.aux_stride, p.aux_stride);
                        store(pu, p.aux2 + block_row * p.aux_stride, p.aux_stride);
                    }
                    // one column group at a time: interleaving the groups for more parallelism
                    // is what runs the scheduler out of registers here
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
        }
        // Everything older than this epilogue's own stores has completed: a wait that costs
        // nothing (the loads it names were needed above) but tells the compiler so.  Without it
        // a spill reload that one of the branches above leaves unused stays "pending" in the
        // compiler's count, and the wait for it lands where its register is next written:
        // inside the caller's steady-state loop, where it would also drain the LDS-DMA stream,
        // which the compiler cannot see, on every iteration.
        FMOE_EPI_STAMP(FM);
        // The number of store instructions issued above, whatever the lanes' predicates: 4 per row
        // block of 64 columns in the staged form, one per column group (and per output tensor) otherwise (as many).
        // The ring kernel's first double step of the next tile skips its own counted wait on the
        // strength of this one (see skip_wait there), which is only sound when every one of these
        // stores was issued unconditionally, i.e. through store16_uniform_base (ALWAYS_VEC).
        constexpr int kStoresIssued = FM * FN_OUT * 2 * (HAS_AUX ? 3 : 1);
        static_assert(kStoresIssued <= 63, "vmcnt is a 6-bit field");
        wait_vmcnt<kStoresIssued>();      // (the element-store path issues more)
        after_stores();
    };
    if (SWIGLU && p.aux) {
        if (p.bias || p.bias2) run(std::true_type{}, std::true_type{});
        else run(std::false_type{}, std::true_type{});
    } else {
        if (p.bias || p.bias2) run(std::true_type{}, std::false_type{});
        else run(std::false_type{}, std::false_type{});
    }
}

// fp32 operands: fp32 bias and output, no intermediate rounding, exact SiLU.
template <int FM, int FN, int TM, int TN, int EPI>
__device__ __forceinline__ void gemm_epilogue_f32(const GemmParams& p, f32x16 (&acc)[FN][FM], int expert,
                                                  int n0, int64_t row0, int rows_valid, int wm, int wn,
                                                  int lane) {
    constexpr bool SWIGLU = EPI == FMOE_EPI_SWIGLU;
    constexpr int FN_OUT = SWIGLU ? FN / 2 : FN;
    const int khalf = lane >> 5;
    const float* bias = reinterpret_cast<const float*>(p.bias);
    const float* bias2 = reinterpret_cast<const float*>(p.bias2);
    float* out = reinterpret_cast<float*>(p.out);
    const int64_t bias_row = (int64_t)expert * p.bias_se;
#pragma unroll
    for (int fn = 0; fn < FN_OUT; ++fn) {
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            const int nb = n0 + (SWIGLU ? wn * (TN / 2) : wn * TN) + fn * 32 + 8 * g + 4 * khalf;
            float bv[4], bv2[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int nc = nb + j < p.N ? nb + j : p.N - 1;
                bv[j] = bias ? bias[bias_row + nc] : 0.0f;
                bv2[j] = (SWIGLU && bias2) ? bias2[bias_row + nc] : 0.0f;
            }
#pragma unroll
            for (int fm = 0; fm < FM; ++fm) {
                const int tile_row = wm * TM + fm * 32 + (lane & 31);
                if (tile_row >= rows_valid) continue;
                float* orow = out + (row0 + tile_row) * p.out_stride;
                float o[4], pg[4], pu[4];
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    float y = acc[fn][fm][4 * g + j] + bv[j];
                    pg[j] = y;
                    pu[j] = SWIGLU ? acc[fn + FN / 2][fm][4 * g + j] + bv2[j] : 0.0f;
                    if (EPI == FMOE_EPI_SILU) y = silu_f32(y);
                    if (SWIGLU) y = silu_f32(y) * pu[j];
                    o[j] = y;
                }
                auto store = [&](const float (&val)[4], float* dst) {
                    if (p.vec_store && nb + 3 < p.N) {
                        *reinterpret_cast<f32x4*>(dst + nb) = f32x4{val[0], val[1], val[2], val[3]};
                    } else {
#pragma unroll
                        for (int j = 0; j < 4; ++j)
                            if (nb + j < p.N) dst[nb + j] = val[j];
                    }
                };
                store(o, orow);
                if (SWIGLU && p.aux) {
                    store(pg, reinterpret_cast<float*>(p.aux) + (row0 + tile_row) * p.aux_stride);
                    store(pu, reinterpret_cast<float*>(p.aux2) + (row0 + tile_row) * p.aux_stride);
                }
            }
        }
    }
}

}  // namespace fmoe
