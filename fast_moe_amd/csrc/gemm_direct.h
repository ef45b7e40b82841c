// Streaming grouped GEMM for a handful of rows per expert and few tiles: weights from memory straight into the registers of the
// wave that multiplies them.
#pragma once

#include "gemm_f32x3.h"

namespace fmoe {

// A block computes up to BM rows x 64 weight columns (SwiGLU: 32 of gate and the same 32 of up), its NW waves split K: wave w takes
// the 128-byte pieces w, w + NW, ... of every row.  A load instruction brings 64 contiguous bytes of each of 16 rows, 16 per lane, as
// the 16 x 16 MFMAs take them: the order of k inside a piece is the same for weights and activations, so it is free.  No LDS and no
// barrier on the way of the weights; the waves' sums meet in LDS once per tile, added in wave order.  A tile multiplies as many
// 16-row fragments as it has rows for (1, 2 or 4): an expert with one row costs its weights, a hot one is not read per 16 rows.
//
// What bounds it: in a launch of few tiles the chain from offsets[] over row_index to the first activations, about 6 us with the
// launch; with all CUs busy the 64-byte pieces a CU can ask for, about 30 KB/us (32 x 32 MFMAs, whose loads touch 32 rows, half as
// fast: 512 rows, 128 experts, 4096 -> 2 x 1536 586 us, now 525 to 529).
template <int DT, int NW_>
struct DirectCfg {
    static constexpr int NW = NW_, SETS = NW == 4 ? 2 : 1;      // pieces of weights a wave has on their way
    static constexpr int FM = DT == kDtF32 ? 2 : 4, BM = 16 * FM;
    static constexpr int NT = kWave * NW;
    static constexpr int LDS_BYTES = NW * 2 * 4 * 64 * 16;      // the sums of two fragments: [wave][2][4][64] x 16 bytes
};

// inclusive prefix sum over the 64 lanes on the DPP network
__device__ __forceinline__ int wave_scan_dpp(int v) {
    v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, true);      // row_shr 1, 2, 4, 8 (rows of 16 lanes)
    v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, true);
    v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, true);
    v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, true);
    v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, true);      // last lane of rows 0 and 2 into rows 1 and 3
    v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, true);      // lane 31 into rows 2 and 3
    return v;
}

// BlockTile (gemm_staged.h) for total_rows < 2^31, in 32-bit arithmetic, everything wave-uniform: a tile is little more than the latency of
// its first loads here, and locating it comes before them.
struct BlockTile32 {
    int expert, nt, row0, rows_valid;

    __device__ __forceinline__ bool locate(const GemmParams& p, int BM) {
        const int lane = threadIdx.x & 63, R = (int)p.total_rows;
        auto rows_of = [&](int e, int& lo) -> int {
            lo = 0;
            if (e >= p.E) return 0;
            lo = (int)clamp_i64(p.offsets[e], 0, R);
            const int hi = (int)clamp_i64(p.offsets[e + 1], 0, R);
            return hi > lo ? hi - lo : 0;
        };
        int total_m = 0, lo, len, inc = 0;
        for (int e0 = 0; e0 < p.E; e0 += kWave) {
            len = rows_of(e0 + lane, lo);
            inc = wave_scan_dpp((len + BM - 1) / BM);
            total_m += __builtin_amdgcn_readlane(inc, 63);
        }
        const int total = total_m * p.n_tiles, per_xcd = (total + kNumXcd - 1) / kNumXcd;
        const int slot = blockIdx.x / kNumXcd, logical = blockIdx.x % kNumXcd * per_xcd + slot;
        if (slot >= per_xcd || logical >= total) return false;
        const int span = kGroupM * p.n_tiles, group = logical / span, within = logical - group * span;
        const int gsize = total_m - group * kGroupM < kGroupM ? total_m - group * kGroupM : kGroupM;
        const int mt = group * kGroupM + within % gsize;
        nt = within / gsize;
        int before = 0;
        for (int e0 = 0; e0 < p.E; e0 += kWave) {
            if (p.E > kWave) {
                len = rows_of(e0 + lane, lo);
                inc = wave_scan_dpp((len + BM - 1) / BM);
            }
            const unsigned long long hit = __ballot(mt < before + inc);
            if (hit) {
                const int src = __builtin_ctzll(hit);
                expert = e0 + src;
                const int tiles = (__builtin_amdgcn_readlane(len, src) + BM - 1) / BM;
                const int skip = (mt - (before + __builtin_amdgcn_readlane(inc, src) - tiles)) * BM;
                row0 = __builtin_amdgcn_readlane(lo, src) + skip;
                const int left = __builtin_amdgcn_readlane(len, src) - skip;
                rows_valid = left < BM ? left : BM;
                return rows_valid > 0;
            }
            before += __builtin_amdgcn_readlane(inc, 63);
        }
        return false;
    }
};

template <typename CF, int DT, int EPI, bool A_SILU, int FM, int SETS>
__device__ __forceinline__ void direct_tile(const GemmParams& p, const BlockTile32& tile) {
    constexpr int NW = CF::NW, NT = CF::NT;
    constexpr bool FP8 = DT == kDtE4m3, F32 = DT == kDtF32, SWIGLU = EPI == FMOE_EPI_SWIGLU;
    constexpr int ESIZE = FP8 ? 1 : F32 ? 4 : 2;
    extern __shared__ __align__(16) uint8_t smem[];
    const int tid = threadIdx.x;
    const int lane = tid & 63, r16 = lane & 15, quarter = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int expert = tile.expert, rows_valid = tile.rows_valid, n0 = tile.nt * (SWIGLU ? 32 : 64);
    const int kbytes = p.K * ESIZE;
    const int pieces = (kbytes + 127) / 128;

    // the lane's 16 bytes of the first half of piece 0 of its row of weight fragment f and of activation fragment fm
    const uint8_t *wrow[4], *xrow[FM];
    bool row_ok[FM];
#pragma unroll
    for (int f = 0; f < 4; ++f) {
        const int n = n0 + 16 * (SWIGLU ? f & 1 : f) + r16;
        wrow[f] = (SWIGLU && f >= 2 ? p.b2 : p.b) + ((int64_t)expert * p.b_se + (int64_t)(n < p.N ? n : p.N - 1) * p.b_sn) * ESIZE + 16 * quarter;
    }
    auto load = [&](const uint8_t* row, int piece, bool ok, u32x4 (&v)[2]) {
        const int at = piece * 128;
        const bool whole = at + 128 <= kbytes;      // uniform
#pragma unroll
        for (int i = 0; i < 2; ++i)
            v[i] = ok && (whole || at + 64 * i + 16 * quarter < kbytes) ? *reinterpret_cast<const u32x4*>(row + at + 64 * i) : u32x4{0, 0, 0, 0};
    };
    u32x4 ws[SETS][4][2], xs[SETS][FM][2];
    auto load_w = [&](int piece, u32x4 (&w)[4][2]) {
#pragma unroll
        for (int f = 0; f < 4; ++f) load(wrow[f], piece, true, w[f]);
    };
    auto load_x = [&](int piece, u32x4 (&x)[FM][2]) {
#pragma unroll
        for (int fm = 0; fm < FM; ++fm) load(xrow[fm], piece, row_ok[fm], x[fm]);
    };
#pragma unroll
    for (int s = 0; s < SETS; ++s)
        if (wave + s * NW < pieces) load_w(wave + s * NW, ws[s]);
#pragma unroll
    for (int fm = 0; fm < FM; ++fm) {
        const int r = 16 * fm + r16;
        row_ok[fm] = r < rows_valid;
        xrow[fm] = p.a + ((int64_t)expert * p.a_stride_e + source_row(p, tile.row0 + (row_ok[fm] ? r : 0)) * p.a_stride_row) * ESIZE + 16 * quarter;
    }
#pragma unroll
    for (int s = 0; s < SETS; ++s)
        if (wave + s * NW < pieces) load_x(wave + s * NW, xs[s]);

    // fp32: the sums of the largest partial products, and of the others (gemm_f32x3.h)
    constexpr int SUMS = F32 ? 2 : 1;
    f32x4 acc[4 * SUMS][FM];
    auto multiply = [&](auto exact_c, const u32x4 (&w)[4][2], u32x4 (&x)[FM][2]) {
        constexpr bool EXACT = decltype(exact_c)::value;        // fp32 operands on fp32 MFMAs
        if constexpr (A_SILU) {
#pragma unroll
            for (int fm = 0; fm < FM; ++fm)
#pragma unroll
                for (int i = 0; i < 2; ++i) x[fm][i] = F32 ? silu_f32x4(x[fm][i]) : silu_bf16x8(x[fm][i]);
        }
        if constexpr (F32 && EXACT) {
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j)
#pragma unroll
                    for (int f = 0; f < 4; ++f)
#pragma unroll
                        for (int fm = 0; fm < FM; ++fm)
                            acc[f][fm] = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(w[f][i][j]), __uint_as_float(x[fm][i][j]),
                                                                             acc[f][fm], 0, 0, 0);
        } else if constexpr (F32) {
            auto parts = [&](const u32x4 (&v)[2], bf16x8 (&out)[3]) {
                u32x4 q[3];
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    uint32_t h, m, l;
                    split3(__uint_as_float(v[j >> 1][2 * (j & 1)]) * kF32x3Scale, __uint_as_float(v[j >> 1][2 * (j & 1) + 1]) * kF32x3Scale, h, m, l);
                    q[0][j] = h;
                    q[1][j] = m;
                    q[2][j] = l;
                }
#pragma unroll
                for (int i = 0; i < 3; ++i) out[i] = __builtin_bit_cast(bf16x8, q[i]);
            };
            bf16x8 xp[FM][3];
#pragma unroll
            for (int fm = 0; fm < FM; ++fm) parts(x[fm], xp[fm]);
            FMOE_F32X3_TERMS;
#pragma unroll
            for (int f = 0; f < 4; ++f) {
                bf16x8 wp[3];
                parts(w[f], wp);
#pragma unroll
                for (int t = 0; t < 8; ++t)
#pragma unroll
                    for (int fm = 0; fm < FM; ++fm) {
                        f32x4& sum = acc[t ? 4 + f : f][fm];
                        sum = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wp[W[t]], xp[fm][X[t]], sum, 0, 0, 0);
                    }
            }
        } else if constexpr (FP8) {
            auto join = [&](const u32x4 (&v)[2]) -> i32x8 {
                return i32x8{(int)v[0][0], (int)v[0][1], (int)v[0][2], (int)v[0][3], (int)v[1][0], (int)v[1][1], (int)v[1][2], (int)v[1][3]};
            };
#pragma unroll
            for (int f = 0; f < 4; ++f)
#pragma unroll
                for (int fm = 0; fm < FM; ++fm)
                    acc[f][fm] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(join(w[f]), join(x[fm]), acc[f][fm], 0, 0, 0, 0, 0, 0);
        } else {
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int f = 0; f < 4; ++f)
#pragma unroll
                    for (int fm = 0; fm < FM; ++fm)
                        acc[f][fm] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, w[f][i]),
                                                                            __builtin_bit_cast(bf16x8, x[fm][i]), acc[f][fm], 0, 0, 0);
        }
    };
    // the first SETS pieces of the wave are in its registers already
    auto contract = [&](auto exact_c) {
#pragma unroll
        for (int f = 0; f < 4 * SUMS; ++f)
#pragma unroll
            for (int fm = 0; fm < FM; ++fm) acc[f][fm] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
        for (int c = wave; c < pieces; c += SETS * NW) {
#pragma unroll
            for (int s = 0; s < SETS; ++s) {
                if (c + s * NW >= pieces) break;
                multiply(exact_c, ws[s], xs[s]);
                const int next = c + (s + SETS) * NW;
                if (next < pieces) {
                    load_w(next, ws[s]);
                    load_x(next, xs[s]);
                }
            }
        }
    };

    // Lane l's sums are columns 16 * f + 4 * (l / 16) .. + 3 of row l % 16 of fragment fm; group c4 = 4 * f + l / 16 of 4 columns lies in
    // slot (l % 16) ^ c4 of its 16, so that neither writing by rows nor reading by columns has bank conflicts.
    f32x4* const red = reinterpret_cast<f32x4*>(smem);
    const int64_t bias_row = (int64_t)expert * p.bias_se;
    constexpr int STEP = FM < 2 || F32 ? 1 : 2;         // fragments whose sums LDS holds at a time
    constexpr int PER_WAVE = STEP * SUMS * 256;
    auto finish = [&](int fm0, float scale) -> bool {
        bool finite = true;
#pragma unroll
        for (int i = 0; i < STEP; ++i)
#pragma unroll
            for (int f = 0; f < 4 * SUMS; ++f) {
                const int c4 = 4 * (f & 3) + quarter;
                red[wave * PER_WAVE + ((i * SUMS + (f >> 2)) * 16 + c4) * 16 + (r16 ^ c4)] = acc[f][fm0 + i];
            }
        __syncthreads();
        constexpr int GROUPS = SWIGLU ? 8 : 16;         // of 4 output columns
        for (int q = tid; q < 16 * STEP * GROUPS; q += NT) {
            const int row = 16 * fm0 + q / GROUPS, c4 = q % GROUPS;
            if (row >= rows_valid) break;
            f32x4 sum[2];
#pragma unroll
            for (int h = 0; h < (SWIGLU ? 2 : 1); ++h) {
                const int c = c4 + 8 * h, at = (((row >> 4) - fm0) * SUMS * 16 + c) * 16 + ((row & 15) ^ c);
                f32x4 total[SUMS];
#pragma unroll
                for (int s = 0; s < SUMS; ++s) {
                    total[s] = red[s * 256 + at];
#pragma unroll
                    for (int i = 1; i < NW; ++i) {
                        const f32x4 part = red[i * PER_WAVE + s * 256 + at];
#pragma unroll
                        for (int j = 0; j < 4; ++j) total[s][j] += part[j];
                    }
                }
                sum[h] = total[0];
                if constexpr (F32) {
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        sum[h][j] += total[1][j];
                        finite &= __builtin_fabsf(sum[h][j]) < __builtin_inff();
                        sum[h][j] *= scale;
                    }
                }
            }
            const int64_t out_row = (int64_t)tile.row0 + row;
            const int n = n0 + 4 * c4;
            float rs_a = 1.0f;
            if constexpr (FP8) rs_a = __builtin_amdgcn_rcpf(p.a_scale[source_row(p, out_row)]);
            float y[4], u[4], o[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int nc = n + j < p.N ? n + j : p.N - 1;
                auto value = [&](float v, const float* w_scale, const uint16_t* bias) -> float {
                    if constexpr (F32) return v + (bias ? reinterpret_cast<const float*>(bias)[bias_row + nc] : 0.0f);
                    if constexpr (FP8) {
                        v = rbf(v * (rs_a * __builtin_amdgcn_rcpf(w_scale[(int64_t)expert * p.N + nc])));
                        return bias ? rbf(v + bf16_bits_to_f32(bias[bias_row + nc])) : v;
                    }
                    return rbf(bias ? v + bf16_bits_to_f32(bias[bias_row + nc]) : v);
                };
                y[j] = value(sum[0][j], p.b_scale, p.bias);
                u[j] = SWIGLU ? value(sum[1][j], p.b2_scale, p.bias2) : 0.0f;
                o[j] = y[j];
                if constexpr (EPI != FMOE_EPI_NONE) o[j] = F32 ? silu_f32(y[j]) : fast_silu_f32(y[j]);
                if constexpr (SWIGLU) o[j] = (F32 ? o[j] : rbf(o[j])) * u[j];
            }
            auto store = [&](const float (&v)[4], uint16_t* base, int64_t stride) {
                const bool whole = p.vec_store && n + 3 < p.N;
                if constexpr (F32) {
                    float* dst = reinterpret_cast<float*>(base) + out_row * stride + n;
                    if (whole) *reinterpret_cast<f32x4*>(dst) = f32x4{v[0], v[1], v[2], v[3]};
                    else
#pragma unroll
                        for (int j = 0; j < 4; ++j)
                            if (n + j < p.N) dst[j] = v[j];
                } else {
                    uint16_t* dst = base + out_row * stride + n;
                    if (whole) *reinterpret_cast<u32x2*>(dst) = u32x2{pack_bf16(v[0], v[1]), pack_bf16(v[2], v[3])};
                    else
#pragma unroll
                        for (int j = 0; j < 4; ++j)
                            if (n + j < p.N) dst[j] = (uint16_t)f32_to_bf16_bits(v[j]);
                }
            };
            store(o, p.out, p.out_stride);
            if (SWIGLU && p.aux) {
                store(y, p.aux, p.aux_stride);
                store(u, p.aux2, p.aux_stride);
            }
        }
        return finite;
    };
    auto finish_all = [&](float scale) -> bool {
        bool finite = true;
#pragma unroll
        for (int fm = 0; fm < FM; fm += STEP) {
            if (fm) __syncthreads();
            finite &= finish(fm, scale);
        }
        return finite;
    };
    contract(std::false_type{});
    const bool finite = finish_all(kF32x3Unscale);
    if constexpr (F32) {            // (gemm_f32x3.h)
        if (__syncthreads_or(!finite)) {
#pragma unroll
            for (int s = 0; s < SETS; ++s)
                if (wave + s * NW < pieces) {
                    load_w(wave + s * NW, ws[s]);
                    load_x(wave + s * NW, xs[s]);
                }
            contract(std::true_type{});
            finish_all(1.0f);
        }
    }
}

template <typename CF, int DT, int EPI, bool A_SILU>
__global__ __launch_bounds__(CF::NT, 2) void grouped_gemm_direct_kernel(const GemmParams p) {
    BlockTile32 tile;
    if (!tile.locate(p, CF::BM)) return;
    if (tile.rows_valid <= 16) return direct_tile<CF, DT, EPI, A_SILU, 1, CF::SETS>(p, tile);
    if (tile.rows_valid <= 32) return direct_tile<CF, DT, EPI, A_SILU, 2, CF::SETS>(p, tile);
    if constexpr (CF::FM == 4) direct_tile<CF, DT, EPI, A_SILU, 4, 1>(p, tile);
}

}  // namespace fmoe
