// fmoe_gate_softmax: the gate of a small batch, scores = softmax(x W^T + b), in one launch.
//
// What it is for: 64 tokens, 8 experts, 128 inputs: the library GEMM with its bias epilogue takes 25 us of host time to issue and 5 us to run, the
// softmax 6 and 3; this kernel 4 us to issue and as long to run.  A batch of few tokens is a chain of such launches (the layer's pass
// 61 us, bound by the host).  Logits are fp32 sums plus bias rounded to the scores' type, as torch.nn.functional.linear rounds
// them, and the softmax is torch's, step by step (one wave per token, expert e in lane e % 64, butterfly sums from the
// widest distance down).
#include "common.h"

namespace fmoe {
namespace {

constexpr int kGateWaves = 8, kGateTokens = 16, kGateMostExperts = 96;

// Block: 16 tokens x all experts on 16 x 16 MFMAs, weights from the A port.  The waves share K in pieces of 64 bytes per row (a lane's
// 16 bytes of row lane % 16 at 16 * (lane / 16); the order of k inside a piece is the same on both sides, so it is free) and
// their sums are added in LDS in wave order.  What bounds it is the chain of loads: 2048 inputs, 64 experts 7 us.
template <bool F32, int NF>
__global__ __launch_bounds__(kGateWaves* kWave) void gate_softmax_kernel(const uint8_t* __restrict__ x, int64_t T, int D, int64_t x_stride,
                                                                       const uint8_t* __restrict__ w, const void* __restrict__ bias,
                                                                       int E, void* __restrict__ scores) {
    constexpr int ESIZE = F32 ? 4 : 2, LD = NF * 16 + 4;
    extern __shared__ float red[];              // [wave][token][LD]
    const int lane = lane_id(), wave = threadIdx.x / kWave, r16 = lane & 15, quarter = lane >> 4;
    const int64_t t0 = (int64_t)blockIdx.x * kGateTokens;
    const int kbytes = D * ESIZE, pieces = (kbytes + 63) / 64;
    const int64_t token = t0 + r16 < T ? t0 + r16 : T - 1;
    const uint8_t* const xrow = x + token * x_stride * ESIZE + 16 * quarter;
    const uint8_t* wrow[NF];
#pragma unroll
    for (int f = 0; f < NF; ++f) wrow[f] = w + (int64_t)(16 * f + r16 < E ? 16 * f + r16 : E - 1) * kbytes + 16 * quarter;
    f32x4 acc[NF];
#pragma unroll
    for (int f = 0; f < NF; ++f) acc[f] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    constexpr int AHEAD = NF <= 2 ? 4 : 2;      // pieces on their way
    u32x4 xv[AHEAD], wv[AHEAD][NF];
    auto load = [&](int c, int i) {
        const bool in = c * 64 + 16 * quarter < kbytes;         // (rows are whole 16-byte chunks)
        const u32x4 zero = {0, 0, 0, 0};
        xv[i] = in ? *reinterpret_cast<const u32x4*>(xrow + c * 64) : zero;
#pragma unroll
        for (int f = 0; f < NF; ++f) wv[i][f] = in ? *reinterpret_cast<const u32x4*>(wrow[f] + c * 64) : zero;
    };
#pragma unroll
    for (int i = 0; i < AHEAD; ++i) load(wave + i * kGateWaves, i);
    for (int c0 = wave; c0 < pieces; c0 += AHEAD * kGateWaves) {
#pragma unroll
        for (int i = 0; i < AHEAD; ++i) {
            const int c = c0 + i * kGateWaves;
            if (c >= pieces) break;
#pragma unroll
            for (int f = 0; f < NF; ++f) {
                if constexpr (F32) {
#pragma unroll
                    for (int j = 0; j < 4; ++j)
                        acc[f] = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(wv[i][f][j]), __uint_as_float(xv[i][j]), acc[f], 0, 0, 0);
                } else {
                    acc[f] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, wv[i][f]), __builtin_bit_cast(bf16x8, xv[i]),
                                                                     acc[f], 0, 0, 0);
                }
            }
            load(c + AHEAD * kGateWaves, i);
        }
    }
    // lane l: experts 16 * f + 4 * (l / 16) .. + 3 of token l % 16
#pragma unroll
    for (int f = 0; f < NF; ++f)
        *reinterpret_cast<f32x4*>(red + (wave * kGateTokens + r16) * LD + 16 * f + 4 * quarter) = acc[f];
    __syncthreads();
    constexpr int PER = (NF * 16 + kWave - 1) / kWave;          // experts of a lane
    for (int t = wave; t < kGateTokens; t += kGateWaves) {
        if (t0 + t >= T) break;
        float v[PER], most = -__builtin_inff();
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            const int e = i * kWave + lane;
            v[i] = -__builtin_inff();
            if (e < E) {
                float s = red[t * LD + e];
#pragma unroll
                for (int j = 1; j < kGateWaves; ++j) s += red[(j * kGateTokens + t) * LD + e];
                if (bias) s += F32 ? reinterpret_cast<const float*>(bias)[e] : bf16_bits_to_f32(reinterpret_cast<const uint16_t*>(bias)[e]);
                v[i] = F32 ? s : round_bf16(s);
            }
            most = most > v[i] ? most : v[i];
        }
#pragma unroll
        for (int o = kWave / 2; o >= 1; o >>= 1) {
            const float other = __shfl_xor(most, o, kWave);
            most = most < other ? other : most;
        }
        float sum = 0.0f;
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            v[i] = i * kWave + lane < E ? expf(v[i] - most) : 0.0f;
            sum += v[i];
        }
#pragma unroll
        for (int o = kWave / 2; o >= 1; o >>= 1) sum += __shfl_xor(sum, o, kWave);
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            const int e = i * kWave + lane;
            if (e >= E) continue;
            const float p = v[i] / sum;
            if constexpr (F32) reinterpret_cast<float*>(scores)[(t0 + t) * E + e] = p;
            else reinterpret_cast<uint16_t*>(scores)[(t0 + t) * E + e] = (uint16_t)f32_to_bf16_bits(p);
        }
    }
}

}  // namespace
}  // namespace fmoe

using namespace fmoe;

static int gate_fragments(int E) { return E <= 16 ? 1 : E <= 32 ? 2 : E <= 64 ? 4 : 6; }

// Batches whose pass is bound by the host (a library GEMM and a softmax take 26 us to issue, this 7) or by its chain of launches; a larger one has
// the library GEMM's rate to lose.  A block's eight waves walk all of K, 3 us and 0.25 for every KB of a gate row times 1 + 2 * fragments, where the
// library's two launches take 7 to 12: us on the GPU, library / kernel, 64 tokens: bf16 128 inputs, 8 experts 7.0 / 3.8; 1024, 64 8.8 / 7.9; 2048, 96
// 8.9 / 16.6; 4096, 64 10.4 / 20.9; 8192, 96 11.6 / 52; fp32 1024, 64 7.9 / 12.6; 2048, 64  - / 20; 8192, 96 18.6 / 101.  The line is where that is as
// much as what issuing them costs a pass.  us of a layer's pass (top-2) among others and alone, library / kernel: bf16, 2048 inputs, 96 experts, 1 token 63 / 42 and
// 85 / 61, 16 tokens 58 / 59 and 94 / 78, 128 tokens 128 / 130 and 164 / 147; beyond it 4096, 64, 1 token 62 / 50 and 90 / 69, 16 tokens 66 / 71 and 102 / 90;
// fp32 4096, 64, 16 tokens 118 / 147 and 153 / 164.
extern "C" int fmoe_gate_softmax_pays(int dtype, int64_t T, int D, int E) {
    if ((dtype != FMOE_BF16 && dtype != FMOE_F32) || T < 1 || T > 128 || E < 1 || E > kGateMostExperts || D < 1) return 0;
    const int chunk = dtype == FMOE_F32 ? 4 : 8;
    return D % chunk == 0 && (int64_t)D * (16 / chunk) * (1 + 2 * gate_fragments(E)) <= 56 * 1024;
}

extern "C" int fmoe_gate_softmax(const void* x, int dtype, int64_t T, int D, int64_t x_stride_row, const void* weight, const void* bias, int E,
                                 void* scores, fmoe_stream_t stream_) {
    FMOE_REQUIRE(dtype == FMOE_BF16 || dtype == FMOE_F32, "fmoe_gate_softmax: bf16 or fp32 expected");
    FMOE_REQUIRE(T >= 0 && D >= 1 && E >= 1, "fmoe_gate_softmax: need T >= 0, D, E >= 1");
    if (T == 0) return FMOE_OK;
    const int chunk = dtype == FMOE_F32 ? 4 : 8;
    FMOE_REQUIRE(x && weight && scores, "fmoe_gate_softmax: NULL tensor pointer");
    FMOE_REQUIRE(E <= kGateMostExperts && D <= (1 << 24) && D % chunk == 0 && x_stride_row >= D && x_stride_row % chunk == 0 && aligned16(x) &&
                     aligned16(weight) && T < ((int64_t)1 << 31),
                 "fmoe_gate_softmax: up to %d experts, rows of whole 16-byte chunks at 16-byte boundaries", kGateMostExperts);
    auto go = [&](auto kern, int nf) {
        const size_t lds = (size_t)kGateWaves * kGateTokens * (nf * 16 + 4) * sizeof(float);
        kern<<<(unsigned)((T + kGateTokens - 1) / kGateTokens), kGateWaves * kWave, lds, (hipStream_t)stream_>>>(
            (const uint8_t*)x, T, D, x_stride_row, (const uint8_t*)weight, bias, E, scores);
        return check_launch("fmoe_gate_softmax");
    };
#define FMOE_GATE(NF) (dtype == FMOE_F32 ? go(gate_softmax_kernel<true, NF>, NF) : go(gate_softmax_kernel<false, NF>, NF))
    switch (gate_fragments(E)) {
        case 1: return FMOE_GATE(1);
        case 2: return FMOE_GATE(2);
        case 4: return FMOE_GATE(4);
        default: return FMOE_GATE(6);
    }
#undef FMOE_GATE
}
