// The gate of a batch of few tokens: logits on 16 x 16 MFMAs, softmax by waves (gate.hip, and with the routing in one block routing.hip).
#pragma once

#include "common.h"

namespace fmoe {

constexpr int kGateWaves = 8, kGateTokens = 16, kGateMostExperts = 96;
inline int gate_fragments(int E) { return E <= 16 ? 1 : E <= 32 ? 2 : E <= 64 ? 4 : 6; }
constexpr int gate_sums_row(int nf) { return nf * 16 + 4; }
constexpr int gate_sums_floats(int nf) { return kGateWaves * kGateTokens * gate_sums_row(nf); }

// The sums of tokens t0 .. t0 + 15 by the eight waves of a group: red [wave][token][gate_sums_row].  The waves share K in pieces of 64 bytes per
// row (a lane's 16 bytes of row lane % 16 at 16 * (lane / 16); the order of k inside a piece is the same on both sides, so it is free).
template <bool F32, int NF>
__device__ __forceinline__ void gate_sums(const uint8_t* __restrict__ x, int64_t T, int D, int64_t x_stride, const uint8_t* __restrict__ w, int E,
                                          int64_t t0, int wave, float* red) {
    constexpr int ESIZE = F32 ? 4 : 2, LD = gate_sums_row(NF);
    const int lane = lane_id(), r16 = lane & 15, quarter = lane >> 4;
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
}

// Softmax of the tokens t .. t + gate_wave_tokens - 1 of a group (those below `tokens`): the waves' sums added in wave order, bias, logits
// rounded to the type; put(token, expert, probability).  A wave has 64 / (16 * NF) tokens side by side (one after the other they are a chain of
// twelve shuffles each); the wider steps of a 64-lane butterfly only add zeros there.
constexpr int gate_lanes(int nf) { return nf * 16 < kWave ? nf * 16 : kWave; }
constexpr int gate_wave_tokens(int nf) { return kWave / gate_lanes(nf); }
template <bool F32, int NF, typename Put>
__device__ __forceinline__ void gate_softmax_tokens(const float* red, int t, int tokens, const void* __restrict__ bias, int E, Put&& put) {
    constexpr int LD = gate_sums_row(NF), LANES = gate_lanes(NF);
    const int lane = lane_id() % LANES;
    t += lane_id() / LANES;
    const bool live = t < tokens;
    if (!live) t = tokens - 1;
    constexpr int PER = (NF * 16 + kWave - 1) / kWave;          // experts of a lane
    float v[PER], most = -__builtin_inff();
#pragma unroll
    for (int i = 0; i < PER; ++i) {
        const int e = i * LANES + lane;
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
    for (int o = LANES / 2; o >= 1; o >>= 1) {
        const float other = __shfl_xor(most, o, kWave);
        most = most < other ? other : most;
    }
    float sum = 0.0f;
#pragma unroll
    for (int i = 0; i < PER; ++i) {
        v[i] = i * LANES + lane < E ? expf(v[i] - most) : 0.0f;
        sum += v[i];
    }
#pragma unroll
    for (int o = LANES / 2; o >= 1; o >>= 1) sum += __shfl_xor(sum, o, kWave);
#pragma unroll
    for (int i = 0; i < PER; ++i) {
        const int e = i * LANES + lane;
        if (live && e < E) put(t, e, v[i] / sum);
    }
}

}  // namespace fmoe
