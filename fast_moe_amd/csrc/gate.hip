// fmoe_gate_softmax: the gate of a small batch, scores = softmax(x W^T + b), in one launch.
//
// What it is for: 64 tokens, 8 experts, 128 inputs: the library GEMM with its bias epilogue takes 25 us of host time to issue and 5 us to run, the
// softmax 6 and 3; this kernel 4 us to issue and as long to run.  A batch of few tokens is a chain of such launches (the layer's pass
// 61 us, bound by the host).  Logits are fp32 sums plus bias rounded to the scores' type, as torch.nn.functional.linear rounds
// them, and the softmax is torch's, step by step (expert e in lane e % 64 of a token's, butterfly sums from the widest
// distance down; up to 32 experts a wave has two tokens, up to 16 four, whose wider steps would only add zeros).
#include "gate.h"

namespace fmoe {
namespace {

// Block: 16 tokens x all experts on 16 x 16 MFMAs, weights from the A port, the eight waves' sums added in LDS in wave order.  What bounds it is the
// chain of loads: 2048 inputs, 64 experts 7 us.
template <bool F32, int NF>
__global__ __launch_bounds__(kGateWaves* kWave) void gate_softmax_kernel(const uint8_t* __restrict__ x, int64_t T, int D, int64_t x_stride,
                                                                       const uint8_t* __restrict__ w, const void* __restrict__ bias,
                                                                       int E, void* __restrict__ scores) {
    extern __shared__ float red[];
    const int wave = threadIdx.x / kWave;
    const int64_t t0 = (int64_t)blockIdx.x * kGateTokens;
    gate_sums<F32, NF>(x, T, D, x_stride, w, E, t0, wave, red);
    __syncthreads();
    const int tokens = T - t0 < kGateTokens ? (int)(T - t0) : kGateTokens;
    constexpr int STEP = gate_wave_tokens(NF);
    for (int first = wave * STEP; first < tokens; first += kGateWaves * STEP)
        gate_softmax_tokens<F32, NF>(red, first, tokens, bias, E, [&](int t, int e, float p) {
            if constexpr (F32) reinterpret_cast<float*>(scores)[(t0 + t) * E + e] = p;
            else reinterpret_cast<uint16_t*>(scores)[(t0 + t) * E + e] = (uint16_t)f32_to_bf16_bits(p);
        });
}

}  // namespace
}  // namespace fmoe

using namespace fmoe;

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
        const size_t lds = (size_t)gate_sums_floats(nf) * sizeof(float);
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
