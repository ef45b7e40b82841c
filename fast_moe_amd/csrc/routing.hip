// Routing for the MoE forward: top-k selection with L1-renormalised gates, the
// per-expert histogram / prefix sum ("jagged offsets") and the stable
// expert-major permutation with its inverse.  All integer outputs are a pure
// function of the selected ids (a stable counting sort), so they are
// reproducible bit for bit.
//
// Two launches on one stream (one for a batch of few tokens, route_block_kernel), no host synchronisation.  The tokens are cut into up to 256
// chunks (one block each: 16 waves up to 256 experts, 4 beyond; a wave owns a contiguous
// share of its chunk):
//   1. topk_hist_kernel (or compact_hist_kernel for caller-supplied ids): a token's scores sit
//      in a group of 8 or 16 lanes (4 to 8 tokens per wave); K rounds of a group argmax on the
//      DPP network select in descending order, ties to the lower expert id; every wave counts
//      the experts of its tokens in LDS -> sub_hist[chunk][wave][e], tot_hist[chunk][e]
//   2. scan_scatter_kernel: every block sums tot_hist over the chunks before it (and over all
//      chunks: lengths; wave scan over the experts: offsets), every wave adds the counts of
//      the waves before it in its chunk and then places its positions: a wave-level
//      match/rank gives each position its slot inside its expert segment
#include "gate.h"

#include <mutex>

namespace fmoe {
namespace {

constexpr int kMaxChunks = 256;
constexpr int kMaxRouteWaves = 16;
// waves per block of both kernels: 16 while the per-wave expert tables fit LDS comfortably
inline int route_waves(int E) { return E <= 256 ? 16 : 4; }
constexpr uint16_t kBadExpert = 0xFFFF;

struct RoutePlan {
    int64_t tokens_per_wave;
    int num_chunks;
    int wpb;                // waves per block
    size_t compact_bytes;   // uint16 expert id per routed position
    size_t sub_bytes;       // int32 [num_chunks][wpb][E]
    size_t tot_bytes;       // int32 [num_chunks][E]
    size_t bad_bytes;       // int32 [num_chunks] out-of-range ids per chunk
    size_t total_bytes;
};

RoutePlan make_plan(int64_t T, int E, int K) {
    RoutePlan p;
    const int kRouteWaves = route_waves(E);
    p.wpb = kRouteWaves;
    const int64_t waves = (int64_t)kMaxChunks * kRouteWaves;
    p.tokens_per_wave = (T + waves - 1) / waves;
    if (p.tokens_per_wave < 1) p.tokens_per_wave = 1;
    const int64_t per_chunk = p.tokens_per_wave * kRouteWaves;
    p.num_chunks = (int)((T + per_chunk - 1) / per_chunk);
    if (p.num_chunks < 1) p.num_chunks = 1;
    auto up = [](size_t v) { return (v + 255) & ~(size_t)255; };
    p.compact_bytes = up((size_t)T * (size_t)K * sizeof(uint16_t));
    p.sub_bytes = up((size_t)p.num_chunks * kRouteWaves * (size_t)E * sizeof(int32_t));
    p.tot_bytes = up((size_t)p.num_chunks * (size_t)E * sizeof(int32_t));
    p.bad_bytes = up((size_t)p.num_chunks * sizeof(int32_t));
    p.total_bytes = p.compact_bytes + p.sub_bytes + p.tot_bytes + p.bad_bytes + 256;
    return p;
}

struct RouteScratch {
    uint16_t* compact;
    int32_t* sub_hist;
    int32_t* tot_hist;
    int32_t* bad_part;
};

RouteScratch carve(void* workspace, const RoutePlan& plan) {
    char* w = (char*)workspace;
    RouteScratch r;
    r.compact = (uint16_t*)w;
    r.sub_hist = (int32_t*)(w + plan.compact_bytes);
    r.tot_hist = (int32_t*)(w + plan.compact_bytes + plan.sub_bytes);
    r.bad_part = (int32_t*)(w + plan.compact_bytes + plan.sub_bytes + plan.tot_bytes);
    return r;
}

template <typename T>
__device__ __forceinline__ float load_score(const T* p);
template <>
__device__ __forceinline__ float load_score<float>(const float* p) { return *p; }
template <>
__device__ __forceinline__ float load_score<uint16_t>(const uint16_t* p) { return bf16_bits_to_f32(*p); }

template <typename T>
__device__ __forceinline__ float round_to(float v);
template <>
__device__ __forceinline__ float round_to<float>(float v) { return v; }
template <>
__device__ __forceinline__ float round_to<uint16_t>(float v) { return round_bf16(v); }

template <typename T>
__device__ __forceinline__ void store_score(T* p, float v);
template <>
__device__ __forceinline__ void store_score<float>(float* p, float v) { *p = v; }
template <>
__device__ __forceinline__ void store_score<uint16_t>(uint16_t* p, float v) { *p = (uint16_t)f32_to_bf16_bits(v); }

// Total order on scores as unsigned keys: NaN above +inf (where torch.topk and torch.sort put
// it), -0 equal to +0, otherwise the order of the values.  With keys every token fills exactly K
// distinct slots whatever its scores hold; a float comparison ranks every NaN first at once.
__device__ __forceinline__ uint32_t order_key(float v) {
    const uint32_t b = __float_as_uint(v);
    if ((b & 0x7FFFFFFFu) > 0x7F800000u) return 0xFFFFFFFFu;     // NaN
    if ((b & 0x7FFFFFFFu) == 0u) return 0x80000000u;             // +-0
    return (b & 0x80000000u) ? ~b : (b | 0x80000000u);
}

// Largest value over each group of LPT (8 or 16) consecutive lanes, in every lane of the group:
// butterfly steps on the DPP network inside a row of 16 lanes (quad permutes, mirrors).
template <int LPT>
__device__ __forceinline__ uint32_t group_max_u32(uint32_t v) {
    static_assert(LPT == 8 || LPT == 16, "a group is half a DPP row or a whole one");
#define FMOE_DPP_MAX(ctrl) v = max(v, (uint32_t)__builtin_amdgcn_update_dpp((int)v, (int)v, ctrl, 0xF, 0xF, false))
    FMOE_DPP_MAX(0xB1);      // quad_perm [1,0,3,2]
    FMOE_DPP_MAX(0x4E);      // quad_perm [2,3,0,1]
    FMOE_DPP_MAX(0x141);     // row_half_mirror
    if (LPT == 16) FMOE_DPP_MAX(0x140);     // row_mirror
#undef FMOE_DPP_MAX
    return v;
}

// Orders this wave's LDS accesses for the compiler.  The hardware runs a wave's LDS instructions in
// order, and the regions touched between two of these belong to one wave: no block barrier needed.
__device__ __forceinline__ void wave_lds_fence() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// One token per LPT lanes (8 or 16: a token's lanes sit in one DPP row), VPL scores per lane
// (expert id = v*LPT + sub).  K rounds of "largest remaining key, lowest expert id among equal
// keys", each two group maxima on the DPP network; the round is the slot (descending score,
// ties -> lower expert id).  A wave takes tokens [w_begin, w_end), TPW of them per pass; compact (global memory or
// LDS) receives the expert ids of its positions, s_hist (this wave's, E entries, zeroed) their counts, s_sel is its scratch.
template <typename T, int LPT, int VPL>
__device__ __forceinline__ void select_experts(const T* __restrict__ scores, int64_t w_begin, int64_t w_end, int64_t tokens_per_wave,
                                               int E, int K, int renorm, int64_t* __restrict__ topk_idx, T* __restrict__ gates,
                                               uint16_t* compact, float (&s_sel)[kWave / LPT][64], int32_t* s_hist) {
    constexpr int TPW = kWave / LPT;          // tokens per wave and pass
    const int lane = lane_id();
    const int sub = lane % LPT;
    const int grp = lane / LPT;
    const int64_t passes = (tokens_per_wave + TPW - 1) / TPW;
    const float ninf = -__builtin_inff();
    // the scores of the next pass are fetched while this one is ranked (as long as registers allow)
    constexpr bool AHEAD = VPL <= 8;
    float ahead[AHEAD ? VPL : 1];
#pragma unroll
    for (int v = 0; v < (AHEAD ? VPL : 0); ++v) {
        const int e = v * LPT + sub;
        const int64_t t0 = w_begin + grp;
        ahead[v] = (t0 < w_end && e < E) ? load_score<T>(scores + t0 * E + e) : ninf;
    }
    for (int64_t pass = 0; pass < passes; ++pass) {
        const int64_t t = w_begin + pass * TPW + grp;
        const bool live = t < w_end;

        float my[VPL];
#pragma unroll
        for (int v = 0; v < VPL; ++v) {
            const int e = v * LPT + sub;
            if (AHEAD) {
                my[v] = ahead[v];
                const int64_t tn = t + TPW;
                ahead[v] = (tn < w_end && e < E) ? load_score<T>(scores + tn * E + e) : ninf;
            } else {
                my[v] = (live && e < E) ? load_score<T>(scores + t * E + e) : ninf;
            }
        }
        // modes 2 and 3: the inputs are logits; they are L2-normalised over the experts first
        // (F.normalize: l / max(||l||, 1e-12), rounded to the logits' dtype), and it is the
        // normalised values that are ranked: rounding can tie values that differed before
        if (renorm >= 2) {
            float sq = 0.0f;
#pragma unroll
            for (int v = 0; v < VPL; ++v) {
                const int e = v * LPT + sub;
                if (live && e < E) sq += my[v] * my[v];
            }
#pragma unroll
            for (int o = LPT / 2; o >= 1; o >>= 1) sq += __shfl_xor(sq, o, kWave);
            const float norm = fmaxf(round_to<T>(sqrtf(sq)), 1e-12f);
#pragma unroll
            for (int v = 0; v < VPL; ++v) {
                const int e = v * LPT + sub;
                if (live && e < E) my[v] = round_to<T>(my[v] / norm);
            }
        }
        int rank[VPL];
        uint32_t work[VPL];
#pragma unroll
        for (int v = 0; v < VPL; ++v) {
            rank[v] = K;                                                   // not selected
            // (a key is never 0: -inf maps to 0x007fffff; 0 marks "taken" and the lanes past E)
            work[v] = (live && v * LPT + sub < E) ? order_key(my[v]) : 0u;
        }
        for (int r = 0; r < K; ++r) {
            uint32_t best = work[0];
            int bv = 0;
#pragma unroll
            for (int v = 1; v < VPL; ++v)
                if (work[v] > best) {                  // strictly: equal keys keep the lower expert id
                    best = work[v];
                    bv = v;
                }
            const uint32_t top = group_max_u32<LPT>(best);
            const uint32_t cand = best == top ? 0x3FFu - (uint32_t)(bv * LPT + sub) : 0u;
            const int win = (int)(0x3FFu - group_max_u32<LPT>(cand));     // this round's winner in the group
#pragma unroll
            for (int v = 0; v < VPL; ++v)
                if (v * LPT + sub == win) {
                    rank[v] = r;
                    work[v] = 0u;
                }
        }
#pragma unroll
        for (int v = 0; v < VPL; ++v) {
            const int e = v * LPT + sub;
            if (live && e < E && rank[v] < K) s_sel[grp][rank[v]] = my[v];
        }
        // gates of modes 2 and 3: softmax of the normalised logits over all experts (2) or over
        // the K selected ones (3)
        float soft_sum = 0.0f;
        wave_lds_fence();
        if (renorm == 2) {
            // the largest normalised logit is slot 0; exp(n_i - n_max) summed over all experts
            const float nmax0 = live ? s_sel[grp][0] : 0.0f;
#pragma unroll
            for (int v = 0; v < VPL; ++v) {
                const int e = v * LPT + sub;
                if (live && e < E) soft_sum += expf(my[v] - nmax0);
            }
#pragma unroll
            for (int o = LPT / 2; o >= 1; o >>= 1) soft_sum += __shfl_xor(soft_sum, o, kWave);
        }
        if (live) {
            float denom = 1.0f;
            if (renorm == 1) {
                float s = 0.0f;
                for (int j = 0; j < K; ++j) s = s + fabsf(s_sel[grp][j]);   // slot order
                // (clamp_min keeps a NaN norm, fmaxf would drop it)
                denom = s != s ? s : fmaxf(round_to<T>(s), round_to<T>(1e-12f));
            }
            float nmax = 0.0f;
            if (renorm >= 2) {
                nmax = s_sel[grp][0];
                if (renorm == 3) {
                    soft_sum = 0.0f;
                    for (int j = 0; j < K; ++j) soft_sum += expf(s_sel[grp][j] - nmax);
                }
            }
#pragma unroll
            for (int v = 0; v < VPL; ++v) {
                const int e = v * LPT + sub;
                if (e < E && rank[v] < K) {
                    const int64_t p = t * K + rank[v];
                    topk_idx[p] = e;
                    compact[p] = (uint16_t)e;
                    atomicAdd(&s_hist[e], 1);      // integer counts in LDS: exact
                    float g = my[v];
                    if (renorm == 1) g = round_to<T>(my[v] / denom);
                    else if (renorm >= 2) g = round_to<T>(expf(my[v] - nmax) / soft_sum);
                    store_score<T>(gates + p, g);
                }
            }
        }
        wave_lds_fence();       // s_sel is rewritten by the next pass
    }
}

template <typename T, int LPT, int VPL, int WPB>
__global__ __launch_bounds__(WPB * kWave) void topk_hist_kernel(const T* __restrict__ scores, int64_t num_tokens,
                                                        int E, int K, int renorm, int64_t tokens_per_wave,
                                                        int64_t* __restrict__ topk_idx,
                                                        T* __restrict__ gates,
                                                        uint16_t* __restrict__ compact,
                                                        int32_t* __restrict__ sub_hist,
                                                        int32_t* __restrict__ tot_hist) {
    constexpr int NT = WPB * kWave;
    __shared__ float s_sel[WPB][kWave / LPT][64];     // selected scores by slot (K <= 64)
    extern __shared__ int32_t s_hist[];       // [WPB][E] experts chosen by this wave's tokens
    const int wave = threadIdx.x / kWave;
    for (int i = threadIdx.x; i < WPB * E; i += NT) s_hist[i] = 0;
    __syncthreads();
    // this wave's tokens: a contiguous range
    const int64_t w_begin = ((int64_t)blockIdx.x * WPB + wave) * tokens_per_wave;
    int64_t w_end = w_begin + tokens_per_wave;
    if (w_end > num_tokens) w_end = num_tokens;
    select_experts<T, LPT, VPL>(scores, w_begin, w_end, tokens_per_wave, E, K, renorm, topk_idx, gates, compact, s_sel[wave],
                                s_hist + wave * E);
    __syncthreads();
    for (int i = threadIdx.x; i < WPB * E; i += NT) sub_hist[(int64_t)blockIdx.x * WPB * E + i] = s_hist[i];
    for (int e = threadIdx.x; e < E; e += NT) {
        int32_t tot = 0;
#pragma unroll
        for (int w = 0; w < WPB; ++w) tot += s_hist[w * E + e];
        tot_hist[(int64_t)blockIdx.x * E + e] = tot;
    }
}

// Expert ids supplied by the caller (int64): narrow to the compact form, count them per wave
// and chunk as above, count the out-of-range ids of the chunk.
__global__ __launch_bounds__(1024) void compact_hist_kernel(const int64_t* __restrict__ topk_idx,
                                                            int64_t num_tokens, int E, int K,
                                                            int64_t tokens_per_wave,
                                                            uint16_t* __restrict__ compact,
                                                            int32_t* __restrict__ sub_hist,
                                                            int32_t* __restrict__ tot_hist,
                                                            int32_t* __restrict__ bad_part) {
    const int WPB = blockDim.x / kWave, NT = blockDim.x;
    extern __shared__ int32_t s_hist[];       // [WPB][E], then [WPB] bad counts
    int32_t* s_bad = s_hist + WPB * E;
    const int lane = lane_id();
    const int wave = threadIdx.x / kWave;
    for (int i = threadIdx.x; i < WPB * E + WPB; i += NT) s_hist[i] = 0;
    __syncthreads();
    const int64_t w_begin = ((int64_t)blockIdx.x * WPB + wave) * tokens_per_wave;
    int64_t w_end = w_begin + tokens_per_wave;
    if (w_end > num_tokens) w_end = num_tokens;
    int bad = 0;
    for (int64_t p = w_begin * K + lane; p < w_end * K; p += kWave) {
        const int64_t e = topk_idx[p];
        const bool ok = e >= 0 && e < E;
        compact[p] = ok ? (uint16_t)e : kBadExpert;
        if (ok) atomicAdd(&s_hist[wave * E + (int)e], 1);
        else ++bad;
    }
    if (bad) atomicAdd(&s_bad[wave], bad);
    __syncthreads();
    for (int i = threadIdx.x; i < WPB * E; i += NT) sub_hist[(int64_t)blockIdx.x * WPB * E + i] = s_hist[i];
    for (int e = threadIdx.x; e < E; e += NT) {
        int32_t tot = 0;
        for (int w = 0; w < WPB; ++w) tot += s_hist[w * E + e];
        tot_hist[(int64_t)blockIdx.x * E + e] = tot;
    }
    if (threadIdx.x == 0) {
        int32_t b = 0;
        for (int w = 0; w < WPB; ++w) b += s_bad[w];
        bad_part[blockIdx.x] = b;
    }
}

// Places the positions of a wave's tokens [t_begin, t_end): next[e] (LDS, this wave's) is the next free slot of expert e.  Each pass
// takes TPI = 64/K whole tokens, lane i <-> position begin + pass*TPI*K + i, so the K slots of a token sit in one pass.
__device__ __forceinline__ void place_positions(const uint16_t* compact, int64_t t_begin, int64_t t_end,
                                                int64_t tokens_per_wave, int K, int ebits, int32_t* next,
                                                int64_t* __restrict__ gate_index, int64_t* __restrict__ token_index,
                                                int64_t* __restrict__ reverse_index) {
    const int lane = lane_id();
    const int tpi = kWave / K;
    const int64_t passes = (tokens_per_wave + tpi - 1) / tpi;
    const int tok_in_iter = lane / K;
    const int slot = lane - tok_in_iter * K;
    const uint64_t lt_mask = lane == 0 ? 0ull : (~0ull >> (64 - lane));
    for (int64_t pass = 0; pass < passes; ++pass) {
        const int64_t t = t_begin + pass * tpi + tok_in_iter;
        const bool live = tok_in_iter < tpi && t < t_end;
        const int64_t p = t * K + slot;
        const uint32_t e = live ? compact[p] : (uint32_t)kBadExpert;
        const bool counted = live && e != kBadExpert;
        // lanes holding the same expert id
        uint64_t same = __ballot(counted);
        for (int b = 0; b < ebits; ++b) {
            const uint64_t bal = __ballot((e >> b) & 1u);
            same &= ((e >> b) & 1u) ? bal : ~bal;
        }
        const int before = __popcll(same & lt_mask);
        const int count = __popcll(same);
        int32_t base = 0;
        if (counted) base = next[e];
        wave_lds_fence();
        if (counted && before == 0) next[e] = base + count;
        wave_lds_fence();
        const int64_t dst = (int64_t)base + before;
        // rank of this slot among the token's K slots, ordered by (expert, slot)
        int rank = 0;
        for (int j = 0; j < K; ++j) {
            const uint32_t oe = __shfl(e, tok_in_iter * K + j, kWave);
            rank += (oe < e || (oe == e && j < slot)) ? 1 : 0;
        }
        if (counted) {
            gate_index[dst] = p;
            token_index[dst] = t;
            reverse_index[t * K + rank] = dst;
        } else if (live) {
            reverse_index[t * K + rank] = 0;    // a dropped position (out-of-range id): sorts last in its token
        }
    }
}

// Block = chunk, 4 or 16 waves.  Phase 1: per expert, the rows of all chunks (lengths) and of the chunks
// before this one.  Phase 2: wave scan over the experts = offsets.  Phase 3: every wave starts
// from offsets + rows of earlier chunks + rows of the earlier waves of its chunk and places its
// positions.
__global__ __launch_bounds__(1024) void scan_scatter_kernel(const uint16_t* __restrict__ compact,
                                                           int64_t num_tokens, int64_t tokens_per_wave,
                                                           int E, int K, int ebits, int num_chunks,
                                                           const int32_t* __restrict__ sub_hist,
                                                           const int32_t* __restrict__ tot_hist,
                                                           const int32_t* __restrict__ bad_part,
                                                           int64_t* __restrict__ lengths,
                                                           int64_t* __restrict__ offsets,
                                                           int64_t* __restrict__ gate_index,
                                                           int64_t* __restrict__ token_index,
                                                           int64_t* __restrict__ reverse_index,
                                                           int64_t* __restrict__ bad_count) {
    const int WPB = blockDim.x / kWave;
    extern __shared__ int32_t smem[];
    int32_t* s_tot = smem;                    // [WPB][E] partial sums over a share of the chunks
    int32_t* s_bef = smem + WPB * E;          // [WPB][E] ... restricted to the chunks before this one
    int32_t* s_base = smem + 2 * WPB * E;     // [E] first slot of this chunk's rows of expert e
    int32_t* s_next = smem + 2 * WPB * E + E; // [WPB][E]: first this chunk's counts per wave, then the next free slots
    const int c = blockIdx.x;
    const int lane = lane_id();
    const int wave = threadIdx.x / kWave;
    {   // phase 1: wave w sums chunks [w * q, (w + 1) * q)
        const int q = (num_chunks + WPB - 1) / WPB;
        const int c_lo = wave * q, c_hi = (wave + 1) * q < num_chunks ? (wave + 1) * q : num_chunks;
        for (int e0 = 0; e0 < E; e0 += kWave) {
            const int e = e0 + lane;
            int32_t tot = 0, bef = 0;
            if (e < E) {
                // (this wave's own counts of the chunk ride along with the first loads)
                s_next[wave * E + e] = sub_hist[((int64_t)c * WPB + wave) * E + e];
#pragma unroll 8
                for (int cc = c_lo; cc < c_hi; ++cc) {
                    const int32_t v = tot_hist[(int64_t)cc * E + e];
                    tot += v;
                    bef += cc < c ? v : 0;
                }
                s_tot[wave * E + e] = tot;
                s_bef[wave * E + e] = bef;
            }
        }
    }
    __syncthreads();
    if (wave == 0) {    // phase 2: exclusive prefix of the lengths over the experts; chunk 0 publishes
        long long run = 0;
        for (int e0 = 0; e0 < E; e0 += kWave) {
            const int e = e0 + lane;
            long long len = 0;
            int32_t bef = 0;
            if (e < E)
                for (int w = 0; w < WPB; ++w) {
                    len += s_tot[w * E + e];
                    bef += s_bef[w * E + e];
                }
            const long long inc = wave_inclusive_scan(len);
            if (e < E) {
                s_base[e] = (int32_t)(run + inc - len) + bef;
                if (c == 0) {
                    lengths[e] = len;
                    offsets[e] = run + inc - len;
                }
            }
            run += wave_bcast(inc, kWave - 1);
        }
        if (c == 0) {
            if (lane == 0) offsets[E] = run;
            // positions dropped for an out-of-range expert id leave a tail behind the last expert's
            // rows: it holds zeros rather than whatever the buffer held (normally the tail is empty)
            for (long long i = run + lane; i < (long long)num_tokens * K; i += kWave) {
                gate_index[i] = 0;
                token_index[i] = 0;
            }
            if (bad_count) {
                long long bad = 0;
                if (bad_part)
                    for (int cc = lane; cc < num_chunks; cc += kWave) bad += bad_part[cc];
#pragma unroll
                for (int o = 32; o >= 1; o >>= 1) bad += __shfl_xor(bad, o, kWave);
                if (lane == 0) *bad_count = bad;
            }
        }
    }
    __syncthreads();
    // phase 3: the counts of the earlier waves of the chunk (LDS) on top of the chunk's base
    int32_t at[16];             // E <= 1024: at most 16 entries per lane
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        const int e = i * kWave + lane;
        at[i] = 0;
        if (e < E) {
            at[i] = s_base[e];
            for (int w = 0; w < wave; ++w) at[i] += s_next[w * E + e];
        }
    }
    __syncthreads();            // every wave has read the counts before anyone overwrites them
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        const int e = i * kWave + lane;
        if (e < E) s_next[wave * E + e] = at[i];
    }
    __syncthreads();
    const int64_t t_begin = ((int64_t)c * WPB + wave) * tokens_per_wave;
    int64_t t_end = t_begin + tokens_per_wave;
    if (t_end > num_tokens) t_end = num_tokens;
    place_positions(compact, t_begin, t_end, tokens_per_wave, K, ebits, s_next + wave * E, gate_index, token_index, reverse_index);
}

// Both launches in one block of 16 waves for a batch of few tokens (route_one_block): the counts and the expert ids stay in LDS, and
// one barrier on either side of the prefix sums takes the place of the second launch.  scores: global memory or LDS.
template <typename T, int LPT, int VPL>
__device__ __forceinline__ void route_in_block(const T* scores, int num_tokens, int E, int K, int ebits, int renorm, int tokens_per_wave,
                                               int64_t* __restrict__ topk_idx, T* __restrict__ gates, int64_t* __restrict__ lengths,
                                               int64_t* __restrict__ offsets, int64_t* __restrict__ gate_index,
                                               int64_t* __restrict__ token_index, int64_t* __restrict__ reverse_index, int32_t* s_hist,
                                               uint16_t* s_ids) {
    constexpr int WPB = kMaxRouteWaves, NT = WPB * kWave;
    __shared__ float s_sel[WPB][kWave / LPT][64];
    const int lane = lane_id();
    const int wave = threadIdx.x / kWave;
    for (int i = threadIdx.x; i < WPB * E; i += NT) s_hist[i] = 0;
    __syncthreads();
    const int t_begin = wave * tokens_per_wave;
    const int t_end = t_begin + tokens_per_wave < num_tokens ? t_begin + tokens_per_wave : num_tokens;
    select_experts<T, LPT, VPL>(scores, t_begin, t_end, tokens_per_wave, E, K, renorm, topk_idx, gates, s_ids, s_sel[wave],
                                s_hist + wave * E);
    __syncthreads();
    if (wave == 0) {
        int run = 0;
        for (int e0 = 0; e0 < E; e0 += kWave) {
            const int e = e0 + lane;
            int count[WPB], len = 0;
#pragma unroll
            for (int w = 0; w < WPB; ++w) count[w] = e < E ? s_hist[w * E + e] : 0;
#pragma unroll
            for (int w = 0; w < WPB; ++w) len += count[w];
            const int inc = wave_inclusive_scan(len);
            if (e < E) {
                int at = run + inc - len;
                lengths[e] = len;
                offsets[e] = at;
#pragma unroll
                for (int w = 0; w < WPB; ++w) {
                    s_hist[w * E + e] = at;
                    at += count[w];
                }
            }
            run += wave_bcast(inc, kWave - 1);
        }
        if (lane == 0) offsets[E] = run;
    }
    __syncthreads();
    place_positions(s_ids, t_begin, t_end, tokens_per_wave, K, ebits, s_hist + wave * E, gate_index, token_index, reverse_index);
}

template <typename T, int LPT, int VPL>
__global__ __launch_bounds__(kMaxRouteWaves* kWave) void route_block_kernel(const T* __restrict__ scores, int num_tokens, int E, int K,
                                                                    int ebits, int renorm, int tokens_per_wave,
                                                                    int64_t* __restrict__ topk_idx, T* __restrict__ gates,
                                                                    int64_t* __restrict__ lengths, int64_t* __restrict__ offsets,
                                                                    int64_t* __restrict__ gate_index,
                                                                    int64_t* __restrict__ token_index,
                                                                    int64_t* __restrict__ reverse_index) {
    extern __shared__ int32_t s_hist[];       // [waves][E] counts per wave, then every wave's next free slots; [T * K] expert ids
    route_in_block<T, LPT, VPL>(scores, num_tokens, E, K, ebits, renorm, tokens_per_wave, topk_idx, gates, lengths, offsets, gate_index,
                                token_index, reverse_index, s_hist, reinterpret_cast<uint16_t*>(s_hist + kMaxRouteWaves * E));
}

// The gate of such a batch as well: the scores never leave LDS.  Groups of eight waves take 16 tokens at a time, as gate_softmax_kernel's blocks
// do (the same sums in the same order), then the block routes them.
constexpr int gate_groups(int nf) { return nf <= 2 ? 2 : 1; }
template <typename T, int NF, int LPT, int VPL>
__global__ __launch_bounds__(kMaxRouteWaves* kWave) void gate_softmax_route_kernel(
    const uint8_t* __restrict__ x, int D, int64_t x_stride, const uint8_t* __restrict__ w, const void* __restrict__ bias, int num_tokens, int E,
    int K, int ebits, int renorm, int tokens_per_wave, int64_t* __restrict__ topk_idx, T* __restrict__ gates, int64_t* __restrict__ lengths,
    int64_t* __restrict__ offsets, int64_t* __restrict__ gate_index, int64_t* __restrict__ token_index, int64_t* __restrict__ reverse_index) {
    constexpr bool F32 = sizeof(T) == 4;
    constexpr int GROUPS = gate_groups(NF), TOKENS = GROUPS * kGateTokens;
    extern __shared__ __align__(16) float red[];                    // [GROUPS] sums of a group; then counts, scores and expert ids
    int32_t* const s_hist = reinterpret_cast<int32_t*>(red + GROUPS * gate_sums_floats(NF));
    T* const s_scores = reinterpret_cast<T*>(s_hist + kMaxRouteWaves * E);
    uint16_t* const s_ids = reinterpret_cast<uint16_t*>(s_scores + num_tokens * E);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), group = wave / kGateWaves;
    for (int t0 = 0; t0 < num_tokens; t0 += TOKENS) {
        if (t0) __syncthreads();                // the sums before have been read
        if (group < GROUPS && t0 + group * kGateTokens < num_tokens)
            gate_sums<F32, NF>(x, num_tokens, D, x_stride, w, E, t0 + group * kGateTokens, wave % kGateWaves, red + group * gate_sums_floats(NF));
        __syncthreads();
        constexpr int STEP = gate_wave_tokens(NF);              // (a wave's tokens lie in one group)
        for (int first = wave * STEP; first < TOKENS && t0 + first < num_tokens; first += kMaxRouteWaves * STEP) {
            const int g0 = first / kGateTokens * kGateTokens, tokens = num_tokens - t0 - g0 < kGateTokens ? num_tokens - t0 - g0 : kGateTokens;
            gate_softmax_tokens<F32, NF>(red + first / kGateTokens * gate_sums_floats(NF), first - g0, tokens, bias, E, [&](int t, int e, float p) {
                if constexpr (F32) s_scores[(t0 + g0 + t) * E + e] = p;
                else s_scores[(t0 + g0 + t) * E + e] = (uint16_t)f32_to_bf16_bits(p);
            });
        }
    }
    // (the barrier behind the clearing of the counts publishes the scores)
    route_in_block<T, LPT, VPL>(s_scores, num_tokens, E, K, ebits, renorm, tokens_per_wave, topk_idx, gates, lengths, offsets, gate_index,
                                token_index, reverse_index, s_hist, s_ids);
}
inline size_t gate_route_lds(int esize, int64_t T, int E, int K) {
    const int nf = gate_fragments(E);
    return (size_t)gate_groups(nf) * gate_sums_floats(nf) * 4 + (size_t)kMaxRouteWaves * E * 4 + (size_t)T * E * esize + (size_t)T * K * 2;
}

int ceil_log2(int v) {
    int b = 0;
    while ((1 << b) < v) ++b;
    return b;
}

int launch_sort(const RouteScratch& ws, const RoutePlan& plan, bool have_bad, int64_t T, int E, int K,
                int64_t* lengths, int64_t* offsets, int64_t* gate_index, int64_t* token_index,
                int64_t* reverse_index, int64_t* bad_count, hipStream_t stream) {
    const size_t lds = (size_t)(3 * plan.wpb + 1) * E * sizeof(int32_t);
    scan_scatter_kernel<<<plan.num_chunks, plan.wpb * kWave, lds, stream>>>(
        ws.compact, T, plan.tokens_per_wave, E, K, ceil_log2(E), plan.num_chunks, ws.sub_hist, ws.tot_hist,
        have_bad ? ws.bad_part : nullptr, lengths, offsets, gate_index, token_index, reverse_index, bad_count);
    return check_launch("routing sort");
}

template <typename T, int LPT, int VPL>
void launch_topk(const void* scores, int64_t T_, int E, int K, int renorm, int64_t* topk_idx,
                 void* gates, const RouteScratch& ws, const RoutePlan& plan, hipStream_t stream) {
    const size_t lds = (size_t)plan.wpb * E * sizeof(int32_t);
    if (plan.wpb == 16)
        topk_hist_kernel<T, LPT, VPL, 16><<<plan.num_chunks, 16 * kWave, lds, stream>>>(
            (const T*)scores, T_, E, K, renorm, plan.tokens_per_wave, topk_idx, (T*)gates, ws.compact, ws.sub_hist,
            ws.tot_hist);
    else
        topk_hist_kernel<T, LPT, VPL, 4><<<plan.num_chunks, 4 * kWave, lds, stream>>>(
            (const T*)scores, T_, E, K, renorm, plan.tokens_per_wave, topk_idx, (T*)gates, ws.compact, ws.sub_hist,
            ws.tot_hist);
}

// One block takes the batch where its 16 waves rank all tokens in one pass (two: up to 64 experts and 8 slots), so that the second
// launch is what it saves.  us, two launches / one block: 64 tokens, 8 experts, top-2 8.9 / 5.0; 256, top-8 11.0 / 9.5; 64 tokens, 32
// experts, top-2 9.4 / 5.5; 128, 64 experts, top-8 12.7 / 12.5; 64, 128 experts, top-8 16.7 / 12.1; 64, 256 experts 27.5 / 22.8.  One pass
// more: 384 tokens, 8 experts, top-8 10.9 / 12.4; 192, 64 experts, top-8 13.0 / 17.4; 100, 128 experts, top-8 16.9 / 18.1.  Beyond
// 16 slots a wave of the block places its four tokens one after the other.
inline bool route_one_block(int64_t T, int E, int K) {
    const int64_t pass = kMaxRouteWaves * (E <= 8 ? 8 : 4);
    return E <= 256 && K <= 16 && T <= (E <= 64 && K <= 8 ? 2 * pass : pass);
}

struct RouteOut {
    int64_t *topk_idx, *lengths, *offsets, *gate_index, *token_index, *reverse_index;
};

template <typename T, int LPT, int VPL>
void launch_one_block(const void* scores, int64_t T_, int E, int K, int renorm, void* gates, const RouteOut& out, hipStream_t stream) {
    const size_t lds = (size_t)kMaxRouteWaves * E * sizeof(int32_t) + (size_t)T_ * K * sizeof(uint16_t);
    route_block_kernel<T, LPT, VPL><<<1, kMaxRouteWaves * kWave, lds, stream>>>(
        (const T*)scores, (int)T_, E, K, ceil_log2(E), renorm, (int)((T_ + kMaxRouteWaves - 1) / kMaxRouteWaves), out.topk_idx,
        (T*)gates, out.lengths, out.offsets, out.gate_index, out.token_index, out.reverse_index);
}

template <typename T>
int dispatch_one_block(const void* scores, int64_t T_, int E, int K, int renorm, void* gates, const RouteOut& out, hipStream_t stream) {
#define FMOE_ROUTE(LPT, VPL) launch_one_block<T, LPT, VPL>(scores, T_, E, K, renorm, gates, out, stream)
    if (E <= 8) FMOE_ROUTE(8, 1);
    else if (E <= 16) FMOE_ROUTE(16, 1);
    else if (E <= 32) FMOE_ROUTE(16, 2);
    else if (E <= 64) FMOE_ROUTE(16, 4);
    else if (E <= 128) FMOE_ROUTE(16, 8);
    else FMOE_ROUTE(16, 16);
#undef FMOE_ROUTE
    return check_launch("routing");
}

template <typename T>
int dispatch_topk(const void* scores, int64_t T_, int E, int K, int renorm, int64_t* topk_idx,
                  void* gates, const RouteScratch& ws, const RoutePlan& plan, hipStream_t stream) {
#define FMOE_TOPK(LPT, VPL) launch_topk<T, LPT, VPL>(scores, T_, E, K, renorm, topk_idx, gates, ws, plan, stream)
    if (E <= 8) FMOE_TOPK(8, 1);
    else if (E <= 16) FMOE_TOPK(16, 1);
    else if (E <= 32) FMOE_TOPK(16, 2);
    else if (E <= 64) FMOE_TOPK(16, 4);
    else if (E <= 128) FMOE_TOPK(16, 8);
    else if (E <= 256) FMOE_TOPK(16, 16);
    else if (E <= 512) FMOE_TOPK(16, 32);
    else return fail(FMOE_ERR_UNSUPPORTED, "fmoe_route_topk: E=%d > 512", E);
#undef FMOE_TOPK
    return FMOE_OK;
}

int check_common(int64_t T, int E, int K, const void* workspace, size_t ws_bytes, const char* who) {
    FMOE_REQUIRE(T >= 0 && E >= 1 && K >= 1, "%s: need T >= 0, E >= 1, K >= 1 (T=%lld E=%d K=%d)", who,
                 (long long)T, E, K);
    FMOE_REQUIRE(K <= 64, "%s: K=%d > 64 is not supported", who, K);
    FMOE_REQUIRE(E <= 1024, "%s: E=%d > 1024 is not supported", who, E);
    FMOE_REQUIRE(T * (int64_t)K < (int64_t)1 << 31, "%s: T*K must be below 2^31", who);
    const RoutePlan plan = make_plan(T, E, K);
    if (T > 0) {
        FMOE_REQUIRE(workspace != nullptr, "%s: workspace is NULL", who);
        if (ws_bytes < plan.total_bytes)
            return fail(FMOE_ERR_WORKSPACE, "%s: workspace %zu B < required %zu B", who, ws_bytes,
                        plan.total_bytes);
    }
    return FMOE_OK;
}

__global__ void empty_routing_kernel(int E, int64_t* lengths, int64_t* offsets, int64_t* bad_count) {
    for (int e = threadIdx.x; e < E; e += blockDim.x) lengths[e] = 0;
    for (int e = threadIdx.x; e <= E; e += blockDim.x) offsets[e] = 0;
    if (bad_count && threadIdx.x == 0) *bad_count = 0;
}

}  // namespace
}  // namespace fmoe

using namespace fmoe;

extern "C" size_t fmoe_route_workspace_bytes(int64_t T, int E, int K) {
    if (T < 0 || E < 1 || K < 1) return 0;
    return make_plan(T, E, K).total_bytes;
}

static int route_topk_impl(const char* who, const void* scores, int score_dtype, int64_t T, int E, int K, int renorm,
                           int64_t* topk_idx, void* gates, int64_t* lengths, int64_t* offsets,
                           int64_t* gate_index, int64_t* token_index, int64_t* reverse_index,
                           void* workspace, size_t workspace_bytes, hipStream_t stream) {
    if (int rc = check_common(T, E, K, workspace, workspace_bytes, who)) return rc;
    FMOE_REQUIRE(K <= E, "%s: K=%d > E=%d", who, K, E);
    FMOE_REQUIRE(renorm >= 0 && renorm <= 3, "%s: gate mode %d is not one of 0..3", who, renorm);
    FMOE_REQUIRE(score_dtype == FMOE_F32 || score_dtype == FMOE_BF16, "%s: scores must be fp32 or bf16", who);
    FMOE_REQUIRE(lengths && offsets, "%s: lengths/offsets are NULL", who);
    if (T == 0) {
        empty_routing_kernel<<<1, 256, 0, stream>>>(E, lengths, offsets, nullptr);
        return check_launch(who);
    }
    FMOE_REQUIRE(scores && topk_idx && gates && gate_index && token_index && reverse_index,
                 "%s: NULL tensor pointer", who);
    if (route_one_block(T, E, K)) {
        const RouteOut out = {topk_idx, lengths, offsets, gate_index, token_index, reverse_index};
        return score_dtype == FMOE_F32 ? dispatch_one_block<float>(scores, T, E, K, renorm, gates, out, stream)
                                       : dispatch_one_block<uint16_t>(scores, T, E, K, renorm, gates, out, stream);
    }
    const RoutePlan plan = make_plan(T, E, K);
    const RouteScratch ws = carve(workspace, plan);
    int rc = score_dtype == FMOE_F32
                 ? dispatch_topk<float>(scores, T, E, K, renorm, topk_idx, gates, ws, plan, stream)
                 : dispatch_topk<uint16_t>(scores, T, E, K, renorm, topk_idx, gates, ws, plan, stream);
    if (rc) return rc;
    return launch_sort(ws, plan, false, T, E, K, lengths, offsets, gate_index, token_index, reverse_index, nullptr,
                       stream);
}

// Where the gate and the routing of a batch are one launch: the one block can hold the scores, and walks the gate's rows in a time that the saved
// launch covers.  Bytes of a gate row times 1 + fragments, for every 16 tokens: us of a layer's pass (256 hidden columns) among others and alone,
// two launches / one: bf16 64 tokens, 128 inputs, 8 experts (2048) 28.8 / 23.9 and 45.1 / 42.7; 1, 128, 8 (512) 27.1 / 22.9 and 41.5 / 37.9; 16, 1024, 8
// (4096) 26.3 / 24.7 and 47.6 / 45.4; 1, 2048, 8 (8192) 27.6 / 26.4 and 49.0 / 47.2; fp32 16, 1024, 8 (8192) 34.1 / 32.9 and 54.1 / 53.8.  Beyond: bf16 1,
// 2048, 32 (12288) 31.1 / 30.0 and 50.2 / 50.6; several groups of tokens: fp32 64, 128, 8 (4096) 27.7 / 28.3 and 50.4 / 48.7; bf16 64, 512, 32 (12288)
// 26.7 / 29.0 and 46.6 / 49.3; 64, 1024, 8 (16384) 28.0 / 31.8.
extern "C" int fmoe_gate_route_pays(int dtype, int64_t T, int D, int E, int K) {
    if (!fmoe_gate_softmax_pays(dtype, T, D, E) || K < 1 || K > E || E > 64 || !route_one_block(T, E, K)) return 0;
    const int esize = dtype == FMOE_F32 ? 4 : 2, nf = gate_fragments(E);
    const size_t selected = (size_t)kMaxRouteWaves * (kWave / (E <= 8 ? 8 : 16)) * 64 * 4;
    if (gate_route_lds(esize, T, E, K) + selected > 65536) return 0;
    const int64_t groups = (T + kGateTokens - 1) / kGateTokens;
    return groups * D * esize * (1 + nf) <= (groups == 1 ? 8192 : 3072);
}

static int gate_route(const fmoe_gate* g, int64_t T, int E, int K, int renorm, int64_t* topk_idx, void* gates, int64_t* lengths, int64_t* offsets,
                      int64_t* gate_index, int64_t* token_index, int64_t* reverse_index, hipStream_t stream) {
    FMOE_REQUIRE(g && fmoe_gate_route_pays(g->dtype, T, g->d, E, K), "fmoe_route_topk: not a gate that fmoe_gate_route_pays takes");
    FMOE_REQUIRE(renorm >= 0 && renorm <= 3, "fmoe_route_topk: gate mode %d is not one of 0..3", renorm);
    const int esize = g->dtype == FMOE_F32 ? 4 : 2;
    FMOE_REQUIRE(g->x && g->weight && topk_idx && gates && lengths && offsets && gate_index && token_index && reverse_index,
                 "fmoe_route_topk: NULL tensor pointer");
    FMOE_REQUIRE(g->x_stride_row >= g->d && g->x_stride_row % (16 / esize) == 0 && aligned16(g->x) && aligned16(g->weight),
                 "fmoe_route_topk: gate rows of whole 16-byte chunks at 16-byte boundaries");
    const size_t lds = gate_route_lds(esize, T, E, K);
#define FMOE_GATE_ROUTE(TYPE, NF, LPT, VPL)                                                                                                     \
    gate_softmax_route_kernel<TYPE, NF, LPT, VPL><<<1, kMaxRouteWaves * kWave, lds, stream>>>(                                                    \
        (const uint8_t*)g->x, g->d, g->x_stride_row, (const uint8_t*)g->weight, g->bias, (int)T, E, K, ceil_log2(E), renorm,                                    \
        (int)((T + kMaxRouteWaves - 1) / kMaxRouteWaves), topk_idx, (TYPE*)gates, lengths, offsets, gate_index, token_index, reverse_index)
#define FMOE_GATE_ROUTE_E(TYPE)                                                                                                                  \
    (E <= 8 ? (void)(FMOE_GATE_ROUTE(TYPE, 1, 8, 1)) : E <= 16 ? (void)(FMOE_GATE_ROUTE(TYPE, 1, 16, 1))                                         \
     : E <= 32 ? (void)(FMOE_GATE_ROUTE(TYPE, 2, 16, 2)) : (void)(FMOE_GATE_ROUTE(TYPE, 4, 16, 4)))
    if (g->dtype == FMOE_F32) FMOE_GATE_ROUTE_E(float);
    else FMOE_GATE_ROUTE_E(uint16_t);
#undef FMOE_GATE_ROUTE_E
#undef FMOE_GATE_ROUTE
    return check_launch("fmoe_route_topk");
}

extern "C" int fmoe_route_topk(const void* scores, int score_dtype, int64_t T, int E, int K, int renorm,
                               int64_t* topk_idx, void* gates, int64_t* lengths, int64_t* offsets,
                               int64_t* gate_index, int64_t* token_index, int64_t* reverse_index,
                               void* workspace, size_t workspace_bytes, fmoe_stream_t stream_) {
    if (score_dtype == FMOE_SCORES_OF_GATE)
        return gate_route((const fmoe_gate*)scores, T, E, K, renorm, topk_idx, gates, lengths, offsets, gate_index, token_index, reverse_index,
                          (hipStream_t)stream_);
    return route_topk_impl("fmoe_route_topk", scores, score_dtype, T, E, K, renorm, topk_idx, gates, lengths,
                           offsets, gate_index, token_index, reverse_index, workspace, workspace_bytes,
                           (hipStream_t)stream_);
}

// ------------------------------------------------------------ allocation-free variant
// The routing scratch (one uint16 expert id per routed position + the per-chunk histograms) in
// device memory that belongs to the library image: one copy per GPU the library runs on, held
// until the process ends.  In host code `scratch` is only a handle for hipGetSymbolAddress;
// the address kernels and copies use is the per-device pointer looked up below.
static constexpr size_t kStaticCompactBytes = (size_t)FMOE_ROUTE_STATIC_MAX_POSITIONS * sizeof(uint16_t);
// (16 waves per block up to 256 experts, 4 beyond: 17 * 256 > 5 * 512)
static constexpr size_t kStaticHistBytes = (size_t)kMaxChunks * (kMaxRouteWaves + 1) * 256 * sizeof(int32_t);
static constexpr size_t kStaticScratchBytes = kStaticCompactBytes + kStaticHistBytes + kMaxChunks * 4 + 1280;
static __device__ __align__(256) unsigned char scratch[kStaticScratchBytes];

static constexpr int kMaxDevices = 64;
static void* g_scratch_ptr[kMaxDevices];     // device address of `scratch` on each GPU, 0 = not looked up yet
static std::mutex g_scratch_mutex;

// Device address of this GPU's copy of `scratch` (looked up once per device, with that device current).
static int static_scratch(void** out, const char* who) {
    int dev = -1;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices)
        return fail(FMOE_ERR_LAUNCH, "%s: no current device (or device index beyond %d)", who, kMaxDevices - 1);
    std::lock_guard<std::mutex> lock(g_scratch_mutex);
    if (g_scratch_ptr[dev] == nullptr) {
        void* ptr = nullptr;
        const hipError_t err = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
        if (err != hipSuccess || ptr == nullptr)
            return fail(FMOE_ERR_LAUNCH, "%s: hipGetSymbolAddress(scratch) failed on device %d: %s", who, dev,
                        hipGetErrorString(err));
        g_scratch_ptr[dev] = ptr;
    }
    *out = g_scratch_ptr[dev];
    return FMOE_OK;
}

extern "C" int fmoe_route_topk_static(const void* scores, int score_dtype, int64_t T, int E, int K, int renorm,
                                      int64_t* topk_idx, void* gates, int64_t* lengths, int64_t* offsets,
                                      int64_t* gate_index, int64_t* token_index, int64_t* reverse_index,
                                      fmoe_stream_t stream_) {
    const char* who = "fmoe_route_topk_static";
    FMOE_REQUIRE(T >= 0 && E >= 1 && K >= 1, "%s: need T >= 0, E >= 1, K >= 1 (T=%lld E=%d K=%d)", who,
                 (long long)T, E, K);
    FMOE_REQUIRE(E <= FMOE_ROUTE_STATIC_MAX_EXPERTS, "%s: E=%d exceeds the %d experts the built-in scratch holds",
                 who, E, FMOE_ROUTE_STATIC_MAX_EXPERTS);
    FMOE_REQUIRE(T <= FMOE_ROUTE_STATIC_MAX_POSITIONS && T * (int64_t)K <= FMOE_ROUTE_STATIC_MAX_POSITIONS,
                 "%s: T*K=%lld routed positions exceed the %d the built-in scratch holds (use fmoe_route_topk "
                 "with a workspace)", who, (long long)T * K, FMOE_ROUTE_STATIC_MAX_POSITIONS);
    // every check that can refuse the call comes before the scratch lookup, so that a refused call
    // never touches the runtime (the first lookup on a device calls hipGetSymbolAddress)
    FMOE_REQUIRE(K <= 64 && K <= E, "%s: K=%d must be at most 64 and at most E=%d", who, K, E);
    FMOE_REQUIRE(renorm >= 0 && renorm <= 3, "%s: gate mode %d is not one of 0..3", who, renorm);
    FMOE_REQUIRE(score_dtype == FMOE_F32 || score_dtype == FMOE_BF16, "%s: scores must be fp32 or bf16", who);
    FMOE_REQUIRE(lengths && offsets, "%s: lengths/offsets are NULL", who);
    if (T > 0)
        FMOE_REQUIRE(scores && topk_idx && gates && gate_index && token_index && reverse_index,
                     "%s: NULL tensor pointer", who);
    if (make_plan(T, E, K).total_bytes > kStaticScratchBytes)
        return fail(FMOE_ERR_WORKSPACE, "%s: the call needs %zu B of scratch, the built-in buffer has %zu B", who,
                    make_plan(T, E, K).total_bytes, kStaticScratchBytes);
    void* ptr = nullptr;
    if (int rc = static_scratch(&ptr, who)) return rc;
    // nothing in the buffer has to start at zero: the first two kernels overwrite every byte the later ones read
    return route_topk_impl(who, scores, score_dtype, T, E, K, renorm, topk_idx, gates, lengths, offsets, gate_index,
                           token_index, reverse_index, ptr, kStaticScratchBytes, (hipStream_t)stream_);
}

extern "C" int fmoe_route_from_topk(const int64_t* topk_idx, int64_t T, int E, int K, int64_t* lengths,
                                    int64_t* offsets, int64_t* gate_index, int64_t* token_index,
                                    int64_t* reverse_index, int64_t* bad_count, void* workspace,
                                    size_t workspace_bytes, fmoe_stream_t stream_) {
    hipStream_t stream = (hipStream_t)stream_;
    if (int rc = check_common(T, E, K, workspace, workspace_bytes, "fmoe_route_from_topk")) return rc;
    FMOE_REQUIRE(lengths && offsets, "fmoe_route_from_topk: lengths/offsets are NULL");
    if (T == 0) {
        empty_routing_kernel<<<1, 256, 0, stream>>>(E, lengths, offsets, bad_count);
        return check_launch("fmoe_route_from_topk");
    }
    FMOE_REQUIRE(topk_idx && gate_index && token_index && reverse_index,
                 "fmoe_route_from_topk: NULL tensor pointer");
    const RoutePlan plan = make_plan(T, E, K);
    const RouteScratch ws = carve(workspace, plan);
    compact_hist_kernel<<<plan.num_chunks, plan.wpb * kWave, ((size_t)plan.wpb * E + plan.wpb) * sizeof(int32_t), stream>>>(
        topk_idx, T, E, K, plan.tokens_per_wave, ws.compact, ws.sub_hist, ws.tot_hist, ws.bad_part);
    return launch_sort(ws, plan, true, T, E, K, lengths, offsets, gate_index, token_index, reverse_index, bad_count,
                       stream);
}
