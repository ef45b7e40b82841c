// Row-wise OCP e4m3fn quantisation with power-of-two multiplier scales.
//
// Fast path (contiguous bf16 rows, cols % 8 == 0): one wavefront per row, the
// row is read once with 16-byte loads and held in registers, so the traffic is
// the algorithmic 2 B in + 1 B out per element (+4 B scale per row).
// Rows too long for that (more than 8192 columns) get one block each and two
// passes.  Generic paths cover any strides, column counts and fp32 inputs.
#include "common.h"

namespace fmoe {
namespace {

// Software e4m3fn encoder: round to nearest even, non-saturating (anything that
// rounds above 448, and inf / NaN, becomes S.1111.111).
__device__ __forceinline__ uint32_t e4m3fn_encode(float f) {
    const uint32_t u = __float_as_uint(f);
    const uint32_t sign = (u >> 24) & 0x80u;
    uint32_t a = u & 0x7fffffffu;
    uint32_t code;
    if (a >= 0x43f00000u) {                 // >= 480, inf, NaN
        code = 0x7fu;
    } else if (a < 0x3c800000u) {           // below 2^-6: subnormal grid of 2^-9
        code = (uint32_t)rintf(__uint_as_float(a) * 512.0f);
    } else {
        a += 0x7ffffu + ((a >> 20) & 1u);
        code = (a >> 20) - (120u << 3);
    }
    return sign | code;
}

// scale = 2^floor(log2(448 / amax)); NaN / inf results -> 2^127; amax = inf -> 0.
// EXACT_EXPONENT: take the exponent field of the fp32 quotient.  For an amax
// that is a bf16 value this equals the reference's bf16 formula for every input.
// Otherwise follow the fp32 formula literally: the fp32 log2 of a quotient just
// below a power of two rounds up to the integer.
template <bool EXACT_EXPONENT>
__device__ __forceinline__ float scale_from_amax(float amax) {
    const float q = 448.0f / amax;
    const float clamp = __uint_as_float(0x7f000000u);  // 2^127
    if (!(q <= 3.4028234664e38f)) return clamp;         // inf or NaN
    if (q == 0.0f) return 0.0f;
    if (EXACT_EXPONENT) return __uint_as_float(__float_as_uint(q) & 0x7f800000u);
    const float fl = floorf((float)log2((double)q));
    if (fl >= 128.0f) return clamp;
    return __uint_as_float((uint32_t)((int)fl + 127) << 23);
}

__device__ __forceinline__ float amax_update(float m, float v, bool& nan) {
    nan |= (v != v);
    return fmaxf(m, fabsf(v));
}

__device__ __forceinline__ float finish_amax(float m, bool nan) {
    m = wave_max(m);
    if (__ballot(nan) != 0ull) m = __uint_as_float(0x7fc00000u);
    return m;
}

// eight bf16 values times the row's scale -> eight e4m3 codes.  Rows without NaN / inf take the
// hardware conversion; a row that holds one goes through the software encoder, which keeps the
// reference's non-saturating codes.
__device__ __forceinline__ u32x2 encode8(const u32x4& v, float s, bool special) {
    float f[8];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        f[2 * j] = bf16_bits_to_f32(v[j] & 0xffffu) * s;
        f[2 * j + 1] = __uint_as_float(v[j] & 0xffff0000u) * s;
    }
    u32x2 o;
    if (!special) {
        int w0 = __builtin_amdgcn_cvt_pk_fp8_f32(f[0], f[1], 0, false);
        w0 = __builtin_amdgcn_cvt_pk_fp8_f32(f[2], f[3], w0, true);
        int w1 = __builtin_amdgcn_cvt_pk_fp8_f32(f[4], f[5], 0, false);
        w1 = __builtin_amdgcn_cvt_pk_fp8_f32(f[6], f[7], w1, true);
        o[0] = (uint32_t)w0;
        o[1] = (uint32_t)w1;
    } else {
        o[0] = e4m3fn_encode(f[0]) | (e4m3fn_encode(f[1]) << 8) | (e4m3fn_encode(f[2]) << 16) |
               (e4m3fn_encode(f[3]) << 24);
        o[1] = e4m3fn_encode(f[4]) | (e4m3fn_encode(f[5]) << 8) | (e4m3fn_encode(f[6]) << 16) |
               (e4m3fn_encode(f[7]) << 24);
    }
    return o;
}

// No row of the call belongs to expert e: no GEMM over these offsets reads what would be written for it.  (A dense call pays the look: 8 x
// 4096 x 1024 weights 21.9 -> 22.0 us; 54 experts, 576 x 3776, two of them with a row 66 -> 6.)
__device__ __forceinline__ bool idle_expert(const int64_t* offsets, int64_t e) { return offsets && offsets[e + 1] <= offsets[e]; }

typedef __attribute__((ext_vector_type(2))) unsigned short u16x2;

// ---- fast path: bf16, contiguous columns, cols % 8 == 0, <= CH*512 columns
// W16: a lane takes pairs of neighbouring 16-byte chunks (32 contiguous input bytes), so that its
// eight-byte results pair up into one 16-byte store (rows of a whole number of such pairs)
template <int CH, bool SILU, bool W16 = false>
__global__ __launch_bounds__(256) void quant_rows_bf16_wave(
    const uint16_t* __restrict__ a, int64_t total_rows, int64_t rows, int cols, int64_t a_sb,
    int64_t a_sr, uint8_t* __restrict__ q, int64_t q_sb, int64_t q_sr, float* __restrict__ scale,
    int store_reciprocal, const int64_t* __restrict__ offsets) {
    const int lane = lane_id();
    const int64_t row = (int64_t)blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    if (row >= total_rows) return;
    const int64_t b = rows == total_rows ? 0 : row / rows, r = row - b * rows;      // (scalar: the loads wait for it)
    if (idle_expert(offsets, b)) return;
    const uint16_t* src = a + b * a_sb + r * a_sr;
    uint8_t* dst = q + b * q_sb + r * q_sr;
    const int chunks = cols >> 3;

    static_assert(!W16 || CH % 2 == 0, "pairs of chunks");
    // chunk held in v[i]
    auto chunk_of = [&](int i) { return W16 ? 2 * (lane + kWave * (i / 2)) + (i & 1) : lane + kWave * i; };
    u32x4 v[CH];
#pragma unroll
    for (int i = 0; i < CH; ++i) {
        const int c = chunk_of(i);
        v[i] = c < chunks ? *reinterpret_cast<const u32x4*>(src + (int64_t)c * 8) : u32x4{0, 0, 0, 0};
    }
    u16x2 most = {0, 0};                            // |value| bits of the low and the high halves: they compare as integers, NaN above inf
#pragma unroll
    for (int i = 0; i < CH; ++i) {
        if (SILU) v[i] = silu_round_bf16_x8(v[i]);
#pragma unroll
        for (int j = 0; j < 4; ++j) most = __builtin_elementwise_max(most, __builtin_bit_cast(u16x2, v[i][j] & 0x7fff7fffu));
    }
    uint32_t bits = max((uint32_t)most[0], (uint32_t)most[1]);
#pragma unroll
    for (int o = kWave / 2; o >= 1; o >>= 1) bits = max(bits, (uint32_t)__shfl_xor((int)bits, o, kWave));
    const float m = bf16_bits_to_f32(bits);
    const float s = scale_from_amax<true>(m);   // every element is a bf16 value
    if (lane == 0) scale[row] = store_reciprocal ? 1.0f / s : s;
    const bool special = !(m <= 3.4028234664e38f);   // NaN or inf in the row
    if constexpr (W16) {
#pragma unroll
        for (int i = 0; i < CH; i += 2) {
            const int c = chunk_of(i);
            if (c >= chunks) continue;
            const u32x2 lo = encode8(v[i], s, special), hi = encode8(v[i + 1], s, special);
            *reinterpret_cast<u32x4*>(dst + (int64_t)c * 8) = u32x4{lo[0], lo[1], hi[0], hi[1]};
        }
    } else {
#pragma unroll
        for (int i = 0; i < CH; ++i) {
            const int c = lane + kWave * i;
            if (c >= chunks) continue;
            const u32x2 o = encode8(v[i], s, special);
            *reinterpret_cast<u32x2*>(dst + (int64_t)c * 8) = o;
        }
    }
}

// ---- long rows (more columns than a wave holds in registers): one block per row, two passes
// with 16-byte loads; the second pass finds most of the row in L2.  The transposed operands of
// the fp8 weight gradient are a few thousand rows of 10^5 columns.
template <bool SILU>
__global__ __launch_bounds__(256) void quant_rows_bf16_block(
    const uint16_t* __restrict__ a, int64_t rows, int64_t cols, int64_t a_sb, int64_t a_sr,
    uint8_t* __restrict__ q, int64_t q_sb, int64_t q_sr, float* __restrict__ scale, int store_reciprocal) {
    __shared__ float s_max[4];
    __shared__ int s_nan[4];
    const int64_t row = blockIdx.x;
    const int64_t b = row / rows, r = row - b * rows;
    const uint16_t* src = a + b * a_sb + r * a_sr;
    uint8_t* dst = q + b * q_sb + r * q_sr;
    const int64_t chunks = cols >> 3;
    auto load = [&](int64_t c) {
        u32x4 v = *reinterpret_cast<const u32x4*>(src + c * 8);
        if (SILU) v = silu_round_bf16_x8(v);
        return v;
    };
    float m = 0.0f;
    bool nan = false;
    for (int64_t c = threadIdx.x; c < chunks; c += 256) {
        const u32x4 v = load(c);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            m = amax_update(m, bf16_bits_to_f32(v[j] & 0xffffu), nan);
            m = amax_update(m, __uint_as_float(v[j] & 0xffff0000u), nan);
        }
    }
    m = wave_max(m);
    const bool any_nan = __ballot(nan) != 0ull;
    if (lane_id() == 0) {
        s_max[threadIdx.x / kWave] = m;
        s_nan[threadIdx.x / kWave] = any_nan;
    }
    __syncthreads();
    m = fmaxf(fmaxf(s_max[0], s_max[1]), fmaxf(s_max[2], s_max[3]));
    if (s_nan[0] | s_nan[1] | s_nan[2] | s_nan[3]) m = __uint_as_float(0x7fc00000u);
    const float s = scale_from_amax<true>(m);
    if (threadIdx.x == 0) scale[row] = store_reciprocal ? 1.0f / s : s;
    const bool special = !(m <= 3.4028234664e38f);
    for (int64_t c = threadIdx.x; c < chunks; c += 256)
        *reinterpret_cast<u32x2*>(dst + c * 8) = encode8(load(c), s, special);
}

template <typename T>
__device__ __forceinline__ float load_as_f32(const T* p);
template <>
__device__ __forceinline__ float load_as_f32<float>(const float* p) { return *p; }
template <>
__device__ __forceinline__ float load_as_f32<uint16_t>(const uint16_t* p) { return bf16_bits_to_f32(*p); }

template <typename T, bool SILU>
__device__ __forceinline__ float fetch(const T* p) {
    float v = load_as_f32<T>(p);
    if (SILU) v = sizeof(T) == 2 ? silu_round_bf16(v) : silu_f32(v);
    return v;
}

// ---- generic: one wave per row, lanes stride over the columns, two passes
template <typename T, bool SILU>
__global__ __launch_bounds__(256) void quant_rows_generic_wave(
    const T* __restrict__ a, int64_t total_rows, int64_t rows, int64_t cols, int64_t a_sb, int64_t a_sr,
    int64_t a_sc, uint8_t* __restrict__ q, int64_t q_sb, int64_t q_sr, int64_t q_sc,
    float* __restrict__ scale, int store_reciprocal) {
    const int lane = lane_id();
    const int64_t row = (int64_t)blockIdx.x * 4 + threadIdx.x / kWave;
    if (row >= total_rows) return;
    const int64_t b = row / rows, r = row - b * rows;
    const T* src = a + b * a_sb + r * a_sr;
    uint8_t* dst = q + b * q_sb + r * q_sr;
    float m = 0.0f;
    bool nan = false;
    for (int64_t c = lane; c < cols; c += kWave) m = amax_update(m, fetch<T, SILU>(src + c * a_sc), nan);
    m = finish_amax(m, nan);
    const float s = sizeof(T) == 2 ? scale_from_amax<true>(m) : scale_from_amax<false>(m);
    if (lane == 0) scale[row] = store_reciprocal ? 1.0f / s : s;
    for (int64_t c = lane; c < cols; c += kWave)
        dst[c * q_sc] = (uint8_t)e4m3fn_encode(fetch<T, SILU>(src + c * a_sc) * s);
}

// ---- generic, rows adjacent in memory (a_sr == 1): one lane per row so that
// the loads of a wave are contiguous
template <typename T, bool SILU>
__global__ __launch_bounds__(256) void quant_rows_generic_lane(
    const T* __restrict__ a, int64_t total_rows, int64_t rows, int64_t cols, int64_t a_sb, int64_t a_sr,
    int64_t a_sc, uint8_t* __restrict__ q, int64_t q_sb, int64_t q_sr, int64_t q_sc,
    float* __restrict__ scale, int store_reciprocal) {
    const int64_t row = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (row >= total_rows) return;
    const int64_t b = row / rows, r = row - b * rows;
    const T* src = a + b * a_sb + r * a_sr;
    uint8_t* dst = q + b * q_sb + r * q_sr;
    float m = 0.0f;
    bool nan = false;
    for (int64_t c = 0; c < cols; ++c) m = amax_update(m, fetch<T, SILU>(src + c * a_sc), nan);
    if (nan) m = __uint_as_float(0x7fc00000u);
    const float s = sizeof(T) == 2 ? scale_from_amax<true>(m) : scale_from_amax<false>(m);
    scale[row] = store_reciprocal ? 1.0f / s : s;
    for (int64_t c = 0; c < cols; ++c)
        dst[c * q_sc] = (uint8_t)e4m3fn_encode(fetch<T, SILU>(src + c * a_sc) * s);
}

// ---- rows that are columns in memory (a_sr == 1: an [E, K, N] weight quantised per output column, q as
// [E, N, K] bytes).  Two launches: the amax of every row over the whole chip, then the transposing
// quantisation, tile by tile.  Bound by HBM: the operand is read twice (the second time mostly from the
// last-level cache where it fits) and its bytes written once.  A lane per row, the form this replaces,
// kept rows / 64 waves in flight, each with a serial walk over its columns and one-byte stores a row apart:
// 8 x 1024 x 4096 took 751 us (N = 4096) and 3147 us (N = 1024).
// Columns that fit a block's registers (kColOneMost) take one launch that reads them once.  us, two launches / one: 8 x 1024 x
// 4096 30.3 / 21.7 (100 MB, 15.7 at copy speed), 8 x 4096 x 1024 32.9 / 23.9; 64 x 2048 x 1408 173 / 120, 64 x 1408 x 2048 191 / 120; 128 x
// 4096 x 1536 804 / 568, 128 x 1536 x 4096 785 / 450; 100 x 200 x 1024 27.7 / 17.9; 4 x 512 x 512 7.0 / 6.1; 4 x 4096 x 64 19.9 / 11.6.

constexpr int kColTileN = 64;       // rows of the result per block: 128 bytes of a memory row
constexpr int kColTileK = 128;      // columns per block of the second launch: a whole line of result bytes
constexpr int kColMaxSplit = 64;
constexpr int64_t kColOneMost = 4096;

// Blocks of the first launch along the columns: enough to fill the chip (4 per CU), at least 64 columns each.
inline int col_splits(int64_t batch, int64_t rows, int64_t cols) {
    const int64_t strips = batch * ((rows + kColTileN - 1) / kColTileN);
    int64_t s = (1024 + strips - 1) / strips;
    const int64_t most = (cols + 63) / 64;
    s = s < most ? s : most;
    return (int)(s < 1 ? 1 : (s > kColMaxSplit ? kColMaxSplit : s));
}

// |value| bits of a bf16 pair, each in the position that compares as an integer (NaN above inf)
__device__ __forceinline__ void amax_bits(uint32_t pair, uint32_t& lo, uint32_t& hi) {
    lo = max(lo, (pair << 16) & 0x7fffffffu);
    hi = max(hi, pair & 0x7fff0000u);
}

// block (strip, split, batch): 8 lanes x 16 bytes across the strip, 32 rows of memory at a time, four loads
// in flight per lane; part[split][batch * rows] receives the strip's |max| bits over the split's columns.
__global__ __launch_bounds__(256) void quant_cols_amax(const uint16_t* __restrict__ a, int64_t rows, int64_t cols,
                                                       int64_t a_sb, int64_t a_sc, uint32_t* __restrict__ part,
                                                       int64_t total_rows, int64_t cols_per_split,
                                                       const int64_t* __restrict__ offsets) {
    if (idle_expert(offsets, blockIdx.z)) return;
    __shared__ uint32_t s_max[4][kColTileN];
    const int lane = lane_id(), wave = threadIdx.x / kWave;
    const int64_t n = (int64_t)blockIdx.x * kColTileN + (lane & 7) * 8;
    const int64_t k_lo = blockIdx.y * cols_per_split;
    const int64_t k_hi = k_lo + cols_per_split < cols ? k_lo + cols_per_split : cols;
    uint32_t m[8] = {0, 0, 0, 0, 0, 0, 0, 0};
    if (n < rows) {             // (rows are whole 8-element chunks on this path)
        const uint16_t* src = a + blockIdx.z * a_sb + n;
        int64_t k = k_lo + threadIdx.x / 8;
        for (; k + 96 < k_hi; k += 128) {
            u32x4 v[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) v[i] = *reinterpret_cast<const u32x4*>(src + (k + 32 * i) * a_sc);
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j) amax_bits(v[i][j], m[2 * j], m[2 * j + 1]);
        }
        for (; k < k_hi; k += 32) {
            const u32x4 v = *reinterpret_cast<const u32x4*>(src + k * a_sc);
#pragma unroll
            for (int j = 0; j < 4; ++j) amax_bits(v[j], m[2 * j], m[2 * j + 1]);
        }
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) {
#pragma unroll
        for (int o = 8; o < kWave; o <<= 1) m[j] = max(m[j], (uint32_t)__shfl_xor((int)m[j], o, kWave));
        if (lane < 8) s_max[wave][lane * 8 + j] = m[j];
    }
    __syncthreads();
    if (threadIdx.x < kColTileN) {
        const int64_t r = (int64_t)blockIdx.x * kColTileN + threadIdx.x;
        if (r < rows)
            part[blockIdx.y * total_rows + blockIdx.z * rows + r] =
                max(max(s_max[0][threadIdx.x], s_max[1][threadIdx.x]), max(s_max[2][threadIdx.x], s_max[3][threadIdx.x]));
    }
}

// block (row tile, column tile, batch): 64 rows x 128 columns.  A lane loads 8 rows of four consecutive columns;
// the conversion instruction packs two values of its choice, so the four columns of a row leave it as one dword
// of consecutive bytes and the transposition costs no instruction of its own.  LDS rows are 33 dwords apart: the
// 64 dwords a wave stores at a time fall into 64 banks.
__global__ __launch_bounds__(256) void quant_cols_store(const uint16_t* __restrict__ a, int64_t rows, int64_t cols,
                                                        int64_t a_sb, int64_t a_sc, const uint32_t* __restrict__ part,
                                                        int splits, int64_t total_rows, uint8_t* __restrict__ q,
                                                        int64_t q_sb, int64_t q_sr, float* __restrict__ scale,
                                                        int store_reciprocal, int wide, const int64_t* __restrict__ offsets) {
    if (idle_expert(offsets, blockIdx.z)) return;
    __shared__ uint32_t tile[kColTileN * 33];
    __shared__ float s_scale[kColTileN];
    __shared__ int s_special;
    const int tid = threadIdx.x;
    const int64_t n0 = (int64_t)blockIdx.x * kColTileN, k0 = (int64_t)blockIdx.y * kColTileK;
    const int ng = tid & 7, kq = tid >> 3;
    const int64_t n = n0 + 8 * ng, k = k0 + 4 * kq;
    // the tile's loads first: they are in flight while the scales are worked out
    u32x4 v[4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
        v[i] = n < rows && k + i < cols ? *reinterpret_cast<const u32x4*>(a + blockIdx.z * a_sb + (k + i) * a_sc + n)
                                        : u32x4{0, 0, 0, 0};
    if (tid == 0) s_special = 0;
    __syncthreads();
    if (tid < kColTileN) {
        const int64_t r = n0 + tid;
        uint32_t bits = 0;
        if (r < rows)
            for (int i = 0; i < splits; ++i) bits = max(bits, part[i * total_rows + blockIdx.z * rows + r]);
        const float s = scale_from_amax<true>(__uint_as_float(bits));
        s_scale[tid] = s;
        if (bits >= 0x7f800000u) s_special = 1;
        if (r < rows && blockIdx.y == 0) scale[blockIdx.z * rows + r] = store_reciprocal ? 1.0f / s : s;
    }
    __syncthreads();
    const bool special = s_special != 0;        // a row with NaN or inf: the software encoder, as in encode8
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        const float s = s_scale[8 * ng + j];
        float f[4];
#pragma unroll
        for (int i = 0; i < 4; ++i)
            f[i] = ((j & 1) ? __uint_as_float(v[i][j / 2] & 0xffff0000u) : bf16_bits_to_f32(v[i][j / 2] & 0xffffu)) * s;
        uint32_t w;
        if (!special) {
            int t = __builtin_amdgcn_cvt_pk_fp8_f32(f[0], f[1], 0, false);
            w = (uint32_t)__builtin_amdgcn_cvt_pk_fp8_f32(f[2], f[3], t, true);
        } else {
            w = e4m3fn_encode(f[0]) | (e4m3fn_encode(f[1]) << 8) | (e4m3fn_encode(f[2]) << 16) | (e4m3fn_encode(f[3]) << 24);
        }
        tile[(8 * ng + j) * 33 + kq] = w;
    }
    __syncthreads();
    // rows out: 8 lanes cover the 128 bytes of one
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const int r = (tid >> 3) + 32 * i, c = 4 * (tid & 7);
        if (n0 + r >= rows) continue;
        uint8_t* dst = q + blockIdx.z * q_sb + (n0 + r) * q_sr + k0 + 4 * c;
        const uint32_t* t = tile + r * 33 + c;
        if (wide && k0 + 4 * c + 16 <= cols) {
            *reinterpret_cast<u32x4*>(dst) = u32x4{t[0], t[1], t[2], t[3]};
        } else {
#pragma unroll
            for (int d = 0; d < 4; ++d)
                if (k0 + 4 * (c + d) < cols) *reinterpret_cast<uint32_t*>(dst + 4 * d) = t[d];     // (cols % 4 == 0)
        }
    }
}

// Both launches in one for columns that fit a block's registers: block (strip of STRIP rows, batch) holds PASSES x 4 x NT / (STRIP / 8)
// columns, 16 bytes of four consecutive columns per lane and pass; the amax meets in LDS, and every pass leaves through the
// transposing tile.  Two blocks and more to a CU where the registers allow, so that one loads under the other's stores; narrow strips
// for that (8 x 3000 x 3000: 32 rows, one block of 1024 threads 92 us, 512 threads of 96 registers 67), and neighbours on one XCD, which
// share the 128-byte lines then (64-row strips dealt round-robin 8 x 4096 x 1024 32, 128 x 4096 x 1536 760; now 24 and 568).
template <int STRIP, int NT, int PASSES>
__global__ __launch_bounds__(NT, 4) void quant_cols_one(const uint16_t* __restrict__ a, int64_t rows, int64_t cols, int64_t a_sb,
                                                     int64_t a_sc, uint8_t* __restrict__ q, int64_t q_sb, int64_t q_sr,
                                                     float* __restrict__ scale, int store_reciprocal, int wide, int strips,
                                                     const int64_t* __restrict__ offsets) {
    constexpr int LPR = STRIP / 8, QUADS = NT / LPR, PASS = 4 * QUADS;      // lanes across the strip, groups of 4 columns in a pass
    // (lanes of a wave store rows 8 * ng + j, dwords q .. of the tile: 8 * DW * ng + q has to name 64 banks)
    constexpr int DW = QUADS + 64 / LPR / 8;
    static_assert((8 * (DW % 64)) % 64 == 64 / LPR, "tile rows");
    constexpr int NW = NT / kWave;
    __shared__ uint32_t tile[STRIP * DW];
    __shared__ uint32_t s_max[NW][STRIP];
    __shared__ float s_scale[STRIP];
    __shared__ int s_special;
    const int tid = threadIdx.x, lane = lane_id(), wave = tid / kWave;
    const int ng = tid % LPR, quad = tid / LPR;
    // neighbouring strips share lines: a run of them to every XCD
    const int strip = gridDim.x > 8 ? (int)(blockIdx.x % 8 * (gridDim.x / 8) + blockIdx.x / 8) : (int)blockIdx.x;
    if (strip >= strips || idle_expert(offsets, blockIdx.y)) return;
    const int64_t n0 = (int64_t)strip * STRIP, n = n0 + 8 * ng;
    const uint16_t* const src = a + blockIdx.y * a_sb + n;
    u32x4 v[PASSES][4];
#pragma unroll
    for (int p = 0; p < PASSES; ++p) {
        const int64_t k = p * PASS + 4 * quad;              // (columns come in fours)
        const bool in = n < rows && k < cols;
#pragma unroll
        for (int i = 0; i < 4; ++i) v[p][i] = in ? *reinterpret_cast<const u32x4*>(src + (k + i) * a_sc) : u32x4{0, 0, 0, 0};
    }
    if (tid == 0) s_special = 0;
    uint32_t m[8] = {0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
    for (int p = 0; p < PASSES; ++p)
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int j = 0; j < 4; ++j) amax_bits(v[p][i][j], m[2 * j], m[2 * j + 1]);
#pragma unroll
    for (int j = 0; j < 8; ++j) {
#pragma unroll
        for (int o = LPR; o < kWave; o <<= 1) m[j] = max(m[j], (uint32_t)__shfl_xor((int)m[j], o, kWave));
        if (lane < LPR) s_max[wave][lane * 8 + j] = m[j];
    }
    __syncthreads();
    if (tid < STRIP) {
        uint32_t bits = 0;
#pragma unroll
        for (int w = 0; w < NW; ++w) bits = max(bits, s_max[w][tid]);
        const float s = scale_from_amax<true>(__uint_as_float(bits));
        s_scale[tid] = s;
        if (bits >= 0x7f800000u) s_special = 1;
        if (n0 + tid < rows) scale[blockIdx.y * rows + n0 + tid] = store_reciprocal ? 1.0f / s : s;
    }
    __syncthreads();
    const bool special = s_special != 0;
    float sc[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) sc[j] = s_scale[8 * ng + j];
#pragma unroll
    for (int p = 0; p < PASSES; ++p) {
        if (p * PASS >= cols) break;
        if (p) __syncthreads();
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            float f[4];
#pragma unroll
            for (int i = 0; i < 4; ++i)
                f[i] = ((j & 1) ? __uint_as_float(v[p][i][j / 2] & 0xffff0000u) : bf16_bits_to_f32(v[p][i][j / 2] & 0xffffu)) * sc[j];
            uint32_t w;
            if (!special) {
                int t = __builtin_amdgcn_cvt_pk_fp8_f32(f[0], f[1], 0, false);
                w = (uint32_t)__builtin_amdgcn_cvt_pk_fp8_f32(f[2], f[3], t, true);
            } else {
                w = e4m3fn_encode(f[0]) | (e4m3fn_encode(f[1]) << 8) | (e4m3fn_encode(f[2]) << 16) | (e4m3fn_encode(f[3]) << 24);
            }
            tile[(8 * ng + j) * DW + quad] = w;
        }
        __syncthreads();
        // rows out: QUADS / 4 lanes cover a pass's bytes of one, 16 each
        constexpr int LANES = QUADS / 4;
#pragma unroll
        for (int i = 0; i < STRIP * LANES / NT; ++i) {
            const int r = tid / LANES + i * (NT / LANES), c = 4 * (tid % LANES);
            const int64_t k = p * PASS + 4 * c;
            if (n0 + r >= rows) continue;
            uint8_t* dst = q + blockIdx.y * q_sb + (n0 + r) * q_sr + k;
            const uint32_t* t = tile + r * DW + c;
            if (wide && k + 16 <= cols) {
                *reinterpret_cast<u32x4*>(dst) = u32x4{t[0], t[1], t[2], t[3]};
            } else {
#pragma unroll
                for (int d = 0; d < 4; ++d)
                    if (k + 4 * d < cols) *reinterpret_cast<uint32_t*>(dst + 4 * d) = t[d];
            }
        }
    }
}

// rows that are whole pairs of chunks, stored 16 bytes at a time
inline bool wide_stores(int64_t cols, const uint8_t* q, int64_t q_sb, int64_t q_sr) {
    return cols % 16 == 0 && (reinterpret_cast<uintptr_t>(q) & 15u) == 0 && q_sb % 16 == 0 && q_sr % 16 == 0;
}

template <int CH>
void launch_fast(bool silu, const uint16_t* a, int64_t total, int64_t rows, int cols, int64_t a_sb,
                 int64_t a_sr, uint8_t* q, int64_t q_sb, int64_t q_sr, float* scale, int recip, const int64_t* offsets,
                 hipStream_t stream) {
    const unsigned blocks = (unsigned)((total + 3) / 4);
    if constexpr (CH % 2 == 0) {
        if (wide_stores(cols, q, q_sb, q_sr)) {
            if (silu)
                quant_rows_bf16_wave<CH, true, true><<<blocks, 256, 0, stream>>>(a, total, rows, cols, a_sb, a_sr, q,
                                                                                 q_sb, q_sr, scale, recip, offsets);
            else
                quant_rows_bf16_wave<CH, false, true><<<blocks, 256, 0, stream>>>(a, total, rows, cols, a_sb, a_sr, q,
                                                                                  q_sb, q_sr, scale, recip, offsets);
            return;
        }
    }
    if (silu)
        quant_rows_bf16_wave<CH, true><<<blocks, 256, 0, stream>>>(a, total, rows, cols, a_sb, a_sr, q,
                                                                   q_sb, q_sr, scale, recip, offsets);
    else
        quant_rows_bf16_wave<CH, false><<<blocks, 256, 0, stream>>>(a, total, rows, cols, a_sb, a_sr, q,
                                                                    q_sb, q_sr, scale, recip, offsets);
}

template <typename T>
void launch_generic(bool silu, bool lane_per_row, const void* a_, int64_t total, int64_t rows,
                    int64_t cols, int64_t a_sb, int64_t a_sr, int64_t a_sc, uint8_t* q, int64_t q_sb,
                    int64_t q_sr, int64_t q_sc, float* scale, int recip, hipStream_t stream) {
    const T* a = (const T*)a_;
#define FMOE_ARGS a, total, rows, cols, a_sb, a_sr, a_sc, q, q_sb, q_sr, q_sc, scale, recip
    if (lane_per_row) {
        const unsigned blocks = (unsigned)((total + 255) / 256);
        if (silu) quant_rows_generic_lane<T, true><<<blocks, 256, 0, stream>>>(FMOE_ARGS);
        else quant_rows_generic_lane<T, false><<<blocks, 256, 0, stream>>>(FMOE_ARGS);
    } else {
        const unsigned blocks = (unsigned)((total + 3) / 4);
        if (silu) quant_rows_generic_wave<T, true><<<blocks, 256, 0, stream>>>(FMOE_ARGS);
        else quant_rows_generic_wave<T, false><<<blocks, 256, 0, stream>>>(FMOE_ARGS);
    }
#undef FMOE_ARGS
}

// Where the one launch is faster than the form of a lane (under 16 rows: a wave) per row, whose time is a serial walk over the columns.  us, lane
// per row / one launch: 64 rows, 12 columns 5.3 / 4.5, 16 6.5 / 4.3, 44 16.4 / 4.5; 32768 rows, 12 6.1 / 5.6, 16 7.6 / 5.4; 2^17 rows, 16 8.4 / 12.0,
// 24 12.0 / 12.5, 32 16.5 / 12.3; 2^19 rows, 24 31 / 40, 32 54 / 39.  Wave per row: 8 rows, 1024 columns 6.2 / 7.3, 2048 9.9 / 7.9.
inline bool cols_one_pays(int64_t total_rows, int64_t rows, int64_t cols) {
    if (rows < 16) return cols > 1024;
    return cols >= (total_rows <= (1 << 15) ? 16 : 32);
}

// What the forms for rows that are columns in memory take: bf16, memory rows of whole aligned 16-byte chunks, result rows of whole dwords.
inline bool takes_cols(int a_dtype, int64_t batch, int64_t rows, int64_t cols, int64_t a_sb, int64_t a_sr, int64_t a_sc, int apply_silu) {
    return a_dtype == FMOE_BF16 && !apply_silu && a_sr == 1 && a_sc >= rows && rows % 8 == 0 && cols % 4 == 0 &&
           a_sc % 8 == 0 && (batch == 1 || a_sb % 8 == 0) && batch >= 1 && batch <= 65535 && rows >= 8 && rows < (1 << 27) &&
           (cols + kColTileK - 1) / kColTileK <= 65535 && (cols > kColOneMost || cols_one_pays(batch * rows, rows, cols));
}
inline bool cols_result(const void* a, const uint8_t* q, int64_t cols, int64_t q_sb, int64_t q_sr, int64_t q_sc) {
    return aligned16(a) && q_sc == 1 && q_sr % 4 == 0 && q_sb % 4 == 0 && q_sr >= cols && (reinterpret_cast<uintptr_t>(q) & 3u) == 0;
}
inline int wide_cols(const uint8_t* q, int64_t q_sb, int64_t q_sr) {
    return (reinterpret_cast<uintptr_t>(q) & 15u) == 0 && q_sr % 16 == 0 && q_sb % 16 == 0;
}

int launch_cols_one(const uint16_t* a, int64_t batch, int64_t rows, int64_t cols, int64_t a_sb, int64_t a_sc, uint8_t* q, int64_t q_sb,
                    int64_t q_sr, float* scale, int recip, const int64_t* offsets, hipStream_t stream) {
    auto one = [&](auto kern, int strip, int threads) {
        const int strips = (int)((rows + strip - 1) / strip);
        kern<<<dim3((unsigned)(strips > 8 ? (strips + 7) / 8 * 8 : strips), (unsigned)batch), threads, 0, stream>>>(
            a, rows, cols, a_sb, a_sc, q, q_sb, q_sr, scale, recip, wide_cols(q, q_sb, q_sr), strips, offsets);
        return check_launch("fmoe_quant_rows_e4m3");
    };
    if (cols <= 256) return one(quant_cols_one<32, 256, 1>, 32, 256);
    if (cols <= 512) return one(quant_cols_one<32, 256, 2>, 32, 256);
    if (cols <= 1024) return one(quant_cols_one<64, 512, 4>, 64, 512);
    if (cols <= 1536) return one(quant_cols_one<32, 512, 3>, 32, 512);
    if (cols <= 2048) return one(quant_cols_one<32, 512, 4>, 32, 512);
    if (cols <= 3072) return one(quant_cols_one<32, 512, 6>, 32, 512);
    return one(quant_cols_one<32, 1024, 4>, 32, 1024);
}

// offsets: NULL, or the experts' rows of the call the result is for (batch + 1); the forms that bring no time leave them aside
int quant_rows(const void* a, int a_dtype, int64_t batch, int64_t rows, int64_t cols, int64_t a_sb, int64_t a_sr, int64_t a_sc,
               int apply_silu, uint8_t* q, int64_t q_sb, int64_t q_sr, int64_t q_sc, float* scale, int store_reciprocal,
               const int64_t* offsets, hipStream_t stream) {
    FMOE_REQUIRE(a_dtype == FMOE_BF16 || a_dtype == FMOE_F32,
                 "fmoe_quant_rows_e4m3: input must be bf16 or fp32");
    FMOE_REQUIRE(batch >= 0 && rows >= 0 && cols >= 1,
                 "fmoe_quant_rows_e4m3: need batch, rows >= 0 and cols >= 1 (got %lld, %lld, %lld)",
                 (long long)batch, (long long)rows, (long long)cols);
    const int64_t total = batch * rows;
    if (total == 0) return FMOE_OK;
    FMOE_REQUIRE(total < ((int64_t)1 << 31) * 4, "fmoe_quant_rows_e4m3: too many rows");
    FMOE_REQUIRE(a && q && scale, "fmoe_quant_rows_e4m3: NULL pointer");

    const bool fast = a_dtype == FMOE_BF16 && a_sc == 1 && q_sc == 1 && (cols % 8) == 0 &&
                      cols <= 16 * 512 && aligned16(a) && (a_sb % 8) == 0 && (a_sr % 8) == 0 &&
                      (reinterpret_cast<uintptr_t>(q) & 7u) == 0 && (q_sb % 8) == 0 && (q_sr % 8) == 0;
    if (fast) {
        int ch = (int)((cols / 8 + kWave - 1) / kWave);
        if (wide_stores(cols, q, q_sb, q_sr)) ch = 2 * (int)((cols / 16 + kWave - 1) / kWave);
#define FMOE_FAST(CH)                                                                              \
    launch_fast<CH>(apply_silu != 0, (const uint16_t*)a, total, rows, (int)cols, a_sb, a_sr, q, q_sb, \
                    q_sr, scale, store_reciprocal, offsets, stream)
        if (ch <= 1) FMOE_FAST(1);
        else if (ch <= 2) FMOE_FAST(2);
        else if (ch <= 3) FMOE_FAST(3);
        else if (ch <= 4) FMOE_FAST(4);
        else if (ch <= 6) FMOE_FAST(6);
        else if (ch <= 8) FMOE_FAST(8);
        else if (ch <= 12) FMOE_FAST(12);
        else FMOE_FAST(16);
#undef FMOE_FAST
        return check_launch("fmoe_quant_rows_e4m3");
    }
    const bool long_rows = a_dtype == FMOE_BF16 && a_sc == 1 && q_sc == 1 && (cols % 8) == 0 && aligned16(a) &&
                           (a_sb % 8) == 0 && (a_sr % 8) == 0 && (reinterpret_cast<uintptr_t>(q) & 7u) == 0 &&
                           (q_sb % 8) == 0 && (q_sr % 8) == 0 && total < ((int64_t)1 << 31);
    if (long_rows) {
        if (apply_silu)
            quant_rows_bf16_block<true><<<(unsigned)total, 256, 0, stream>>>((const uint16_t*)a, rows, cols, a_sb, a_sr,
                                                                             q, q_sb, q_sr, scale, store_reciprocal);
        else
            quant_rows_bf16_block<false><<<(unsigned)total, 256, 0, stream>>>((const uint16_t*)a, rows, cols, a_sb, a_sr,
                                                                              q, q_sb, q_sr, scale, store_reciprocal);
        return check_launch("fmoe_quant_rows_e4m3");
    }
    if (cols <= kColOneMost && takes_cols(a_dtype, batch, rows, cols, a_sb, a_sr, a_sc, apply_silu) && cols_result(a, q, cols, q_sb, q_sr, q_sc))
        return launch_cols_one((const uint16_t*)a, batch, rows, cols, a_sb, a_sc, q, q_sb, q_sr, scale, store_reciprocal, offsets, stream);
    const bool lane_per_row = a_sc != 1 && a_sr == 1 && rows >= 16;
    if (a_dtype == FMOE_BF16)
        launch_generic<uint16_t>(apply_silu != 0, lane_per_row, a, total, rows, cols, a_sb, a_sr, a_sc, q,
                                 q_sb, q_sr, q_sc, scale, store_reciprocal, stream);
    else
        launch_generic<float>(apply_silu != 0, lane_per_row, a, total, rows, cols, a_sb, a_sr, a_sc, q,
                              q_sb, q_sr, q_sc, scale, store_reciprocal, stream);
    return check_launch("fmoe_quant_rows_e4m3");
}

int quant_rows_ws(const void* a, int a_dtype, int64_t batch, int64_t rows, int64_t cols, int64_t a_sb, int64_t a_sr, int64_t a_sc,
                  int apply_silu, uint8_t* q, int64_t q_sb, int64_t q_sr, int64_t q_sc, float* scale, int store_reciprocal,
                  const int64_t* offsets, void* workspace, size_t workspace_bytes, hipStream_t stream) {
    const size_t need = fmoe_quant_rows_workspace_bytes(a_dtype, batch, rows, cols, a_sb, a_sr, a_sc, apply_silu);
    if (need == 0 || workspace_bytes < need || !workspace || !a || !q || !scale || !cols_result(a, q, cols, q_sb, q_sr, q_sc))
        return quant_rows(a, a_dtype, batch, rows, cols, a_sb, a_sr, a_sc, apply_silu, q, q_sb, q_sr, q_sc, scale, store_reciprocal,
                          offsets, stream);
    const int splits = col_splits(batch, rows, cols);
    const int64_t per_split = (cols + splits - 1) / splits;
    const int64_t strips = (rows + kColTileN - 1) / kColTileN;
    uint32_t* part = (uint32_t*)workspace;
    quant_cols_amax<<<dim3((unsigned)strips, (unsigned)splits, (unsigned)batch), 256, 0, stream>>>(
        (const uint16_t*)a, rows, cols, a_sb, a_sc, part, batch * rows, per_split, offsets);
    quant_cols_store<<<dim3((unsigned)strips, (unsigned)((cols + kColTileK - 1) / kColTileK), (unsigned)batch), 256, 0,
                       stream>>>((const uint16_t*)a, rows, cols, a_sb, a_sc, part, splits, batch * rows, q, q_sb, q_sr,
                                 scale, store_reciprocal, wide_cols(q, q_sb, q_sr), offsets);
    return check_launch("fmoe_quant_rows_e4m3_ws");
}

}  // namespace
}  // namespace fmoe

using namespace fmoe;

extern "C" int fmoe_quant_rows_e4m3(const void* a, int a_dtype, int64_t batch, int64_t rows, int64_t cols,
                                    int64_t a_sb, int64_t a_sr, int64_t a_sc, int apply_silu, uint8_t* q,
                                    int64_t q_sb, int64_t q_sr, int64_t q_sc, float* scale,
                                    int store_reciprocal, fmoe_stream_t stream) {
    return quant_rows(a, a_dtype, batch, rows, cols, a_sb, a_sr, a_sc, apply_silu, q, q_sb, q_sr, q_sc, scale, store_reciprocal, nullptr,
                      (hipStream_t)stream);
}

extern "C" size_t fmoe_quant_rows_workspace_bytes(int a_dtype, int64_t batch, int64_t rows, int64_t cols, int64_t a_sb,
                                                  int64_t a_sr, int64_t a_sc, int apply_silu) {
    if (cols <= kColOneMost || !takes_cols(a_dtype, batch, rows, cols, a_sb, a_sr, a_sc, apply_silu)) return 0;
    return (size_t)col_splits(batch, rows, cols) * (size_t)(batch * rows) * sizeof(uint32_t);
}

extern "C" int fmoe_quant_rows_e4m3_ws(const void* a, int a_dtype, int64_t batch, int64_t rows, int64_t cols,
                                       int64_t a_sb, int64_t a_sr, int64_t a_sc, int apply_silu, uint8_t* q,
                                       int64_t q_sb, int64_t q_sr, int64_t q_sc, float* scale, int store_reciprocal,
                                       void* workspace, size_t workspace_bytes, fmoe_stream_t stream) {
    return quant_rows_ws(a, a_dtype, batch, rows, cols, a_sb, a_sr, a_sc, apply_silu, q, q_sb, q_sr, q_sc, scale, store_reciprocal, nullptr,
                         workspace, workspace_bytes, (hipStream_t)stream);
}

extern "C" int fmoe_quant_expert_weights_e4m3(const void* a, int a_dtype, int64_t batch, int64_t rows, int64_t cols,
                                              int64_t a_sb, int64_t a_sr, int64_t a_sc, uint8_t* q,
                                              int64_t q_sb, int64_t q_sr, int64_t q_sc, float* scale, const int64_t* offsets,
                                              void* workspace, size_t workspace_bytes, fmoe_stream_t stream) {
    FMOE_REQUIRE(offsets, "fmoe_quant_expert_weights_e4m3: NULL pointer");
    return quant_rows_ws(a, a_dtype, batch, rows, cols, a_sb, a_sr, a_sc, 0, q, q_sb, q_sr, q_sc, scale, 0, offsets, workspace,
                         workspace_bytes, (hipStream_t)stream);
}
