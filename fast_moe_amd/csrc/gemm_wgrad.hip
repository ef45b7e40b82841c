// fmoe_weight_grad: weight gradients of experts with few rows, both operands row-major.
#include "gemm_wgrad.h"
#include "gemm_kernel.h"

using namespace fmoe;

// Where the kernel is taken, against the ring on the tensors in place (bf16) or the fp32 GEMM on transposed copies: a short contraction,
// whose cost is the stores, and matrices that leave the ring's 256 x 256 tiles less than half the CUs (up to 1024 rows per expert).
// us, the ring / it:
//   330 rows, 77 experts, 704 x 1896, Zipf 97 / 40; 490 rows, 52 experts, 1648 x 368 34 / 16.5; 469 rows, 10 experts, 2720 x 3136 56.5 / 35;
//   128 experts, 1536 x 4096 (1.6 GB, 252 at copy speed): 8 rows each 421 / 279, 32 500 / 334 (Zipf 473 / 385, one hot expert 740 / 543), 64
//   511 / 465, 96 491 / 542; 64 experts, 2816 x 2048, 96 each 217 / 249; 16 experts, 2048 x 2048, 128 each 40.7 / 37.3, 192 45.1 / 47.1
//   8 experts, 512 x 256, 1024 rows each 25.7 / 19.2, one hot expert 124 / 115; 1024 x 512, 512 each 18.8 / 13.5; 4096 x 1024, 256 each (two
//   rounds of the ring) 30.0 / 33.7
// fp32 against the transposed copies, their index launches and the three-part GEMM, us of a layer's whole training step: 847 tokens, 5 experts,
// top-2, 576 x 792 882 / 592; 2000 tokens, 8 experts, 512 x 1024 856 / 568; 2048, 1024 x 2048 1372 / 1359; 600 tokens, 5 experts, 2048 x 4096
// 1566 / 1418; not taken: 1000 tokens, 8 experts, top-4, 2048 x 2048 (1.7e10 products a matrix) 2378 / 2274; 4096 tokens, 4 experts, top-3, 1024 x
// 4096 (5.2e10) 5819 / 5851.
extern "C" int fmoe_weight_grad_pays(int dtype, int num_experts, int m, int n, int64_t rows) {
    if (num_experts < 1 || m < 1 || n < 1 || rows < 1) return 0;
    if (rows <= 64 * (int64_t)num_experts) return 1;
    if (dtype == FMOE_F32) return (double)rows * m * n <= 1.2e10;
    const int64_t ring_tiles = (int64_t)num_experts * ((m + 255) / 256) * ((n + 255) / 256);
    return rows <= 1024 * (int64_t)num_experts && 2 * ring_tiles <= compute_units();
}

extern "C" int fmoe_weight_grad(const void* a, const void* b, int dtype, int num_experts, int m, int n, int64_t rows,
                                int64_t a_stride_row, int64_t b_stride_row, const int64_t* offsets, void* out, void* out2,
                                fmoe_stream_t stream_) {
    FMOE_REQUIRE(num_experts >= 1 && m >= 1 && n >= 1 && rows >= 0, "fmoe_weight_grad: need E, m, n >= 1 and rows >= 0");
    FMOE_REQUIRE(dtype == FMOE_BF16 || dtype == FMOE_F32, "fmoe_weight_grad: operands must be bf16 or fp32");
    FMOE_REQUIRE(a && b && offsets && out, "fmoe_weight_grad: NULL tensor pointer");
    const int chunk = dtype == FMOE_F32 ? 4 : 8;
    FMOE_REQUIRE(m % chunk == 0 && n % chunk == 0 && a_stride_row >= m && b_stride_row >= n && a_stride_row % chunk == 0 &&
                     b_stride_row % chunk == 0 && aligned16(a) && aligned16(b) && aligned16(out) && aligned16(out2) && n < (1 << 25),
                 "fmoe_weight_grad: rows of whole 16-byte chunks at 16-byte boundaries");
    FMOE_REQUIRE(!out2 || m % 64 == 0, "fmoe_weight_grad: out2 takes the second half of m, whole blocks of 32 rows each");
    FMOE_REQUIRE(rows < ((int64_t)1 << 31) && num_experts * (int64_t)m < ((int64_t)1 << 31), "fmoe_weight_grad: more than 2^31 rows");
    GemmParams p = {};
    p.E = num_experts;
    p.N = n;
    p.K = (int)rows;
    p.total_rows = num_experts * (int64_t)m;
    p.a = (const uint8_t*)a;
    p.b = (const uint8_t*)b;
    p.a_sk = a_stride_row;
    p.b_sk = b_stride_row;
    p.k_window = offsets;
    p.out = (uint16_t*)out;
    p.out2 = (uint16_t*)out2;
    p.out_half = out2 ? m / 2 : 0;
    p.out_stride = n;
    p.vec_store = 1;
    WgradTile t;
    const int col_tiles = (n + WgradTile::BN - 1) / WgradTile::BN;
    t.m = m;
    t.row_tiles = (m + WgradTile::BM - 1) / WgradTile::BM;
    // column tiles to a block: up to four, as long as there are two rounds and a half of blocks (three to a CU)
    t.strip = 1;
    while (t.strip < 4 && (int64_t)num_experts * t.row_tiles * ((col_tiles + 2 * t.strip - 1) / (2 * t.strip)) >= 8 * (int64_t)compute_units())
        t.strip *= 2;
    t.strips = (col_tiles + t.strip - 1) / t.strip;
    const int64_t tiles = (int64_t)t.row_tiles * t.strips;
    t.per_xcd = tiles >= kNumXcd ? (int)((tiles + kNumXcd - 1) / kNumXcd) : 0;
    const int64_t grid = num_experts * (t.per_xcd ? (int64_t)t.per_xcd * kNumXcd : tiles);
    if (grid >= ((int64_t)1 << 31)) return fail(FMOE_ERR_UNSUPPORTED, "fmoe_weight_grad: grid too large");
    hipStream_t stream = (hipStream_t)stream_;
    if (dtype == FMOE_F32) grouped_wgrad_kernel<true><<<(unsigned)grid, WgradTile::NT, WgradTile::LDS_BYTES, stream>>>(p, t);
    else grouped_wgrad_kernel<false><<<(unsigned)grid, WgradTile::NT, WgradTile::LDS_BYTES, stream>>>(p, t);
    return check_launch("fmoe_weight_grad");
}
