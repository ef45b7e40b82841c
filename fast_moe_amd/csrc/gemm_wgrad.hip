// Weight gradients of experts with few rows (bf16, row-major operands).
#include "gemm_wgrad.h"
#include "gemm_kernel.h"

namespace fmoe {

// Column tiles to a block: up to four, as long as there are two rounds and a half of blocks (three to a CU).
int run_wgrad_short(GemmParams p, hipStream_t stream) {
    const int64_t row_tiles = most_row_tiles(p.total_rows, p.E, WgradTile::BM), col_tiles = (p.N + WgradTile::BN - 1) / WgradTile::BN;
    int strip = 1;
    while (strip < 4 && row_tiles * ((col_tiles + 2 * strip - 1) / (2 * strip)) >= 8 * (int64_t)compute_units()) strip *= 2;
    p.n_tiles = (int)((col_tiles + strip - 1) / strip);
    const int64_t groups = (row_tiles + kGroupM - 1) / kGroupM;
    const int64_t grid = (groups + kNumXcd - 1) / kNumXcd * kNumXcd * kGroupM * p.n_tiles;
    if (grid >= ((int64_t)1 << 31)) return fail(FMOE_ERR_UNSUPPORTED, "fmoe_grouped_gemm: grid too large");
    grouped_wgrad_kernel<<<(unsigned)grid, WgradTile::NT, WgradTile::LDS_BYTES, stream>>>(p, strip);
    return check_launch("fmoe_grouped_gemm");
}

}  // namespace fmoe
