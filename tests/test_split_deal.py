"""The tall ring's last round cut along K (csrc/gemm_split.h), walked on the host: every tile once, whole or as parts that cover every
pair of its K-slices once, no more pieces than blocks and none of fewer than two pairs; no block has work behind a piece.
And the fp32 kernel's (csrc/gemm_f32x3.h), a block of which takes one tile or piece: up to two pieces to a CU."""
import os
import subprocess

PROGRAM = r"""
#include <cstdio>
#include <vector>
#include "gemm_f32x3.h"

int check(int total, int slots, int pairs, int f32) {
    std::vector<std::vector<int>> seen(total, std::vector<int>(pairs, 0));
    std::vector<int> pieces_seen(2 * fmoe::kSplitMost, 0);
    for (int xcd = 0; xcd < 8; ++xcd) {
        const fmoe::SplitDeal d = f32 ? fmoe::SplitDeal(total, slots, xcd, pairs, [&](int r, int p, int b) { return f32 == 128 ? fmoe::f32x3_split_pieces<128>(r, p, b) : fmoe::f32x3_split_pieces<64>(r, p, b); })
                                      : fmoe::SplitDeal(total, slots, xcd, pairs);
        if (f32 && d.count > (total / (8 * slots) + 2) * slots) return printf("%d blocks of an XCD\n", d.count), 1;   // the launch's grid
        for (int j = 0; j < d.count; ++j) {
            int piece, part, first = 0, number = 2 * pairs;
            const int t = d.tile(j, piece, part);
            if (t < 0 || t >= total) return printf("tile %d of %d\n", t, total), 1;
            if (piece >= 0) {
                if (piece >= (f32 ? 16 * slots : fmoe::kSplitMost) || pieces_seen[piece]++) return printf("piece %d\n", piece), 1;
                if (!f32 && j + slots < d.count) return printf("work behind a piece\n"), 1;
                if (piece % d.rest != t - d.base || piece / d.rest != part) return printf("piece %d is not part %d of %d\n", piece, part, t), 1;
                d.slices(part, pairs, first, number);
                if (number < 4) return printf("%d slices\n", number), 1;
            }
            if (first % 2 || number % 2) return printf("half a pair\n"), 1;
            for (int k = first / 2; k < (first + number) / 2; ++k) ++seen[t][k];
        }
    }
    for (auto& t : seen)
        for (int n : t)
            if (n != 1) return printf("a pair of slices computed %d times\n", n), 1;
    return 0;
}

int main() {
    for (int slots : {32, 31, 4, 1})
        for (int pairs : {4, 5, 16, 61, 64, 200})
            for (int total = 0; total <= 40 * slots; total += total < 300 ? 1 : 37)
                if (check(total, slots, pairs, 0) || check(total, slots, pairs, 64) || check(total, slots, pairs, 128)) return printf("total %d, slots %d, pairs %d\n", total, slots, pairs), 1;
    return 0;
}
"""


def test_every_tile_and_every_pair_of_slices_once(tmp_path):
    from fast_moe_amd import build
    src, exe = str(tmp_path / "split.hip"), str(tmp_path / "split")
    with open(src, "w") as f:
        f.write(PROGRAM)
    res = subprocess.run([build._hipcc(), "--offload-host-only", "-O2", "-std=c++17", "-w", "-I" + build.CSRC, src, "-o", exe],
                         capture_output=True, text=True)
    assert res.returncode == 0, res.stderr
    res = subprocess.run([exe], capture_output=True, text=True)
    assert res.returncode == 0, res.stdout
