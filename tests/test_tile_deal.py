"""The ring kernel's tile order (csrc/gemm_deal.h), walked on the host: every XCD's share, for every kind of launch, together
names each tile of the launch once; and the share of the busiest XCD where the left-over groups go out as equal runs."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = r"""
#include <cstdio>
#include <cstdlib>
#include <vector>
#include "gemm_deal.h"

template <typename T, bool EQUAL_COST>
int check(int row_tiles, int n_tiles, int slots, bool groups) {
    std::vector<int> seen((size_t)row_tiles * n_tiles, 0);
    for (int xcd = 0; xcd < 8; ++xcd) {
        using Deal = fmoe::TileDeal<T, 8, 4, EQUAL_COST>;
        const Deal d = groups ? Deal(row_tiles, n_tiles, xcd, slots) : Deal::contiguous(row_tiles, n_tiles, xcd);
        for (T j = 0; j < d.count; ++j) {
            const T t = groups ? d.tile(j, j / d.span) : d.run_base + j;
            if (t < 0 || t >= (T)seen.size()) return printf("tile %lld of %zu\n", (long long)t, seen.size()), 1;
            ++seen[t];
        }
    }
    for (size_t t = 0; t < seen.size(); ++t)
        if (seen[t] != 1) return printf("tile %zu computed %d times\n", t, seen[t]), 1;
    return 0;
}

int main(int argc, char** argv) {
    if (argc > 1) {     // row_tiles n_tiles slots equal_cost -> tiles of every XCD
        const int m = atoi(argv[1]), n = atoi(argv[2]), slots = atoi(argv[3]);
        for (int xcd = 0; xcd < 8; ++xcd)
            printf("%d ", atoi(argv[4]) ? fmoe::TileDeal<int, 8, 4>(m, n, xcd, slots).count
                                        : fmoe::TileDeal<int, 8, 4, false>(m, n, xcd, slots).count);
        return 0;
    }
    for (int n_tiles : {1, 2, 3, 4, 6, 11, 16, 40})
        for (int slots : {32, 31, 4, 1})
            for (int row_tiles = 0; row_tiles <= 230; ++row_tiles)
                for (bool groups : {true, false})
                    if (check<int, true>(row_tiles, n_tiles, slots, groups) || check<long long, true>(row_tiles, n_tiles, slots, groups) ||
                        check<int, false>(row_tiles, n_tiles, slots, groups))
                        return printf("row tiles %d, column tiles %d, slots %d, groups %d\n", row_tiles, n_tiles, slots, groups), 1;
    return 0;
}
"""


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    from fast_moe_amd import build
    where = tmp_path_factory.mktemp("deal")
    src, exe = str(where / "deal.hip"), str(where / "deal")
    with open(src, "w") as f:
        f.write(PROGRAM)
    res = subprocess.run([build._hipcc(), "--offload-host-only", "-O2", "-std=c++17", "-I" + build.CSRC, src, "-o", exe],
                         capture_output=True, text=True)
    assert res.returncode == 0, res.stderr
    return exe


def test_every_tile_is_dealt_once(program):
    res = subprocess.run([program], capture_output=True, text=True)
    assert res.returncode == 0, res.stdout


@pytest.mark.parametrize("row_tiles,n_tiles,busiest,equal_cost", [(*c, True) for c in [
    (42, 10, 53), (11, 16, 22),     # runs: a round of tiles fewer on the busiest XCD (of 80, of 64)
    (39, 4, 20),                    # all tiles at once
    (81, 10, 102),                  # the last round of 120 three quarters full
    (33, 16, 80), (130, 6, 108), (34, 8, 48), (67, 8, 88),       # groups: a run would give every XCD a last round of its own
    (64, 8, 64), (28, 4, 16),       # nothing left; seven groups
]] + [(42, 10, 80, False), (48, 11, 88, False), (11, 16, 22, False)])     # contraction windows: runs without a whole round only
def test_left_over_groups(program, row_tiles, n_tiles, busiest, equal_cost):
    out = subprocess.run([program, str(row_tiles), str(n_tiles), "32", str(int(equal_cost))], capture_output=True, text=True, check=True).stdout
    assert max(int(v) for v in out.split()) == busiest
