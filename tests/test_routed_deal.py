"""How the tiles of expert-routed rows are dealt to the XCDs (csrc/routed_deal.h, which the tile kernels call), on the host compiler: with
any numbers of row tiles per height class and of column tiles, every tile is dealt once inside the launch's grid, and every
XCD gets an even share of each class, the highest first. Dealt as one sequence, one XCD gets all the high tiles of a skewed routing
(128 experts of 2048 x 768, 16384 rows, half of
them with one expert: 139 us, 110 with even shares)."""
import itertools
import os
import subprocess

from tests.test_stream_loop_waits import CSRC

SRC = r"""
#include "routed_deal.h"
#include <cstdio>
#include <cstdlib>
#include <vector>
using namespace mtq;
int main(int argc, char** argv) {
    for (int i = 1; i + 4 < argc; i += 5) {
        uint32_t count[QD_HEIGHTS], all_rows = 0;
        for (int h = 0; h < 4; h++) all_rows += count[h] = (uint32_t)atoi(argv[i + h]);
        const uint32_t n_tiles = (uint32_t)atoi(argv[i + 4]), total = all_rows * n_tiles, grid = (total + 7) & ~7u, stride = all_rows + 5;
        std::vector<int> seen(4 * stride * n_tiles, 0);
        for (uint32_t x = 0; x < 8; x++) {
            uint32_t of[4] = {0}, all = 0, last = 0;
            for (uint32_t at = 0; at < grid / 8 + 3; at++) {
                const uint32_t t = routed_deal(count, stride, n_tiles, x, at);
                if (t == 0xFFFFFFFFu) continue;
                const uint32_t h = t / n_tiles / stride;
                if (h > 3 || t / n_tiles - h * stride >= count[h] || seen[t]++ || at >= grid / 8 || at != all) return printf("bad tile %u\n", t), 1;
                if (h < last) return printf("a higher tile behind a lower one\n"), 1;
                last = h; of[h]++; all++;
            }
            for (int h = 0; h < 4; h++) {
                const uint32_t c = count[h] * n_tiles;
                if (of[h] < c / 8 || of[h] > (c + 7) / 8) return printf("uneven\n"), 1;
            }
            if (all < total / 8) return printf("uneven in all\n"), 1;
        }
        uint32_t dealt = 0;
        for (int s : seen) dealt += s;
        if (dealt != total) return printf("tile left out\n"), 1;
    }
    printf("ok\n");
    return 0;
}
"""


def test_every_tile_once_and_even_shares(tmp_path):
    src, exe = str(tmp_path / "deal.cpp"), str(tmp_path / "deal")
    open(src, "w").write(SRC)
    r = subprocess.run(["g++", "-std=c++17", "-O1", "-fsanitize=address,undefined", "-fno-sanitize-recover=all", "-I", CSRC, src, "-o", exe], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-2000:]
    cases = [(*h, n) for h in itertools.product((0, 1, 3, 8, 13), repeat=4) for n in (1, 5, 16)] + [(52, 0, 0, 127, 16), (0, 2, 0, 7, 32)]
    r = subprocess.run([exe, *(str(v) for c in cases for v in c)], capture_output=True, text=True)
    assert r.returncode == 0 and r.stdout == "ok\n", r.stdout + r.stderr[-2000:]
