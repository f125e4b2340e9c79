"""The walk of every wave of the weight-gradient kernel, replayed on the CPU with
the kernel's own index functions: whatever a wave loads lies inside the tensor,
also for the waves past the last unit, and every pixel of dy is met exactly
once, together with the rows of x around it."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SOURCE = r"""
#include "wgrad_walk.h"
#include <cstdio>
#include <cstdlib>
#include <vector>
using namespace gr;

template <int HALO, int SEG>
static int replay(int n, int H, int W, int cin, int cout, int forced)
{
    const long long tiles = (long long)((cout + 31) / 32) * ((cin + 31) / 32);
    const long long columns = (long long)n * ((W + SEG - 1) / SEG);
    const int rows = forced > 0 ? forced : wgrad_rows(columns, H, tiles);
    const long long units = columns * ((H + rows - 1) / rows);
    std::vector<int> met((size_t)n * H * W, 0);
    std::vector<char> read(met.size());
    for (long long unit = 0; unit < 4 * ((units + 3) / 4); ++unit) {
        const WgradUnit U = wgrad_unit<SEG>((int)unit, n, H, W, rows);
        std::vector<size_t> x;
        auto load = [&](int t) {
            for (int is_x = 0; is_x < 2; ++is_x) {
                const int row = wgrad_row(U.r0, t, is_x, HALO);
                if (!wgrad_row_ok(row, t, U.nrows, H, is_x)) continue;
                const int extra = is_x ? 2 * HALO : 0;  // pixels beyond the segment
                for (int i = 0; i < SEG + extra; ++i) {
                    const int px = U.x0 + i - (is_x ? HALO : 0);
                    if (px < 0 || px >= W) continue;
                    if (U.img < 0 || U.img >= n || row < 0 || row >= H) {
                        std::printf("unit %lld of %lld reads image %d row %d of %d x %d rows\n",
                                    unit, units, U.img, row, n, H);
                        return false;
                    }
                    const size_t at = ((size_t)U.img * H + row) * W + px;
                    if (is_x) { read[at] = 1; x.push_back(at); }
                    else ++met[at];
                }
            }
            return true;
        };
        const int first = wgrad_first(U.nrows, HALO);
        if (first < U.nrows && !load(first)) return 1;
        for (int t = first; t < U.nrows; ++t)
            if (!load(t + 1)) return 1;
        // the taps of each row of the walk find their rows of x
        for (int r = 0; r < U.nrows; ++r)
            for (int dr = -HALO; dr <= HALO; ++dr)
                for (int i = -HALO; i < SEG + HALO; ++i) {
                    const int row = U.r0 + r + dr, px = U.x0 + i;
                    if (row < 0 || row >= H || px < 0 || px >= W) continue;
                    if (!read[((size_t)U.img * H + row) * W + px]) return 2;
                }
        for (size_t at : x) read[at] = 0;
    }
    for (int m : met)
        if (m != 1) return 3;
    return 0;
}

int main(int argc, char** argv)
{
    int a[8];
    for (int i = 0; i < 8; ++i) a[i] = std::atoi(argv[i + 1]);
    const int halo = a[0], seg = a[1];
    return halo == 0 ? replay<0, 64>(a[2], a[3], a[4], a[5], a[6], a[7])
           : seg == 32 ? replay<1, 32>(a[2], a[3], a[4], a[5], a[6], a[7])
                       : replay<1, 64>(a[2], a[3], a[4], a[5], a[6], a[7]);
}
"""

# (n, H, W, cin, cout, rows per wave; 0: the launch's own choice)
CASES = [(n, 3, 5, 32, 32, rows) for n in range(1, 9) for rows in (1, 2, 3)]  # 1 .. 24 units
CASES += [
    (1, 64, 64, 384, 128, 0),    # 22 units
    (3, 128, 128, 64, 64, 0),    # 258
    (13, 32, 32, 256, 256, 0),   # 26
    (25, 32, 32, 256, 256, 0),   # 25, one walk an image
    (1, 1, 1, 8, 8, 0), (5, 60, 130, 40, 64, 0), (9, 90, 129, 32, 32, 0),
]


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    d = tmp_path_factory.mktemp("wgrad")
    src, exe = d / "walk.cpp", d / "walk"
    src.write_text(SOURCE)
    subprocess.run(["g++", "-O1", "-std=c++17", "-I", os.path.join(ROOT, "graptor_amd", "csrc"),
                    "-o", str(exe), str(src)], check=True)
    return str(exe)


@pytest.mark.parametrize("halo,seg", [(1, 64), (1, 32), (0, 64)])
def test_every_wave_stays_inside(program, halo, seg):
    for case in CASES:
        r = subprocess.run([program, str(halo), str(seg), *map(str, case)],
                           capture_output=True, text=True)
        assert r.returncode == 0, (case, r.returncode, r.stdout)
