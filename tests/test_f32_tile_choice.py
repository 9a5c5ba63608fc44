"""Which tile shape fp32 products take (csrc/tiles_f32.hpp), on the CPU: by the table of the kernel that their depth runs."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PROGRAM = r"""
#include <cassert>
#include "tiles_f32.hpp"
using namespace sd3;
int pick(int M, int N, int K) {
    const F32Layer l{M, N, K};
    return pick_f32_tile(&l, 1, 256, K % 32 == 0);
}
int main() {
    // Depths that are not whole K tiles, us with 128x128 | 128x64 | 64x64 | 32x64 | 32x32 tiles: the choice is the fastest one or within 2 % of it
    const struct { int M, N, K; double us[F32_TILES]; } ragged[] = {
        {1178, 6144, 1548, {194.22, 202.06, 209.57, 205.79, 230.25}}, {1178, 3072, 6156, {384.38, 392.64, 408.05, 398.80, 440.74}},
        {2356, 1536, 1548, {103.21, 104.11, 107.46, 107.51, 116.54}}, {2356, 4608, 1548, {287.76, 300.79, 287.09, 307.09, 342.61}},
        {6000, 4608, 1548, {661.83, 690.60, 696.12, 771.14, 859.68}}, {8500, 768, 6156, {739.37, 772.14, 707.63, 725.73, 789.03}},
        {8500, 2304, 1548, {474.10, 495.15, 494.00, 551.98, 610.80}}, {200, 4096, 6156, {381.36, 206.47, 114.39, 119.92, 127.41}},
        {1024, 1024, 1548, {99.85, 56.77, 33.75, 34.61, 36.21}},      {512, 4608, 6156, {381.31, 389.83, 307.12, 283.89, 284.09}},
        {1178, 1536, 6156, {382.27, 208.74, 208.97, 230.04, 227.55}}, {77, 1536, 6156, {378.61, 206.01, 113.47, 69.74, 44.36}},
    };
    for (const auto& c : ragged) {
        double best = c.us[0];
        for (double us : c.us) best = us < best ? us : best;
        assert(c.us[pick(c.M, c.N, c.K)] <= 1.02 * best);
    }
    // the same sizes of whole K tiles go by the other table
    assert(pick(1178, 6144, 1536) == 3 && pick(1178, 6144, 1548) == 0 && pick(6000, 4608, 1536) == 2 && pick(6000, 4608, 1548) == 0);
    return 0;
}
"""


def test_tile_shape_by_depth(tmp_path):
    src, exe = tmp_path / "tiles.cpp", tmp_path / "tiles"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-Wall", "-I", os.path.join(ROOT, "sd3.c_amd", "csrc"), str(src), "-o", str(exe)], check=True)
    subprocess.run([str(exe)], check=True)
