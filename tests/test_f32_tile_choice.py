"""Which kernel and which tile shape fp32 products take (csrc/tiles_f32.hpp), on the CPU: by the table of the kernel that their depth runs."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PROGRAM = r"""
#include <cassert>
#include <initializer_list>
#include "tiles_f32.hpp"
using namespace sd3;
int pick(int M, int N, int K) {
    const F32Layer l{M, N, K};
    return pick_f32_tile(&l, 1, 256, K % 32 == 0);
}
bool by_pieces(int K, int K2 = 0) {
    const F32Layer l[2] = {{1178, 1536, K}, {333, 1536, K2}};
    return f32_by_pieces(l, K2 ? 2 : 1);
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
    assert(pick(1178, 6144, 1568) == 3 && pick(1178, 6144, 1548) == 0 && pick(6000, 4608, 1568) == 2 && pick(6000, 4608, 1548) == 0);

    // Whole groups of four K tiles from 512 on go by pieces, a launch only if all its layers do
    for (int K : {32, 128, 256, 384, 544, 576, 608, 1548, 1568, 6156}) assert(!by_pieces(K));
    for (int K : {512, 640, 768, 1024, 1536, 6144}) assert(by_pieces(K));
    assert(!by_pieces(1536, 256) && !by_pieces(1548, 1536) && by_pieces(512, 6144));
    // us with 128x128 | 128x64 | 64x64 | 32x64 | 32x32 | 256x128 tiles: the choice is the fastest one or within 13 % of it (times of one shape differ by up to 9 % with the clock)
    const struct { int M, N, K; double us[F32_PIECE_TILES]; } pieces[] = {
        {64, 1536, 1536, {51.58, 31.88, 20.81, 16.66, 12.67, 97.06}},       {154, 1536, 1536, {52.56, 32.21, 21.12, 16.95, 13.25, 96.27}},
        {333, 1536, 1536, {53.37, 32.77, 21.95, 27.03, 27.82, 97.48}},      {333, 6144, 1536, {56.01, 69.22, 65.90, 68.89, 77.09, 99.92}},
        {666, 1536, 1536, {54.41, 33.98, 43.34, 30.96, 39.39, 98.32}},      {1178, 1536, 1536, {57.00, 38.83, 48.05, 56.42, 62.63, 99.59}},
        {1178, 4608, 1536, {116.33, 111.29, 138.85, 151.13, 180.12, 102.45}}, {1178, 6144, 1536, {125.23, 147.84, 182.02, 191.54, 237.36, 115.80}},
        {1178, 1536, 6144, {196.84, 137.84, 158.88, 203.57, 227.95, 371.42}}, {2356, 4608, 1536, {190.43, 222.40, 253.80, 287.45, 352.39, 210.64}},
        {2356, 1536, 6144, {232.77, 266.49, 317.84, 364.80, 446.48, 374.52}}, {8192, 3072, 768, {214.38, 251.91, 302.41, 340.54, 419.54, 188.95}},
        {10656, 768, 1536, {130.15, 153.62, 183.64, 213.74, 264.52, 120.54}}, {4250, 6144, 1536, {439.13, 487.60, 591.00, 675.71, 834.06, 439.84}},
        {1000, 1024, 512, {22.06, 15.15, 10.90, 12.35, 14.88, 38.12}},      {4096, 512, 512, {23.23, 16.88, 19.92, 22.30, 27.10, 38.46}},
        {154, 6144, 1536, {54.25, 34.53, 43.05, 32.69, 37.69, 99.21}},      {154, 1536, 6144, {191.84, 111.76, 69.51, 54.66, 41.67, 363.54}},
        {8192, 1536, 512, {79.26, 93.16, 110.55, 119.62, 148.46, 81.82}},   {3300, 256, 1024, {37.69, 24.67, 17.14, 20.70, 25.33, 67.29}},
    };
    for (const auto& c : pieces) {
        double best = c.us[0];
        for (double us : c.us) best = us < best ? us : best;
        const F32Layer l{c.M, c.N, c.K};
        assert(c.us[pick_f32_piece_tile(&l, 1, 256)] <= 1.13 * best);
    }
    return 0;
}
"""


def test_tile_shape_by_depth(tmp_path):
    src, exe = tmp_path / "tiles.cpp", tmp_path / "tiles"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-Wall", "-I", os.path.join(ROOT, "sd3.c_amd", "csrc"), str(src), "-o", str(exe)], check=True)
    subprocess.run([str(exe)], check=True)
