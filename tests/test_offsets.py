"""Which rows the tiles of the matrix products address by 32-bit offsets (csrc/offsets.hpp), on the CPU."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PROGRAM = r"""
#include <cassert>
#include <cstdint>
#include <initializer_list>
#include "offsets.hpp"
using namespace sd3;
int main() {
    for (int rows : {64, 128, 192, 256})
        for (long long row_bytes = 128; row_bytes <= 1LL << 32; row_bytes += row_bytes < 8192 ? 128 : row_bytes / 64 / 128 * 128) {
            const long long last = (rows - 1) * row_bytes + 127;  // the last byte of the first K tile
            assert(offsets_fit(rows, row_bytes) == (last <= UINT32_MAX));
        }
    // bf16: tiles of 256, 128 and 64 rows up to 2^23, 2^24 and 2^25 values a row; fp8: twice that
    for (long long k : {1LL << 22, (1LL << 22) + 64, 1LL << 23}) assert(offsets_fit(256, 2 * k));
    assert(offsets_fit(128, 2LL << 24) && offsets_fit(64, 2LL << 25) && offsets_fit(256, 1LL << 24) && offsets_fit(128, 1LL << 25));
    assert(!offsets_fit(256, 2LL << 24) && !offsets_fit(128, 2LL << 25) && !offsets_fit(64, 2LL << 26));
    return 0;
}
"""


def test_rows_that_32_bit_offsets_reach(tmp_path):
    src, exe = tmp_path / "offsets.cpp", tmp_path / "offsets"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-Wall", "-I", os.path.join(ROOT, "sd3.c_amd", "csrc"), str(src), "-o", str(exe)], check=True)
    subprocess.run([str(exe)], check=True)
