"""How many modulation panels a launch takes along (csrc/passengers.hpp), on the CPU."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PROGRAM = r"""
#include <initializer_list>
#include "passengers.hpp"
#include <cassert>
using namespace sd3;
int main() {
    // what a panel of K x 64 took a workgroup, alone on a device: in proportion, with 6.5 us at 1536, within an eighth
    const double measured[][2] = {{512, 2.43}, {768, 4.04}, {1024, 4.00}, {1536, 5.71}, {2048, 7.35}, {2432, 9.00}, {3072, 10.34}, {4096, 12.92}};
    for (auto& m : measured) {
        const double want = m[1] * 6.5 / 5.71, got = passenger_panel_us((int)m[0]);
        assert(got > want * 0.875 && got < want * 1.125);
    }
    for (int K = 64; K <= 4096; K += 64)
        for (double us : {0.0, 3.0, 6.0, 12.7, 20.0, 45.0, 150.0})
            for (int want : {0, 1, 7, 60, 360})
                for (int idle : {0, 1, 16, 100, 255})
                    for (bool last : {false, true}) {
                        const int n = passenger_panels(us, K, want, idle, last);
                        assert(n >= 0 && (want && idle ? true : n == 0));
                        if (!n) continue;
                        assert((n - 1) * idle < want);  // no more than there are
                        assert(PASSENGER_START + n * passenger_panel_us(K) <= us + (last ? PASSENGER_OVERTIME : 0) + 1e-9);  // they end with the launch
                        if (!last && n * idle < want) assert(PASSENGER_START + (n + 1) * passenger_panel_us(K) > us);        // and fill it
                    }
    // width 1536 in the launches of a 512px forward: 16 idle units, a launch of 41 us and the block's last
    assert(passenger_panels(41.0, 1536, 360, 16, false) == 5 && passenger_panels(41.0, 1536, 160, 16, true) == 10 && passenger_panels(41.0, 1536, 176, 16, true) == 5);
    // what was taken is worth a launch for the rest from 6 us of streaming at 5.4 TB/s on
    assert(!passengers_pay(0, 1536) && !passengers_pay(164, 1536) && passengers_pay(165, 1536) && !passengers_pay(180, 768) && passengers_pay(83, 3072));
    return 0;
}
"""


def test_panels_taken_along_fit_the_launch(tmp_path):
    src, exe = tmp_path / "passengers.cpp", tmp_path / "passengers"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-Wall", "-I", os.path.join(ROOT, "sd3.c_amd", "csrc"), str(src), "-o", str(exe)], check=True)
    subprocess.run([str(exe)], check=True)
