"""What the host side keeps per device (csrc/device.hpp), on the CPU: the HIP calls are stand-ins that count and answer by device."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PROGRAM = r"""
#include "device.hpp"
#include <cassert>
#include <thread>
static thread_local int device = 0;
static std::atomic<int> queries{0}, settings{0}, failing{0};
extern "C" {
hipError_t hipGetDevice(int* d) { *d = device; return hipSuccess; }
hipError_t hipDeviceGetAttribute(int* n, hipDeviceAttribute_t, int d) { queries++; *n = 100 + d; return hipSuccess; }
hipError_t hipFuncSetAttribute(const void*, hipFuncAttribute, int) { settings++; return failing ? hipErrorInvalidValue : hipSuccess; }
const char* hipGetErrorString(hipError_t) { return ""; }
}
int sd3::fail(int status, const char*, ...) { return status; }
int main() {
    for (int round = 0; round < 2; round++)
        for (int d : {0, 1, 7, 63, 64, 200}) { device = d; assert(sd3::compute_units() == 100 + d); }
    assert(queries == 4 + 2 * 2);  // asked once for each of the devices whose answers are kept
    std::thread other([] { device = 5; assert(sd3::compute_units() == 105); });
    other.join();
    sd3::DynamicLds lds, second;
    for (int round = 0; round < 2; round++)
        for (int d : {0, 1, 63}) { device = d; assert(lds.allow(nullptr, 65536) == SD3_OK && lds.allow(nullptr, 65537) == SD3_OK); }
    assert(settings == 3);  // once per device, and not at all where no more than 64 KiB are needed
    device = 2;
    failing = 1;
    assert(lds.allow(nullptr, 100000) == SD3_ERR_HIP && second.allow(nullptr, 100000) == SD3_ERR_HIP);
    failing = 0;
    assert(lds.allow(nullptr, 100000) == SD3_OK && settings == 6);  // a failed setting is tried again
    return 0;
}
"""


def test_answers_are_kept_by_device(tmp_path):
    src, exe = tmp_path / "device_state.cpp", tmp_path / "device_state"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-Wall", "-pthread", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", "-I", os.path.join(ROOT, "sd3.c_amd", "csrc"), str(src),
                    "-o", str(exe)], check=True)
    subprocess.run([str(exe)], check=True)
