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


LDS_SIZES = r"""
#include "device.hpp"
#include <cassert>
#include <algorithm>
#include <thread>
#include <vector>
static thread_local int device = 0;
static int set_to[256], settings = 0, failing = 0;
extern "C" {
hipError_t hipGetDevice(int* d) { *d = device; return hipSuccess; }
hipError_t hipDeviceGetAttribute(int* n, hipDeviceAttribute_t, int) { *n = 1; return hipSuccess; }
hipError_t hipFuncSetAttribute(const void*, hipFuncAttribute, int bytes) { settings++; if (failing) return hipErrorInvalidValue; set_to[device] = bytes; return hipSuccess; }
const char* hipGetErrorString(hipError_t) { return ""; }
}
int sd3::fail(int status, const char*, ...) { return status; }
int main() {
    sd3::DynamicLds lds;
    for (int d : {0, 1, 63, 64, 200}) {  // (the last two are beyond the devices whose answers are kept)
        device = d;
        for (int bytes : {90112, 114688, 70000, 114688, 98304, 160 * 1024, 90112}) {
            assert(lds.allow(nullptr, bytes) == SD3_OK && set_to[d] >= bytes);  // what is set now covers this launch ...
            assert(set_to[d] >= 114688 || bytes == 90112);                      // ... and those that were allowed before
        }
    }
    const int before = settings;
    for (int d : {0, 1, 63}) { device = d; assert(lds.allow(nullptr, 100000) == SD3_OK); }
    assert(settings == before);
    sd3::DynamicLds other;  // a size that was refused is not taken for allowed, and does not become the one that smaller requests set
    device = 2;
    assert(other.allow(nullptr, 80000) == SD3_OK);
    failing = 1;
    assert(other.allow(nullptr, 200000) == SD3_ERR_HIP && other.allow(nullptr, 80000) == SD3_OK);
    failing = 0;
    device = 3;
    assert(other.allow(nullptr, 80000) == SD3_OK && set_to[3] == 80000);
    sd3::DynamicLds shared;
    std::vector<std::thread> threads;
    for (int i = 0; i < 8; i++)
        threads.emplace_back([&, i] { device = 5; for (int n = 0; n < 2000; n++) assert(shared.allow(nullptr, 65537 + (n * 37 + i * 911) % 90000) == SD3_OK); });
    for (auto& t : threads) t.join();
    int most = 0;
    for (int i = 0; i < 8; i++) for (int n = 0; n < 2000; n++) most = std::max(most, 65537 + (n * 37 + i * 911) % 90000);
    assert(set_to[5] == most);
    return 0;
}
"""


def test_a_kernel_keeps_the_largest_lds_size_it_was_allowed(tmp_path):
    src, exe = tmp_path / "lds_sizes.cpp", tmp_path / "lds_sizes"
    src.write_text(LDS_SIZES)
    subprocess.run(["g++", "-std=c++17", "-Wall", "-pthread", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", "-I", os.path.join(ROOT, "sd3.c_amd", "csrc"), str(src),
                    "-o", str(exe)], check=True)
    subprocess.run([str(exe)], check=True)
