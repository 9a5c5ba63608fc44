"""A context's workspace (csrc/workspace.hpp), on the CPU: the HIP calls are stand-ins that count, refuse sizes and capture as they are told to."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PROGRAM = r"""
#include "workspace.hpp"
#include <cassert>
#include <cstdlib>
#include <set>
static size_t limit = SIZE_MAX;  // the largest size that can be had
static hipError_t refusal = hipErrorOutOfMemory;
static int allocations = 0, frees = 0, waits = 0, capturing = 0;
static std::set<void*> live;
extern "C" {
hipError_t hipMalloc(void** p, size_t n) {
    allocations++;
    if (n > limit) return refusal;
    *p = std::malloc(1);
    live.insert(*p);
    return hipSuccess;
}
hipError_t hipFree(void* p) { frees++; assert(live.erase(p) == 1 && waits > 0); std::free(p); return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { assert(!capturing); waits++; return hipSuccess; }
hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus* s) { *s = capturing ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone; return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
const char* hipGetErrorString(hipError_t) { return ""; }
}
int sd3::fail(int status, const char*, ...) { return status; }
static sd3::Workspace* ws;
static bool prefers(size_t least, size_t better) {  // whether the better size was had; the buffer is always good for what was said
    bool had = false;
    assert(ws->prefer(nullptr, least, better, &had) == SD3_OK);
    assert(ws->get() && live.count(ws->get()) && ws->bytes() >= (had ? better : least) && live.size() == 1);
    return had;
}
static void unmoved(int calls, size_t least, size_t better, bool had) {  // calls like the one before: nothing is asked of the device
    void* const p = ws->get();
    const int before = allocations + frees + waits;
    for (int i = 0; i < calls; i++) assert(prefers(least, better) == had && ws->get() == p);
    assert(allocations + frees + waits == before);
}
static void fresh() {
    if (ws) { waits++; ws->release(); delete ws; }
    assert(live.empty());
    ws = new sd3::Workspace;
    limit = SIZE_MAX;
    refusal = hipErrorOutOfMemory;
    capturing = allocations = frees = waits = 0;
}
int main() {
    fresh();  // the better size, a larger one, the same again
    assert(prefers(100, 150) && allocations == 1);
    unmoved(3, 100, 150, true);
    assert(prefers(140, 210) && allocations == 2 && frees == 1 && waits == 1);
    unmoved(3, 100, 150, true);
    assert(prefers(300, 300) && ws->bytes() == 300);

    fresh();  // no memory for it: asked for once
    limit = 120;
    assert(!prefers(100, 150) && allocations == 2);
    unmoved(3, 100, 150, false);
    assert(!prefers(110, 165) && ws->bytes() == 110);  // more than what was refused is not asked for, what is needed is
    limit = SIZE_MAX;
    unmoved(3, 110, 165, false);
    assert(prefers(112, 149));
    assert(ws->require(nullptr, 400) == SD3_OK && prefers(100, 150));

    fresh();  // no memory for it beside a buffer that will do: that one stays
    assert(ws->require(nullptr, 100) == SD3_OK);
    limit = 120;
    void* const kept = ws->get();
    assert(!prefers(90, 150) && ws->get() == kept && allocations == 2 && frees == 0 && waits == 0);
    unmoved(3, 90, 150, false);

    fresh();  // what is not for lack of memory is asked for again
    assert(ws->require(nullptr, 100) == SD3_OK);
    limit = 120;
    refusal = hipErrorInvalidValue;
    assert(!prefers(90, 150));
    limit = SIZE_MAX;
    assert(prefers(90, 150));

    fresh();  // not even what is needed
    limit = 50;
    bool had = true;
    assert(ws->prefer(nullptr, 100, 150, &had) == SD3_ERR_OOM && !had && !ws->get() && ws->bytes() == 0);
    limit = SIZE_MAX;
    assert(prefers(100, 150));

    fresh();  // a capture that goes without, and eager calls of the same sizes behind it: the graph's buffer stays
    assert(ws->require(nullptr, 100) == SD3_OK);
    capturing = 1;
    unmoved(1, 90, 150, false);
    ws->captured();
    capturing = 0;
    unmoved(3, 90, 150, false);
    assert(prefers(200, 300) && prefers(300, 450));  // a call that it is too small for moves it, and the graph is no longer asked about

    fresh();  // a graph of another call holds it
    assert(ws->require(nullptr, 100) == SD3_OK);
    ws->captured();
    unmoved(3, 90, 150, false);

    fresh();  // a captured call of the better size
    assert(prefers(100, 150));
    capturing = 1;
    unmoved(1, 100, 150, true);
    ws->captured();
    capturing = 0;
    unmoved(3, 100, 150, true);
    fresh();
    delete ws;
    return 0;
}
"""


def test_a_call_like_one_before_leaves_the_workspace_in_place(tmp_path):
    src, exe = tmp_path / "workspace.cpp", tmp_path / "workspace"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-Wall", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", "-I", os.path.join(ROOT, "sd3.c_amd", "csrc"), str(src),
                    "-o", str(exe)], check=True)
    subprocess.run([str(exe)], check=True)
