// A context's workspace: one buffer for the intermediates of a call, kept from call to call, moved only by a call that it is too small for. Host code only (no device
// code, so that it also compiles without hipcc).
#pragma once
#include <hip/hip_runtime_api.h>

#include <cstddef>
#include <cstdint>

#include "../../include/sd3_hip.h"

namespace sd3 {

int fail(int status, const char* fmt, ...);

class Workspace {
    void* p_ = nullptr;
    size_t bytes_ = 0;
    bool captured_ = false;        // a HIP graph holds this buffer's address
    size_t refused_ = SIZE_MAX;    // the last size that there was no memory for when a smaller one would do

    static hipError_t allocate(void** p, size_t bytes) {
        const hipError_t e = hipMalloc(p, bytes);
        if (e != hipSuccess) {
            *p = nullptr;
            (void)hipGetLastError();
        }
        return e;
    }
    // Waits for the work that uses the buffer, all of it on `stream` or before what is there, and frees it
    int give_back(hipStream_t stream) {
        hipError_t e = hipStreamSynchronize(stream);
        if (e == hipSuccess) e = hipFree(p_);
        if (e != hipSuccess) {
            (void)hipGetLastError();
            return fail(SD3_ERR_HIP, "workspace: %s", hipGetErrorString(e));
        }
        p_ = nullptr;
        bytes_ = 0;
        captured_ = false;
        return SD3_OK;
    }

  public:
    void* get() const { return p_; }
    size_t bytes() const { return bytes_; }
    void captured() { captured_ = p_ != nullptr; }

    // At least `bytes`
    int require(hipStream_t stream, size_t bytes) {
        if (bytes <= bytes_) return SD3_OK;
        if (p_) {
            const int rc = give_back(stream);
            if (rc != SD3_OK) return rc;
        }
        const hipError_t e = allocate(&p_, bytes);
        if (e != hipSuccess) return fail(SD3_ERR_OOM, "workspace of %zu bytes: %s", bytes, hipGetErrorString(e));
        bytes_ = bytes;
        return SD3_OK;
    }

    // At least `least`, and `better` where it can be had: *had. A buffer that does for `least` is given up for `better` only once the larger one is there, not again in this
    // context after that was refused, and never while a graph holds its address or the call is being captured into one: a call like one that was made
    // before neither allocates nor moves the buffer, whichever of the two it got.
    int prefer(hipStream_t stream, size_t least, size_t better, bool* had) {
        *had = better <= least || better <= bytes_;
        if (*had || better >= refused_) return require(stream, least);
        if (least > bytes_) {
            int rc = require(stream, better);
            *had = rc == SD3_OK;
            if (rc != SD3_ERR_OOM) return rc;
            rc = require(stream, least);
            if (rc == SD3_OK) refused_ = better;
            return rc;
        }
        hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
        if (captured_ || hipStreamIsCapturing(stream, &capture) != hipSuccess || capture != hipStreamCaptureStatusNone) {
            (void)hipGetLastError();
            return SD3_OK;
        }
        void* larger = nullptr;
        const hipError_t e = allocate(&larger, better);
        if (e != hipSuccess) {  // (other errors may be gone the next time: another thread's capture)
            if (e == hipErrorOutOfMemory) refused_ = better;
            return SD3_OK;
        }
        const int rc = give_back(stream);
        if (rc != SD3_OK) {
            (void)hipFree(larger);
            return rc;
        }
        p_ = larger;
        bytes_ = better;
        *had = true;
        return SD3_OK;
    }

    void release() {
        if (p_) (void)hipFree(p_);
        p_ = nullptr;
        bytes_ = 0;
    }
};

}  // namespace sd3
