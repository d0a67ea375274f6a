// Error handling and device buffers shared by the host files of the C ABI
// (no exceptions cross the ABI: every entry point runs under guarded()).
#pragma once
#include <hip/hip_runtime.h>
#include <algorithm>
#include <stdexcept>
#include <string>

#include "../../include/atm_mi355x.h"

namespace atm {

// The message atm_last_error() returns (one per calling thread).
std::string& last_error();

struct AtmError : std::runtime_error {
    int code;
    AtmError(int c, const std::string& m) : std::runtime_error(m), code(c) {}
};

#define HIPCHK(expr)                                                                                   \
    do {                                                                                               \
        hipError_t e_ = (expr);                                                                        \
        if (e_ != hipSuccess)                                                                          \
            throw ::atm::AtmError(ATM_ERR_DEVICE, std::string(#expr) + ": " + hipGetErrorString(e_));  \
    } while (0)

[[noreturn]] inline void fail(int code, const std::string& msg) { throw AtmError(code, msg); }

template <typename F>
int guarded(F&& f) {
    try {
        f();
        return ATM_OK;
    } catch (const AtmError& e) {
        last_error() = e.what();
        return e.code;
    } catch (const std::exception& e) {
        last_error() = e.what();
        return ATM_ERR_INVALID_ARGUMENT;
    }
}

// Device allocation owned by a host object.
struct DevBuf {
    void* p = nullptr;
    size_t bytes = 0;
    void alloc(size_t n) {
        release();
        bytes = std::max<size_t>(n, 256);
        HIPCHK(hipMalloc(&p, bytes));
    }
    void release() {
        if (p) (void)hipFree(p);
        p = nullptr;
        bytes = 0;
    }
    DevBuf() = default;
    DevBuf(const DevBuf&) = delete;
    DevBuf& operator=(const DevBuf&) = delete;
    ~DevBuf() { release(); }
    template <typename T> T* as() const { return static_cast<T*>(p); }
};

// Page-locked host memory that kernels read and write in place (coherent: a kernel's
// stores are seen by the host once its stream has been waited for).  A copy to or from
// ordinary host memory is staged by the runtime and waited for, 20 to 85 us each; a
// kernel's own stores to this memory cost only their bytes over the link.
struct HostBuf {
    void* p = nullptr;
    size_t bytes = 0;
    void alloc(size_t n) {
        release();
        n = std::max<size_t>(n, 256);
        HIPCHK(hipHostMalloc(&p, n, hipHostMallocPortable | hipHostMallocMapped | hipHostMallocCoherent));
        bytes = n;
    }
    void release() {
        if (p) (void)hipHostFree(p);
        p = nullptr;
        bytes = 0;
    }
    HostBuf() = default;
    HostBuf(const HostBuf&) = delete;
    HostBuf& operator=(const HostBuf&) = delete;
    ~HostBuf() { release(); }
    template <typename T> T* as() const { return static_cast<T*>(p); }
};

// Host data on its way to a kernel that reads it in place, without a wait after the
// launch: begin() waits for the kernel that still reads the previous contents (and
// refuses a stream under capture, whose replays would read whatever is here by then),
// end() marks the launch of the reader.
struct Upload {
    void* p = nullptr;  // page-locked memory, the owner's
    hipEvent_t done = nullptr;
    bool used = false;
    void create(void* memory) {
        p = memory;
        HIPCHK(hipEventCreateWithFlags(&done, hipEventDisableTiming));
    }
    void* begin(hipStream_t st) {
        hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
        HIPCHK(hipStreamIsCapturing(st, &cap));
        if (cap != hipStreamCaptureStatusNone) fail(ATM_ERR_DEVICE, "host data cannot be set on a stream under capture");
        if (used) HIPCHK(hipEventSynchronize(done));
        used = false;
        return p;
    }
    void end(hipStream_t st) {
        used = true;
        HIPCHK(hipEventRecord(done, st));
    }
    Upload() = default;
    Upload(const Upload&) = delete;
    Upload& operator=(const Upload&) = delete;
    ~Upload() {
        if (done) (void)hipEventDestroy(done);
    }
};

}  // namespace atm
