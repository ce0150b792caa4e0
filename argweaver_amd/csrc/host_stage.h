// host_stage.h -- pinned host memory that uploads and tables pass through.
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>

#include "hip_check.h"

namespace aw {

// Makes a device current while it lives: streams, events and memory of one
// device are used together, whichever the caller has current.
class OnDevice {
public:
    explicit OnDevice(int dev)
    {
        if (hipGetDevice(&was_) != hipSuccess || was_ == dev || hipSetDevice(dev) != hipSuccess) was_ = -1;
    }
    ~OnDevice()
    {
        if (was_ >= 0) (void)hipSetDevice(was_);
    }
    OnDevice(const OnDevice &) = delete;
    OnDevice &operator=(const OnDevice &) = delete;

private:
    int was_ = -1;
};

// The pool's device memory that no call uses, in bytes, and its release
// (engine.hip): true if there was any.  A device allocation that finds no memory
// releases it and tries again.
size_t idle_stage_bytes();
bool free_idle_stage_memory();

// hipMalloc, with the pool's idle memory given up where memory is short
inline hipError_t device_malloc(void **p, size_t n)
{
    hipError_t e = hipMalloc(p, n);
    if (e == hipSuccess || !free_idle_stage_memory()) return e;
    (void)hipGetLastError();   // of the first try
    return hipMalloc(p, n);
}

// Two halves of pinned memory with an event each, of one device, and device
// memory for a call's arrays, kept up to DEV_KEEP bytes: allocating 36 MB, the
// copies into pages not mapped yet and freeing it cost a call 2 ms.
struct HostStage {
    static constexpr size_t HALF = size_t(2) << 20;   // bytes; a table row has at most 16 KB
    static constexpr size_t DEV_KEEP = size_t(64) << 20;
    char *p = nullptr;
    int dev = 0;
    hipEvent_t filled[2];
    char *dbuf = nullptr;
    size_t dcap = 0;
    // device memory of n bytes, null when there is none
    char *device(size_t n)
    {
        if (n > dcap) {
            drop();
            if (device_malloc((void **)&dbuf, n) != hipSuccess) dbuf = nullptr;
            else dcap = n;
        }
        return dbuf;
    }
    // gives the device memory back; true if there was any
    bool drop()
    {
        const bool any = dbuf != nullptr;
        if (any) (void)hipFree(dbuf);
        dbuf = nullptr;
        dcap = 0;
        return any;
    }
    void trim()
    {
        if (dcap > DEV_KEEP) drop();
    }
    double *half(int k) const { return reinterpret_cast<double *>(p + k * HALF); }
};

// A stage for the current device, and back (engine.hip).  Up to STAGE_KEEP stages
// are kept for later calls of any thread, more are freed when given back; their
// user has waited for the work on them.  Null when there is no memory.
constexpr size_t STAGE_KEEP = 8;
HostStage *take_stage();
void give_stage(HostStage *s);

// A stage while in use; `own` is one that the caller keeps, or null.
struct StageUse {
    HostStage *const own, *const s;
    explicit StageUse(HostStage *own_ = nullptr) : own(own_), s(own_ ? own_ : take_stage()) {}
    ~StageUse()
    {
        if (!own && s) give_stage(s);
    }
    StageUse(const StageUse &) = delete;
    StageUse &operator=(const StageUse &) = delete;
};

// Host arrays on their way to the device.  A copy from pageable memory costs the
// caller 5-50 us, however small (the rows of 100 sequences, 100 KB each: 45 us each);
// put() gathers arrays in pinned memory, and what lies close together on the device
// goes in one copy of up to 2 MB, beside which the next half is filled.  The
// arrays may be released after put().
class Uploader {
public:
    static constexpr size_t ALIGN = 256;   // of the arrays put (Plan, DevBufs)
    Uploader(HostStage &s, hipStream_t st) : s_(s), st_(st) {}
    ~Uploader()
    {
        for (int k = 0; k < 2; k++)
            if (busy_[k]) (void)hipEventSynchronize(s_.filled[k]);
    }
    int put(void *dst, const void *src, size_t n)
    {
        char *d = static_cast<char *>(dst);
        const char *x = static_cast<const char *>(src);
        while (n > 0) {
            // gaps less than the 256 bytes that arrays are aligned to hold nothing, and go along
            if (base_ && (d < base_ + used_ || d >= base_ + used_ + ALIGN || d >= base_ + HostStage::HALF))
                if (flush()) return 1;
            if (!base_) {
                if (busy_[half_]) HIP_OK(hipEventSynchronize(s_.filled[half_]));
                busy_[half_] = false;
                base_ = d;
            }
            const size_t off = d - base_, m = std::min(n, HostStage::HALF - off);
            memcpy(s_.p + half_ * HostStage::HALF + off, x, m);
            used_ = off + m;
            d += m;
            x += m;
            n -= m;
        }
        return 0;
    }
    // sends what is gathered
    int flush()
    {
        if (!base_) return 0;
        HIP_OK(hipMemcpyAsync(base_, s_.p + half_ * HostStage::HALF, used_, hipMemcpyHostToDevice, st_));
        HIP_OK(hipEventRecord(s_.filled[half_], st_));
        busy_[half_] = true;
        half_ ^= 1;
        base_ = nullptr;
        used_ = 0;
        return 0;
    }

private:
    HostStage &s_;
    hipStream_t st_;
    char *base_ = nullptr;   // device address of the half's first byte
    size_t used_ = 0;
    int half_ = 0;
    bool busy_[2] = {false, false};
};

}  // namespace aw
