// A HIP runtime of two devices in host memory, for checks of the library's host
// code: a check that defines it and links the library has it called in the
// runtime's place.  Kernels are counted and do nothing (device memory starts as
// zeros); copies happen at once.  As in HIP, an event belongs to the device that was
// current when it was made, and is not recorded on another device's stream.
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <string>
#include <vector>

using std::max;   // as hipcc's headers have them
using std::min;

namespace fake {

struct Stream {
    int dev;
    long issued = 0, done = 0;   // kernels
};
struct Event {
    int dev;
    Stream *s = nullptr;
    long at = 0;
};

inline int device = 0;
inline int live_events = 0;
inline int kernels = 0, copies = 0;
inline int good_events = -1, good_launches = -1;   // calls that still succeed, -1: all
inline size_t device_bytes = 0, device_limit = size_t(1) << 40;
inline std::map<void *, size_t> allocated;
inline std::vector<Stream *> streams;
inline hipError_t last = hipSuccess;
inline Stream null_stream{0};

inline Stream *stream(hipStream_t s) { return s ? reinterpret_cast<Stream *>(s) : &null_stream; }
inline hipError_t fail(hipError_t e)
{
    last = e;
    return e;
}
inline long pending()
{
    long n = 0;
    for (Stream *s : streams) n += s->issued - s->done;
    return n;
}
inline bool use(int &left)
{
    if (left == 0) return false;
    if (left > 0) left--;
    return true;
}

}  // namespace fake

extern "C" {

hipError_t hipGetDeviceCount(int *n) { return *n = 2, hipSuccess; }
hipError_t hipGetDevice(int *d) { return *d = fake::device, hipSuccess; }
hipError_t hipSetDevice(int d) { return fake::device = d, hipSuccess; }
hipError_t hipGetDeviceProperties(hipDeviceProp_t *p, int)
{
    memset(p, 0, sizeof *p);
    p->multiProcessorCount = 256;
    return hipSuccess;
}
hipError_t hipGetLastError(void)
{
    const hipError_t e = fake::last;
    fake::last = hipSuccess;
    return e;
}
const char *hipGetErrorString(hipError_t e) { return e == hipSuccess ? "no error" : "an error of the check's runtime"; }

hipError_t hipMalloc(void **p, size_t n)
{
    if (fake::device_bytes + n > fake::device_limit) return *p = nullptr, fake::fail(hipErrorOutOfMemory);
    *p = calloc(n ? n : 1, 1);
    fake::device_bytes += fake::allocated[*p] = n;
    return hipSuccess;
}
hipError_t hipFree(void *p)
{
    if (p) fake::device_bytes -= fake::allocated.at(p);
    fake::allocated.erase(p);
    free(p);
    return hipSuccess;
}
hipError_t hipHostMalloc(void **p, size_t n, unsigned) { return *p = calloc(n, 1), hipSuccess; }
hipError_t hipHostFree(void *p) { return free(p), hipSuccess; }
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind) { return memcpy(d, s, n), hipSuccess; }
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t)
{
    fake::copies++;
    return memcpy(d, s, n), hipSuccess;
}

hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned)
{
    fake::streams.push_back(new fake::Stream{fake::device});
    return *s = reinterpret_cast<hipStream_t>(fake::streams.back()), hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t s)
{
    return fake::stream(s)->done = fake::stream(s)->issued, hipSuccess;
}

hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned)
{
    if (!fake::use(fake::good_events)) return fake::fail(hipErrorOutOfMemory);
    fake::live_events++;
    return *e = reinterpret_cast<hipEvent_t>(new fake::Event{fake::device}), hipSuccess;
}
hipError_t hipEventCreate(hipEvent_t *e) { return hipEventCreateWithFlags(e, 0); }
hipError_t hipEventDestroy(hipEvent_t e)
{
    fake::live_events--;
    delete reinterpret_cast<fake::Event *>(e);
    return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s)
{
    fake::Event *v = reinterpret_cast<fake::Event *>(e);
    fake::Stream *st = fake::stream(s);
    if (s && v->dev != st->dev) return fake::fail(hipErrorInvalidHandle);
    v->s = st;
    v->at = st->issued;
    return hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t e)
{
    fake::Event *v = reinterpret_cast<fake::Event *>(e);
    if (v->s && v->s->done < v->at) v->s->done = v->at;
    return hipSuccess;
}
hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t) { return *ms = 0, hipSuccess; }

hipError_t hipFuncSetAttribute(const void *, hipFuncAttribute, int) { return hipSuccess; }
hipError_t hipGetSymbolAddress(void **p, const void *) { return *p = calloc(size_t(64) << 20, 1), hipSuccess; }
hipError_t hipLaunchKernel(const void *, dim3, dim3, void **, size_t, hipStream_t s)
{
    if (!fake::use(fake::good_launches)) return fake::fail(hipErrorLaunchFailure);
    fake::kernels++;
    fake::stream(s)->issued++;
    return hipSuccess;
}
hipError_t __hipPushCallConfiguration(dim3, dim3, size_t, hipStream_t s);
hipError_t __hipPopCallConfiguration(dim3 *g, dim3 *b, size_t *sh, hipStream_t *s);

}  // extern "C"

namespace fake {
inline hipStream_t launch_stream = nullptr;
}
hipError_t __hipPushCallConfiguration(dim3, dim3, size_t, hipStream_t s)
{
    return fake::launch_stream = s, hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3 *g, dim3 *b, size_t *sh, hipStream_t *s)
{
    *g = *b = dim3(1);
    *sh = 0;
    return *s = fake::launch_stream, hipSuccess;
}

#define REQUIRE(x)                                              \
    do {                                                        \
        if (!(x)) {                                             \
            printf("%s:%d: %s\n", __FILE__, __LINE__, #x);      \
            exit(1);                                            \
        }                                                       \
    } while (0)
