/* The HIP calls of csrc/devbuf.hip over a device of `fake::room` bytes, for
 * tests/c/devbuf_test.cpp. */
#pragma once
#include <stddef.h>

#include <map>

typedef struct fake_stream *hipStream_t;
typedef enum { hipSuccess = 0, hipErrorOutOfMemory = 2, hipErrorUnknown = 999 } hipError_t;
typedef enum { hipStreamCaptureStatusNone = 0, hipStreamCaptureStatusActive = 1 } hipStreamCaptureStatus;

namespace fake {
inline size_t room = 0;
inline std::map<void *, size_t> live;
inline bool capturing = false, sync_fails = false;
inline int mallocs = 0, syncs = 0, bad_frees = 0;
inline char heap[64];
} // namespace fake

inline hipError_t hipMalloc(void **p, size_t n)
{
    fake::mallocs++;
    if (n > fake::room)
        return hipErrorOutOfMemory;
    for (char &c : fake::heap)
        if (!fake::live.count(&c)) {
            *p = &c;
            fake::live[&c] = n;
            fake::room -= n;
            return hipSuccess;
        }
    return hipErrorOutOfMemory;
}
inline hipError_t hipFree(void *p)
{
    if (!fake::live.count(p)) {
        fake::bad_frees++;
        return hipErrorUnknown;
    }
    fake::room += fake::live[p];
    fake::live.erase(p);
    return hipSuccess;
}
inline hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus *s)
{
    *s = fake::capturing ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone;
    return hipSuccess;
}
inline hipError_t hipStreamSynchronize(hipStream_t)
{
    fake::syncs++;
    return fake::sync_fails ? hipErrorUnknown : hipSuccess;
}
inline hipError_t hipGetLastError() { return hipSuccess; }
inline const char *hipGetErrorString(hipError_t) { return "fake"; }
