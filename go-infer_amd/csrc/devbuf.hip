// Growable device buffers (devbuf.h): host code only.
#include "../../include/goinfer_paged.h"
#include "devbuf.h"

#include <algorithm>

namespace gi {

int devbuf_reserve(DevBuffer &b, size_t need, hipStream_t st, const char *what, size_t ahead)
{
    hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
    hipError_t e = hipStreamIsCapturing(st, &cs);
    if (e != hipSuccess)
        return set_error(GI_ERR_HIP, std::string(what) + ": hipStreamIsCapturing: " + hipGetErrorString(e));
    const bool capturing = cs != hipStreamCaptureStatusNone;
    if (capturing)
        b.captured = true;
    if (need <= b.bytes)
        return GI_OK;
    if (capturing)
        return set_error(GI_ERR_BAD_ARG,
                         std::string(what) + ": needs " + std::to_string(need) + " bytes of workspace (holds " +
                             std::to_string(b.bytes) +
                             ") while the stream is capturing a graph; make one eager call of this shape "
                             "before capturing");
    size_t got = 0;
    void *p = nullptr;
    for (size_t want : {ahead ? std::max(ahead, need) : need + need / 4, need}) {
        if (hipMalloc(&p, want) == hipSuccess) {
            got = want;
            break;
        }
        p = nullptr;
        (void)hipGetLastError(); // the error is this call's to report
    }
    if (!p)
        return set_error(GI_ERR_OOM, std::string(what) + ": hipMalloc(" + std::to_string(need) + ") failed");
    if (b.ptr) {
        if (b.captured) {
            // a captured graph may still address it: keep it until release
            b.retired.push_back(b.ptr);
        } else {
            // work already queued may still read it
            e = hipStreamSynchronize(st);
            if (e != hipSuccess) {
                (void)hipFree(p);
                return set_error(GI_ERR_HIP, std::string(what) + ": " + hipGetErrorString(e));
            }
            (void)hipFree(b.ptr);
        }
    }
    b.ptr = p;
    b.bytes = got;
    return GI_OK;
}

int devbuf_reserve_plan(DevBuffer &b, size_t need, size_t lean, size_t ahead, hipStream_t st, const char *what,
                        bool *use_lean)
{
    *use_lean = false;
    if (need == 0 && lean == 0)
        return GI_OK; // nothing is used, nothing to note
    hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
    hipError_t e = hipStreamIsCapturing(st, &cs);
    if (e != hipSuccess)
        return set_error(GI_ERR_HIP, std::string(what) + ": hipStreamIsCapturing: " + hipGetErrorString(e));
    if (cs != hipStreamCaptureStatusNone) {
        *use_lean = need > b.bytes;
        const size_t used = *use_lean ? lean : need;
        return used ? devbuf_reserve(b, used, st, what) : GI_OK;
    }
    if (std::max(need, lean) <= b.bytes)
        return GI_OK;
    // room for either plan, or for the better one, or for the lean one
    int rc = devbuf_reserve(b, std::max(need, lean), st, what, ahead);
    if (rc != GI_ERR_OOM)
        return rc;
    if (need < lean) {
        rc = devbuf_reserve(b, need, st, what);
    } else if (lean < need) {
        *use_lean = true;
        rc = devbuf_reserve(b, lean, st, what);
    }
    if (rc == GI_OK)
        clear_error();
    return rc;
}

void devbuf_release(DevBuffer &b)
{
    if (b.ptr)
        (void)hipFree(b.ptr);
    for (void *p : b.retired)
        (void)hipFree(p);
    b.retired.clear();
    b.ptr = nullptr;
    b.bytes = 0;
}

} // namespace gi
