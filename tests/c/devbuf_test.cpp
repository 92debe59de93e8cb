// Workspaces on a device with little room: what devbuf_reserve and
// devbuf_reserve_plan keep, take and refuse (csrc/devbuf.hip over the calls
// of fakehip/).
#include "goinfer_paged.h"
#include "devbuf.h"

#include <stdio.h>

using namespace gi;

static std::string last;
namespace gi {
int set_error(int code, const std::string &msg)
{
    last = msg;
    return code;
}
void clear_error() { last.clear(); }
} // namespace gi

static int failed = 0;
#define CHECK(x) \
    if (!(x)) failed++, printf("line %d: %s\n", __LINE__, #x)

static DevBuffer held(size_t bytes, size_t room) // a buffer of `bytes` and room for `room` more
{
    fake::live.clear();
    fake::capturing = fake::sync_fails = false;
    fake::mallocs = fake::syncs = 0;
    fake::room = bytes + room;
    DevBuffer b;
    if (bytes) {
        (void)hipMalloc(&b.ptr, bytes);
        b.bytes = bytes;
    }
    last.clear();
    return b;
}

static int plan(DevBuffer &b, size_t need, size_t lean, bool *use_lean, size_t ahead = 0)
{
    return devbuf_reserve_plan(b, need, lean, ahead, nullptr, "test", use_lean);
}

int main()
{
    bool lean;
    { // a quarter more where it fits, the size itself where that does not
        DevBuffer b = held(0, 1000);
        CHECK(devbuf_reserve(b, 400, nullptr, "test") == GI_OK && b.bytes == 500);
        DevBuffer c = held(0, 410);
        CHECK(devbuf_reserve(c, 400, nullptr, "test") == GI_OK && c.bytes == 400 && last.empty());
    }
    { // a growth that fails leaves the buffer as it was
        DevBuffer b = held(100, 150);
        void *p = b.ptr;
        CHECK(devbuf_reserve(b, 200, nullptr, "test") == GI_ERR_OOM && !last.empty());
        CHECK(b.ptr == p && b.bytes == 100 && fake::live.count(p) && b.retired.empty());
        fake::room = 1000;
        fake::sync_fails = true;
        CHECK(devbuf_reserve(b, 200, nullptr, "test") == GI_ERR_HIP);
        CHECK(b.ptr == p && b.bytes == 100 && fake::live.size() == 1);
    }
    { // the fallback is the larger one and has no room: the plan itself is held, or fits, or does not
        DevBuffer b = held(100, 50);
        void *p = b.ptr;
        CHECK(plan(b, 100, 300, &lean) == GI_OK && !lean && b.ptr == p && last.empty());
        DevBuffer c = held(0, 130);
        CHECK(plan(c, 120, 300, &lean) == GI_OK && !lean && c.bytes == 120 && last.empty());
        DevBuffer d = held(0, 0);
        CHECK(plan(d, 0, 300, &lean) == GI_OK && !lean && last.empty());
        DevBuffer e = held(50, 80);
        CHECK(plan(e, 120, 300, &lean) == GI_ERR_OOM && e.bytes == 50);
    }
    { // the fallback is the smaller one
        DevBuffer b = held(0, 130);
        CHECK(plan(b, 300, 100, &lean) == GI_OK && lean && b.bytes == 125 && last.empty());
        DevBuffer c = held(0, 0);
        CHECK(plan(c, 300, 0, &lean) == GI_OK && lean && last.empty());
        DevBuffer d = held(0, 90);
        CHECK(plan(d, 300, 100, &lean) == GI_ERR_OOM);
        DevBuffer e = held(0, 1000);
        CHECK(plan(e, 300, 100, &lean) == GI_OK && !lean && e.bytes == 375);
        CHECK(plan(e, 200, 375, &lean) == GI_OK && !lean && fake::mallocs == 1);
        CHECK(plan(e, 0, 0, &lean) == GI_OK && !lean);
    }
    { // what later calls can need is allocated with the first growth, where it fits
        DevBuffer b = held(0, 1000);
        CHECK(plan(b, 0, 0, &lean, 800) == GI_OK && fake::mallocs == 0);
        for (size_t need = 50; need <= 800; need += 50)
            CHECK(plan(b, need, 40, &lean, 800) == GI_OK && !lean && b.bytes == 800 && fake::mallocs == 1);
        DevBuffer c = held(0, 500);
        CHECK(plan(c, 300, 100, &lean, 800) == GI_OK && !lean && c.bytes == 300);
        CHECK(plan(c, 900, 100, &lean, 800) == GI_OK && lean && c.bytes == 300);
    }
    { // a capturing stream never allocates, synchronises or frees
        DevBuffer b = held(200, 1000);
        void *p = b.ptr;
        fake::capturing = true;
        fake::mallocs = 0;
        CHECK(plan(b, 0, 900, &lean) == GI_OK && !lean && !b.captured);
        CHECK(plan(b, 150, 900, &lean) == GI_OK && !lean && b.captured);
        CHECK(plan(b, 300, 200, &lean) == GI_OK && lean);
        CHECK(plan(b, 300, 0, &lean) == GI_OK && lean);
        CHECK(plan(b, 300, 201, &lean) == GI_ERR_BAD_ARG && last.find("capturing") != std::string::npos);
        CHECK(devbuf_reserve(b, 201, nullptr, "test") == GI_ERR_BAD_ARG);
        CHECK(fake::mallocs == 0 && fake::syncs == 0 && b.ptr == p);
        // what a graph may hold stays until release
        fake::capturing = false;
        CHECK(plan(b, 300, 0, &lean) == GI_OK && !lean && b.ptr != p);
        CHECK(fake::live.count(p) && b.retired.size() == 1 && fake::syncs == 0);
        devbuf_release(b);
        CHECK(fake::live.empty() && fake::bad_frees == 0 && b.ptr == nullptr && b.bytes == 0);
    }
    if (!failed)
        printf("ok\n");
    return failed != 0;
}
