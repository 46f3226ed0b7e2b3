// Host test of fgt::DBuf over a runtime whose allocations can be made to
// fail: a failed allocation leaves an empty buffer, so a holder that compares
// its size with what it needs allocates again, and no stale error.
#include "device_buffer.h"

#include <cstdio>
#include <cstdlib>
#include <cstring>

static bool fail_next = false;
static hipError_t last_error = hipSuccess;
static int live = 0;

extern "C" {
hipError_t hipMalloc(void** p, size_t n) {
    if (fail_next) {
        fail_next = false;
        return last_error = hipErrorOutOfMemory;   // *p is left alone
    }
    *p = std::malloc(n);
    ++live;
    return hipSuccess;
}
hipError_t hipFree(void* p) {
    std::free(p);
    --live;
    return hipSuccess;
}
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) {
    std::memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipGetLastError() {
    const hipError_t e = last_error;
    last_error = hipSuccess;
    return e;
}
const char* hipGetErrorString(hipError_t) { return "error"; }
}

#define CHECK(c)                                               \
    if (!(c)) {                                                \
        std::printf("line %d: %s\n", __LINE__, #c);            \
        return 1;                                              \
    }

template <class F>
static bool throws(F&& f) {
    try {
        f();
    } catch (const std::exception&) {
        return true;
    }
    return false;
}

int main() {
    {
        fgt::DBuf w;
        fail_next = true;
        CHECK(throws([&] { w.alloc(1000); }));
        CHECK(w.p == nullptr && w.bytes == 0);
        CHECK(last_error == hipSuccess);
        // a smaller request afterwards, as a workspace's holder makes it
        const size_t need = 100;
        if (w.bytes < need) w.alloc(need);
        CHECK(w.p != nullptr && w.bytes == need);
        // growing fails: the smaller buffer is gone, and known to be gone
        fail_next = true;
        CHECK(throws([&] { w.alloc(1000); }));
        CHECK(w.p == nullptr && w.bytes == 0 && live == 0);
        w.alloc(8);
        w.release();
        CHECK(w.p == nullptr && w.bytes == 0 && live == 0);
        fail_next = true;
        CHECK(throws([&] { w.upload(std::vector<int>{1, 2, 3}); }));
        CHECK(w.p == nullptr && w.bytes == 0);
        w.upload(std::vector<int>{1, 2, 3});
        CHECK(w.bytes == 12 && w.as<int>()[2] == 3);
        // an arena that is too small
        char range[512];
        fgt::Arena a{range, sizeof range};
        fgt::g_arena = &a;
        fgt::DBuf v;
        CHECK(throws([&] { v.alloc(1000); }));
        CHECK(v.p == nullptr && v.bytes == 0);
        v.alloc(100);
        CHECK(v.p != nullptr && v.bytes == 100 && v.from_arena);
        fgt::g_arena = nullptr;
        w = std::move(v);
        CHECK(w.bytes == 100 && v.p == nullptr && v.bytes == 0);
    }
    CHECK(live == 0);
    return 0;
}
