// device_buffer.h -- device memory of the host side (api.cpp): a buffer owned
// by its holder, or carved from a caller's range while an arena is installed.
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>
#include <stdexcept>
#include <string>
#include <vector>

namespace fgt {

// Throws on an error.  The runtime keeps an error until it is asked for: read
// here, it is not taken for that of a later launch (a caller may go on after
// an allocation that failed).
inline void hcheck(hipError_t e, const char* what) {
    if (e == hipSuccess) return;
    (void)hipGetLastError();
    throw std::runtime_error(std::string(what) + ": " + hipGetErrorString(e));
}

// Bump allocator over a caller-provided device range (the no-allocation
// entry point's scratch): while one is installed on this thread, device
// buffers are carved from it instead of hipMalloc'd.
struct Arena {
    char* base = nullptr;
    size_t cap = 0, used = 0;
    void* take(size_t b) {
        const size_t off = (used + 255) & ~size_t(255);
        if (off + b > cap)
            throw std::invalid_argument("problem needs more device workspace than the " +
                                        std::to_string(cap >> 20) + " MiB no-allocation scratch");
        used = off + b;
        return base + off;
    }
};
inline thread_local Arena* g_arena = nullptr;
// device bytes allocated on this thread by DBuf::alloc (the server's
// admission accounting reads it around a solver build)
inline thread_local size_t g_tally = 0;

// A device buffer owned by the solver (or carved from the installed arena).
// bytes is the size of the memory at p: zero whenever there is none, also
// after an allocation that failed (holders compare it with what they need).
struct DBuf {
    void* p = nullptr;
    size_t bytes = 0;
    bool from_arena = false;
    DBuf() = default;
    DBuf(const DBuf&) = delete;
    DBuf& operator=(const DBuf&) = delete;
    DBuf& operator=(DBuf&& o) noexcept {
        if (this != &o) {
            release();
            p = o.p;
            bytes = o.bytes;
            from_arena = o.from_arena;
            o.p = nullptr;
            o.bytes = 0;
            o.from_arena = false;
        }
        return *this;
    }
    ~DBuf() { release(); }
    void release() {
        if (p && !from_arena) (void)hipFree(p);
        p = nullptr;
        bytes = 0;
        from_arena = false;
    }
    void alloc(size_t b) {
        release();
        if (!b) return;
        if (g_arena) {
            p = g_arena->take(b);
            from_arena = true;
        } else {
            void* q = nullptr;
            hcheck(hipMalloc(&q, b), "hipMalloc");
            p = q;
            g_tally += b;
        }
        bytes = b;
    }
    template <class T>
    void upload(const std::vector<T>& v) {
        alloc(sizeof(T) * v.size());
        if (!v.empty()) hcheck(hipMemcpy(p, v.data(), bytes, hipMemcpyHostToDevice), "hipMemcpy H2D");
    }
    template <class T>
    T* as() const { return static_cast<T*>(p); }
};

}  // namespace fgt
