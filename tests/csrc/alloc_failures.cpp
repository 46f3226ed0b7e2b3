// Host test of a change of precision whose allocations fail, through the
// public interface, over a runtime that runs no kernel: after a failed change
// nothing is launched until a change succeeds.  Every allocation of the change
// is made to fail in turn.
//   alloc_failures <problem file: ints nboxes nlevels ltree norder, itree, iptr, centers, boxsize>
#include <hip/hip_runtime.h>

#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <vector>

#include "fgt.h"

static long fail_at = -1;   // the allocation to fail, counted down
static long allocs = 0, launches = 0;
static hipError_t last_error = hipSuccess;

extern "C" {
hipError_t hipMalloc(void** p, size_t n) {
    ++allocs;
    if (fail_at >= 0 && fail_at-- == 0) return last_error = hipErrorOutOfMemory;
    *p = std::calloc(1, n);
    return hipSuccess;
}
hipError_t hipFree(void* p) { std::free(p); return hipSuccess; }
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) { std::memcpy(d, s, n); return hipSuccess; }
hipError_t hipMemset(void* d, int v, size_t n) { std::memset(d, v, n); return hipSuccess; }
hipError_t hipMemsetAsync(void* d, int v, size_t n, hipStream_t) { std::memset(d, v, n); return hipSuccess; }
hipError_t hipGetLastError() { const hipError_t e = last_error; last_error = hipSuccess; return e; }
hipError_t hipGetDevice(int* d) { *d = 0; return hipSuccess; }
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t, int) { *v = 160 * 1024; return hipSuccess; }
hipError_t hipDeviceSynchronize() { return hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) { *s = nullptr; return hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t* e) { *e = nullptr; return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { *e = nullptr; return hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) { *ms = 0; return hipSuccess; }
hipError_t __hipPushCallConfiguration(dim3, dim3, size_t, hipStream_t) { return hipSuccess; }
hipError_t __hipPopCallConfiguration(dim3*, dim3*, size_t*, hipStream_t*) { return hipSuccess; }
hipError_t hipLaunchKernel(const void*, dim3, dim3, void**, size_t, hipStream_t) { ++launches; return hipSuccess; }
}

#define CHECK(c)                                                                     \
    if (!(c)) {                                                                      \
        char m[256];                                                                 \
        fgt_last_status(m, sizeof m);                                                \
        std::printf("line %d (failing allocation %ld): %s [%s]\n", __LINE__, k, #c, m); \
        return 1;                                                                    \
    }

template <class T>
static std::vector<T> get(FILE* f, size_t n) {
    std::vector<T> v(n);
    if (std::fread(v.data(), sizeof(T), n, f) != n) std::exit(3);
    return v;
}

int main(int argc, char** argv) {
    FILE* f = argc == 2 ? std::fopen(argv[1], "rb") : nullptr;
    if (!f) return 2;
    const std::vector<int> dim = get<int>(f, 4);
    const int nb = dim[0], nl = dim[1], ltree = dim[2], n = dim[3];
    const std::vector<int> itree = get<int>(f, ltree), iptr = get<int>(f, 8);
    const std::vector<double> centers = get<double>(f, 3 * (size_t)nb), boxsize = get<double>(f, nl + 1);
    const double delta = 1e-2, eps = 1e-3;
    long k = -1;
    // a solver: FP64 -> FP32 -> BF16 -> FP64, each change failing at every allocation
    fgt_solver* s = nullptr;
    CHECK(fgt_solver_create(1, 3, delta, eps, 0, 0, n, nb, nl, ltree, itree.data(), iptr.data(), centers.data(),
                            boxsize.data(), &s) == 0);
    CHECK(fgt_solver_execute(s, nullptr, 0) == 0 && launches > 0);
    for (int mode : {1, 0, 2, 0}) {
        bool done = false;
        for (k = 0; !done; ++k) {
            fail_at = k;
            done = fgt_solver_set_precision(s, mode) == 0;
            fail_at = -1;
            launches = 0;
            const int rc = fgt_solver_execute(s, nullptr, 0);
            CHECK((rc == 0) == done && (launches > 0) == done);
            if (!done) {
                // the other precision may be asked for instead
                CHECK(fgt_solver_set_precision(s, mode ? 0 : 1) == 0);
                CHECK(fgt_solver_execute(s, nullptr, 0) == 0 && launches > 0);
            }
        }
        CHECK(k > 1);
    }
    // a batch of two problems
    fgt_problem q{1, 3, delta, eps, 0, 0, n, nb, nl, ltree, itree.data(), iptr.data(), centers.data(), boxsize.data()};
    const fgt_problem qs[2] = {q, q};
    fgt_batch* b = nullptr;
    k = -1;
    CHECK(fgt_batch_create(2, qs, 1, &b) == 0 && fgt_batch_set_graph(b, 0) == 0 && fgt_batch_execute(b) == 0);
    for (int mode : {1, 0, 3, 0}) {
        bool done = false;
        for (k = 0; !done; ++k) {
            fail_at = k;
            done = fgt_batch_set_precision(b, mode, 0.0, nullptr) == 0;
            fail_at = -1;
            launches = 0;
            const int rc = fgt_batch_execute(b);
            CHECK((rc == 0) == done && (launches > 0) == done);
            if (!done) {
                CHECK(fgt_batch_set_precision(b, mode ? 0 : 1, 0.0, nullptr) == 0);
                CHECK(fgt_batch_execute(b) == 0 && launches > 0);
            }
        }
        CHECK(k > 1);
    }
    fgt_batch_destroy(b);
    fgt_solver_destroy(s);
    return 0;
}
