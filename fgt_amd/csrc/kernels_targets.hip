// kernels_targets.hip -- extra-target evaluation (STEP 11, ifpghtarg >= 1).
//
// Values on the leaves -> orthogonal-polynomial coefficients
// (treedata_trans_nd, src/common/tree_data_routs_nd.f:16-95) -> values at
// arbitrary targets (treedata_evalt_nd, tree_data_routs_nd.f:582-686).  The
// targets are grouped by leaf on the device: each descends the tree (the
// reference's root-to-leaf descent) and takes a place in its leaf's count, a
// scan over the boxes turns the counts into ranges and tasks of at most 256
// targets, and a block per task transforms its leaf's values in LDS and
// evaluates its targets.  (20000 targets on 547 leaves: descent and sort on
// the host 1.48 ms, coefficients of every leaf and evaluation 0.41; now 0.08
// together.)
#include <algorithm>

#include "kernels.h"

namespace fgt {

namespace {

constexpr int kTaskTargets = 256;

// leaf of every target and its place among the leaf's targets; *missing is
// set when a target's path ends at a missing child
__global__ void __launch_bounds__(256) k_target_leaf(int nt, int ndim, int nlevels, const double* __restrict__ targs,
                                                     const double* __restrict__ centers,
                                                     const int* __restrict__ child, int* __restrict__ count,
                                                     int2* __restrict__ place, int* __restrict__ missing) {
    const int it = blockIdx.x * blockDim.x + threadIdx.x;
    if (it >= nt) return;
    double x[3];
    for (int a = 0; a < ndim; ++a) x[a] = targs[(size_t)it * ndim + a];
    // child[b << ndim | k]; -1 in every place of a leaf, -2 where a parent has none
    int b = 0;
    for (int l = 0; l <= nlevels; ++l) {
        int k = 0;
        for (int a = 0; a < ndim; ++a)
            if (x[a] - centers[(size_t)b * ndim + a] >= 0) k |= 1 << a;
        const int c = child[((size_t)b << ndim) | k];
        if (c == -2) *missing = 1;
        if (c < 0) break;
        b = c;
    }
    place[it] = make_int2(b, atomicAdd(count + b, 1));
}

// one block: first[b] = targets in boxes before b, and the tasks {box, first
// target, count, 0}; *ntask their number
__global__ void __launch_bounds__(1024) k_target_tasks(int nboxes, const int* __restrict__ count,
                                                       int* __restrict__ first, int4* __restrict__ tasks,
                                                       int* __restrict__ ntask) {
    __shared__ int2 s[1024];
    const int tid = threadIdx.x;
    int2 base = make_int2(0, 0);   // targets, tasks before this chunk
    for (int b0 = 0; b0 < nboxes; b0 += 1024) {
        const int b = b0 + tid;
        const int c = b < nboxes ? count[b] : 0, k = (c + kTaskTargets - 1) / kTaskTargets;
        int2 v = make_int2(c, k);
        s[tid] = v;
        __syncthreads();
        for (int d = 1; d < 1024; d <<= 1) {
            const int2 u = tid >= d ? s[tid - d] : make_int2(0, 0);
            __syncthreads();
            v.x += u.x;
            v.y += u.y;
            s[tid] = v;
            __syncthreads();
        }
        const int f = base.x + v.x - c;
        if (b < nboxes) first[b] = f;
        for (int q = 0; q < k; ++q)
            tasks[base.y + v.y - k + q] =
                make_int4(b, f + q * kTaskTargets, min(kTaskTargets, c - q * kTaskTargets), 0);
        base.x += s[1023].x;
        base.y += s[1023].y;
        __syncthreads();
    }
    if (tid == 0) *ntask = base.y;
}

__global__ void __launch_bounds__(256) k_target_perm(int nt, const int2* __restrict__ place,
                                                     const int* __restrict__ first, int* __restrict__ perm) {
    const int it = blockIdx.x * blockDim.x + threadIdx.x;
    if (it < nt) perm[first[place[it].x] + place[it].y] = it;
}

// p[k], k < N: Legendre or Chebyshev polynomials at x
template <int N>
__device__ __forceinline__ void polys(int ipoly, double x, double (&p)[N]) {
    p[0] = 1.0;
    p[1] = x;
#pragma unroll
    for (int k = 1; k + 1 < N; ++k)
        p[k + 1] = ipoly == 0 ? ((2 * k + 1) * x * p[k] - k * p[k - 1]) / (k + 1) : 2 * x * p[k] - p[k - 1];
}

// Per value component: the leaf's values become coefficients in LDS, one axis
// after another (a thread takes whole lines of N values in registers; the
// matrix u(k, j) = u[k + j N] is uniform and comes through the scalar cache),
// then the targets are evaluated 64 at a time, wave w taking every fourth
// index of the last axis from w on.
template <int N>
__global__ void __launch_bounds__(256) k_targets(int ndim, int ipoly, int ncd, const double* __restrict__ u,
                                                 const int4* __restrict__ tasks, const int* __restrict__ ntask,
                                                 const double* __restrict__ centers,
                                                 const double* __restrict__ bsize_of_box,
                                                 const double* __restrict__ targs, const int* __restrict__ perm,
                                                 const double* __restrict__ vals, double* __restrict__ out) {
    extern __shared__ double sc[];   // npbox values, then coefficients
    __shared__ double part[4][64], poly[2][N][64];
    if ((int)blockIdx.x >= *ntask) return;
    const int4 task = tasks[blockIdx.x];
    const int b = task.x, first = task.y, cnt = task.z;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int nlines = ndim == 3 ? N * N : ndim == 2 ? N : 1, npbox = nlines * N;
    const CTab1 U = ctab(u);
    const double s = 2.0 / bsize_of_box[b];
    double cen[3];
    for (int a = 0; a < 3; ++a) cen[a] = centers[(size_t)b * ndim + min(a, ndim - 1)];
    for (int q = 0; q < ncd; ++q) {
        for (int i = tid; i < npbox; i += 256) sc[i] = vals[((size_t)b * npbox + i) * ncd + q];
        __syncthreads();
        int stride = 1;
        for (int a = 0; a < ndim; ++a, stride *= N) {
            if (tid < nlines) {   // (N^2 <= 256)
                const int base = tid / stride * stride * N + tid % stride;
                double f[N];
#pragma unroll
                for (int j = 0; j < N; ++j) f[j] = sc[base + j * stride];
#pragma unroll
                for (int k = 0; k < N; ++k) {
                    double d = 0.0;
#pragma unroll
                    for (int j = 0; j < N; ++j) d += U[k + j * N] * f[j];
                    sc[base + k * stride] = d;
                }
            }
            __syncthreads();
        }
        for (int t0 = 0; t0 < cnt; t0 += 64) {
            const int t = min(t0 + lane, cnt - 1), it = perm[first + t];
            // x polynomials in every wave's registers; the others' go through
            // LDS, one wave forming them (indexed by loop counters)
            double p[N];
            polys<N>(ipoly, (targs[(size_t)it * ndim] - cen[0]) * s, p);
            if (wave > 0 && wave < ndim) {
                double r[N];
                polys<N>(ipoly, (targs[(size_t)it * ndim + wave] - cen[wave]) * s, r);
#pragma unroll
                for (int k = 0; k < N; ++k) poly[wave - 1][k][lane] = r[k];
            }
            __syncthreads();
            double v = 0.0;
            // line (j, i) of N coefficients; the last axis' index from the wave on
            const int ni = ndim == 1 ? 1 : N, nj = ndim == 3 ? N : 1;
            for (int i = wave; i < ni; i += 4) {
                double t2 = 0.0;
                for (int j = 0; j < nj; ++j) {
                    const double* c = sc + N * (j + nj * i);
                    double d = 0.0;
#pragma unroll
                    for (int k = 0; k < N; ++k) d += c[k] * p[k];
                    t2 += ndim == 3 ? d * poly[0][j][lane] : d;
                }
                v += ndim == 1 ? t2 : t2 * poly[ndim - 2][i][lane];
            }
            part[wave][lane] = v;
            __syncthreads();
            if (wave == 0 && t0 + lane < cnt)
                out[(size_t)it * ncd + q] = ((part[0][lane] + part[1][lane]) + part[2][lane]) + part[3][lane];
            __syncthreads();
        }
    }
}

}  // namespace

int target_tasks_max(int nt, int nend) { return (int)std::min<long long>(nt, (long long)nend + nt / kTaskTargets); }

bool launch_target_groups(int nt, int ndim, int nlevels, int nboxes, const double* targs, const double* centers,
                          const int* child, int* count, int* first, int2* place, int* perm, int4* tasks, int* ntask,
                          int* missing, hipStream_t s) {
    const dim3 grid((unsigned)((nt + 255LL) / 256));
    hipLaunchKernelGGL(k_target_leaf, grid, dim3(256), 0, s, nt, ndim, nlevels, targs, centers, child, count, place,
                       missing);
    hipLaunchKernelGGL(k_target_tasks, dim3(1), dim3(1024), 0, s, nboxes, count, first, tasks, ntask);
    hipLaunchKernelGGL(k_target_perm, grid, dim3(256), 0, s, nt, place, first, perm);
    return hipGetLastError() == hipSuccess;
}

bool launch_targets(int ndim, int n, int ipoly, int ncd, int maxtask, const double* u, const int4* tasks,
                    const int* ntask, const double* centers, const double* bsize_of_box, const double* targs,
                    const int* perm, const double* vals, double* out, hipStream_t s) {
    size_t lds = sizeof(double);
    for (int a = 0; a < ndim; ++a) lds *= n;
    switch (n) {
#define FGT_TARGETS(N)                                                                                             \
    case N:                                                                                                        \
        hipLaunchKernelGGL((k_targets<N>), dim3(maxtask), dim3(256), lds, s, ndim, ipoly, ncd, u, tasks, ntask,    \
                           centers, bsize_of_box, targs, perm, vals, out);                                         \
        break;
        FGT_TARGETS(2) FGT_TARGETS(3) FGT_TARGETS(4) FGT_TARGETS(5) FGT_TARGETS(6) FGT_TARGETS(7) FGT_TARGETS(8)
        FGT_TARGETS(9) FGT_TARGETS(10) FGT_TARGETS(11) FGT_TARGETS(12) FGT_TARGETS(13) FGT_TARGETS(14)
        FGT_TARGETS(15) FGT_TARGETS(16)
#undef FGT_TARGETS
        default: return false;
    }
    return hipGetLastError() == hipSuccess;
}

}  // namespace fgt
