// kernels_plane.hip -- 2-D kernels for gfx950 (FP64): STEP 1 + 2, STEP 4 + 5
// and STEP 6.
//
// A plane problem is small: its stages take microseconds each, and what it
// waits for is launches (one per level for the merges and for the splits) and
// dependent loads.  The cutoff level is the only one whose expansions
// interact, and every phase between a leaf and its cutoff box is a product of
// 1-D phases, so STEP 1 sums the leaves of a cutoff box into its expansion
// directly and STEP 5 evaluates the cutoff box's local expansion at the leaf:
// no expansion of a level below the cutoff exists and neither pass grows with
// the depth.  Frequencies k and npw-1-k are opposite and nodes i and n-1-i
// mirror images, so a 1-D table (and a phase) is known from a quarter (half)
// of it: with S and D the sum and difference of a pair's operands, both
// results of a pair are Re(T) S +- i Im(T) D, a quarter of the products and of
// the LDS reads that bound these kernels.  Whole calls (order 8): 595 leaves on
// four levels 72 -> 32 us, 4363 leaves on six with three densities 572 -> 125.
#include <algorithm>

#include "kernels.h"

namespace fgt {

namespace {

constexpr int kBlock = 256;

__device__ __forceinline__ double2 cmul(double2 a, double2 b) {
    return make_double2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}
__device__ __forceinline__ double2 cfma(double2 a, double2 b, double2 c) {
    c.x += a.x * b.x - a.y * b.y;
    c.y += a.x * b.y + a.y * b.x;
    return c;
}

// 1-D phase of frequency k between the cutoff box and a leaf `depth` levels
// below it: the product of the levels' merge phases (conjugated where the
// path's bit i, coarse to fine, says so).  w: the cutoff level's phase row;
// each finer level's is one row (npw) before.
__device__ __forceinline__ double2 path_phase(const double2* __restrict__ w, int npw, int depth, unsigned conj,
                                              int k) {
    double2 p = make_double2(1.0, 0.0);
    for (int i0 = 0; i0 < depth; i0 += 4) {   // four loads in flight
        double2 q[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) q[i] = gload(w - (ptrdiff_t)min(i0 + i, depth - 1) * npw, (unsigned)k);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            if (i0 + i >= depth) break;
            if ((conj >> (i0 + i)) & 1) q[i].y = -q[i].y;
            p = i0 + i ? cmul(p, q[i]) : q[i];
        }
    }
    return p;
}

// ---------------------------------------------------------------- STEP 1 + 2
// g2d_tens_prod_to_pw (bfgt_pwrouts.f:81-140) per leaf, then the merges of
// STEP 2 up to the cutoff level.  Block = (group of leaves of one cutoff box,
// density and chunk of half-spectrum rows): per leaf the half axis is
// contracted and phased into LDS, and each thread adds its frequencies (the
// pair k1 = tid mod nh, kRows rows k3) of the x contraction times the x phase
// to registers.  A cutoff box with several groups keeps the first group's sum
// in its own slot and the others' in the slots of their first leaves, which
// k_plane_sum then adds up.
// LDS: sT [m][k] (h*nh complex, h = ceil(n/2)); two buffers each of the
// leaf's phases sP (nh x, then R z), sff [k3][m1 pair][S, D] (2*R*h complex)
// and the values sf [m2][m1].
constexpr int kRows = 3;

__global__ void __launch_bounds__(kBlock) k_p2pw2(Geom g, const double2* __restrict__ tab, int n,
                                                  const double2* __restrict__ wms, int nlev,
                                                  const PlaneGroup* __restrict__ groups,
                                                  const PlaneLeaf* __restrict__ leaves, int R, int y0,
                                                  const double* __restrict__ fvals, double2* __restrict__ expn) {
    extern __shared__ double2 sm[];
    const int npw = g.npw, nh = g.pz, nn = n * n, h = (n + 1) / 2;
    const PlaneGroup grp = groups[blockIdx.x];
    const int y = blockIdx.y + y0, ind = y % g.nd, k30 = y / g.nd * R;
    const int rows = min(R, nh - k30);
    double2* sT = sm;
    double2* sP = sT + (size_t)nh * h;
    double2* sff = sP + 2 * (nh + R);
    double* sf = reinterpret_cast<double*>(sff + 4 * (size_t)R * h);
    const int tid = threadIdx.x;
    const int tpr = kBlock / nh;   // rows of threads
    const int k1 = tid % nh, q = tid / nh;
    const int zm0 = tid % h, zr0 = tid / h, zstep = kBlock / h;   // half axis: column pair, row
    const double2* __restrict__ w = wms + (size_t)(nlev - 1) * npw;
    double2 ap[kRows], am[kRows];   // frequencies k1 and npw-1-k1
#pragma unroll
    for (int j = 0; j < kRows; ++j) ap[j] = am[j] = make_double2(0.0, 0.0);
    int lev = -1;
    PlaneLeaf leaf = leaves[grp.first];
    double fv = tid < nn ? gload(fvals + (size_t)leaf.box * nn * g.nd + ind, tid * g.nd) : 0.0;
    for (int i = 0; i < grp.count; ++i) {
        if (leaf.lev != lev) {
            lev = leaf.lev;
            if (i) __syncthreads();   // the last leaf's x contraction has read the table
            const double2* __restrict__ T = tab + (size_t)lev * npw * n;
            for (int o = tid; o < nh * h; o += kBlock) sT[o] = gload(T, (o % nh) * n + o / nh);
        }
        const int buf = i & 1;
        double* f = sf + buf * nn;
        double2* ph = sP + buf * (nh + R);
        double2* ff = sff + (size_t)buf * 2 * R * h;
        if (tid < nn) f[tid] = fv;
        for (int o = tid; o < nh + rows; o += kBlock)
            ph[o] = o < nh ? path_phase(w, npw, leaf.depth, leaf.sx, o)
                           : path_phase(w, npw, leaf.depth, leaf.sz, k30 + o - nh);
        leaf = leaves[grp.first + min(i + 1, grp.count - 1)];
        if (tid < nn) fv = gload(fvals + (size_t)leaf.box * nn * g.nd + ind, tid * g.nd);
        __syncthreads();
        // half axis: F[k3][m1] = P[k3] sum_m2 T[k3][m2] f[m1, m2], then the
        // column pair's sum and difference (a middle column or node is its
        // own mirror image: half of twice it, and zero)
        if (zr0 < zstep)
            for (int r = zr0; r < rows; r += zstep) {
                double2 a = make_double2(0.0, 0.0), b = a;
                for (int m2 = 0; m2 < h; ++m2) {
                    double2 t = sT[m2 * nh + k30 + r];
                    if (2 * m2 + 1 == n) t.x *= 0.5;
                    const double* lo = f + n * m2;
                    const double* hi = f + n * (n - 1 - m2);
                    a.x += t.x * (lo[zm0] + hi[zm0]);
                    a.y += t.y * (lo[zm0] - hi[zm0]);
                    b.x += t.x * (lo[n - 1 - zm0] + hi[n - 1 - zm0]);
                    b.y += t.y * (lo[n - 1 - zm0] - hi[n - 1 - zm0]);
                }
                if (2 * zm0 + 1 == n) b = make_double2(0.0, 0.0);
                const double2 S = cmul(make_double2(a.x + b.x, a.y + b.y), ph[nh + r]);
                const double2 D = cmul(make_double2(a.x - b.x, a.y - b.y), ph[nh + r]);
                ff[2 * (r * h + zm0)] = S;
                // (a middle column's table entries are real: D multiplies zero)
                ff[2 * (r * h + zm0) + 1] = D;
            }
        __syncthreads();
        // x: E[k3][k1] += P[k1] sum_m1 T[k1][m1] F[k3][m1]
        if (q < tpr) {
            double2 s[kRows], d[kRows];   // sum Re(T) S, sum Im(T) D
#pragma unroll
            for (int j = 0; j < kRows; ++j) s[j] = d[j] = make_double2(0.0, 0.0);
            for (int m1 = 0; m1 < h; ++m1) {
                const double2 t = sT[m1 * nh + k1];
#pragma unroll
                for (int j = 0; j < kRows; ++j) {
                    const double2* v = ff + 2 * (min(q + tpr * j, rows - 1) * h + m1);
                    s[j].x += t.x * v[0].x;
                    s[j].y += t.x * v[0].y;
                    d[j].x += t.y * v[1].x;
                    d[j].y += t.y * v[1].y;
                }
            }
            const double2 p = ph[k1], pc = make_double2(p.x, -p.y);
#pragma unroll
            for (int j = 0; j < kRows; ++j) {
                ap[j] = cfma(p, make_double2(s[j].x - d[j].y, s[j].y + d[j].x), ap[j]);
                am[j] = cfma(pc, make_double2(s[j].x + d[j].y, s[j].y - d[j].x), am[j]);
            }
        }
    }
    double2* __restrict__ E = expn + ((size_t)grp.slot * 2 * g.nd + ind) * g.nexp + (size_t)k30 * npw;
    if (q < tpr)
#pragma unroll
        for (int j = 0; j < kRows; ++j)
            if (q + tpr * j < rows) {
                E[(q + tpr * j) * npw + k1] = ap[j];
                if (2 * k1 + 1 != npw) E[(q + tpr * j) * npw + npw - 1 - k1] = am[j];
            }
}

// Cutoff boxes with several groups: task i adds the expansions in
// slots[off[i] ..] into the first of them.  32 elements per block, eight
// threads each.
__global__ void __launch_bounds__(kBlock) k_plane_sum(long long tot, int y0, const int* __restrict__ off,
                                                      const int* __restrict__ slots, double2* __restrict__ expn) {
    __shared__ double2 part[8][32];
    const int a = off[blockIdx.x], b = off[blockIdx.x + 1];
    const int el = threadIdx.x & 31, p = threadIdx.x >> 5;
    const long long e = (long long)(blockIdx.y + y0) * 32 + el;
    double2 s = make_double2(0.0, 0.0);
    if (e < tot) {
#pragma unroll 4
        for (int i = a + p; i < b; i += 8) {
            const double2 v = expn[(size_t)slots[i] * 2 * tot + e];
            s.x += v.x;
            s.y += v.y;
        }
    }
    part[p][el] = s;
    __syncthreads();
    if (p == 0 && e < tot) {
        for (int i = 1; i < 8; ++i) {
            s.x += part[i][el].x;
            s.y += part[i][el].y;
        }
        expn[(size_t)slots[a] * 2 * tot + e] = s;
    }
}

// ---------------------------------------------------------------- STEP 4 + 5
// g2d_pw2pot (bfgt_pwrouts.f:473-526): pot[kk1][kk2] += 2 Re sum_{k1, k3}
// Ux[kk1][k1] Uz[kk2][k3] loc[k3][k1] over the half axis k3 (the last one
// halved when npw is odd), loc being the cutoff box's local expansion times
// the path's phases.  Block = (leaf, output component and density): the
// expansion's frequency pairs, phased along x as they are read, and the 1-D
// tables are staged in LDS, then x runs with one thread per node pair and k3
// and the half axis with one per kk1 and node pair kk2.  The first-derivative
// tables of mirror nodes are minus conjugate.
// LDS: sE [k3][k1 pair][S, D] (2*nh*nh complex), sU [k1][kk1] and sZ
// [k3][kk2] (nh*h each, h = ceil(n/2)), sff [k3][kk1] (nh*n), sP (2*nh).
__global__ void __launch_bounds__(kBlock) k_pw2pot2(Geom g, const double2* __restrict__ tab, size_t ks, int n,
                                                    const double2* __restrict__ wms, int nlev,
                                                    const PlaneLeaf* __restrict__ leaves,
                                                    const double2* __restrict__ expn, PlaneComps pc, int y0) {
    extern __shared__ double2 sm[];
    const PlaneLeaf leaf = leaves[blockIdx.x];
    const int y = blockIdx.y + y0, ind = y % g.nd, c = y / g.nd;
    const int npw = g.npw, nh = g.pz, nn = n * n, h = (n + 1) / 2;
    double2* sE = sm;
    double2* sU = sE + 2 * (size_t)nh * nh;
    double2* sZ = sU + (size_t)nh * h;
    double2* sff = sZ + (size_t)nh * h;
    double2* sP = sff + (size_t)nh * n;
    const size_t lo = (size_t)leaf.lev * n * npw;
    const double2* __restrict__ Ux = tab + pc.kx[c] * ks + lo;   // [i][k]
    const double2* __restrict__ Uz = tab + pc.kz[c] * ks + lo;
    const double2* __restrict__ E = expn + ((size_t)leaf.slot * 2 * g.nd + g.nd + ind) * g.nexp;
    const double2* __restrict__ w = wms + (size_t)(nlev - 1) * npw;
    const int tid = threadIdx.x;
    // the split phases are the conjugates of the merge phases
    for (int o = tid; o < 2 * nh; o += kBlock)
        sP[o] = o < nh ? path_phase(w, npw, leaf.depth, ~leaf.sx, o)
                       : path_phase(w, npw, leaf.depth, ~leaf.sz, o - nh);
    for (int o = tid; o < nh * h; o += kBlock) {
        const int i = o / nh, k = o % nh;
        sU[k * h + i] = gload(Ux, i * npw + k);
        sZ[k * h + i] = gload(Uz, i * npw + k);
    }
    __syncthreads();
    const bool odd = (npw & 1) == 1;
    for (int o = tid; o < nh * nh; o += kBlock) {
        const int k1 = o % nh, k3 = o / nh;
        const double2 p = sP[k1];
        const double2 a = cmul(gload(E, k3 * npw + k1), p);
        double2 b = cmul(gload(E, k3 * npw + npw - 1 - k1), make_double2(p.x, -p.y));
        if (odd && k1 == nh - 1) b = make_double2(0.0, 0.0);   // the zero frequency is its own opposite
        sE[2 * o] = make_double2(a.x + b.x, a.y + b.y);
        sE[2 * o + 1] = make_double2(a.x - b.x, a.y - b.y);
    }
    __syncthreads();
    const double sgx = pc.kx[c] == 1 ? -1.0 : 1.0;
    for (int o = tid; o < nh * h; o += kBlock) {
        const int kk1 = o % h, k3 = o / h;
        const double2* __restrict__ e = sE + 2 * (size_t)k3 * nh;
        double2 s = make_double2(0.0, 0.0), d = s;
#pragma unroll 4
        for (int k1 = 0; k1 < nh; ++k1) {
            const double2 u = sU[k1 * h + kk1], S = e[2 * k1], D = e[2 * k1 + 1];
            s.x += u.x * S.x;
            s.y += u.x * S.y;
            d.x += u.y * D.x;
            d.y += u.y * D.y;
        }
        const double t = (odd && k3 == nh - 1) ? 1.0 : 2.0;
        const double2 p = make_double2(t * sP[nh + k3].x, t * sP[nh + k3].y);
        sff[k3 * n + kk1] = cmul(make_double2(s.x - d.y, s.y + d.x), p);
        if (2 * kk1 + 1 != n) sff[k3 * n + n - 1 - kk1] = cmul(make_double2(sgx * (s.x + d.y), sgx * (s.y - d.x)), p);
    }
    __syncthreads();
    const double sgz = pc.kz[c] == 1 ? -1.0 : 1.0;
    if (tid < n * h) {
        const int kk1 = tid % n, kk2 = tid / n;
        double a = 0.0, b = 0.0;
#pragma unroll 4
        for (int k3 = 0; k3 < nh; ++k3) {
            const double2 u = sZ[k3 * h + kk2], f = sff[k3 * n + kk1];
            a += u.x * f.x;
            b += u.y * f.y;
        }
        const OutDesc& od = pc.od[c];
        double* __restrict__ out = od.p + (size_t)leaf.box * nn * od.ns + od.coff + ind;
        out[tid * od.ns] += a - b;
        if (2 * kk2 + 1 != n) out[(kk1 + n * (n - 1 - kk2)) * od.ns] += sgz * (a + b);
    }
}

// ---------------------------------------------------------------- STEP 6
// g2d_tens_prod_to_potloc_fast (bfgt_local.f:1230-1315): per source
// out[k1][k3] += sum_j1 Ax[k1][j1] sum_j3 Az[k3][j3] f[j1][j3].  Block =
// (target, output component and density), four waves; a wave takes four
// sources at a time, one in each block of the 4x4x4 FP64 matrix products
// (lane = 16 k + 4 b + i: A[i][k], B[k][i], result D[k][i] of block b), where
// the result of the half-axis contraction is the operand of the x contraction
// as it stands.  Sixteen sources are in flight, so a target's list is one or
// two rounds of dependent loads (list, then values and tables) -- what a plane
// problem's near field waits for: a call with 154 leaves of order 16 took 26 us
// with one source after another through LDS, now 10; 22 leaves with two
// densities and all six components 237, now 15.  Tables [j][k] (source node, target
// node).  At the end the sixteen partial sums meet in LDS.
template <int NB>
__global__ void __launch_bounds__(kBlock) k_direct2(int n, int nd, const double* __restrict__ loctab, size_t ks,
                                                    int nls, const int* __restrict__ tgt,
                                                    const int* __restrict__ lev, const int* __restrict__ off,
                                                    const int* __restrict__ src, const int* __restrict__ code,
                                                    const double* __restrict__ fvals, PlaneComps pc, int y0) {
    constexpr int ROW = 4 * NB + 1, PART = 4 * NB * ROW;
    __shared__ double buf[16][PART];
    const int task = blockIdx.x, y = blockIdx.y + y0, ind = y % nd, c = y / nd;
    const int nn = n * n;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int i = lane & 3, b = (lane >> 2) & 3, k = lane >> 4;
    const int l = lev[task], j0 = off[task], j1 = off[task + 1];
    const double* __restrict__ tabx = loctab + (pc.kx[c] * ks + (size_t)l * nls * nn);
    const double* __restrict__ tabz = loctab + (pc.kz[c] * ks + (size_t)l * nls * nn);
    double X[NB][NB];
#pragma unroll
    for (int m = 0; m < NB; ++m)
#pragma unroll
        for (int r = 0; r < NB; ++r) X[m][r] = 0.0;
    // element (row 4 h + k, column 4 m + i); past n a valid one
    int el[NB][NB];
#pragma unroll
    for (int h = 0; h < NB; ++h)
#pragma unroll
        for (int m = 0; m < NB; ++m) el[h][m] = min(4 * h + k, n - 1) * n + min(4 * m + i, n - 1);
    for (int j = j0 + 4 * wave; j < j1; j += 16) {
        const int e = min(j + b, j1 - 1);
        const bool on = j + b < j1;
        const int cd = code[e];
        const double* __restrict__ f = fvals + (size_t)src[e] * nn * nd + ind;
        double F[NB][NB], T[NB][NB], U[NB][NB];
        const unsigned to = ((cd >> 16) & 255) * nn, uo = (cd & 255) * nn;
#pragma unroll
        for (int h = 0; h < NB; ++h)
#pragma unroll
            for (int m = 0; m < NB; ++m) {
                // (zero past n and past the list: the products need no more)
                const double v = gload(f, el[h][m] * nd);
                F[m][h] = on && 4 * m + i < n && 4 * h + k < n ? v : 0.0;
                T[m][h] = gload(tabz, to + el[h][m]);
                U[m][h] = gload(tabx, uo + el[h][m]);
            }
        // Y[j1][k3] = sum_j3 f[j1][j3] Az[k3][j3]
        double Y[NB][NB];
#pragma unroll
        for (int m = 0; m < NB; ++m)
#pragma unroll
            for (int r = 0; r < NB; ++r) Y[m][r] = 0.0;
#pragma unroll
        for (int h = 0; h < NB; ++h)
#pragma unroll
            for (int m = 0; m < NB; ++m)
#pragma unroll
                for (int r = 0; r < NB; ++r)
                    Y[m][r] = __builtin_amdgcn_mfma_f64_4x4x4f64(F[m][h], T[r][h], Y[m][r], 0, 0, 0);
        // X[k1][k3] += sum_j1 Ax[k1][j1] Y[j1][k3]
#pragma unroll
        for (int h = 0; h < NB; ++h)
#pragma unroll
            for (int m = 0; m < NB; ++m)
#pragma unroll
                for (int r = 0; r < NB; ++r)
                    X[m][r] = __builtin_amdgcn_mfma_f64_4x4x4f64(U[m][h], Y[h][r], X[m][r], 0, 0, 0);
    }
    // lane: k1 = 4 m + k, k3 = 4 r + i
    double* __restrict__ o = buf[4 * wave + b];
#pragma unroll
    for (int m = 0; m < NB; ++m)
#pragma unroll
        for (int r = 0; r < NB; ++r) o[(4 * r + i) * ROW + 4 * m + k] = X[m][r];
    __syncthreads();
    if (tid < nn) {
        const int at = tid / n * ROW + tid % n;
        double v = 0.0;
#pragma unroll
        for (int p = 0; p < 16; ++p) v += buf[p][at];
        const OutDesc& od = pc.od[c];
        od.p[((size_t)tgt[task] * nn + tid) * od.ns + od.coff + ind] += v;
    }
}

// grid rows [0, n) in launches of at most HIP's y limit
template <class F>
void for_y(int n, F&& launch) {
    for (int y0 = 0; y0 < n; y0 += 65535) launch(y0, std::min(n - y0, 65535));
}

bool ok_launch() { return hipGetLastError() == hipSuccess; }

// rows k3 of a STEP 1 block: as its threads take them, of those there are (LDS
// holds the rows: three plane waves at order 16, 256 / nh threads a row, would
// ask for 209 KB and go the general way, 166 leaves 63 us and not 22)
int plane_rows(int nh) { return std::min(kBlock / nh * kRows, nh); }
size_t p2pw2_lds(int n, int nh) {
    const size_t R = plane_rows(nh), h = (n + 1) / 2;
    return sizeof(double2) * (nh * h + 2 * (nh + R) + 4 * R * h) + sizeof(double) * 2 * n * n;
}
size_t pw2pot2_lds(int n, int nh) {
    const size_t h = (n + 1) / 2;
    return sizeof(double2) * nh * (2 * (size_t)nh + 2 * h + n + 2);
}

}  // namespace

bool plane_supported(const Geom& g, const DevTables& t, int nlev) {
    return g.ndim == 2 && t.npw > 0 && g.pz <= kBlock && nlev <= 32 && p2pw2_lds(t.n, g.pz) <= t.lds_limit &&
           pw2pot2_lds(t.n, g.pz) <= t.lds_limit;
}

bool launch_p2pw_plane(const Geom& g, const DevTables& t, int nlev, int ngroup, const PlaneGroup* groups,
                       const PlaneLeaf* leaves, int nsum, const int* sum_off, const int* sum_slots,
                       const double* fvals, double2* expn, hipStream_t s) {
    if (ngroup > 0) {
        const int R = plane_rows(g.pz);
        for_y(g.nd * ((g.pz + R - 1) / R), [&](int y0, int ny) {
            hipLaunchKernelGGL(k_p2pw2, dim3(ngroup, ny), dim3(kBlock), p2pw2_lds(t.n, g.pz), s, g, t.p2pw, t.n, t.wms,
                               nlev, groups, leaves, R, y0, fvals, expn);
        });
    }
    if (nsum > 0) {
        const long long tot = (long long)g.nd * g.nexp;
        for_y((int)((tot + 31) / 32), [&](int y0, int ny) {
            hipLaunchKernelGGL(k_plane_sum, dim3(nsum, ny), dim3(kBlock), 0, s, tot, y0, sum_off, sum_slots, expn);
        });
    }
    return ok_launch();
}

bool launch_pw2pot_plane(const Geom& g, const DevTables& t, int nlev, int nleaf, const PlaneLeaf* leaves,
                         const double2* expn, const PlaneComps& pc, hipStream_t s) {
    if (nleaf > 0)
        for_y(pc.n * g.nd, [&](int y0, int ny) {
            hipLaunchKernelGGL(k_pw2pot2, dim3(nleaf, ny), dim3(kBlock), pw2pot2_lds(t.n, g.pz), s, g, t.pw2pot,
                               t.pw2pot_ks, t.n, t.wms, nlev, leaves, expn, pc, y0);
        });
    return ok_launch();
}

bool launch_direct_plane(const Geom& g, const DevTables& t, int ntask, const int* tgt, const int* lev, const int* off,
                         const int* src, const int* code, const double* fvals, const PlaneComps& pc, hipStream_t s) {
    if (ntask <= 0) return true;
    for_y(pc.n * g.nd, [&](int y0, int ny) {
        const dim3 grid(ntask, ny);
#define FGT_DIRECT2(NB)                                                                                             \
    hipLaunchKernelGGL((k_direct2<NB>), grid, dim3(kBlock), 0, s, t.n, g.nd, t.loctab, t.loctab_ks, t.loc_slots, tgt, \
                       lev, off, src, code, fvals, pc, y0)
        switch ((t.n + 3) / 4) {
            case 1: FGT_DIRECT2(1); break;
            case 2: FGT_DIRECT2(2); break;
            case 3: FGT_DIRECT2(3); break;
            default: FGT_DIRECT2(4); break;
        }
#undef FGT_DIRECT2
    });
    return ok_launch();
}

}  // namespace fgt
