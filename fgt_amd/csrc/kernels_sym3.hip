// kernels_sym3.hip -- 3-D STEP 1 (values -> PW) and STEP 5 (PW -> values) in
// FP64 through the symmetries of the 1-D tables (gfx950).
//
// Replaces g3d_tens_prod_to_pw (bfgt_pwrouts.f:153-222) with the STEP 2
// shift of leaf children folded in, and g3d_pw2pgh (bfgt_pwrouts.f:719-1065)
// with the STEP 4 shift into leaves folded in.
//
// The plane-wave frequencies come in pairs (k, npw-1-k) of opposite sign and
// the nodes in pairs (i, n-1-i) about the box centre, so a 1-D table obeys
//   T[npw-1-k][i] = conj T[k][i],   T[k][n-1-i] = conj T[k][i]
// (first-derivative tables: -conj).  The same holds for the two children of
// a box along an axis: the node i of one and n-1-i of the other lie
// symmetric about the parent's centre, and their tables, which carry the
// parent-child phase, are conjugates.  A "pair" below is two such nodes:
// side a is node i (of the child whose table variant is 1), side b its mirror
// image.  A leaf evaluated by itself has ceil(n/2) pairs per axis; the
// (up to eight) leaf children of one parent together have n.
//
// With E = sums and D = differences over the pair being contracted,
//   sum = Re(T) E + i Im(T) D,   the partner's sum = Re(T) E - i Im(T) D
// (E, D complex, the table real): four real multiply-adds serve two inputs
// and two outputs, where the plain complex form takes sixteen.  A quarter
// of the arithmetic leaves both steps bound by the expansion bytes they
// write and read.  Orders 4 to 16 (lower ones, and 1-D and 2-D, take the
// general kernels: one barrier-separated pass per half-axis frequency; at
// order 6, npw 18, 1972 leaves with two densities these took 94 us for STEP 1
// and 304 us for STEP 5, 19 and 29 us here).
#include "kernels.h"

#include <algorithm>
#include <type_traits>

namespace fgt {

namespace {

constexpr int kThreads = 256;

__device__ __forceinline__ double2 cplus(double2 a, double2 b) { return make_double2(a.x + b.x, a.y + b.y); }
__device__ __forceinline__ double2 cminus(double2 a, double2 b) { return make_double2(a.x - b.x, a.y - b.y); }
__device__ __forceinline__ double2 cprod(double2 a, double2 b) {
    return make_double2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}

// Touches every 64-byte line of n table entries once, eight scalar loads at a
// time, the lines dealt to the block's waves: the scalar cache starts a
// kernel empty, and the stages below would take its misses one by one.
__device__ __forceinline__ void warm_table(CTab2 t, int n, int wave) {
    const int lines = (n + 3) >> 2;
    for (int i = 8 * wave; i < lines; i += 8 * (kThreads / 64)) {
        double d[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) d[j] = t[4 * (long long)min(i + j, lines - 1)].x;
        asm volatile("" ::"s"(d[0]), "s"(d[1]), "s"(d[2]), "s"(d[3]), "s"(d[4]), "s"(d[5]), "s"(d[6]), "s"(d[7]));
    }
}

// pairs per axis of a task: a family (the leaf children of one parent) or one leaf
template <int N, bool FAM>
constexpr int sym_pairs() { return FAM ? N : (N + 1) / 2; }

// ---------------------------------------------------------------- STEP 5
// x pairs per block: a task's x pairs are split over blocks so that the
// block's output columns (2 NX x nodes, 2 NP y nodes) are at most one per
// thread and the x stage's sums stay in registers
template <int N, bool FAM>
constexpr int sym5_parts() { return sym_pairs<N, FAM>() <= 6 ? 1 : (sym_pairs<N, FAM>() + 3) / 4; }
template <int N, bool FAM>
constexpr int sym5_nx() { return (sym_pairs<N, FAM>() + sym5_parts<N, FAM>() - 1) / sym5_parts<N, FAM>(); }

// k3 slabs per round: about one (slab, k2) column of the x stage per thread,
// at most 8, the rounds of equal length
__host__ __device__ inline int sym5_slabs(int npw) {
    const int nh = (npw + 1) / 2;
    const int most = kThreads / npw < 1 ? 1 : (kThreads / npw > 8 ? 8 : kThreads / npw);
    const int rounds = (nh + most - 1) / most;
    return (nh + rounds - 1) / rounds;
}
// double2 entries of the block's LDS: sff [k2][slab][x node] and yres
// [slab][x node][y node] share it (rows padded by one entry: odd strides)
inline size_t sym5_lds_entries(int npw, int nodx, int nody) {
    const size_t sr = (size_t)sym5_slabs(npw);
    return std::max(npw * (sr * nodx + 1), sr * nodx * (nody + 1));
}

// One block: x pairs [px0, px0 + NX) of one task, all k3.  Per round of SR
// slabs:
//   x: thread = (slab, k2) column; E rows k1 and npw-1-k1 stream from HBM,
//      two steps ahead of their use, into 2 NX node sums;
//   y: lane = (slab, x node), the y pairs split over the waves;
//   z: thread = (x node, y node), all z pairs of every z kind in registers.
// The tables are wave-uniform (scalar loads); LDS carries the transposes.
// Bound by the expansion reads and by the latency of each round's three
// stages (norder 8, npw 28, 8382 leaves: 84 us for 210 MB, 2.5 TB/s; the
// sixteen-multiply-add form over half the siblings 244 us; norder 12, npw 60,
// 4250 leaves: 402 us, 1182 before).  A family whose box's expansion is not
// formed reads the one above it and splits it on the way: the x phase on each
// row pair's sum and difference, the y and z phases on the column's results
// (77 and 360 us, with the siblings' rows shared through the caches).  x pairs over more blocks at eight pairs
// (two of four rather than one of eight: smaller LDS tiles, four blocks per
// CU instead of three) measured 106 -> 102 us, the scalar cache's warm-up,
// the unrolled y and z stages and one launch for both kinds of task 102 -> 84.
template <int N, bool FAM, int NZ, typename ET>
__device__ __forceinline__ void pw2pot_sym_block(int npw, int nd, const double2* __restrict__ tabS,
                                                 const SymTask* __restrict__ T, int part,
                                                 const ET* __restrict__ expn, const double2* __restrict__ wms,
                                                 size_t ks, Kinds kd, const ZOut& zo,
                                                 const ProbPtrs* __restrict__ prob, double2* __restrict__ sm) {
    constexpr int NP = sym_pairs<N, FAM>(), NX = sym5_nx<N, FAM>();
    // (FP32 expansions round after every split: none is folded in)
    constexpr bool FOLD = FAM && std::is_same<ET, double2>::value;
    constexpr int NODX = 2 * NX, NODY = 2 * NP, COLS = NODX * NODY;
    static_assert(COLS <= kThreads, "one output column per thread");
    constexpr int YS = NODX <= 8 ? 4 : 2;                  // waves sharing one y row batch
    constexpr int YP = (NP + YS - 1) / YS;                 // y pairs per wave
    constexpr int ZS = COLS <= 64 ? 4 : (COLS <= 128 ? 2 : 1);   // thread groups sharing the z pairs
    constexpr int ZP = (NP + ZS - 1) / ZS;
    constexpr int V = FAM ? 1 : 0;
    constexpr int KU = 3;
    const int nh = (npw + 1) >> 1;
    const int SR = sym5_slabs(npw);
    const int ST = SR * NODX + 1;
    const bool odd = (npw & 1) != 0;
    const long long per = (long long)npw * N;
    const long long row3 = (3LL * __builtin_amdgcn_readfirstlane(T->lev) + V) * per;
    const int px0 = min(part * NX, NP - NX);
    const CTab2 UX = ctab(tabS) + ((long long)(kd.x * ks) + row3 + px0);
    const CTab2 UY = ctab(tabS) + ((long long)(kd.y * ks) + row3);
    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lane = tid & 63;
    const int slot = __builtin_amdgcn_readfirstlane(T->slot);
    const double sgx = kd.x == 1 ? -1.0 : 1.0, sgy = kd.y == 1 ? -1.0 : 1.0;
    // the split of the expansion to the family's box: per axis the phase row,
    // conjugated as the box lies (only the imaginary parts' signs)
    const int klev = FOLD ? __builtin_amdgcn_readfirstlane(T->klev) : 0;
    const int fsg = FOLD ? __builtin_amdgcn_readfirstlane(T->sign) : 0;
    const double2* __restrict__ W = wms + (long long)(klev > 0 ? klev - 1 : 0) * npw;
    const CTab2 WX = ctab(W);
    const double wsx = fsg & 1 ? -1.0 : 1.0, wsy = fsg & 2 ? -1.0 : 1.0, wsz = fsg & 4 ? -1.0 : 1.0;
    CTab2 UZ[NZ];
#pragma unroll
    for (int z = 0; z < NZ; ++z) UZ[z] = ctab(tabS) + ((long long)(zo.kz[z] * ks) + row3);
    warm_table(UX, nh * N - px0, wave);
    if (kd.y != kd.x) warm_table(UY, nh * N, wave);
#pragma unroll
    for (int z = 0; z < NZ; ++z)
        if (zo.kz[z] != kd.x && zo.kz[z] != kd.y) warm_table(UZ[z], nh * N, wave);
    // y rows and output column of this thread
    const int yset = YS == 4 ? wave : wave >> 1, yrow0 = YS == 4 ? 0 : 64 * (wave & 1);
    const int zset = ZS == 1 ? 0 : (ZS == 2 ? wave >> 1 : wave);
    const int col = ZS == 1 ? tid : (ZS == 2 ? (tid & 127) : lane);
    const bool zact = col < COLS;
    const int zx = zact ? col % NODX : 0, zy = zact ? col / NODX : 0;
    for (int ind = 0; ind < nd; ++ind) {
        double GP[NZ][ZP], GQ[NZ][ZP];
#pragma unroll
        for (int z = 0; z < NZ; ++z)
#pragma unroll
            for (int q = 0; q < ZP; ++q) GP[z][q] = GQ[z][q] = 0.0;
        const ET* __restrict__ E = expn + (size_t)(slot * 2 * nd + nd + ind) * (size_t)(nh * npw * npw);
        for (int r = 0; r < nh; r += SR) {
            const int cols = SR * npw;
            // ---- x
            for (int cb = 64 * wave; cb < cols; cb += kThreads) {
                const int c = min(cb + lane, cols - 1);   // past the end: a duplicate of the last column
                const int s = c / npw, k2 = c - s * npw;
                // row base scalar, column offset per lane
                const unsigned co = (unsigned)(min(r + s, nh - 1) * npw * npw + k2);
                double2 P[NX], Q[NX];
#pragma unroll
                for (int p = 0; p < NX; ++p) P[p] = Q[p] = make_double2(0.0, 0.0);
                ET u[KU][2], v[KU][2];   // two sets of KU frequency pairs
                auto load = [&](ET (&e)[KU][2], int k) {
#pragma unroll
                    for (int j = 0; j < KU; ++j) {
                        const int kc = min(k + j, nh - 1);
                        e[j][0] = gload(E + (size_t)(kc * npw), co);
                        e[j][1] = gload(E + (size_t)((npw - 1 - kc) * npw), co);
                    }
                };
                auto apply = [&](const ET (&e)[KU][2], int k) {
#pragma unroll
                    for (int j = 0; j < KU; ++j) {
                        if (k + j >= nh) break;
                        const double2 a = ldE(e[j][0]), b = ldE(e[j][1]);
                        // the zero frequency of an odd count pairs with itself
                        double2 S = (odd && k + j == nh - 1) ? a : cplus(a, b);
                        double2 D = cminus(a, b);
                        if (FOLD && klev > 0) {
                            // sum and difference of a w and b conj(w)
                            const double2 w = WX[k + j];
                            const double wi = wsx * w.y;
                            const double2 S0 = S;
                            S = make_double2(S0.x * w.x - D.y * wi, S0.y * w.x + D.x * wi);
                            D = make_double2(D.x * w.x - S0.y * wi, D.y * w.x + S0.x * wi);
                        }
#pragma unroll
                        for (int p = 0; p < NX; ++p) {
                            const double2 t = UX[(long long)(k + j) * N + p];
                            P[p].x += t.x * S.x;
                            P[p].y += t.x * S.y;
                            Q[p].x += t.y * D.x;
                            Q[p].y += t.y * D.y;
                        }
                    }
                };
                load(u, 0);
                for (int k = 0; k < nh; k += 2 * KU) {
                    load(v, k + KU);
                    __builtin_amdgcn_sched_barrier(0);
                    apply(u, k);
                    if (k + KU >= nh) break;
                    load(u, k + 2 * KU);
                    __builtin_amdgcn_sched_barrier(0);
                    apply(v, k + KU);
                }
                double2* __restrict__ o = sm + k2 * ST + s * NODX;
                double2 yz = make_double2(1.0, 0.0);   // the column's y and z phases
                if (FOLD && klev > 0) {
                    const double2 wy = gload(W, (unsigned)k2), wz = gload(W, (unsigned)min(r + s, nh - 1));
                    yz = cprod(make_double2(wy.x, wsy * wy.y), make_double2(wz.x, wsz * wz.y));
                }
#pragma unroll
                for (int p = 0; p < NX; ++p) {
                    double2 a = make_double2(P[p].x - Q[p].y, P[p].y + Q[p].x);
                    double2 b = make_double2(sgx * (P[p].x + Q[p].y), sgx * (P[p].y - Q[p].x));
                    if (FOLD && klev > 0) a = cprod(a, yz), b = cprod(b, yz);
                    o[p] = a;
                    o[NX + p] = b;
                }
            }
            __syncthreads();
            // ---- y
            const int rows = SR * NODX;
            const int row = yrow0 + lane;
            {
                const double2* __restrict__ f = sm + min(row, rows - 1);
                double2 P[YP], Q[YP];
#pragma unroll
                for (int p = 0; p < YP; ++p) P[p] = Q[p] = make_double2(0.0, 0.0);
                if (yrow0 < rows) {
                    // several steps' table and LDS reads together
                    constexpr int YU = YP <= 2 ? 4 : 2;
                    for (int k0 = 0; k0 < nh; k0 += YU) {
                        double2 a[YU], b[YU], t[YU][YP];
#pragma unroll
                        for (int j = 0; j < YU; ++j) {
                            const int k = min(k0 + j, nh - 1);
                            a[j] = f[k * ST];
                            b[j] = f[(npw - 1 - k) * ST];
#pragma unroll
                            for (int p = 0; p < YP; ++p) t[j][p] = UY[(long long)k * N + min(yset * YP + p, NP - 1)];
                        }
#pragma unroll
                        for (int j = 0; j < YU; ++j) {
                            if (k0 + j >= nh) break;
                            const double2 S = (odd && k0 + j == nh - 1) ? a[j] : cplus(a[j], b[j]);
                            const double2 D = cminus(a[j], b[j]);
#pragma unroll
                            for (int p = 0; p < YP; ++p) {
                                P[p].x += t[j][p].x * S.x;
                                P[p].y += t[j][p].x * S.y;
                                Q[p].x += t[j][p].y * D.x;
                                Q[p].y += t[j][p].y * D.y;
                            }
                        }
                    }
                }
                __syncthreads();   // sff is read; yres takes its place
                if (row < rows) {
                    double2* __restrict__ o = sm + row * (NODY + 1);
#pragma unroll
                    for (int p = 0; p < YP; ++p) {
                        const int q = yset * YP + p;
                        if (q < NP) {
                            o[q] = make_double2(P[p].x - Q[p].y, P[p].y + Q[p].x);
                            o[NP + q] = make_double2(sgy * (P[p].x + Q[p].y), sgy * (P[p].y - Q[p].x));
                        }
                    }
                }
            }
            __syncthreads();
            // ---- z
            if (zact) {
                constexpr int ZU = NZ * ZP <= 4 ? 4 : (NZ * ZP <= 8 ? 2 : 1);
                const int ns = min(SR, nh - r);
                for (int s0 = 0; s0 < ns; s0 += ZU) {
                    double2 yv[ZU], t[ZU][NZ][ZP];
#pragma unroll
                    for (int j = 0; j < ZU; ++j) {
                        const int s = min(s0 + j, ns - 1);
                        yv[j] = sm[(s * NODX + zx) * (NODY + 1) + zy];
#pragma unroll
                        for (int z = 0; z < NZ; ++z)
#pragma unroll
                            for (int q = 0; q < ZP; ++q)
                                t[j][z][q] = UZ[z][(long long)(r + s) * N + min(zset * ZP + q, NP - 1)];
                    }
#pragma unroll
                    for (int j = 0; j < ZU; ++j) {
                        if (s0 + j >= ns) break;
                        const double w = (odd && r + s0 + j == nh - 1) ? 0.5 : 1.0;
                        const double yr = yv[j].x * w, yi = yv[j].y * w;
#pragma unroll
                        for (int z = 0; z < NZ; ++z)
#pragma unroll
                            for (int q = 0; q < ZP; ++q) {
                                GP[z][q] += t[j][z][q].x * yr;
                                GQ[z][q] += t[j][z][q].y * yi;
                            }
                    }
                }
            }
            __syncthreads();
        }
        if (zact) {
            // node pair -> (child bit, node): side b is the mirrored node, of
            // the other child (family) or of the same leaf; a leaf's middle
            // node (odd n) is its own mirror, side a
            const int bx = zx >= NX, by = zy >= NP;
            const int px = px0 + zx - bx * NX, py = zy - by * NP;
            const int ix = bx ? N - 1 - px : px, iy = by ? N - 1 - py : py;
            const bool own = px >= part * NX && (FAM || !((bx && 2 * px + 1 == N) || (by && 2 * py + 1 == N)));
            if (own) {
                const int cxy = FAM ? bx | by << 1 : 0;
                const int ba = T->box[cxy], bb = T->box[FAM ? cxy | 4 : 0];
                int node = ix + N * iy;
                // opaque: the output addresses are formed here, not held
                // through the whole task
                asm volatile("" : "+v"(node));
#pragma unroll
                for (int z = 0; z < NZ; ++z) {
                    double* const op = (prob ? prob->pot : zo.od[z].p) + zo.od[z].coff + ind;
                    const int ns = zo.od[z].ns;
                    const double sgz = zo.kz[z] == 1 ? -2.0 : 2.0;
#pragma unroll
                    for (int q = 0; q < ZP; ++q) {
                        const int pz = zset * ZP + q;
                        if (pz >= NP) break;
                        if (ba >= 0)
                            gadd(op + (size_t)ba * (N * N * N) * ns, (node + N * N * pz) * ns,
                                 2.0 * (GP[z][q] - GQ[z][q]));
                        if (bb >= 0 && (FAM || 2 * pz + 1 != N))
                            gadd(op + (size_t)bb * (N * N * N) * ns, (node + N * N * (N - 1 - pz)) * ns,
                                 sgz * (GP[z][q] + GQ[z][q]));
                    }
                }
            }
        }
    }
}

// The families' blocks first, then the single leaves', in one launch; each
// kind is dealt to the XCDs in contiguous runs (blocks of one task, and tasks
// of one region, share an L2).
template <int N, int NZ, typename ET>
__global__ void __launch_bounds__(kThreads, (NZ > 1 && NZ * N >= 16) ? 2 : 3)
    k_pw2pot_sym(int nd, const double2* __restrict__ tabS, int npw, const SymTask* __restrict__ tasks, int nfam,
                 int nown, const ET* __restrict__ expn, const double2* __restrict__ wms, size_t ks, ZGroups zg, Multi mu) {
    constexpr int PF = sym5_parts<N, true>(), PO = sym5_parts<N, false>();
    extern __shared__ double2 sm[];
    const int nfb = nfam * PF, per = nfb + nown * PO;
    const int grp = blockIdx.x / per, b = blockIdx.x - grp * per;   // blocks of one group after another's
    const bool fam = b < nfb;
    const int lin = fam ? xcd_task(b, nfb) : xcd_task(b - nfb, nown * PO);
    const Kinds kd = zg.kd[grp];
    const ZOut& zo = zg.zo[grp];
    const int tix = fam ? lin / PF : nfam + lin / PO, part = fam ? lin % PF : lin % PO;
    const ProbPtrs* prob = nullptr;
    if (mu.pp) {
        prob = mu.pp + mu.tprob[tix];
        npw = prob->g.npw;
        tabS = prob->pw2potS;
        wms = prob->wms;
        expn = static_cast<const ET*>(prob->expn);
    }
    if (fam) pw2pot_sym_block<N, true, NZ, ET>(npw, nd, tabS, tasks + tix, part, expn, wms, ks, kd, zo, prob, sm);
    else pw2pot_sym_block<N, false, NZ, ET>(npw, nd, tabS, tasks + tix, part, expn, wms, ks, kd, zo, prob, sm);
}

// f(std::integral_constant<int, n>) for the orders covered here
template <class F>
bool for_order(int n, F&& f) {
    switch (n) {
        case 4: f(std::integral_constant<int, 4>{}); return true;
        case 5: f(std::integral_constant<int, 5>{}); return true;
        case 6: f(std::integral_constant<int, 6>{}); return true;
        case 7: f(std::integral_constant<int, 7>{}); return true;
        case 8: f(std::integral_constant<int, 8>{}); return true;
        case 9: f(std::integral_constant<int, 9>{}); return true;
        case 10: f(std::integral_constant<int, 10>{}); return true;
        case 11: f(std::integral_constant<int, 11>{}); return true;
        case 12: f(std::integral_constant<int, 12>{}); return true;
        case 13: f(std::integral_constant<int, 13>{}); return true;
        case 14: f(std::integral_constant<int, 14>{}); return true;
        case 15: f(std::integral_constant<int, 15>{}); return true;
        case 16: f(std::integral_constant<int, 16>{}); return true;
        default: return false;
    }
}
// FP32 expansions exist at the orders with reduced-precision kernels
constexpr bool has_fp32(int n) { return n == 8 || n == 12 || n == 16; }

template <int N, int NZ>
void launch_sym5_z(const Geom& g, const DevTables& t, int nfam, int nown, const SymTask* tasks, const double2* expn,
                   const ZGroups& zg, hipStream_t s, const Multi& mu) {
    size_t lds = 0;
    // a batch class holds smaller plane-wave counts too
    for (int p = mu.pp ? 1 : t.npw; p <= t.npw; ++p) {
        if (nfam) lds = std::max(lds, sym5_lds_entries(p, 2 * sym5_nx<N, true>(), 2 * sym_pairs<N, true>()));
        if (nown) lds = std::max(lds, sym5_lds_entries(p, 2 * sym5_nx<N, false>(), 2 * sym_pairs<N, false>()));
    }
    lds *= sizeof(double2);
    const dim3 grid((unsigned)(zg.n * (nfam * sym5_parts<N, true>() + nown * sym5_parts<N, false>())));
    const dim3 block(kThreads);
    if constexpr (has_fp32(N)) {
        if (t.expn_f32) {
            hipLaunchKernelGGL((k_pw2pot_sym<N, NZ, float2>), grid, block, lds, s, g.nd, t.pw2potS, t.npw, tasks, nfam,
                               nown, reinterpret_cast<const float2*>(expn), t.wms, t.pw2potS_ks, zg, mu);
            return;
        }
    }
    hipLaunchKernelGGL((k_pw2pot_sym<N, NZ, double2>), grid, block, lds, s, g.nd, t.pw2potS, t.npw, tasks, nfam, nown,
                       expn, t.wms, t.pw2potS_ks, zg, mu);
}

template <int N>
void launch_sym5(const Geom& g, const DevTables& t, int nfam, int nown, const SymTask* tasks, const double2* expn,
                 const ZGroups& zg, hipStream_t s, const Multi& mu) {
    const int nz = zg.zo[0].nz;
    if (nz == 1) {
        launch_sym5_z<N, 1>(g, t, nfam, nown, tasks, expn, zg, s, mu);
    } else if (nz == 2) {
        launch_sym5_z<N, 2>(g, t, nfam, nown, tasks, expn, zg, s, mu);
    } else if constexpr (N <= 12) {
        launch_sym5_z<N, 3>(g, t, nfam, nown, tasks, expn, zg, s, mu);
    } else {
        // the sums of three z kinds exceed the registers
        launch_sym5_z<N, 2>(g, t, nfam, nown, tasks, expn, z_kinds(zg, 0, 2), s, mu);
        launch_sym5_z<N, 1>(g, t, nfam, nown, tasks, expn, z_kinds(zg, 2, 1), s, mu);
    }
}

// ---------------------------------------------------------------- STEP 1
// k3 slabs per round: one row (slab, x node) of the y stage per lane
template <int N, bool FAM>
constexpr int sym1_slabs() { return 32 / sym_pairs<N, FAM>() > 8 ? 8 : 32 / sym_pairs<N, FAM>(); }
// double2 entries of the block's LDS: sH [slab][y node][x node] and sF
// [slab][x node][k2] (odd row length) share it
template <int N, bool FAM>
size_t sym1_lds_entries(int npw) {
    const size_t nod = 2 * sym_pairs<N, FAM>(), sr = sym1_slabs<N, FAM>();
    return std::max(sr * nod * nod, sr * nod * (size_t)(npw | 1));
}

// One block: part kp of kparts of the k3 rounds of one task, whose expansion
// (the leaf's, or the parent's with the STEP 2 shift folded in) it overwrites.
// Per round of SR slabs:
//   z: thread = (x node, y node) column, its values folded over the z pairs
//      (kept in registers for all rounds where a thread has one column);
//   y: lane = (slab, x node), folded over the y pairs, k2 pairs dealt to the
//      waves;
//   x: lane = (slab, k2) column, folded over the x pairs, k1 pairs split over
//      the waves that share a batch of columns; both frequencies of a pair
//      are stored as they are formed.
// Bound by the expansion writes and each round's latency (norder 8, npw 28,
// 8382 leaves: 68 us for 210 MB, 171 us with the plain complex products;
// norder 12, npw 60, 4250 leaves: 314 us for 1 GB, 639 before).  The part
// count fills the device four blocks deep at most: each part reads the
// values again.
template <int N, bool FAM, typename ET>
__device__ __forceinline__ void p2pw_sym_block(int npw, int nd, const double2* __restrict__ tabS,
                                               const SymTask* __restrict__ T, int kp, int kparts,
                                               const double* __restrict__ fvals, ET* __restrict__ expn,
                                               double2* __restrict__ sm) {
    constexpr int NP = sym_pairs<N, FAM>(), NOD = 2 * NP, COLS = NOD * NOD, SR = sym1_slabs<N, FAM>();
    constexpr int NC = (COLS + kThreads - 1) / kThreads;   // columns per thread
    constexpr int ZG = COLS <= 64 ? 4 : (COLS <= 128 ? 2 : 1);   // thread groups sharing the slabs
    constexpr int V = FAM ? 1 : 0;
    static_assert(SR * NOD <= 64, "one y row per lane");
    const int nh = (npw + 1) >> 1;
    const int nround = (nh + SR - 1) / SR;
    const int rb = SR * (kp * nround / kparts), re = min(nh, SR * ((kp + 1) * nround / kparts));
    if (rb >= re) return;
    const int PW = npw | 1;
    const long long row3 = (3LL * __builtin_amdgcn_readfirstlane(T->lev) + V) * ((long long)npw * N);
    const CTab2 U = ctab(tabS) + row3;   // U[k*N + pair]
    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lane = tid & 63;
    const int slot = __builtin_amdgcn_readfirstlane(T->slot);
    warm_table(U, nh * N, wave);
    // one folded z column: values of side a plus / minus those of side b
    auto fold = [&](int col, int ind, double (&fe)[NP], double (&fo)[NP]) {
        const int zx = col % NOD, zy = col / NOD;
        const int bx = zx >= NP, by = zy >= NP;
        const int px = zx - bx * NP, py = zy - by * NP;
        // the middle node of a leaf with odd n has no mirror image
        const bool on = FAM || !((bx && 2 * px + 1 == N) || (by && 2 * py + 1 == N));
        const int cxy = FAM ? bx | by << 1 : 0;
        const int ba = on ? T->box[cxy] : -1, bb = on ? T->box[FAM ? cxy | 4 : 0] : -1;
        const int node = (bx ? N - 1 - px : px) + N * (by ? N - 1 - py : py);
        const double* __restrict__ pa = fvals + ((size_t)max(ba, 0) * (N * N * N) + node) * nd + ind;
        const double* __restrict__ pb = fvals + ((size_t)max(bb, 0) * (N * N * N) + node) * nd + ind;
        const int st = N * N * nd;
        double a[NP], b[NP];
#pragma unroll
        for (int q = 0; q < NP; ++q) {
            a[q] = ba >= 0 ? gload(pa, q * st) : 0.0;
            b[q] = (bb >= 0 && (FAM || 2 * q + 1 != N)) ? gload(pb, (N - 1 - q) * st) : 0.0;
        }
#pragma unroll
        for (int q = 0; q < NP; ++q) {
            fe[q] = a[q] + b[q];
            fo[q] = a[q] - b[q];
        }
    };
    const int zgrp = ZG == 1 ? 0 : (ZG == 2 ? wave >> 1 : wave);
    const int zcol = ZG == 1 ? tid : (ZG == 2 ? (tid & 127) : lane);
    for (int ind = 0; ind < nd; ++ind) {
        ET* __restrict__ E = expn + (size_t)(slot * 2 * nd + ind) * (size_t)(nh * npw * npw);
        double fe[NP], fo[NP];
        if (NC == 1 && zcol < COLS) fold(zcol, ind, fe, fo);
        for (int r = rb; r < re; r += SR) {
            // ---- z
#pragma unroll 1
            for (int c = 0; c < NC; ++c) {
                const int col = zcol + c * kThreads;
                if (col < COLS) {
                    if (NC > 1) fold(col, ind, fe, fo);
                    for (int s = zgrp; s < SR; s += ZG) {
                        const CTab2 u = U + (long long)min(r + s, nh - 1) * N;
                        double hr = 0.0, hi = 0.0;
#pragma unroll
                        for (int q = 0; q < NP; ++q) {
                            const double2 t = u[q];
                            hr += t.x * fe[q];
                            hi += t.y * fo[q];
                        }
                        sm[s * COLS + col] = make_double2(hr, hi);
                    }
                }
            }
            __syncthreads();
            // ---- y
            {
                const int row = min(lane, SR * NOD - 1);
                const double2* __restrict__ h = sm + (row / NOD) * COLS + row % NOD;
                double2 S[NP], D[NP];
#pragma unroll
                for (int q = 0; q < NP; ++q) {
                    const double2 a = h[q * NOD], b = h[(NP + q) * NOD];
                    S[q] = cplus(a, b);
                    D[q] = cminus(a, b);
                }
                __syncthreads();   // sH is read; sF takes its place
                double2* __restrict__ o = sm + row * PW;
                for (int k = wave; k < nh; k += kThreads / 64) {
                    double2 P = make_double2(0.0, 0.0), Q = make_double2(0.0, 0.0);
#pragma unroll
                    for (int q = 0; q < NP; ++q) {
                        const double2 t = U[(long long)k * N + q];
                        P.x += t.x * S[q].x;
                        P.y += t.x * S[q].y;
                        Q.x += t.y * D[q].x;
                        Q.y += t.y * D[q].y;
                    }
                    if (lane < SR * NOD) {
                        o[npw - 1 - k] = make_double2(P.x + Q.y, P.y - Q.x);
                        o[k] = make_double2(P.x - Q.y, P.y + Q.x);
                    }
                }
            }
            __syncthreads();
            // ---- x
            {
                const int cols = min(SR, nh - r) * npw;
                const int nb = (cols + 63) >> 6;
                const int ks = nb == 1 ? 4 : (nb == 2 ? 2 : 1);   // waves per batch of columns
                const int kq = ks == 4 ? wave : (ks == 2 ? wave >> 1 : 0);
                const int ka = kq * nh / ks, kb = (kq + 1) * nh / ks;
                for (int b = ks == 4 ? 0 : (ks == 2 ? wave & 1 : wave); b < nb; b += 4 / ks) {
                    const int c = min(64 * b + lane, cols - 1);
                    const bool act = 64 * b + lane < cols;
                    const int s = c / npw, k2 = c - s * npw;
                    const double2* __restrict__ f = sm + s * NOD * PW + k2;
                    double2 S[NP], D[NP];
#pragma unroll
                    for (int q = 0; q < NP; ++q) {
                        const double2 u = f[q * PW], v = f[(NP + q) * PW];
                        S[q] = cplus(u, v);
                        D[q] = cminus(u, v);
                    }
                    // row base scalar, column offset per lane
                    const unsigned co = (unsigned)((r + s) * npw * npw + k2);
                    for (int k = ka; k < kb; ++k) {
                        double2 P = make_double2(0.0, 0.0), Q = make_double2(0.0, 0.0);
#pragma unroll
                        for (int q = 0; q < NP; ++q) {
                            const double2 t = U[(long long)k * N + q];
                            P.x += t.x * S[q].x;
                            P.y += t.x * S[q].y;
                            Q.x += t.y * D[q].x;
                            Q.y += t.y * D[q].y;
                        }
                        if (act) {
                            gstore(E + (size_t)(k * npw), co, make_double2(P.x - Q.y, P.y + Q.x));
                            if (2 * k + 1 != npw)
                                gstore(E + (size_t)((npw - 1 - k) * npw), co, make_double2(P.x + Q.y, P.y - Q.x));
                        }
                    }
                }
            }
            __syncthreads();
        }
    }
}

// The families' blocks first, then the single leaves' (see k_pw2pot_sym).
template <int N, typename ET>
__global__ void __launch_bounds__(kThreads, 2)
    k_p2pw_sym(int nd, const double2* __restrict__ tabS, int npw, const SymTask* __restrict__ tasks, int nfam,
               int nown, int kfam, int kown, const double* __restrict__ fvals, ET* __restrict__ expn, Multi mu) {
    extern __shared__ double2 sm[];
    const int b = blockIdx.x, nfb = nfam * kfam;
    const bool fam = b < nfb;
    const int lin = fam ? xcd_task(b, nfb) : xcd_task(b - nfb, nown * kown);
    const int tix = fam ? lin / kfam : nfam + lin / kown, kp = fam ? lin % kfam : lin % kown;
    if (mu.pp) {
        const ProbPtrs* prob = mu.pp + mu.tprob[tix];
        npw = prob->g.npw;
        tabS = prob->p2pwS;
        fvals = prob->fvals;
        expn = static_cast<ET*>(prob->expn);
    }
    if (fam) p2pw_sym_block<N, true, ET>(npw, nd, tabS, tasks + tix, kp, kfam, fvals, expn, sm);
    else p2pw_sym_block<N, false, ET>(npw, nd, tabS, tasks + tix, kp, kown, fvals, expn, sm);
}

template <int N>
void launch_sym1(const Geom& g, const DevTables& t, int nfam, int nown, const SymTask* tasks, const double* fvals,
                 double2* expn, hipStream_t s, const Multi& mu) {
    size_t lds = 0;
    if (nfam) lds = std::max(lds, sym1_lds_entries<N, true>(t.npw));
    if (nown) lds = std::max(lds, sym1_lds_entries<N, false>(t.npw));
    lds *= sizeof(double2);
    // parts of the rounds per task: enough blocks to fill the device
    const auto parts = [&](int n, int sr) {
        const int rounds = ((t.npw + 1) / 2 + sr - 1) / sr;
        return n > 0 ? std::max(1, std::min(std::min(4, rounds), 4096 / n)) : 1;
    };
    const int kf = parts(nfam, sym1_slabs<N, true>()), ko = parts(nown, sym1_slabs<N, false>());
    const dim3 grid((unsigned)(nfam * kf + nown * ko)), block(kThreads);
    if constexpr (has_fp32(N)) {
        if (t.expn_f32) {
            hipLaunchKernelGGL((k_p2pw_sym<N, float2>), grid, block, lds, s, g.nd, t.p2pwS, t.npw, tasks, nfam, nown,
                               kf, ko, fvals, reinterpret_cast<float2*>(expn), mu);
            return;
        }
    }
    hipLaunchKernelGGL((k_p2pw_sym<N, double2>), grid, block, lds, s, g.nd, t.p2pwS, t.npw, tasks, nfam, nown, kf, ko,
                       fvals, expn, mu);
}

}  // namespace

bool launch_p2pw_sym(const Geom& g, const DevTables& t, int nfam, int nown, const SymTask* tasks, const double* fvals,
                     double2* expn, hipStream_t s, const Multi& mu) {
    if (g.ndim != 3 || nfam + nown <= 0) return false;
    return for_order(t.n, [&](auto n) { launch_sym1<n()>(g, t, nfam, nown, tasks, fvals, expn, s, mu); });
}

bool launch_pw2pot_sym(const Geom& g, const DevTables& t, int nfam, int nown, const SymTask* tasks,
                       const double2* expn, const ZGroups& zg, hipStream_t s, const Multi& mu) {
    if (g.ndim != 3 || zg.n < 1 || zg.n > kMaxZGroups || zg.zo[0].nz < 1 || zg.zo[0].nz > 3 || nfam + nown <= 0)
        return false;
    return for_order(t.n, [&](auto n) { launch_sym5<n()>(g, t, nfam, nown, tasks, expn, zg, s, mu); });
}

bool sym3_supported(const Geom& g, const DevTables& t) {
    if (g.ndim != 3) return false;
    size_t need = 0;
    const bool ok = for_order(t.n, [&](auto n) {
        constexpr int N = n();
        for (int p = 1; p <= t.npw; ++p)
            need = std::max({need, sym1_lds_entries<N, true>(p), sym1_lds_entries<N, false>(p),
                             sym5_lds_entries(p, 2 * sym5_nx<N, true>(), 2 * sym_pairs<N, true>()),
                             sym5_lds_entries(p, 2 * sym5_nx<N, false>(), 2 * sym_pairs<N, false>())});
    });
    return ok && need * sizeof(double2) <= t.lds_limit;
}

}  // namespace fgt
