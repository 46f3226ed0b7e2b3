// kernels_pw3.hip -- 3-D plane-wave kernels with a reduced-precision x stage
// on the matrix cores (gfx950); the FP64 forms are in kernels_sym3.hip.
//
// STEP 1 (values -> PW, g3d_tens_prod_to_pw, bfgt_pwrouts.f:153-222) and
// STEP 5 (PW -> values, g3d_pw2pot, bfgt_pwrouts.f:719-790) for norder
// N in {8, 12, 16}, one 256-thread block (4 waves) per task (a leaf, a
// quarter of a parent with leaf children, or one side of such a family).
//
// The y and z stages run on the FP64 VALU with a wave-uniform 1-D table
// operand (its address depends only on loop counters and the wave index, so
// it comes from the scalar cache into SGPRs); LDS only carries the transposes
// between stages.  The half (z) axis is processed in rounds of slabs.
#include "kernels.h"

#include <algorithm>
#include <cstdlib>
#include <type_traits>

namespace fgt {

int lowp_stages(int prec);

namespace {

__device__ __forceinline__ double2 zfma(double2 t, double2 f, double2 c) {
    return make_double2(c.x + t.x * f.x - t.y * f.y, c.y + t.x * f.y + t.y * f.x);
}

// Reduced-precision matrix-core contractions (mixed-precision forms).  A
// complex product C[row][kk] = sum_k A[row][k] U[kk][k] becomes a real GEMM
// with columns (kk, part) -- part 0 the real, 1 the imaginary part of C:
//   C = Ar * B1 + Ai * B2,  B1[k][(kk,0|1)] = (Ur | Ui),  B2 = (-Ui | Ur),
// so a column tile of 16 holds 8 complex outputs (norder 8 fills one tile).
// FP32: v_mfma_f32_16x16x4_f32, A lane l = A[l%16][l/16], B lane l =
// B[l/16][l%16], result lane l element v = D[4(l/16)+v][l%16].
// BF16 hi/lo: v_mfma_f32_16x16x32_bf16 with K = (k, part) interleaved, lane l
// holding K entries 8(l/16)..8(l/16)+7 of row (A) or column (B) l%16; each
// FP32 operand x is split as hi = bf16(x), lo = bf16(x - hi) and the product
// is Ah Bh + Ah Bl + Al Bh (relative error ~1e-5), accumulated in FP32.
typedef float flt4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf8 __attribute__((ext_vector_type(8)));
// largest plane-wave count of the reduced-precision stages (row tiles of 16)
constexpr int kLowpMaxPw = 80;

__device__ __forceinline__ flt4 mfma32(float a, float b, flt4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ flt4 mfma_bf(bf8 a, bf8 b, flt4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}
// hi/lo split of eight FP32 values
__device__ __forceinline__ void split_bf(const float (&x)[8], bf8& hi, bf8& lo) {
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const __bf16 h = (__bf16)x[i];
        hi[i] = h;
        lo[i] = (__bf16)(x[i] - (float)h);
    }
}
// B entry of column c = (kk, part) for K entry (k, kpart) of the expanded
// real GEMM, from the complex table value u = U[kk][k]
__device__ __forceinline__ float bcol(double2 u, int part, int kpart) {
    return kpart == 0 ? (part == 0 ? (float)u.x : (float)u.y) : (part == 0 ? -(float)u.y : (float)u.x);
}

// x stage of STEP 1 in reduced precision on the matrix cores (one wave):
//   E[k1][k2] = sum_{kk < KN} B(kk, k1) A(k2, kk)
// rows k2 (tiles of 16), columns (k1, part) interleaved (a tile holds 8
// frequencies k1), K = kk (KN complex terms: N values of m1, or 2N for the
// fused form's two x signs).  fa(k2, kk) / fb(kk, k1) return the FP64
// operands (stage buffer in LDS / 1-D table); fw(k2, k1, v) stores one
// complex result.  The wave does column tiles ct0, ct0 + ctstep, ... in
// pairs (FP32: a last tile without a partner alone).  Each lane trades its part
// with the neighbouring lane (the other part of the same output) so every
// result is written once as a complex pair: part-0 lanes write rows v = 0, 1
// of their four, part-1 lanes 2, 3.
constexpr int kLowpColGroup = 2;

// BF16: the table operands of every column tile and K step, split, in LDS once
// per task: tab[(ct * KB + st) * 64 + lane], KB = K steps of 16 (prepared per
// row tile and round, with the result's part picked by an index through
// scratch, k_p2pw3 over the 779 leaves of an order-8 problem took 39 us, per
// column group and round 30; in LDS STEP 1 beside the near field 66 -> 41 us)
struct BfPair { bf8 hi, lo; };
__host__ __device__ constexpr size_t x1_tab_entries(int KN, int npw) {
    return (size_t)((2 * npw + 15) >> 4) * ((KN + 15) / 16) * 64;
}
template <int KN, class FB>
__device__ __forceinline__ void x1_fill(BfPair* __restrict__ tab, int npw, int tid, FB fb) {
    constexpr int KB = (KN + 15) / 16;
    const int n = (int)x1_tab_entries(KN, npw);
    for (int o = tid; o < n; o += 256) {
        const int lane = o & 63, st = (o >> 6) % KB, c = 16 * ((o >> 6) / KB) + (lane & 15), lq = lane >> 4;
        const bool cval = (c >> 1) < npw;
        float bx[8];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int kk = 16 * st + 4 * lq + j;
            const bool ok = kk < KN && cval;
            const double2 u = fb(kk < KN ? kk : KN - 1, cval ? (c >> 1) : 0);
            bx[2 * j] = ok ? bcol(u, c & 1, 0) : 0.f;
            bx[2 * j + 1] = ok ? bcol(u, c & 1, 1) : 0.f;
        }
        split_bf(bx, tab[o].hi, tab[o].lo);
    }
}

// column tiles c0, c0 + ctstep, ... (CG of them, all below CT)
template <int KN, int XS, int CG, class FA, class FB, class FW>
__device__ __forceinline__ void x1_lowp_group(int npw, int lane, int c0, int ctstep, FA fa, FB fb, FW fw,
                                              const BfPair* __restrict__ tab) {
    const int MT = (npw + 15) >> 4;
    const int CT = (2 * npw + 15) >> 4;
    const int li = lane & 15, lq = lane >> 4;
    {
        int k1c[CG], part[CG];
        bool cval[CG];
#pragma unroll
        for (int gi = 0; gi < CG; ++gi) {
            const int c = 16 * (c0 + gi * ctstep) + li;
            part[gi] = c & 1;
            cval[gi] = (c >> 1) < npw && c0 + gi * ctstep < CT;
            k1c[gi] = cval[gi] ? (c >> 1) : 0;
        }
        // FP32: the column tiles' table operands of every K step, read once for
        // all row tiles
        constexpr int KS = (KN + 3) / 4, KB = (KN + 15) / 16;
        float tb1[CG][XS == 2 ? KS : 1], tb2[CG][XS == 2 ? KS : 1];
        if constexpr (XS == 2) {
#pragma unroll
            for (int st = 0; st < KS; ++st) {
                const int kk = 4 * st + lq;
                const bool kv = kk < KN;
                const int kkc = kv ? kk : KN - 1;
#pragma unroll
                for (int gi = 0; gi < CG; ++gi) {
                    const double2 u = fb(kkc, k1c[gi]);
                    const bool ok = kv && cval[gi];
                    tb1[gi][st] = ok ? bcol(u, part[gi], 0) : 0.f;
                    tb2[gi][st] = ok ? bcol(u, part[gi], 1) : 0.f;
                }
            }
        }
        // one row tile at a time (few live accumulators, high occupancy)
        for (int mt = 0; mt < MT; ++mt) {
            // two accumulator chains per tile (real / imaginary A parts, or
            // hi*hi / the correction products) so dependent MFMAs interleave
            flt4 acc[CG][2];
#pragma unroll
            for (int gi = 0; gi < CG; ++gi) acc[gi][0] = acc[gi][1] = flt4{0.f, 0.f, 0.f, 0.f};
            const int k2r = min(16 * mt + li, npw - 1);
            if constexpr (XS == 2) {
#pragma unroll
                for (int st = 0; st < KS; ++st) {
                    const int kk = 4 * st + lq;
                    const double2 a = fa(k2r, kk < KN ? kk : KN - 1);
#pragma unroll
                    for (int gi = 0; gi < CG; ++gi) {
                        acc[gi][0] = mfma32((float)a.x, tb1[gi][st], acc[gi][0]);
                        acc[gi][1] = mfma32((float)a.y, tb2[gi][st], acc[gi][1]);
                    }
                }
            } else {
#pragma unroll
                for (int st = 0; st < KB; ++st) {
                    float ax[8];
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        const int kk = 16 * st + 4 * lq + j;
                        const double2 a = fa(k2r, kk < KN ? kk : KN - 1);
                        ax[2 * j] = (float)a.x;
                        ax[2 * j + 1] = (float)a.y;
                    }
                    bf8 ah, al;
                    split_bf(ax, ah, al);
#pragma unroll
                    for (int gi = 0; gi < CG; ++gi) {
                        // (a group's tile past the last is discarded)
                        const BfPair* __restrict__ b = tab + (min(c0 + gi * ctstep, CT - 1) * KB + st) * 64 + lane;
                        const bf8 bh = b->hi, bl = b->lo;
                        acc[gi][0] = mfma_bf(ah, bh, acc[gi][0]);
                        acc[gi][1] = mfma_bf(ah, bl, acc[gi][1]);
                        acc[gi][1] = mfma_bf(al, bh, acc[gi][1]);
                    }
                }
            }
            // lane holds rows 16 mt + 4 lq + v of column (k1, part)
#pragma unroll
            for (int gi = 0; gi < CG; ++gi) {
                float o[4], q[4];
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    o[v] = acc[gi][0][v] + acc[gi][1][v];
                    q[v] = __shfl_xor(o[v], 1);
                }
                if (cval[gi])
#pragma unroll
                    for (int h = 0; h < 2; ++h) {
                        // (selects of fixed elements: an index by lane goes through scratch)
                        const int k2 = 16 * mt + 4 * lq + 2 * part[gi] + h;
                        const float2 v = part[gi] ? make_float2(q[2 + h], o[2 + h]) : make_float2(o[h], q[h]);
                        if (k2 < npw) fw(k2, k1c[gi], v);
                    }
            }
        }
    }
}

template <int KN, int XS, class FA, class FB, class FW>
__device__ __forceinline__ void x1_lowp(int npw, int lane, int ct0, int ctstep, FA fa, FB fb, FW fw,
                                        const BfPair* __restrict__ tab) {
    constexpr int CG = kLowpColGroup;
    const int CT = (2 * npw + 15) >> 4;
    for (int c0 = ct0; c0 < CT; c0 += CG * ctstep) {
        // (BF16: the one-tile form's registers would cost a block per CU)
        if (XS != 2 || c0 + (CG - 1) * ctstep < CT)
            x1_lowp_group<KN, XS, CG>(npw, lane, c0, ctstep, fa, fb, fw, tab);
        else
            x1_lowp_group<KN, XS, 1>(npw, lane, c0, ctstep, fa, fb, fw, tab);
    }
}

// ---------------------------------------------------------------- STEP 1
// LDS: sff [m2][s][m1] (N*4*N complex) and sff2 [s][m1][k2] (4*N*npw
// complex) share one buffer: the y stage reads its sff column into registers
// and passes a barrier before writing sff2 (more blocks fit on a CU).
__host__ __device__ constexpr size_t p2pw3_entries(int n, int npw) {
    return 4 * (size_t)n * (npw > n ? npw : n);
}
template <int N, int XS>
__global__ void __launch_bounds__(256) k_p2pw3(Geom g, const double2* __restrict__ tab_a, int npw,
                                              const int* __restrict__ box, const int* __restrict__ lev,
                                              const int* __restrict__ slot,
                                              const double* __restrict__ fvals_a,
                                              float2* __restrict__ expn_a, Multi mu) {
    extern __shared__ double2 sm[];
    double2* sff = sm;
    double2* sff2 = sm;
    const int task = blockIdx.x;
    const double2* __restrict__ tab = tab_a;
    const double* __restrict__ fvals = fvals_a;
    float2* __restrict__ expn = expn_a;
    if (mu.pp) {
        const ProbPtrs& q = mu.pp[mu.tprob[task]];
        g = q.g;
        npw = q.g.npw;
        tab = q.p2pw;
        fvals = q.fvals;
        expn = static_cast<float2*>(q.expn);
    }
    const int b = box[task], l = lev[task], sl = slot[task];
    const CTab2 T = ctab(tab) + (long long)l * npw * N;   // T[k][m]
    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lane = tid & 63;
    const int nh = g.pz, nd = g.nd;
    BfPair* xtab = reinterpret_cast<BfPair*>(sm + p2pw3_entries(N, npw));
    if (XS == 3) x1_fill<N>(xtab, npw, tid, [&](int m1, int k1) { return T[k1 * N + m1]; });   // (a barrier follows)
    for (int ind = 0; ind < nd; ++ind) {
        double fr[N];
        if (tid < N * N) {
#pragma unroll
            for (int m3 = 0; m3 < N; ++m3)
                fr[m3] = fvals[((size_t)b * g.npbox + tid + N * N * m3) * nd + ind];
        }
        float2* __restrict__ E = expn + ((size_t)sl * 2 * nd + ind) * g.nexp;
        for (int r = 0; r < nh; r += 4) {
            // z: ff[s][m1][m2] = sum_m3 T[k3_s][m3] f[m1,m2,m3], thread = (m1,m2)
            if (tid < N * N) {
                const int m1 = tid % N, m2 = tid / N;
#pragma unroll
                for (int s = 0; s < 4; ++s) {
                    const int k3 = r + s;
                    if (k3 < nh) {
                        double ar = 0.0, ai = 0.0;
#pragma unroll
                        for (int m3 = 0; m3 < N; ++m3) {
                            const double2 t = T[k3 * N + m3];
                            ar += t.x * fr[m3];
                            ai += t.y * fr[m3];
                        }
                        sff[(m2 * 4 + s) * N + m1] = make_double2(ar, ai);
                    }
                }
            }
            __syncthreads();
            // y: ff2[s][m1][k2] = sum_m2 T[k2][m2] ff[s][m1][m2]; lane = (m1, s), wave strides k2
            {
                const int m1 = lane & 15, s = lane >> 4;
                const bool act = (m1 < N) && (r + s < nh);
                double2 ff[N];
#pragma unroll
                for (int m2 = 0; m2 < N; ++m2)
                    ff[m2] = act ? sff[(m2 * 4 + s) * N + m1] : make_double2(0.0, 0.0);
                __syncthreads();   // sff consumed; sff2 (same memory) may be written
                for (int k2 = wave; k2 < npw; k2 += 4) {
                    // two partial sums: four independent FMA chains
                    double2 a0 = make_double2(0.0, 0.0), a1 = make_double2(0.0, 0.0);
#pragma unroll
                    for (int m2 = 0; m2 < N; m2 += 2) {
                        a0 = zfma(T[k2 * N + m2], ff[m2], a0);
                        a1 = zfma(T[k2 * N + m2 + 1], ff[m2 + 1], a1);
                    }
                    if (act) sff2[(s * N + m1) * npw + k2] = make_double2(a0.x + a1.x, a0.y + a1.y);
                }
            }
            __syncthreads();
            // x: E[k3][k1][k2] = sum_m1 T[k1][m1] ff2[s][m1][k2]; wave = slab, lane = k2
            {
                const int k3 = r + wave;
                if (k3 < nh) {
                    float2* __restrict__ Ek = E + (size_t)k3 * npw * npw;
                    x1_lowp<N, XS>(
                        npw, lane, 0, 1,
                        [&](int k2, int m1) { return sff2[(wave * N + m1) * npw + k2]; },
                        [&](int m1, int k1) { return T[k1 * N + m1]; },
                        [&](int k2, int k1, float2 v) { Ek[(size_t)k1 * npw + k2] = v; }, xtab);
                }
            }
            __syncthreads();
        }
    }
}

// ------------------------------------------------------- STEP 1 + STEP 2
// Parent expansion formed directly from its leaf children (STEP 1 of each
// leaf child and its STEP 2 shift into the parent, fused):
//   mp_P = sum_c (Tx o w_x^{c}) (Ty o w_y^{c}) (Tz o w_z^{c}) f_c
// with w^{c} the child->parent merge phase of each axis.  Children are grouped
// by their x and y signs: the z stage runs per child and is summed into four
// (sx,sy) groups, the y stage runs per x sign over both y signs, the x stage
// runs once over both x signs (K = 2N) -- four times fewer x-stage flops than
// eight separate leaf transforms, and no leaf expansion reaches HBM.
// tabS[l][v][k][m]: child-level table, v = 0 plain, 1 = + phase, 2 = conjugate.
// Task lists: kids (up to 8 leaf children), ksg (merge sign bits, x = bit0).
// Rounds of SR slabs.  SR = 2: wave w takes slab w & 1 and half (w >> 1) of
// the x stage's k1 range; the y stage's lanes are (m1 < 16, slab, sx).  SR = 4
// (norder 8, matrix-core x stage, npw <= 48): wave w takes slab w, and the y
// stage's 64 lanes are (m1 < 8, slab, sx) with none idle.
// Each parent is split over kFusedParts blocks, each taking a contiguous run
// of rounds (the parts of one parent are adjacent in launch order and land on
// one XCD, so the children's values they all read meet in its L2).
// LDS: sH [4 groups][SR slabs][m2][m1] and sF [2 sx][SR slabs][m1][npw]
// share one buffer: sH is fully read into registers before sF is written.
constexpr int kFusedParts = 4;

__host__ __device__ constexpr size_t p2pwF3_entries(int n, int sr, int npw) {
    return 2 * (size_t)sr * n * (npw > 2 * n ? npw : 2 * n);
}
template <int N, int XS, int SR = 2>
__global__ void __launch_bounds__(256) k_p2pwF3(Geom g, const double2* __restrict__ tabS_a, int npw,
                                               const int* __restrict__ plev, const int* __restrict__ pslot,
                                               const int* __restrict__ kids, const int* __restrict__ ksg,
                                               const double* __restrict__ fvals_a,
                                               float2* __restrict__ expn_a, Multi mu) {
    static_assert(SR == 2 || (SR == 4 && N == 8 && XS >= 2), "four-slab rounds: norder 8, matrix-core x stage");
    extern __shared__ double2 sm[];
    double2* sH = sm;                     // 4*SR*N*N
    double2* sF = sm;                     // 2*SR*N*npw (aliases sH)
    const int lin = xcd_task(blockIdx.x, gridDim.x);
    const int task = lin / kFusedParts, part = lin % kFusedParts;
    const double2* __restrict__ tabS = tabS_a;
    const double* __restrict__ fvals = fvals_a;
    float2* __restrict__ expn = expn_a;
    if (mu.pp) {
        const ProbPtrs& q = mu.pp[mu.tprob[task]];
        g = q.g;
        npw = q.g.npw;
        tabS = q.p2pwS;
        fvals = q.fvals;
        expn = static_cast<float2*>(q.expn);
    }
    const int l = plev[task] + 1, sl = pslot[task];
    const int per = npw * N;
    const int base0 = __builtin_amdgcn_readfirstlane(3 * l * per);
    const CTab2 T = ctab(tabS);
    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lane = tid & 63;
    const int nh = g.pz, nd = g.nd;
    int nk = 0;
    while (nk < 8 && kids[8 * task + nk] >= 0) ++nk;   // leaf children are packed first
    const int nround = (nh + SR - 1) / SR;
    const int rb = SR * (part * nround / kFusedParts), re = SR * ((part + 1) * nround / kFusedParts);
    BfPair* xtab = reinterpret_cast<BfPair*>(sm + p2pwF3_entries(N, SR, npw));
    if (XS == 3) {   // (barriers follow)
        const CTab2 Txp = T + base0 + 1 * per;
        const CTab2 Txm = T + base0 + 2 * per;
        x1_fill<2 * N>(xtab, npw, tid,
                       [&](int kk, int k1) { return kk >= N ? Txm[k1 * N + kk - N] : Txp[k1 * N + kk]; });
    }
    for (int ind = 0; ind < nd; ++ind) {
        float2* __restrict__ E = expn + ((size_t)sl * 2 * nd + ind) * g.nexp;
        // norder 8: one wave per group g = (sx, sy) of children; the values
        // of its (up to two) children -- the z sign tells them apart -- stay
        // in registers for every round
        double frg[2][N];
        bool has0 = false, has1 = false;
        if constexpr (N * N == 64) {
            for (int c = 0; c < nk; ++c) {
                const int sg = ksg[8 * task + c];
                if ((sg & 3) != wave) continue;
                const int b = kids[8 * task + c];
                const double* __restrict__ fb = fvals + ((size_t)b * g.npbox + lane) * nd + ind;
                if ((sg >> 2) & 1) {
                    has1 = true;
#pragma unroll
                    for (int m3 = 0; m3 < N; ++m3) frg[1][m3] = fb[(size_t)N * N * m3 * nd];
                } else {
                    has0 = true;
#pragma unroll
                    for (int m3 = 0; m3 < N; ++m3) frg[0][m3] = fb[(size_t)N * N * m3 * nd];
                }
            }
        }
        for (int r = rb; r < re; r += SR) {
            // z: H[g][s][m2][m1] = sum_{c in g} sum_m3 Tz_c[k3_s][m3] f_c[m1,m2,m3]
            if constexpr (N * N == 64) {
                const int q = wave;
                double2 H[SR];
#pragma unroll
                for (int s = 0; s < SR; ++s) H[s] = make_double2(0.0, 0.0);
#pragma unroll
                for (int z = 0; z < 2; ++z) {
                    if (!(z ? has1 : has0)) continue;
                    const CTab2 Tz = T + base0 + (1 + z) * per;
#pragma unroll
                    for (int s = 0; s < SR; ++s) {
                        const int k3 = min(r + s, nh - 1);
                        double ar = 0.0, ai = 0.0;
#pragma unroll
                        for (int m3 = 0; m3 < N; ++m3) {
                            const double2 t = Tz[k3 * N + m3];
                            ar += t.x * frg[z][m3];
                            ai += t.y * frg[z][m3];
                        }
                        H[s].x += ar;
                        H[s].y += ai;
                    }
                }
#pragma unroll
                for (int s = 0; s < SR; ++s) sH[((q * SR + s) * N) * N + lane] = H[s];
            } else if (tid < N * N) {
                double2 H[4][2];
#pragma unroll
                for (int q = 0; q < 4; ++q) H[q][0] = H[q][1] = make_double2(0.0, 0.0);
                for (int c = 0; c < nk; ++c) {
                    const int b = kids[8 * task + c], sg = ksg[8 * task + c];
                    const int vz = 1 + ((sg >> 2) & 1);
                    const CTab2 Tz = T + base0 + vz * per;
                    double fr[N];
#pragma unroll
                    for (int m3 = 0; m3 < N; ++m3)
                        fr[m3] = fvals[((size_t)b * g.npbox + tid + N * N * m3) * nd + ind];
                    const int q = sg & 3;
#pragma unroll
                    for (int s = 0; s < 2; ++s) {
                        const int k3 = min(r + s, nh - 1);
                        double ar = 0.0, ai = 0.0;
#pragma unroll
                        for (int m3 = 0; m3 < N; ++m3) {
                            const double2 t = Tz[k3 * N + m3];
                            ar += t.x * fr[m3];
                            ai += t.y * fr[m3];
                        }
                        // q is the same for all lanes (uniform per child)
#pragma unroll
                        for (int qq = 0; qq < 4; ++qq)
                            if (qq == q) { H[qq][s].x += ar; H[qq][s].y += ai; }
                    }
                }
#pragma unroll
                for (int q = 0; q < 4; ++q)
#pragma unroll
                    for (int s = 0; s < 2; ++s) sH[((q * 2 + s) * N) * N + tid] = H[q][s];
            }
            __syncthreads();
            // y: F[sx][s][m1][k2] = sum_sy sum_m2 Ty^{sy}[k2][m2] H[(sx,sy)][s][m2][m1]
            // lane = (m1 < MS, s < SR, sx in 0..1), wave strides k2
            {
                constexpr int MS = 32 / SR;
                const int m1 = lane % MS, s = (lane / MS) % SR, sx = lane / (MS * SR);
                const bool act = (m1 < N) && (r + s < nh);
                double2 hp[N], hm[N];
#pragma unroll
                for (int m2 = 0; m2 < N; ++m2) {
                    hp[m2] = act ? sH[(((sx + 0) * SR + s) * N + m2) * N + m1] : make_double2(0.0, 0.0);
                    hm[m2] = act ? sH[(((sx + 2) * SR + s) * N + m2) * N + m1] : make_double2(0.0, 0.0);
                }
                const CTab2 Typ = T + base0 + 1 * per;
                const CTab2 Tym = T + base0 + 2 * per;
                __syncthreads();   // sH consumed; sF (same memory) may be written
                for (int k2 = wave; k2 < npw; k2 += 4) {
                    double2 a0 = make_double2(0.0, 0.0), a1 = make_double2(0.0, 0.0);
#pragma unroll
                    for (int m2 = 0; m2 < N; ++m2) {
                        a0 = zfma(Typ[k2 * N + m2], hp[m2], a0);
                        a1 = zfma(Tym[k2 * N + m2], hm[m2], a1);
                    }
                    if (act) sF[((sx * SR + s) * N + m1) * npw + k2] = make_double2(a0.x + a1.x, a0.y + a1.y);
                }
            }
            __syncthreads();
            // x: E[k3][k1][k2] = sum_sx sum_m1 Tx^{sx}[k1][m1] F[sx][s][m1][k2]
            {
                // K = (sx, m1); SR = 2: the two waves of a slab take alternate
                // column tiles, SR = 4: one wave per slab takes them all
                const int s = SR == 4 ? wave : (wave & 1), hlf = SR == 4 ? 0 : wave >> 1;
                const int k3 = r + s;
                if (k3 < nh) {
                    float2* __restrict__ Ek = E + (size_t)k3 * npw * npw;
                    const CTab2 Txp = T + base0 + 1 * per;
                    const CTab2 Txm = T + base0 + 2 * per;
                    x1_lowp<2 * N, XS>(
                        npw, lane, hlf, SR == 4 ? 1 : 2,
                        [&](int k2, int kk) {
                            const int sx = kk >= N ? 1 : 0;
                            return sF[((sx * SR + s) * N + (kk - N * sx)) * npw + k2];
                        },
                        [&](int kk, int k1) { return kk >= N ? Txm[k1 * N + kk - N] : Txp[k1 * N + kk]; },
                        [&](int k2, int k1, float2 v) { Ek[(size_t)k1 * npw + k2] = v; }, xtab);
                }
            }
            __syncthreads();
        }
    }
}

// The x table of a STEP 5 task as the operands of its matrix products, in LDS
// once per task (read from memory and converted again for every row tile, the
// wait for them had set the x stage's time): XS 2 (FP32) per K step, column
// tile and lane the two parts' entries, XS 3 (BF16) the hi and lo halves of
// the lane's eight K entries.  Zero past npw and past the last column.
template <int XS> struct XEntry;
template <> struct XEntry<2> { typedef float2 type; };
template <> struct XEntry<3> { typedef BfPair type; };
template <int N, int XS> struct XTable {
    static constexpr int NT = (2 * N + 15) / 16;
    typedef typename XEntry<XS>::type E;
    static __host__ __device__ int steps(int npw) { return XS == 2 ? (npw + 3) >> 2 : (npw + 15) >> 4; }
    static __host__ __device__ size_t bytes(int npw) { return sizeof(E) * steps(npw) * NT * 64; }
    static __device__ __forceinline__ void fill(E* __restrict__ tab, const CTab2 UX, int npw, int tid) {
        const int n = steps(npw) * NT * 64;
        for (int o = tid; o < n; o += 256) {
            const int lane = o & 63, t = (o >> 6) % NT, st = (o >> 6) / NT;
            const int c = 16 * t + (lane & 15), lq = lane >> 4;
            const bool cval = c < 2 * N;
            const int part = c >= N ? 1 : 0, kk = cval ? c - N * part : 0;
            if constexpr (XS == 2) {
                const int k1 = 4 * st + lq;
                const double2 u = UX[min(k1, npw - 1) * N + kk];
                const bool ok = k1 < npw && cval;
                tab[o] = make_float2(ok ? bcol(u, part, 0) : 0.f, ok ? bcol(u, part, 1) : 0.f);
            } else {
                float bx[8];
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const int k1 = 16 * st + 4 * lq + j;
                    const double2 u = UX[min(k1, npw - 1) * N + kk];
                    const bool ok = k1 < npw && cval;
                    bx[2 * j] = ok ? bcol(u, part, 0) : 0.f;
                    bx[2 * j + 1] = ok ? bcol(u, part, 1) : 0.f;
                }
                split_bf(bx, tab[o].hi, tab[o].lo);
            }
        }
    }
};

// x stage of STEP 5 in reduced precision on the matrix cores (wave w takes
// the round's slabs w, w + 4, ... of SR):
//   ff[k2][kk1] = sum_k1 Ux[kk1][k1] E[k3][k1][k2],
// rows k2 (row tiles of 16, up to 80 frequencies), columns (kk1, part), K =
// k1.  XS 2: FP32 operands; XS 3: BF16 hi/lo operands.  The result goes to
// sff[(k2*SR + slab)*KW + (kk1 ^ (k2 & (KW-1)))], KW = 64 / SR (FP32
// complex: the two accumulator chains' FP32 sum, stored exactly), where the y
// stage reads it.  Lanes past npw read a valid duplicate row (discarded).
template <int N, int XS, int SR>
__device__ __forceinline__ void pw2pot_x_lowp(const float2* __restrict__ E,
                                              const typename XTable<N, XS>::E* __restrict__ tab, int npw, int nh,
                                              int r, int wave, int lane, float2* sff) {
    constexpr int KW = 64 / SR;
    static_assert(KW >= N, "a (k2, slab) row of sff holds the N values kk1");
    if (r + wave >= nh) return;
    constexpr int NT = XTable<N, XS>::NT;
    const int MT = (npw + 15) >> 4;
    const int li = lane & 15, lq = lane >> 4;
    int ckk[NT], cpart[NT];
    bool cval[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) {
        const int c = 16 * t + li;
        cval[t] = c < 2 * N;
        cpart[t] = c >= N ? 1 : 0;
        ckk[t] = cval[t] ? c - N * cpart[t] : 0;
    }
    float* __restrict__ sffd = reinterpret_cast<float*>(sff);
    const int ks = XTable<N, XS>::steps(npw);
    for (int sl = wave; sl < SR; sl += 4) {
        const int k3 = r + sl;
        if (k3 >= nh) break;
        const float2* __restrict__ Ek = E + (size_t)k3 * npw * npw;
        // one row tile (16 frequencies k2) at a time, two accumulator chains per
        // column tile
        for (int mt = 0; mt < MT; ++mt) {
            const int k2r = min(16 * mt + li, npw - 1);
            flt4 acc[NT][2];
#pragma unroll
            for (int t = 0; t < NT; ++t) acc[t][0] = acc[t][1] = flt4{0.f, 0.f, 0.f, 0.f};
            // K steps in chunks of KC, the next chunk's rows of E loaded (from
            // valid clamped addresses, past npw against zero table entries)
            // before this chunk's products
            constexpr int KC = XS == 2 ? 8 : 2, KE = XS == 2 ? 1 : 4;
            float2 ea[KC][KE], eb[KC][KE];
            auto load = [&](float2 (&e)[KC][KE], int st0) {
#pragma unroll
                for (int j = 0; j < KC; ++j)
#pragma unroll
                    for (int i = 0; i < KE; ++i)
                        e[j][i] = gload(Ek, (unsigned)(min(4 * KE * (st0 + j) + KE * lq + i, npw - 1) * npw + k2r));
            };
            auto apply = [&](const float2 (&e)[KC][KE], int st0) {
#pragma unroll
                for (int j = 0; j < KC; ++j) {
                    if (st0 + j >= ks) break;
                    const typename XTable<N, XS>::E* __restrict__ b = tab + (st0 + j) * NT * 64 + lane;
                    if constexpr (XS == 2) {
#pragma unroll
                        for (int t = 0; t < NT; ++t) {
                            const float2 u = b[64 * t];
                            acc[t][0] = mfma32(e[j][0].x, u.x, acc[t][0]);
                            acc[t][1] = mfma32(e[j][0].y, u.y, acc[t][1]);
                        }
                    } else {
                        // K = (k1, part): 16 frequencies per step; lane K entries 8 lq .. 8 lq + 7
                        float ax[8];
#pragma unroll
                        for (int i = 0; i < 4; ++i) {
                            ax[2 * i] = e[j][i].x;
                            ax[2 * i + 1] = e[j][i].y;
                        }
                        bf8 ah, al;
                        split_bf(ax, ah, al);
#pragma unroll
                        for (int t = 0; t < NT; ++t) {
                            const bf8 bh = b[64 * t].hi, bl = b[64 * t].lo;
                            acc[t][0] = mfma_bf(ah, bh, acc[t][0]);
                            acc[t][1] = mfma_bf(ah, bl, acc[t][1]);
                            acc[t][1] = mfma_bf(al, bh, acc[t][1]);
                        }
                    }
                }
            };
            load(ea, 0);
            for (int st = 0; st < ks; st += 2 * KC) {
                if (st + KC < ks) load(eb, st + KC);
                __builtin_amdgcn_sched_barrier(0);
                apply(ea, st);
                if (st + KC >= ks) break;
                if (st + 2 * KC < ks) load(ea, st + 2 * KC);
                __builtin_amdgcn_sched_barrier(0);
                apply(eb, st + KC);
            }
#pragma unroll
            for (int t = 0; t < NT; ++t)
                if (cval[t])
#pragma unroll
                    for (int v = 0; v < 4; ++v) {
                        const int k2 = 16 * mt + 4 * lq + v;
                        if (k2 < npw)
                            sffd[2 * ((k2 * SR + sl) * KW + (ckk[t] ^ (k2 & (KW - 1)))) + cpart[t]] =
                                acc[t][0][v] + acc[t][1][v];
                    }
        }
    }
}

// ---------------------------------------------------------------- STEP 5
// The reduced-precision form (FP32 expansions, x stage on the matrix cores;
// the FP64 form is k_pw2pot_sym).  Tables: tabS[kind][l][v][k][i] (frequency k,
// node i), v = 0 the plain PW->value table, 1 / 2 the table times the + /
// conjugate parent->child split phase (STEP 4 folded into STEP 5).
// A block evaluates one expansion at the leaf children of its box that share
// their x side (FAM; SymTask families, two blocks each, whose x contraction is
// that of the side's table) or at the leaf that holds it.
// Per round of SR k3 slabs (4; 8 for norder 8):
//   x: ff[k2][s][kk1] = sum_k1 Ux[kk1][k1] E[k3][k1][k2]   (wave = slab,
//      or slabs w and w + 4), FP32 products of FP32 or BF16 hi/lo operands;
//   y, z: FP64, through the tables' symmetries as in k_pw2pot_sym (pairs of
//      opposite frequencies and of mirror nodes, these of the two children
//      along the axis where there are two): y lane = (kk1, slab), the pairs
//      split over the waves; z thread = output column, all (or ZP) pairs of
//      every z kind in registers.
// Bound by the latencies of each round's three stages.  Order 12, npw 28, 3423
// leaves: 253 us with the plain complex y and z stages, one leaf after another,
// and the x table read per row tile; 188 with the symmetric stages, 119 with
// the x table in LDS as well.  BF16 order 8, npw 20, 1332 leaves: 51, 39, 32.
// LDS: sff [k2][s][KW] (npw*64 complex, KW = 64 / SR; the x stage's FP32
// results, held exactly), yres [s][kk1][y node] (rows padded by one), the x
// table's operands (XTable).
// NZ: output components that differ in their z kind zo.kz[q] only share the x
// and y stages.
template <int N> constexpr int mix_slabs() { return N == 8 ? 8 : 4; }
template <int N, int XS, bool FAM, int NZ>
__global__ void __launch_bounds__(256, 2) k_pw2pot3(Geom g, const double2* __restrict__ tabS, int npw,
                                                    const SymTask* __restrict__ tasks,
                                                    const float2* __restrict__ expn, size_t ks, Kinds kd, ZOut zo,
                                                    Multi mu) {
    constexpr int SR = mix_slabs<N>(), KW = 64 / SR;
    constexpr int NP = FAM ? N : N / 2, NODY = 2 * NP, COLS = N * NODY;
    constexpr int YP = (NP + 3) / 4;                                       // y pairs per wave
    constexpr int ZS = COLS <= 64 ? 4 : (COLS <= 128 ? 2 : 1);             // thread groups sharing the z pairs
    constexpr int ZP = (NP + ZS - 1) / ZS, CPT = (COLS + 255) / 256;       // pairs, columns per thread
    constexpr int V = FAM ? 1 : 0;
    extern __shared__ double2 sm[];
    float2* sff = reinterpret_cast<float2*>(sm);
    double2* yres = reinterpret_cast<double2*>(sff + (size_t)npw * 64);
    auto* xtab = reinterpret_cast<typename XTable<N, XS>::E*>(yres + SR * N * (2 * N + 1));
    const int lin = xcd_task(blockIdx.x, gridDim.x);
    const int tix = FAM ? lin >> 1 : lin, sx = FAM ? lin & 1 : 0;
    const SymTask* __restrict__ T = tasks + tix;
    const ProbPtrs* prob = nullptr;
    if (mu.pp) {
        prob = mu.pp + mu.tprob[tix];
        npw = prob->g.npw;
        tabS = prob->pw2potS;
        expn = static_cast<const float2*>(prob->expn);
    }
    if (FAM && T->box[sx] < 0 && T->box[sx | 2] < 0 && T->box[sx | 4] < 0 && T->box[sx | 6] < 0) return;
    const int nh = (npw + 1) >> 1, nd = g.nd;
    const bool odd = (npw & 1) != 0;
    const long long per = (long long)npw * N;
    const long long row3 = 3LL * __builtin_amdgcn_readfirstlane(T->lev) * per;
    const CTab2 UX = ctab(tabS) + ((long long)(kd.x * ks) + row3 + (FAM ? 1 + sx : 0) * per);
    const CTab2 UY = ctab(tabS) + ((long long)(kd.y * ks) + row3 + V * per);
    CTab2 UZ[NZ];
#pragma unroll
    for (int z = 0; z < NZ; ++z) UZ[z] = ctab(tabS) + ((long long)(zo.kz[z] * ks) + row3 + V * per);
    const double sgy = kd.y == 1 ? -1.0 : 1.0;
    const int slot = __builtin_amdgcn_readfirstlane(T->slot);
    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lane = tid & 63;
    const int kk1 = lane & (KW - 1), s = lane / KW;
    const bool yact = kk1 < N;
    const int kk1c = yact ? kk1 : N - 1;
    const int zset = ZS == 1 ? 0 : (ZS == 2 ? wave >> 1 : wave);
    const int col0 = ZS == 1 ? tid : (ZS == 2 ? (tid & 127) : lane);
    XTable<N, XS>::fill(xtab, UX, npw, tid);
    __syncthreads();
    for (int ind = 0; ind < nd; ++ind) {
        double GP[CPT][NZ][ZP], GQ[CPT][NZ][ZP];
#pragma unroll
        for (int c = 0; c < CPT; ++c)
#pragma unroll
            for (int z = 0; z < NZ; ++z)
#pragma unroll
                for (int q = 0; q < ZP; ++q) GP[c][z][q] = GQ[c][z][q] = 0.0;
        const float2* __restrict__ E = expn + (size_t)(slot * 2 * nd + nd + ind) * (size_t)(nh * npw * npw);
        for (int r = 0; r < nh; r += SR) {
            pw2pot_x_lowp<N, XS, SR>(E, xtab, npw, nh, r, wave, lane, sff);
            __syncthreads();   // (and the last round's z stage is done with yres)
            {
                double2 P[YP], Q[YP];
#pragma unroll
                for (int p = 0; p < YP; ++p) P[p] = Q[p] = make_double2(0.0, 0.0);
                // several steps' table and LDS reads together (a slab past nh
                // holds stale values, never read back)
                constexpr int YU = YP <= 2 ? 4 : 2;
                for (int k0 = 0; k0 < nh; k0 += YU) {
                    float2 a[YU], b[YU];
                    double2 t[YU][YP];
#pragma unroll
                    for (int j = 0; j < YU; ++j) {
                        const int k = min(k0 + j, nh - 1), m = npw - 1 - k;
                        a[j] = sff[(k * SR + s) * KW + (kk1c ^ (k & (KW - 1)))];
                        b[j] = sff[(m * SR + s) * KW + (kk1c ^ (m & (KW - 1)))];
#pragma unroll
                        for (int p = 0; p < YP; ++p) t[j][p] = UY[(long long)k * N + min(wave * YP + p, NP - 1)];
                    }
#pragma unroll
                    for (int j = 0; j < YU; ++j) {
                        if (k0 + j >= nh) break;
                        const double ax = a[j].x, ay = a[j].y, bx = b[j].x, by = b[j].y;
                        const bool self = odd && k0 + j == nh - 1;   // the zero frequency pairs with itself
                        const double Sx = self ? ax : ax + bx, Sy = self ? ay : ay + by, Dx = ax - bx, Dy = ay - by;
#pragma unroll
                        for (int p = 0; p < YP; ++p) {
                            P[p].x += t[j][p].x * Sx;
                            P[p].y += t[j][p].x * Sy;
                            Q[p].x += t[j][p].y * Dx;
                            Q[p].y += t[j][p].y * Dy;
                        }
                    }
                }
                if (yact && r + s < nh) {
                    double2* __restrict__ o = yres + (s * N + kk1) * (NODY + 1);
#pragma unroll
                    for (int p = 0; p < YP; ++p) {
                        const int q = wave * YP + p;
                        if (q < NP) {
                            o[q] = make_double2(P[p].x - Q[p].y, P[p].y + Q[p].x);
                            o[NP + q] = make_double2(sgy * (P[p].x + Q[p].y), sgy * (P[p].y - Q[p].x));
                        }
                    }
                }
            }
            __syncthreads();
            const int ns = min(SR, nh - r);
#pragma unroll
            for (int c = 0; c < CPT; ++c) {
                const int col = col0 + 256 * c;
                if (col < COLS) {
                    const double2* __restrict__ yc = yres + (col % N) * (NODY + 1) + col / N;
                    constexpr int ZU = NZ * ZP <= 4 ? 4 : (NZ * ZP <= 8 ? 2 : 1);
                    for (int s0 = 0; s0 < ns; s0 += ZU) {
                        double2 yv[ZU], t[ZU][NZ][ZP];
#pragma unroll
                        for (int j = 0; j < ZU; ++j) {
                            const int s2 = min(s0 + j, ns - 1);
                            yv[j] = yc[s2 * N * (NODY + 1)];
#pragma unroll
                            for (int z = 0; z < NZ; ++z)
#pragma unroll
                                for (int q = 0; q < ZP; ++q)
                                    t[j][z][q] = UZ[z][(long long)(r + s2) * N + min(zset * ZP + q, NP - 1)];
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
                                    GP[c][z][q] += t[j][z][q].x * yr;
                                    GQ[c][z][q] += t[j][z][q].y * yi;
                                }
                        }
                    }
                }
            }
        }
        // node pair -> (child bit, node): side b is the mirrored node, of the
        // other child (FAM) or of the same leaf
#pragma unroll
        for (int c = 0; c < CPT; ++c) {
            const int col = col0 + 256 * c;
            if (col >= COLS) continue;
            const int ix = col % N, zy = col / N, by = zy >= NP, py = zy - by * NP, iy = by ? N - 1 - py : py;
            const int cxy = FAM ? sx | by << 1 : 0;
            const int ba = T->box[cxy], bb = T->box[FAM ? cxy | 4 : 0];
            int node = ix + N * iy;
            // opaque: the output addresses are formed here, not held through
            // the whole task
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
                             2.0 * (GP[c][z][q] - GQ[c][z][q]));
                    if (bb >= 0)
                        gadd(op + (size_t)bb * (N * N * N) * ns, (node + N * N * (N - 1 - pz)) * ns,
                             sgz * (GP[c][z][q] + GQ[c][z][q]));
                }
            }
        }
    }
}

// slabs per round of the fused STEP 1 kernel: four for norder 8 while sF (8 n npw complex) leaves room for three blocks
// per CU, else two
int p2pwF3_slabs(int n, int npw) { return n == 8 && npw <= 48 ? 4 : 2; }

// LDS of the STEP 1 kernels, the BF16 table included: the launchers and
// pw2pot_3d_supported, which answers before anything is launched, ask the same
size_t p2pw3_lds(int n, int npw, int prec) {
    return sizeof(double2) * p2pw3_entries(n, npw) + (prec == 2 ? sizeof(BfPair) * x1_tab_entries(n, npw) : 0);
}
size_t p2pwF3_lds(int n, int npw, int prec) {
    return sizeof(double2) * p2pwF3_entries(n, p2pwF3_slabs(n, npw), npw) +
           (prec == 2 ? sizeof(BfPair) * x1_tab_entries(2 * n, npw) : 0);
}

template <int N>
bool try_p2pw3(const Geom& g, const DevTables& t, int ntask, const int* box, const int* lev, const int* slot,
               const double* fvals, double2* expn, hipStream_t s, size_t lds_limit, const Multi& mu) {
    const size_t lds = p2pw3_lds(N, t.npw, t.prec);
    if (lds > lds_limit) return false;
    float2* e32 = reinterpret_cast<float2*>(expn);
    if (t.prec == 2)
        hipLaunchKernelGGL((k_p2pw3<N, 3>), dim3(ntask), dim3(256), lds, s, g, t.p2pw, t.npw, box, lev, slot,
                           fvals, e32, mu);
    else
        hipLaunchKernelGGL((k_p2pw3<N, 2>), dim3(ntask), dim3(256), lds, s, g, t.p2pw, t.npw, box, lev, slot,
                           fvals, e32, mu);
    return true;
}

size_t pw2pot3_lds(int n, int npw, int xs) {
    // sff, yres (a family's, the larger), x table
    const size_t sr = n == 8 ? 8 : 4;
    const size_t tab = n == 8 ? (xs == 2 ? XTable<8, 2>::bytes(npw) : XTable<8, 3>::bytes(npw))
                              : (xs == 2 ? XTable<16, 2>::bytes(npw) : XTable<16, 3>::bytes(npw));
    return sizeof(float2) * (size_t)npw * 64 + sizeof(double2) * sr * n * (2 * (size_t)n + 1) + tab;
}

template <int N, int XS, bool FAM, int NZ>
void launch_pw2pot3_z(const Geom& g, const DevTables& t, int nblk, const SymTask* tasks, const double2* expn,
                      Kinds kd, const ZOut& zo, hipStream_t s, size_t lds, const Multi& mu) {
    hipLaunchKernelGGL((k_pw2pot3<N, XS, FAM, NZ>), dim3(nblk), dim3(256), lds, s, g, t.pw2potS, t.npw, tasks,
                       reinterpret_cast<const float2*>(expn), t.pw2potS_ks, kd, zo, mu);
}

// components zo.kz[a..a+nz) of zo as a group of their own
ZOut zsub(const ZOut& zo, int a, int nz) {
    ZOut r{};
    r.nz = nz;
    for (int q = 0; q < nz; ++q) {
        r.kz[q] = zo.kz[a + q];
        r.od[q] = zo.od[a + q];
    }
    return r;
}

// nblk blocks of one kind of task: the z kinds together, or (a family's z
// sums of several kinds exceed the registers above norder 8) one after another
template <int N, int XS, bool FAM>
void launch_pw2pot3_kind(const Geom& g, const DevTables& t, int nblk, const SymTask* tasks, const double2* expn,
                         Kinds kd, const ZOut& zo, hipStream_t s, size_t lds, const Multi& mu) {
    if (nblk <= 0) return;
    if constexpr (!FAM || N == 8) {
        switch (zo.nz) {
            case 3: launch_pw2pot3_z<N, XS, FAM, 3>(g, t, nblk, tasks, expn, kd, zo, s, lds, mu); return;
            case 2: launch_pw2pot3_z<N, XS, FAM, 2>(g, t, nblk, tasks, expn, kd, zo, s, lds, mu); return;
            default: launch_pw2pot3_z<N, XS, FAM, 1>(g, t, nblk, tasks, expn, kd, zo, s, lds, mu); return;
        }
    } else {
        for (int q = 0; q < zo.nz; ++q)
            launch_pw2pot3_z<N, XS, FAM, 1>(g, t, nblk, tasks, expn, kd, zsub(zo, q, 1), s, lds, mu);
    }
}

template <int N, int XS>
void launch_pw2pot3_typed(const Geom& g, const DevTables& t, int nfam, int nown, const SymTask* tasks,
                          const double2* expn, Kinds kd, const ZOut& zo, hipStream_t s, size_t lds,
                          const Multi& mu) {
    launch_pw2pot3_kind<N, XS, true>(g, t, 2 * nfam, tasks, expn, kd, zo, s, lds, mu);
    Multi m1 = mu;
    if (m1.tprob) m1.tprob += nfam;
    launch_pw2pot3_kind<N, XS, false>(g, t, nown, tasks + nfam, expn, kd, zo, s, lds, m1);
}

template <int N>
bool try_pw2pot3(const Geom& g, const DevTables& t, int nfam, int nown, const SymTask* tasks,
                 const double2* expn, Kinds kd, const ZOut& zo, hipStream_t s, size_t lds_limit, const Multi& mu) {
    const size_t lds = pw2pot3_lds(N, t.npw, t.prec == 2 ? 3 : 2);
    if (lds > lds_limit || nfam > 0x3fffffff) return false;
    // BF16 hi/lo, or FP32
    if (t.prec == 2) launch_pw2pot3_typed<N, 3>(g, t, nfam, nown, tasks, expn, kd, zo, s, lds, mu);
    else launch_pw2pot3_typed<N, 2>(g, t, nfam, nown, tasks, expn, kd, zo, s, lds, mu);
    return true;
}

template <int N>
void launch_p2pwF3_typed(const Geom& g, const DevTables& t, unsigned nblk, size_t lds, const int* plev,
                         const int* pslot, const int* kids, const int* ksg, const double* fvals, double2* expn,
                         hipStream_t s, const Multi& mu) {
    float2* e32 = reinterpret_cast<float2*>(expn);
    if constexpr (N == 8) {
        if (p2pwF3_slabs(N, t.npw) == 4) {
            if (t.prec == 2)
                hipLaunchKernelGGL((k_p2pwF3<N, 3, 4>), dim3(nblk), dim3(256), lds, s, g, t.p2pwS, t.npw, plev,
                                   pslot, kids, ksg, fvals, e32, mu);
            else
                hipLaunchKernelGGL((k_p2pwF3<N, 2, 4>), dim3(nblk), dim3(256), lds, s, g, t.p2pwS, t.npw, plev,
                                   pslot, kids, ksg, fvals, e32, mu);
            return;
        }
    }
    if (t.prec == 2)
        hipLaunchKernelGGL((k_p2pwF3<N, 3>), dim3(nblk), dim3(256), lds, s, g, t.p2pwS, t.npw, plev, pslot,
                           kids, ksg, fvals, e32, mu);
    else
        hipLaunchKernelGGL((k_p2pwF3<N, 2>), dim3(nblk), dim3(256), lds, s, g, t.p2pwS, t.npw, plev, pslot,
                           kids, ksg, fvals, e32, mu);
}

}  // namespace

// FGT_LOWP_STAGES (bit 0 STEP 1, bit 1 STEP 5): which stages run their x
// contraction on the reduced-precision matrix cores in the FP32 / BF16
// modes; the others keep the FP64 VALU contraction on FP32 expansions
// (tuning and comparison runs).
int lowp_stages(int prec) {
    static const int v = [] {
        const char* e = std::getenv("FGT_LOWP_STAGES");
        return e ? (std::atoi(e) & 3) : -1;
    }();
    // defaults by mode: FP32 runs STEP 5's x stage on the matrix cores, BF16
    // hi/lo both steps'.  The FP64 arithmetic of the symmetric kernels on FP32
    // expansions is a quarter of the plain products, and at order 8 with up to
    // 48 plane waves (35 problems in one launch) the faster one: STEP 1 2.0 ms
    // against 4.4, STEP 5 2.7 against 3.7.  A batch's autotuner times both; a
    // single solver keeps the arithmetic that its mode names.
    return v >= 0 ? v : (prec == 2 ? 3 : 2);
}

bool p2pw_lowp(const DevTables& t) {
    if (t.prec < 1 || t.npw > kLowpMaxPw) return false;
    return t.xs1 >= 0 ? t.xs1 == 2 : (lowp_stages(t.prec) & 1) != 0;
}

bool pw2pot_lowp(const DevTables& t) {
    if (t.prec < 1 || t.npw > kLowpMaxPw) return false;
    return t.xs5 >= 0 ? t.xs5 == 2 : (lowp_stages(t.prec) & 2) != 0;
}

bool launch_p2pw_3d(const Geom& g, const DevTables& t, int ntask, const int* box, const int* lev,
                    const int* slot, const double* fvals, double2* expn, hipStream_t s, size_t lds_limit,
                    const Multi& mu) {
    if (g.ndim != 3 || ntask <= 0) return false;
    switch (t.n) {
        case 8: return try_p2pw3<8>(g, t, ntask, box, lev, slot, fvals, expn, s, lds_limit, mu);
        case 12: return try_p2pw3<12>(g, t, ntask, box, lev, slot, fvals, expn, s, lds_limit, mu);
        case 16: return try_p2pw3<16>(g, t, ntask, box, lev, slot, fvals, expn, s, lds_limit, mu);
        default: return false;
    }
}

bool p2pw_fused_3d(const Geom& g, const DevTables& t, int ntask, const int* plev, const int* pslot,
                   const int* kids, const int* ksg, const double* fvals, double2* expn, hipStream_t s,
                   const Multi& mu) {
    if (g.ndim != 3 || ntask <= 0) return ntask <= 0;
    const int N = t.n;
    const size_t lds = p2pwF3_lds(N, t.npw, t.prec);
    if (lds > t.lds_limit) return false;
    if ((long long)ntask * kFusedParts > 0x7fffffffLL) return false;
    const unsigned nblk = (unsigned)(ntask * kFusedParts);
    switch (N) {
        case 8: launch_p2pwF3_typed<8>(g, t, nblk, lds, plev, pslot, kids, ksg, fvals, expn, s, mu); return true;
        case 12: launch_p2pwF3_typed<12>(g, t, nblk, lds, plev, pslot, kids, ksg, fvals, expn, s, mu); return true;
        case 16: launch_p2pwF3_typed<16>(g, t, nblk, lds, plev, pslot, kids, ksg, fvals, expn, s, mu); return true;
        default: return false;
    }
}

bool pw2pot_3d_supported(const Geom& g, const DevTables& t) {
    if (g.ndim != 3 || (t.n != 8 && t.n != 12 && t.n != 16)) return false;
    size_t need = std::max(pw2pot3_lds(t.n, t.npw, 2), pw2pot3_lds(t.n, t.npw, 3));
    // (beyond kLowpMaxPw both steps stay in FP64 arithmetic)
    if (t.npw <= kLowpMaxPw)
        for (int prec = 1; prec <= 2; ++prec)
            need = std::max({need, p2pw3_lds(t.n, t.npw, prec), p2pwF3_lds(t.n, t.npw, prec)});
    return need <= t.lds_limit;
}

bool launch_pw2pot_3d_z(const Geom& g, const DevTables& t, int nfam, int nown, const SymTask* tasks,
                        const double2* expn, Kinds kd, const ZOut& zo, hipStream_t s, size_t lds_limit,
                        const Multi& mu) {
    if (g.ndim != 3 || nfam + nown <= 0 || zo.nz < 1 || zo.nz > 3) return false;
    switch (t.n) {
        case 8: return try_pw2pot3<8>(g, t, nfam, nown, tasks, expn, kd, zo, s, lds_limit, mu);
        case 12: return try_pw2pot3<12>(g, t, nfam, nown, tasks, expn, kd, zo, s, lds_limit, mu);
        case 16: return try_pw2pot3<16>(g, t, nfam, nown, tasks, expn, kd, zo, s, lds_limit, mu);
        default: return false;
    }
}

}  // namespace fgt
