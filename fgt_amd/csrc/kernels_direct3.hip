// kernels_direct3.hip -- 3-D near-field (STEP 6) kernel for gfx950 (FP64).
//
// Replaces the per-pair banded contraction of g3d_tens_prod_to_potloc_fast
// (src/bfgt/bfgt_local.f:1322-1618) summed over a target's list-1 sources
// (boxfgt.f:904-928).  Sources of one target are pre-sorted on the host by
// their (z, x, y) table slots; since the near-field operator is the
// separable product A_z (x) A_x (x) A_y, sources that share the x and z
// tables are summed after their y contraction, and x-results that share the
// z table are summed before it:
//     pot += sum_z A_z ( sum_{x | z} A_x ( sum_{y | x,z} A_y f_s ) )
// which needs one y contraction per source, one x contraction per (x,z)
// group and one z contraction per z group.  y goes first because the values'
// fastest index then stays a row index of the product: neighbouring lanes
// load neighbouring values (with x first every lane of a load fell into a
// cache line of its own, and the L1 bounded the kernel).
//
// The contractions run on the FP64 matrix cores as 4x4x4 products (four
// independent blocks per instruction).  On this card they reach the FP64
// peak from one dependent chain (77 of 78.6 TFLOP/s; v_fma_f64 61 with four
// waves per SIMD) and take the table as a per-lane operand: with the table in
// SGPRs, each loaded double served one multiply-add of a wave, and the scalar
// cache bounded the kernel at a third of the peak.  Measured (alone, then
// beside STEP 1): order 16, 60255 pairs 460 -> 357 us, 45 % of the FP64 peak (the
// table and output latencies at each z group are left); order 12 Hessian,
// 4774 pairs 620 -> 187 us; order 8 gradient, 21347 pairs 228 -> 112 us.
#include <cstdlib>

#include "kernels.h"

namespace fgt {

namespace {

// Task order: runs of eight consecutive targets per XCD (neighbours of one
// problem, whose list-1 sources overlap, read them through one L2) or the
// launch order.  Batches take the runs (their many small near-field-only
// problems: 1.1-1.8 vs 4.4 ms for a norder-16 class), single problems the
// launch order (0.71 vs 0.88 ms on a norder-16 periodic problem);
// FGT_DIRECT_RUNS=0/1 forces one.
int direct_runs(const Multi& mu) {
    static const int v = [] {
        const char* e = std::getenv("FGT_DIRECT_RUNS");
        return e ? std::atoi(e) : -1;
    }();
    return v >= 0 ? v : (mu.pp ? 1 : 0);
}

// A target's source entries, staged in LDS kChunk at a time: read back at a
// wave-uniform address they keep the vector-memory counter for the values
// and tables alone (read from global memory between the products, every step
// waited for all loads in flight).  z group g of the chunk goes to team
// g % TEAMS; a chunk's last entry closes its groups.  (The lists of list 1 are
// one chunk: a leaf has at most 26 colleagues, each a leaf or its 8 children,
// itself, and 27 colleagues of its parent, 236 entries.)
// flags per entry: bit0 = last of its (x,z) group, bit1 = last of its z group.
constexpr int kChunk = 256;
template <int TEAMS>
struct Entries {
    int2 e[TEAMS][kChunk];   // source box; slot codes | flags << 24
    int n[TEAMS];
};
struct Entry {
    int src, code;
    __device__ __forceinline__ int x() const { return code & 255; }
    __device__ __forceinline__ int y() const { return (code >> 8) & 255; }
    __device__ __forceinline__ int z() const { return (code >> 16) & 255; }
    __device__ __forceinline__ bool xz_end() const { return (code >> 24) & 1; }
    __device__ __forceinline__ bool z_end() const { return (code >> 25) & 1; }
};
__device__ __forceinline__ Entry uniform(int2 v) {
    return Entry{__builtin_amdgcn_readfirstlane(v.x), __builtin_amdgcn_readfirstlane(v.y)};
}
// What one lane of a wave wrote to LDS and another reads after: the wave's LDS
// accesses complete in program order, so only the compiler has to keep it.  The
// barrier alone stops the scheduler, not the passes that move memory accesses.
__device__ __forceinline__ void wave_lds_exchange() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront", "local");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront", "local");
}

// entries [j0, j0 + n), n <= kChunk, by the block's first wave; the caller's
// barrier follows
template <int TEAMS>
__device__ __forceinline__ void stage_entries(Entries<TEAMS>& en, const int* __restrict__ src,
                                              const int* __restrict__ code, const int* __restrict__ flags, int j0,
                                              int n, int lane) {
    int cnt[TEAMS], g0 = 0;
#pragma unroll
    for (int t = 0; t < TEAMS; ++t) cnt[t] = 0;
    for (int q = 0; q < n; q += 64) {
        const int j = q + lane;
        const bool on = j < n;
        const int fl = on ? (j == n - 1 ? 3 : flags[j0 + j]) : 0;
        const int2 v = on ? make_int2(src[j0 + j], code[j0 + j] | fl << 24) : make_int2(0, 0);
        const unsigned long long before = (1ull << lane) - 1;
        const unsigned long long m = __ballot(fl & 2);
        const int team = TEAMS == 1 ? 0 : (g0 + __popcll(m & before)) % TEAMS;
#pragma unroll
        for (int t = 0; t < TEAMS; ++t) {
            const unsigned long long mt = __ballot(on && team == t);
            if (on && team == t) en.e[t][cnt[t] + __popcll(mt & before)] = v;
            cnt[t] += __popcll(mt);
        }
        g0 += __popcll(m);
    }
#pragma unroll
    for (int t = 0; t < TEAMS; ++t)
        if (lane == 0) en.n[t] = cnt[t];
}

// Runs a team's entries: the operands of the next entry load (always, past
// the end the last entry's again, so every path waits with exactly one set in
// flight) during the products of this one.  OP: an entry's operands; load(e,
// op), step(e, op).
template <class OP, class L, class S>
__device__ __forceinline__ void run_entries(const int2* list, int n, L&& load, S&& step) {
    if (n <= 0) return;
    OP a, b;
    Entry ea = uniform(list[0]), eb = ea;
    load(ea, a);
    int2 nx = list[min(1, n - 1)];   // the entry after the one being loaded
    for (int q = 0; q < n; q += 2) {
        eb = uniform(nx);
        load(eb, b);
        nx = list[min(q + 2, n - 1)];
        __builtin_amdgcn_sched_barrier(0);
        step(ea, a);
        __builtin_amdgcn_sched_barrier(0);
        if (q + 1 >= n) break;
        ea = uniform(nx);
        load(ea, a);
        nx = list[min(q + 3, n - 1)];
        __builtin_amdgcn_sched_barrier(0);
        step(eb, b);
        __builtin_amdgcn_sched_barrier(0);
    }
}

// ------------------------------------------------------------ orders to 12
// v_mfma_f64_4x4x4_4b (lane = 16 k + 4 b + i, block b): operands A[i][k],
// B[k][i], result D[k][i].

// T[r][h] = P[(4 h + k) * N + 4 r + i], zero past n: one 1-D table (stored
// [source node][target node]) as the operand of its contraction.  P is
// wave-uniform and the lane offset 32-bit (one address register, the rest
// immediate offsets).
template <int N, int NB>
__device__ __forceinline__ void load_table(const double* __restrict__ P, int i, int k, double (&T)[NB][NB]) {
#pragma unroll
    for (int r = 0; r < NB; ++r)
#pragma unroll
        for (int h = 0; h < NB; ++h) {
            const int j = 4 * h + k, row = 4 * r + i;
            if (N % 4 == 0) {
                T[r][h] = gload(P, j * N + row);
            } else {
                const double v = gload(P, min(j, N - 1) * N + min(row, N - 1));
                T[r][h] = row < N && j < N ? v : 0.0;
            }
        }
}

template <int N> constexpr int direct3_nb() { return (N + 3) / 4; }
// a team's exchange buffer [z][y][x] (doubles): odd rows and planes of 4
// mod 16 put the sixteen lanes of a write into different banks
template <int N> constexpr int direct3_row() { return 4 * direct3_nb<N>() + 1; }
template <int N> constexpr int direct3_plane() {
    return (4 * direct3_nb<N>() * direct3_row<N>() + 11) / 16 * 16 + 4;
}
template <int N> constexpr int direct3_buf() { return 4 * direct3_nb<N>() * direct3_plane<N>(); }

// One block per target: TEAMS teams of W waves, each team taking every
// TEAMS-th z group.  Wave w of a team holds the z slabs j3 = 4 (w S + s) + b,
// s < S = NB / W, of the source values and of the y and x sums, where the
// result of one contraction is the operand of the next as it stands; the z
// contraction takes the x sums through LDS, the wave its rows k2 of the same
// blocks.  A team of one wave (orders to 8) needs no barrier for that.
// nls table slots per level, slot codes 8 bits per axis.
// NZ output components that differ only in their z kind (ZOut) share the x
// and y sums.
template <int N> constexpr int direct3_waves() { return direct3_nb<N>() <= 2 ? 1 : direct3_nb<N>(); }
// three teams where a team is one wave: one per z offset of same-level
// neighbours, so a target's list takes a third of the time (one team measured
// the same on lists that fill the device)
template <int N> constexpr int direct3_teams() { return direct3_waves<N>() == 1 ? 3 : 1; }

template <int N, int NZ>
__global__ void __launch_bounds__(64 * direct3_waves<N>() * direct3_teams<N>())
    k_direct3(int nd, const double* __restrict__ loctab, int nls, const int* __restrict__ tgt,
              const int* __restrict__ lev, const int* __restrict__ off, const int* __restrict__ src,
              const int* __restrict__ code, const int* __restrict__ flags, const double* __restrict__ fvals,
              size_t ks, ZGroups zg, int ntask, Multi mu, int runs) {
    constexpr int NB = direct3_nb<N>(), W = direct3_waves<N>(), TEAMS = direct3_teams<N>(), S = NB / W;
    constexpr int NN = N * N, NPB = N * N * N;
    constexpr int ROW = direct3_row<N>(), PLANE = direct3_plane<N>();
    static_assert(W == 1 || TEAMS == 1, "the teams of a block share its barriers");
    __shared__ double s_buf[TEAMS][direct3_buf<N>()];   // exchange [j3][k2][k1]
    __shared__ Entries<TEAMS> en;
    // blocks of one group after another's
    const int grp = blockIdx.x / ntask, bt = blockIdx.x - grp * ntask;
    const int task = runs ? xcd_run_task<8>(bt, ntask) : bt;
    const Kinds kd = zg.kd[grp];
    const ZOut& zo = zg.zo[grp];
    const ProbPtrs* prob = nullptr;
    if (mu.pp) {
        prob = mu.pp + mu.tprob[task];
        loctab = prob->loctab;
        fvals = prob->fvals;
    }
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int team = wave / W, w = wave % W;
    const int i = lane & 3, b = (lane >> 2) & 3, k = lane >> 4;
    const int tb = tgt[task], l = lev[task];
    const int j0 = off[task], j1 = off[task + 1];
    // table kind per axis (value / first / second derivative): stride ks
    const double* __restrict__ tabx = loctab + (kd.x * ks + (size_t)l * nls * NN);
    const double* __restrict__ taby = loctab + (kd.y * ks + (size_t)l * nls * NN);
    double* __restrict__ buf = s_buf[team];
    struct Op {
        double F[S][NB][NB], T[NB][NB];
    };
    for (int ind = 0; ind < nd; ++ind) {
        double Z[NZ][S][NB][NB];
#pragma unroll
        for (int c = 0; c < NZ; ++c)
#pragma unroll
            for (int s = 0; s < S; ++s)
#pragma unroll
                for (int m = 0; m < NB; ++m)
#pragma unroll
                    for (int r = 0; r < NB; ++r) Z[c][s][m][r] = 0.0;
        double Y[S][NB][NB], X[S][NB][NB];
#pragma unroll
        for (int s = 0; s < S; ++s)
#pragma unroll
            for (int m = 0; m < NB; ++m)
#pragma unroll
                for (int r = 0; r < NB; ++r) Y[s][m][r] = X[s][m][r] = 0.0;
        auto load = [&](Entry e, Op& op) {
            const double* __restrict__ f = fvals + (size_t)e.src * NPB * nd + ind;
            // lane (i = j1, k = j2), slab j3; past n: a valid value, zeroed
#pragma unroll
            for (int s = 0; s < S; ++s)
#pragma unroll
                for (int m = 0; m < NB; ++m)
#pragma unroll
                    for (int h = 0; h < NB; ++h) {
                        const int jx = 4 * m + i, jy = 4 * h + k, jz = 4 * (w * S + s) + b;
                        if (N % 4 == 0) {
                            op.F[s][m][h] = gload(f, (NN * jz + N * jy + jx) * nd);
                        } else {
                            const double v =
                                gload(f, (NN * min(jz, N - 1) + N * min(jy, N - 1) + min(jx, N - 1)) * nd);
                            op.F[s][m][h] = jx < N && jy < N && jz < N ? v : 0.0;
                        }
                    }
            load_table<N, NB>(taby + e.y() * NN, i, k, op.T);
        };
        auto step = [&](Entry e, Op& op) {
            // y: Y[j1][k2] += sum_j2 f[j1][j2] Ay[k2][j2]
#pragma unroll
            for (int h = 0; h < NB; ++h)
#pragma unroll
                for (int r = 0; r < NB; ++r)
#pragma unroll
                    for (int s = 0; s < S; ++s)
#pragma unroll
                        for (int m = 0; m < NB; ++m)
                            Y[s][m][r] =
                                __builtin_amdgcn_mfma_f64_4x4x4f64(op.F[s][m][h], op.T[r][h], Y[s][m][r], 0, 0, 0);
            if (!e.xz_end()) return;
            // x: X[k1][k2] += sum_j1 Ax[k1][j1] Y[j1][k2]
            double U[NB][NB];   // (prefetched too it took a third of the registers and gained nothing)
            load_table<N, NB>(tabx + e.x() * NN, i, k, U);
#pragma unroll
            for (int h = 0; h < NB; ++h)
#pragma unroll
                for (int r = 0; r < NB; ++r)
#pragma unroll
                    for (int s = 0; s < S; ++s)
#pragma unroll
                        for (int m = 0; m < NB; ++m)
                            X[s][m][r] =
                                __builtin_amdgcn_mfma_f64_4x4x4f64(U[m][h], Y[s][h][r], X[s][m][r], 0, 0, 0);
#pragma unroll
            for (int s = 0; s < S; ++s)
#pragma unroll
                for (int m = 0; m < NB; ++m)
#pragma unroll
                    for (int r = 0; r < NB; ++r) Y[s][m][r] = 0.0;
            if (!e.z_end()) return;
            // lane: k1 = 4 m + k, k2 = 4 r + i, slab j3
#pragma unroll
            for (int s = 0; s < S; ++s)
#pragma unroll
                for (int m = 0; m < NB; ++m)
#pragma unroll
                    for (int r = 0; r < NB; ++r) {
                        buf[(4 * (w * S + s) + b) * PLANE + (4 * r + i) * ROW + 4 * m + k] = X[s][m][r];
                        X[s][m][r] = 0.0;
                    }
            if (W > 1) __syncthreads();
            else wave_lds_exchange();
            // z: Z[k3][k1] += sum_j3 Az[k3][j3] X[j3][k1], rows k2
            double V[S][NB][NB];
#pragma unroll
            for (int s = 0; s < S; ++s)
#pragma unroll
                for (int h = 0; h < NB; ++h)
#pragma unroll
                    for (int r = 0; r < NB; ++r)
                        V[s][h][r] = buf[(4 * h + k) * PLANE + (4 * (w * S + s) + b) * ROW + 4 * r + i];
#pragma unroll
            for (int c = 0; c < NZ; ++c) {
                double A[NB][NB];
                load_table<N, NB>(loctab + (zo.kz[c] * ks + ((size_t)l * nls + e.z()) * NN), i, k, A);
#pragma unroll
                for (int h = 0; h < NB; ++h)
#pragma unroll
                    for (int r = 0; r < NB; ++r)
#pragma unroll
                        for (int s = 0; s < S; ++s)
#pragma unroll
                            for (int m = 0; m < NB; ++m)
                                Z[c][s][m][r] =
                                    __builtin_amdgcn_mfma_f64_4x4x4f64(A[m][h], V[s][h][r], Z[c][s][m][r], 0, 0, 0);
            }
            if (W > 1) __syncthreads();   // the x sums are read
            else wave_lds_exchange();
        };
        for (int c0 = j0; c0 < j1; c0 += kChunk) {
            if (ind == 0 || j1 - j0 > kChunk) {
                __syncthreads();
                if (wave == 0) stage_entries<TEAMS>(en, src, code, flags, c0, min(kChunk, j1 - c0), lane);
                __syncthreads();
            }
            run_entries<Op>(en.e[team], __builtin_amdgcn_readfirstlane(en.n[team]), load, step);
        }
        // lane: k3 = 4 m + k, k1 = 4 r + i, rows k2; the teams' sums go to
        // the first team in order
#pragma unroll
        for (int c = 0; c < NZ; ++c) {
            if (TEAMS > 1) {
                __syncthreads();
                if (team > 0) {
#pragma unroll
                    for (int s = 0; s < S; ++s)
#pragma unroll
                        for (int m = 0; m < NB; ++m)
#pragma unroll
                            for (int r = 0; r < NB; ++r)
                                buf[(4 * m + k) * PLANE + (4 * (w * S + s) + b) * ROW + 4 * r + i] = Z[c][s][m][r];
                }
                __syncthreads();
            }
            if (team == 0) {
                // (batches evaluate the potential only)
                double* __restrict__ o =
                    (prob ? prob->pot : zo.od[c].p) + (size_t)tb * NPB * zo.od[c].ns + zo.od[c].coff + ind;
                const int ns = zo.od[c].ns;
                int node = i + N * (4 * w * S + b) + NN * k;
                // opaque: the output addresses are formed here, not held
                // through the whole target
                asm volatile("" : "+v"(node));
#pragma unroll
                for (int s = 0; s < S; ++s)
#pragma unroll
                    for (int m = 0; m < NB; ++m)
#pragma unroll
                        for (int r = 0; r < NB; ++r) {
                            const int k1 = 4 * r + i, k2 = 4 * (w * S + s) + b, k3 = 4 * m + k;
                            double v = Z[c][s][m][r];
#pragma unroll
                            for (int t = 1; t < TEAMS; ++t) v += s_buf[t][k3 * PLANE + k2 * ROW + k1];
                            if (N % 4 == 0 || (k1 < N && k2 < N && k3 < N))
                                gadd(o, (node + 4 * r + 4 * N * s + 4 * NN * m) * ns, v);
                        }
            }
        }
        if (TEAMS > 1) __syncthreads();   // the buffers are read
    }
}

// ------------------------------------------------------------ orders 13-16
// v_mfma_f64_16x16x4 (lane = 16 k + i): operands A[i][k], B[k][i], result
// element v D[k + 4 v][i].
typedef double dbl4 __attribute__((ext_vector_type(4)));

// T[s] = P[((4 s + k) * N + i) * nd], zero where !ok or past n
template <int N>
__device__ __forceinline__ void load_tile(const double* __restrict__ P, int i, int k, bool ok, int nd,
                                          double (&T)[4]) {
#pragma unroll
    for (int s = 0; s < 4; ++s) {
        const int j = 4 * s + k;
        if (N == 16) {
            T[s] = gload(P, (j * N + i) * nd);
        } else {
            const double v = gload(P, (min(j, N - 1) * N + min(i, N - 1)) * nd);
            T[s] = ok && i < N && j < N ? v : 0.0;
        }
    }
}

// One block of four waves per target, wave w the z slabs j3 = 4 w .. 4 w + 3
// (one tile each: rows j1, columns k2), then in the z contraction the rows
// k2 = 4 w .. 4 w + 3; otherwise as k_direct3.
template <int N, int NZ>
__global__ void __launch_bounds__(256, 2)
    k_direct3w(int nd, const double* __restrict__ loctab, int nls, const int* __restrict__ tgt,
               const int* __restrict__ lev, const int* __restrict__ off, const int* __restrict__ src,
               const int* __restrict__ code, const int* __restrict__ flags, const double* __restrict__ fvals,
               size_t ks, ZGroups zg, int ntask, Multi mu, int runs) {
    constexpr int NN = N * N, NPB = N * N * N;
    constexpr int ROW = 17, PLANE = 16 * ROW;
    __shared__ double buf[16 * PLANE];   // exchange [j3][k2][k1]
    __shared__ Entries<1> en;
    // blocks of one group after another's
    const int grp = blockIdx.x / ntask, bt = blockIdx.x - grp * ntask;
    const int task = runs ? xcd_run_task<8>(bt, ntask) : bt;
    const Kinds kd = zg.kd[grp];
    const ZOut& zo = zg.zo[grp];
    const ProbPtrs* prob = nullptr;
    if (mu.pp) {
        prob = mu.pp + mu.tprob[task];
        loctab = prob->loctab;
        fvals = prob->fvals;
    }
    const int tid = threadIdx.x, lane = tid & 63;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int i = lane & 15, k = lane >> 4;
    const int tb = tgt[task], l = lev[task];
    const int j0 = off[task], j1 = off[task + 1];
    const double* __restrict__ tabx = loctab + (kd.x * ks + (size_t)l * nls * NN);
    const double* __restrict__ taby = loctab + (kd.y * ks + (size_t)l * nls * NN);
    struct Op {
        double F[4][4], T[4], U[4];
    };
    static_assert(NZ <= 2, "the sums of three z kinds exceed the registers");
    for (int ind = 0; ind < nd; ++ind) {
        dbl4 Y[4], X[4], Z[NZ][4];
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            Y[t] = X[t] = dbl4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
            for (int c = 0; c < NZ; ++c) Z[c][t] = dbl4{0.0, 0.0, 0.0, 0.0};
        }
        auto load = [&](Entry e, Op& op) {
            const double* __restrict__ f = fvals + (size_t)e.src * NPB * nd + ind;
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                const int j3 = 4 * w + t;
                load_tile<N>(f + (size_t)NN * min(j3, N - 1) * nd, i, k, j3 < N, nd, op.F[t]);
            }
            load_tile<N>(taby + e.y() * NN, i, k, true, 1, op.T);
            load_tile<N>(tabx + e.x() * NN, i, k, true, 1, op.U);
        };
        auto step = [&](Entry e, const Op& op) {
            // y: Y[j1][k2] += sum_j2 f[j1][j2] Ay[k2][j2]
#pragma unroll
            for (int s = 0; s < 4; ++s)
#pragma unroll
                for (int t = 0; t < 4; ++t)
                    Y[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(op.F[t][s], op.T[s], Y[t], 0, 0, 0);
            if (!e.xz_end()) return;
            // x: X[k1][k2] += sum_j1 Ax[k1][j1] Y[j1][k2], element s of Y: j1 = k + 4 s
#pragma unroll
            for (int s = 0; s < 4; ++s)
#pragma unroll
                for (int t = 0; t < 4; ++t)
                    X[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(op.U[s], Y[t][s], X[t], 0, 0, 0);
#pragma unroll
            for (int t = 0; t < 4; ++t) Y[t] = dbl4{0.0, 0.0, 0.0, 0.0};
            if (!e.z_end()) return;
            // lane: k1 = k + 4 v, k2 = i
#pragma unroll
            for (int t = 0; t < 4; ++t) {
#pragma unroll
                for (int v = 0; v < 4; ++v) buf[(4 * w + t) * PLANE + i * ROW + k + 4 * v] = X[t][v];
                X[t] = dbl4{0.0, 0.0, 0.0, 0.0};
            }
            __syncthreads();
            double V[4][4];
#pragma unroll
            for (int t = 0; t < 4; ++t)
#pragma unroll
                for (int s = 0; s < 4; ++s) V[t][s] = buf[(4 * s + k) * PLANE + (4 * w + t) * ROW + i];
#pragma unroll
            for (int c = 0; c < NZ; ++c) {
                // z: Z[k3][k1] += sum_j3 Az[k3][j3] X[j3][k1], rows k2
                double A[4];
                load_tile<N>(loctab + (zo.kz[c] * ks + ((size_t)l * nls + e.z()) * NN), i, k, true, 1, A);
#pragma unroll
                for (int s = 0; s < 4; ++s)
#pragma unroll
                    for (int t = 0; t < 4; ++t)
                        Z[c][t] = __builtin_amdgcn_mfma_f64_16x16x4f64(A[s], V[t][s], Z[c][t], 0, 0, 0);
            }
            __syncthreads();   // the x sums are read
        };
        for (int c0 = j0; c0 < j1; c0 += kChunk) {
            if (ind == 0 || j1 - j0 > kChunk) {
                __syncthreads();
                if (w == 0) stage_entries<1>(en, src, code, flags, c0, min(kChunk, j1 - c0), lane);
                __syncthreads();
            }
            run_entries<Op>(en.e[0], __builtin_amdgcn_readfirstlane(en.n[0]), load, step);
        }
        // lane: k3 = k + 4 v, k1 = i, rows k2 = 4 w + t (batches evaluate the
        // potential only)
#pragma unroll
        for (int c = 0; c < NZ; ++c) {
            const OutDesc& od = zo.od[c];
            double* __restrict__ o = (prob ? prob->pot : od.p) + (size_t)tb * NPB * od.ns + od.coff + ind;
            const int ns = od.ns;
            int node = i + N * (4 * w) + NN * k;
            asm volatile("" : "+v"(node));
#pragma unroll
            for (int t = 0; t < 4; ++t)
#pragma unroll
                for (int v = 0; v < 4; ++v)
                    if (N == 16 || (i < N && 4 * w + t < N && k + 4 * v < N))
                        gadd(o, (node + N * t + 4 * NN * v) * ns, Z[c][t][v]);
        }
    }
}

template <int N, int NZ>
void launch_direct3(const Geom& g, const DevTables& t, int ntask, const int* tgt, const int* lev, const int* off,
                    const int* src, const int* code, const int* flags, const double* fvals, const ZGroups& zg,
                    hipStream_t s, const Multi& mu) {
    const int runs = direct_runs(mu);
    const dim3 grid((unsigned)(ntask * zg.n));
    if constexpr (N > 12) {
        hipLaunchKernelGGL((k_direct3w<N, NZ>), grid, dim3(256), 0, s, g.nd, t.loctab, t.loc_slots, tgt, lev, off, src,
                           code, flags, fvals, t.loctab_ks, zg, ntask, mu, runs);
    } else {
        hipLaunchKernelGGL((k_direct3<N, NZ>), grid, dim3(64 * direct3_waves<N>() * direct3_teams<N>()), 0, s, g.nd,
                           t.loctab, t.loc_slots, tgt, lev, off, src, code, flags, fvals, t.loctab_ks, zg, ntask, mu,
                           runs);
    }
}

template <int N>
bool try_direct3(const Geom& g, const DevTables& t, int ntask, const int* tgt, const int* lev, const int* off,
                 const int* src, const int* code, const int* flags, const double* fvals, const ZGroups& zg,
                 hipStream_t s, const Multi& mu) {
    switch (zg.zo[0].nz) {
        case 1: launch_direct3<N, 1>(g, t, ntask, tgt, lev, off, src, code, flags, fvals, zg, s, mu); return true;
        case 2: launch_direct3<N, 2>(g, t, ntask, tgt, lev, off, src, code, flags, fvals, zg, s, mu); return true;
        case 3:
            if constexpr (N > 12) {
                // (three z kinds' sums exceed the registers)
                launch_direct3<N, 2>(g, t, ntask, tgt, lev, off, src, code, flags, fvals, z_kinds(zg, 0, 2), s, mu);
                launch_direct3<N, 1>(g, t, ntask, tgt, lev, off, src, code, flags, fvals, z_kinds(zg, 2, 1), s, mu);
            } else {
                launch_direct3<N, 3>(g, t, ntask, tgt, lev, off, src, code, flags, fvals, zg, s, mu);
            }
            return true;
        default: return false;
    }
}

}  // namespace

bool launch_direct_3d(const Geom& g, const DevTables& t, int ntask, const int* tgt, const int* lev,
                      const int* off, const int* src, const int* code, const int* flags,
                      const double* fvals, const ZGroups& zg, hipStream_t s, const Multi& mu) {
    if (!direct3_orders(g.ndim, t.n) || ntask <= 0 || !flags || zg.n < 1 || zg.n > kMaxZGroups) return false;
    if ((long long)ntask * zg.n > 0x7fffffffLL) return false;
    switch (t.n) {
        case 4: return try_direct3<4>(g, t, ntask, tgt, lev, off, src, code, flags, fvals, zg, s, mu);
        case 5: return try_direct3<5>(g, t, ntask, tgt, lev, off, src, code, flags, fvals, zg, s, mu);
        case 6: return try_direct3<6>(g, t, ntask, tgt, lev, off, src, code, flags, fvals, zg, s, mu);
        case 7: return try_direct3<7>(g, t, ntask, tgt, lev, off, src, code, flags, fvals, zg, s, mu);
        case 8: return try_direct3<8>(g, t, ntask, tgt, lev, off, src, code, flags, fvals, zg, s, mu);
        case 9: return try_direct3<9>(g, t, ntask, tgt, lev, off, src, code, flags, fvals, zg, s, mu);
        case 10: return try_direct3<10>(g, t, ntask, tgt, lev, off, src, code, flags, fvals, zg, s, mu);
        case 11: return try_direct3<11>(g, t, ntask, tgt, lev, off, src, code, flags, fvals, zg, s, mu);
        case 12: return try_direct3<12>(g, t, ntask, tgt, lev, off, src, code, flags, fvals, zg, s, mu);
        case 13: return try_direct3<13>(g, t, ntask, tgt, lev, off, src, code, flags, fvals, zg, s, mu);
        case 14: return try_direct3<14>(g, t, ntask, tgt, lev, off, src, code, flags, fvals, zg, s, mu);
        case 15: return try_direct3<15>(g, t, ntask, tgt, lev, off, src, code, flags, fvals, zg, s, mu);
        case 16: return try_direct3<16>(g, t, ntask, tgt, lev, off, src, code, flags, fvals, zg, s, mu);
        default: return false;
    }
}

}  // namespace fgt
