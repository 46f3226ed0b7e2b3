// kernels.h -- launch interface of the box-FGT HIP kernels (gfx950).
//
// Geometry is expressed with three axes (x, y, z); the plane-wave half
// spectrum always lives on z.  A 3-D problem uses (n,n,n) nodes and
// (npw,npw,nh) frequencies; a 2-D problem maps (x,y) -> (x,z) with a unit
// y axis; a 1-D problem maps x -> z.  Unit axes carry the 1x1 identity
// table and unit phases, so one set of kernels serves every dimension.
//
// Expansion layout in HBM (one "slot" = mp then loc, nd densities each):
//   E[ind][k3][k1][k2], k2 fastest  (k3 < Pz = nh, k1 < Px, k2 < Py)
#pragma once

#include <hip/hip_runtime.h>

namespace fgt {

struct Geom {
    int nd;
    int nx, ny, nz;      // nodes per axis
    int px, py, pz;      // frequencies per axis (pz = half spectrum)
    int npw;             // full 1-D frequency count (odd => zero-frequency halving)
    int npbox;           // nx*ny*nz
    long long nexp;      // px*py*pz
    int ndim;
};

#ifdef __HIPCC__
// Expansion storage: FP64 (double2) or, in the mixed-precision form, FP32
// (float2) complex numbers; the arithmetic is FP64 either way.
__device__ __forceinline__ double2 ldE(const double2& v) { return v; }
__device__ __forceinline__ double2 ldE(const float2& v) { return make_double2(v.x, v.y); }
__device__ __forceinline__ void stE(double2* p, double2 v) { *p = v; }
__device__ __forceinline__ void stE(float2* p, double2 v) { *p = make_float2((float)v.x, (float)v.y); }

// Read-only 1-D tables viewed through the constant address space: loads
// there are invariant for the kernel, so wave-uniform reads become scalar
// loads into SGPRs whether the table pointer is a kernel argument or comes
// from a per-problem descriptor in memory (where the compiler could not
// otherwise rule out a clobbering store).  CTab2: complex (double2) entries,
// CTab1: real.
typedef const double __attribute__((address_space(4))) cdouble_t;
typedef double dvec2_t __attribute__((ext_vector_type(2)));
typedef const dvec2_t __attribute__((address_space(4))) cdvec2_t;
struct CTab2 {
    cdvec2_t* p;
    __device__ __forceinline__ CTab2 operator+(long long o) const { return CTab2{p + o}; }
    __device__ __forceinline__ double2 operator[](long long i) const {
        const dvec2_t v = p[i];   // one 16-byte load
        return make_double2(v.x, v.y);
    }
};
struct CTab1 {
    cdouble_t* p;
    __device__ __forceinline__ CTab1 operator+(long long o) const { return CTab1{p + o}; }
    __device__ __forceinline__ double operator[](long long i) const { return p[i]; }
};
__device__ __forceinline__ CTab2 ctab(const double2* q) { return CTab2{(cdvec2_t*)q}; }
__device__ __forceinline__ CTab1 ctab(const double* q) { return CTab1{(cdouble_t*)q}; }

// Global memory through its own address space.  A pointer that is either a
// kernel argument or read from a per-problem descriptor is generic to the
// compiler, which then emits flat accesses: they count on the LDS counter as
// well, so every wait for one of them waits for all loads in flight.
// gload / gstore: element o of a wave-uniform base (scalar base, 32-bit lane
// offset).
typedef float fvec2_t __attribute__((ext_vector_type(2)));
#define FGT_GLOBAL __attribute__((address_space(1)))
__device__ __forceinline__ double gload(const double* p, unsigned o) {
    return ((const FGT_GLOBAL double*)p)[o];
}
__device__ __forceinline__ double2 gload(const double2* p, unsigned o) {
    const dvec2_t v = ((const FGT_GLOBAL dvec2_t*)p)[o];
    return make_double2(v.x, v.y);
}
__device__ __forceinline__ float2 gload(const float2* p, unsigned o) {
    const fvec2_t v = ((const FGT_GLOBAL fvec2_t*)p)[o];
    return make_float2(v.x, v.y);
}
__device__ __forceinline__ void gadd(double* p, unsigned o, double v) {
    FGT_GLOBAL double* q = (FGT_GLOBAL double*)p + o;
    *q += v;
}
__device__ __forceinline__ void gstore(double2* p, unsigned o, double2 v) {
    ((FGT_GLOBAL dvec2_t*)p)[o] = dvec2_t{v.x, v.y};
}
__device__ __forceinline__ void gstore(float2* p, unsigned o, double2 v) {
    ((FGT_GLOBAL fvec2_t*)p)[o] = fvec2_t{(float)v.x, (float)v.y};
}

// Workgroups are dealt to the 8 XCDs round-robin; give each XCD a contiguous
// range of tasks so that tasks sharing data (children of one parent,
// neighbouring targets, one element range of many targets) meet in the same L2.
__device__ __forceinline__ int xcd_task(int b, int nb) {
    const int x = b & 7, i = b >> 3, per = nb >> 3, rem = nb & 7;
    return x * per + min(x, rem) + i;
}
// Runs of C consecutive tasks per XCD, dealt round-robin: the XCDs work on
// the same region of the task list at any time (balanced when task costs
// drift along the list) while each run (e.g. the children of one parent)
// shares one L2.  Blocks past the last whole round keep their own index.
template <int C>
__device__ __forceinline__ int xcd_run_task(int b, int nb) {
    const int whole = nb / (8 * C) * (8 * C);
    if (b >= whole) return b;
    const int x = b & 7, i = b >> 3;
    return (i / C) * (8 * C) + x * C + (i % C);
}
#endif

// One output component of STEP 5 / STEP 6 (potential, one gradient or one
// Hessian entry): value of node `node` of box b, density ind, goes to
// p[(b*npbox + node)*ns + coff + ind] (ns = nd * components of the array).
struct OutDesc {
    double* p;
    int ns;
    int coff;
};

// Per kernel axis (x, y, z): which 1-D table kind a component uses
// (0 value, 1 first derivative, 2 second derivative).
struct Kinds {
    int x, y, z;
};

// Output components that differ only in their z table kind (up to three:
// value, first, second derivative) share one STEP 5 or STEP 6 pass: the x
// and y sums are formed once and each z kind zo.kz[q] contracts them into
// its own output zo.od[q].
struct ZOut {
    int nz;
    int kz[3];
    OutDesc od[3];
};

// Up to three such groups with equally many z kinds run in one launch (their
// blocks side by side: a group alone leaves the device idle on small trees).
constexpr int kMaxZGroups = 3;
struct ZGroups {
    int n;
    Kinds kd[kMaxZGroups];   // x and y kinds (z unused)
    ZOut zo[kMaxZGroups];    // equal nz
};
// z kinds [a, a + nz) of every group
inline ZGroups z_kinds(const ZGroups& zg, int a, int nz) {
    ZGroups r = zg;
    for (int k = 0; k < zg.n; ++k) {
        r.zo[k].nz = nz;
        for (int q = 0; q < nz; ++q) {
            r.zo[k].kz[q] = zg.zo[k].kz[a + q];
            r.zo[k].od[q] = zg.zo[k].od[a + q];
        }
    }
    return r;
}

// One task of the 3-D STEP 1 (FP64) and STEP 5 kernels: a leaf with an
// expansion of its own (box[0]), or a family, the leaf children of the box
// whose expansion is in `slot`.  A family's child c has bit a (x, y, z) set
// when it is the side whose table carries the conjugate parent-child phase
// along axis a (-1: no leaf there); lev is the leaves' level.  STEP 5 of FP64
// expansions (klev > 0): slot holds the expansion of that box's parent, still
// to be split to it with phase row klev and the signs of k_split.
struct SymTask {
    int slot, lev;
    int box[8];
    int klev = 0, sign = 0;
};

// 2-D: a leaf with an expansion (at `depth` levels below its cutoff box, whose
// expansion is in `slot`; bit i of sx / sz set when the merge phase of the
// path's level i, coarse to fine, is conjugated along that axis), and a group
// of consecutive leaves of one cutoff box, summed into expansion `slot`.
struct PlaneLeaf {
    int box, lev, slot, depth;
    unsigned sx, sz;
};
struct PlaneGroup {
    int slot, first, count;
};
// 2-D output components: x and z table kinds, outputs
constexpr int kPlaneComps = 6;
struct PlaneComps {
    int n;
    int kx[kPlaneComps], kz[kPlaneComps];
    OutDesc od[kPlaneComps];
};

// Several problems of one shape class (3-D, same norder, density count and
// precision; plane-wave counts may differ) in one launch.  Task i of a launch belongs
// to problem tprob[i]; the kernel then takes that problem's tables, values,
// outputs and expansion workspace from pp[tprob[i]] instead of its
// single-problem arguments.  tklev[i]: the merge/split level code of task i
// (STEPs 2 and 4, whose phase rows depend on the problem's depth).  All
// pointers device pointers; pp == nullptr means a single-problem launch.
struct ProbPtrs {
    Geom g;                   // the problem's geometry (plane-wave count, nexp)
    const double2* p2pw;      // value->PW tables [l][k][m]
    const double2* p2pwS;     // the same times the merge phases [l][v][k][m]
    const double2* pw2potS;   // PW->value tables [l][v][k][i] (value kind)
    const double2* wms;       // merge/split 1-D phases [klev-1][k]
    const double2* wm2l;      // M2L 1-D phases [o][k]
    const double* loctab;     // near-field tables [l][slot][j][k] (value kind)
    const double* fvals;      // (nd, npbox, nboxes)
    double* pot;              // (nd, npbox, nboxes), accumulated into
    void* expn;               // expansion slots (FP64 or FP32 complex)
    long long zero_off;       // element offset of the all-zero slot
};
struct Multi {
    const ProbPtrs* pp = nullptr;
    const int* tprob = nullptr;
    const int* tklev = nullptr;
};

// Device-resident tables (all pointers are device pointers).
struct DevTables {
    // per level l: value->PW  T[l][k][m] (k < npw, m < n) complex (double2)
    const double2* p2pw;
    // per kind and level l: PW->value  U[kind][l][i][k] (i < n, k < npw)
    const double2* pw2pot;
    // its transpose and that times the parent->child split phase of each
    // level: pw2potS[kind][l][v][k][i], v = 0 plain, 1 = + phase, 2 = conjugate
    const double2* pw2potS;
    // p2pw and its products with the child->parent merge phase of each level:
    // p2pwS[l][v][k][m], v = 0 plain, 1 = + phase, 2 = conjugate phase
    const double2* p2pwS;
    // merge/split 1-D phases wms[klev-1][k], M2L 1-D phases wm2l[o][k]
    const double2* wms;
    const double2* wm2l;
    // near-field masked tables loc[kind][l][slot][k][j] ([j][k] where
    // loctab_by_source), else with bands [l][slot][k][2];
    // loc_slots table slots per level (13 for the solve, 193 for the
    // refinement of a new tree); a pair's table slots are packed 8 bits per
    // kernel axis: x | y << 8 | z << 16
    const double* loctab;
    const int* locband;
    int loc_slots = 13;
    // kind strides (elements): pw2pot, pw2potS, loctab
    size_t pw2pot_ks, pw2potS_ks, loctab_ks;
    int n;     // norder
    int npw;
    // 1: expansions are stored as FP32 complex (mixed precision; 3-D
    // register-blocked path only), 0: FP64
    int expn_f32;
    // contraction precision of the mixed-precision forms: 0 FP64, 1 FP32
    // matrix cores, 2 BF16 hi/lo matrix cores (prec >= 1 implies expn_f32)
    int prec;
    // x-stage variant of STEP 1 / STEP 5 (tuned per shape class; -1 = the
    // default policy): 0 FP64 (VALU), 2 the reduced-precision matrix cores
    // (prec >= 1)
    int xs1 = -1, xs5 = -1;
    size_t lds_limit;  // device LDS bytes per block
};

// 3-D STEP 1 / STEP 5 kernels; each returns false (nothing launched) when the
// shape is not covered.
// STEP 1 with a reduced-precision x stage, leaves of the cutoff level
bool launch_p2pw_3d(const Geom& g, const DevTables& t, int ntask, const int* box, const int* lev,
                    const int* slot, const double* fvals, double2* expn, hipStream_t s, size_t lds_limit,
                    const Multi& mu = Multi{});
// STEP 5 with a reduced-precision x stage: tasks [0, nfam) families, then
// nown single leaves; the components of zo (x and y kinds kd.x, kd.y)
bool launch_pw2pot_3d_z(const Geom& g, const DevTables& t, int nfam, int nown, const SymTask* tasks,
                        const double2* expn, Kinds kd, const ZOut& zo, hipStream_t s, size_t lds_limit,
                        const Multi& mu = Multi{});
// STEP 5 in FP64 arithmetic (FP64 or FP32 expansions) through the tables'
// symmetries: tasks [0, nfam) families, then nown single leaves
bool launch_pw2pot_sym(const Geom& g, const DevTables& t, int nfam, int nown, const SymTask* tasks,
                       const double2* expn, const ZGroups& zg, hipStream_t s, const Multi& mu = Multi{});
// the symmetric kernels cover this shape (norder 4..16, LDS)
bool sym3_supported(const Geom& g, const DevTables& t);
// the reduced-precision kernels cover it too (norder 8, 12, 16, LDS)
bool pw2pot_3d_supported(const Geom& g, const DevTables& t);
// STEP 5 runs its x stage on the reduced-precision matrix cores (else it
// takes launch_pw2pot_sym)
bool pw2pot_lowp(const DevTables& t);
// STEP 1 runs its x stage on the reduced-precision matrix cores (else it
// takes launch_p2pw_sym)
bool p2pw_lowp(const DevTables& t);
// STEP 1 in FP64 arithmetic through the tables' symmetries: tasks [0, nfam)
// families (their parent's expansion, STEP 2 folded in), then nown leaves of
// the cutoff level
bool launch_p2pw_sym(const Geom& g, const DevTables& t, int nfam, int nown, const SymTask* tasks, const double* fvals,
                     double2* expn, hipStream_t s, const Multi& mu = Multi{});
// Fused STEP 1 + 2 with a reduced-precision x stage, for parents with leaf
// children (3-D, N in {8,12,16}):
// plev/pslot per parent, kids/ksg 8 per parent (leaf child box or -1, merge
// sign bits).  Writes (overwrites) the parent's mp; returns false if not covered.
bool p2pw_fused_3d(const Geom& g, const DevTables& t, int ntask, const int* plev, const int* pslot,
                   const int* kids, const int* ksg, const double* fvals, double2* expn, hipStream_t s,
                   const Multi& mu = Multi{});

// 3-D STEP 1 in the form p2pw_lowp picks (throws when the shape is not
// covered): leaves of the cutoff level, and parents with leaf children
struct Step1Lists {
    int n_s1;                 // reduced precision: leaves, then parents
    const int *s1_box, *s1_lev, *s1_slot, *s1_prob;
    int n_fz;
    const int *fz_lev, *fz_slot, *fz_kids, *fz_ksg, *fz_prob;
    int nfam, nown;           // SymTask list
    const SymTask* sym;
    const int* symprob;
};
void launch_p2pw_tasks(const Geom& g, const DevTables& t, const Step1Lists& l, const double* fvals, double2* expn,
                       hipStream_t s, const ProbPtrs* pp = nullptr);

// Stage launchers (stream-ordered; all arguments device pointers).
void launch_p2pw(const Geom& g, const DevTables& t, int ntask, const int* box,
                 const int* lev, const int* slot, const double* fvals,
                 double2* expn, hipStream_t s);
// par_acc (nullable): per parent, nonzero = add to the parent's current mp
void launch_merge(const Geom& g, const DevTables& t, int ntask, const int* par_slot,
                  const int* par_first, const int* par_count, const int* pc_child,
                  const int* pc_sign, const int* par_acc, int klev, double2* expn, hipStream_t s,
                  const Multi& mu = Multi{});
// STEP 3, kM2lGroup targets per block.  toff[i]: element offset of target
// i's slot (slot * 2 * nd * nexp); gent: per group, the range of its entry
// stream (each target's own expansion, then its list; padded to a multiple
// of kM2lBatch); soff[j]: element offset of the entry's source slot (padding
// points at an all-zero slot, whose element offset is zero_off); scode[j] =
// o | last << 5 with o = ox + 3 oy + 9 oz in 0..26 and last set on each
// target's final entry.
// (2-D with entries in batches of two: 1062 targets x 16 densities 204 / 175 /
// 176 / 180 / 187 us in groups of 1 / 2 / 4 / 5 / 8, 3184 targets 43 / 36 / 36 /
// 41 / 49, periodic 2933 x 4 107 / 93 / 92 / 97 / 105)
constexpr int kM2lGroup = 4;
constexpr int kM2lGroupMax = 12;
// targets per STEP 3 block of a problem with `blocks` targets x element
// ranges: kM2lGroup, or one where even that leaves each CU fewer than sixteen
// blocks (178 targets of 800 elements: 13 us in groups of four, now 9), or
// FGT_M2L_GROUP (1..kM2lGroupMax, tuning runs)
int m2l_group(long long blocks);
// source loads per register batch (STEP 3 in groups and over bricks): the
// grouped kernel keeps two batches in flight, and with four loads in each
// measured the same or slower (2-D, 1062 / 3184 targets 19.8 -> 20.4 / 36.4 ->
// 38.4 us; 3-D without bricks, 752 targets 158 -> 164)
constexpr int kM2lBatch = 2;
// longest entry stream of a group: kM2lGroupMax targets x (own + 26 list
// entries), padded
constexpr int kM2lMaxEntries = kM2lGroupMax * 27 + kM2lBatch;
// ept: elements per thread, 1 or 2 (2 needs an even nd * nexp in every
// problem of the launch)
void launch_m2l27(const Geom& g, const DevTables& t, int ngroup, int group, long long zero_off,
                  const long long* toff, const int* gent, const long long* soff, const int* scode, double2* expn,
                  hipStream_t s, const Multi& mu = Multi{}, int ept = 1);
// FGT_M2L_EPT (1 or 2) forces the elements per thread of STEP 3; 0 = policy
int m2l_ept_env();
// STEP 3 over sibling bricks (3-D): per brick 8 loc element offsets (-1 =
// none), an entry stream of source mp offsets and codes (position 6 bits |
// target mask << 6), padded to a multiple of kM2lBatch
constexpr int kM2lBrickMax = 64 + kM2lBatch;
void launch_m2l_brick(const Geom& g, const DevTables& t, int nbrick, long long zero_off, const long long* toff,
                      const int* gent, const long long* soff, const int* scode, double2* expn, hipStream_t s,
                      const Multi& mu = Multi{});
// The same bricks as a separable stencil (the brick's lists must be
// geometric: every source holds every sibling whose 3x3x3 neighbourhood
// contains it): the phase of offset (ox, oy, oz) is w_x(ox) w_y(oy)
// w_z(oz) with w(0) = conj(w(2)), w(1) = 1, so the sum over a sibling's 27
// neighbours runs as three 3-tap passes along x, y and z over the brick's
// 4x4x4 source grid, each source loaded once.  Same arrays as
// launch_m2l_brick.
void launch_m2l_sep(const Geom& g, const DevTables& t, int nbrick, long long zero_off, const long long* toff,
                    const int* gent, const long long* soff, const int* scode, double2* expn, hipStream_t s,
                    const Multi& mu = Multi{});
// FGT_M2L_BRICK: 0 keeps STEP 3 on the target groups, 1 on sibling bricks
// (entry streams), 2 on sibling bricks as a separable stencil, where a
// problem allows them; unset (-1) = policy (entry-stream bricks: the
// separable form does a sixth of the arithmetic but was measured slower,
// 1.17 vs 0.74 ms on a norder-16 periodic problem, bound by the cache
// traffic of the source loads that both forms share)
int m2l_brick_env();
void launch_split(const Geom& g, const DevTables& t, int nentry, const int* pc_parent,
                  const int* pc_child, const int* pc_sign, int klev, double2* expn,
                  hipStream_t s, const Multi& mu = Multi{});
void launch_pw2pot(const Geom& g, const DevTables& t, int ntask, const int* box,
                   const int* lev, const int* slot, const double2* expn,
                   Kinds kd, OutDesc od, hipStream_t s);
// 3-D STEP 5 for the components of zg, in the form pw2pot_lowp picks (throws
// when the shape is not covered)
struct Step5Lists {
    int nfam, nown;           // SymTask list
    const SymTask* sym;
    const int* symprob;       // its problem indices (batches)
};
void launch_pw2pot_tasks(const Geom& g, const DevTables& t, const Step5Lists& l, const double2* expn,
                         const ZGroups& zg, hipStream_t s, const ProbPtrs* pp = nullptr);
// flags (nullable): per entry bit0 = last of its (x,z) table group, bit1 =
// last of its z group; entries must then be grouped in that order.
void launch_direct(const Geom& g, const DevTables& t, int ntask, const int* tgt,
                   const int* lev, const int* off, const int* src, const int* code,
                   const int* flags, const double* fvals, Kinds kd, OutDesc od, hipStream_t s,
                   const Multi& mu = Multi{});
// the 3-D near-field kernels cover this order (4..16); they read the near-
// field tables as [j][k] (source node, target node)
inline bool direct3_orders(int ndim, int n) { return ndim == 3 && n >= 4 && n <= 16; }
// the near-field tables of a problem are [j][k] (the 2-D kernel reads them so
// for every order)
inline bool loctab_by_source(int ndim, int n) { return ndim == 2 || direct3_orders(ndim, n); }
// orders covered, with flags; false when not (nothing launched)
bool launch_direct_3d(const Geom& g, const DevTables& t, int ntask, const int* tgt, const int* lev,
                      const int* off, const int* src, const int* code, const int* flags,
                      const double* fvals, const ZGroups& zg, hipStream_t s, const Multi& mu = Multi{});

// 2-D STEP 1 + 2, STEP 4 + 5 and STEP 6 (kernels_plane.hip); nlev: levels
// below the cutoff.  The launchers return false on a launch error.
bool plane_supported(const Geom& g, const DevTables& t, int nlev);
// leaves grouped by cutoff box; sum_slots[sum_off[i] ..]: the group slots of
// the i-th cutoff box with more than one group, its own first
bool launch_p2pw_plane(const Geom& g, const DevTables& t, int nlev, int ngroup, const PlaneGroup* groups,
                       const PlaneLeaf* leaves, int nsum, const int* sum_off, const int* sum_slots,
                       const double* fvals, double2* expn, hipStream_t s);
bool launch_pw2pot_plane(const Geom& g, const DevTables& t, int nlev, int nleaf, const PlaneLeaf* leaves,
                         const double2* expn, const PlaneComps& pc, hipStream_t s);
bool launch_direct_plane(const Geom& g, const DevTables& t, int ntask, const int* tgt, const int* lev, const int* off,
                         const int* src, const int* code, const double* fvals, const PlaneComps& pc, hipStream_t s);

// Device workspace of the no-allocation entry point: a file-scope device
// array of kScratchBytes per GPU.  scratch_region() returns its address on
// the current device (looked up once per device); launch_zero() clears a
// byte range (8-byte aligned) with a fill kernel on stream s.
constexpr size_t kScratchBytes = size_t(128) << 20;
void* scratch_region(size_t* bytes);
void launch_zero(void* p, size_t bytes, hipStream_t s);

// Extra targets (STEP 11).  launch_target_groups groups them by leaf: child
// [box][2^ndim] (-1 leaf, -2 missing child), count zeroed by the caller;
// perm the targets by leaf, tasks {box, first, count, -} of at most 256 and
// their number *ntask (<= target_tasks_max); *missing set when a target's path
// ends at a missing child.  launch_targets evaluates values (ncd, npbox,
// nboxes) at the targets, out[t*ncd + q] (u = values->coefficients, u(k,j) at
// u[k + j*n]).
// (nend: boxes where a target's path can end, leaves and boxes that lack a child)
int target_tasks_max(int nt, int nend);
bool launch_target_groups(int nt, int ndim, int nlevels, int nboxes, const double* targs, const double* centers,
                          const int* child, int* count, int* first, int2* place, int* perm, int4* tasks, int* ntask,
                          int* missing, hipStream_t s);
bool launch_targets(int ndim, int n, int ipoly, int ncd, int maxtask, const double* u, const int4* tasks,
                    const int* ntask, const double* centers, const double* bsize_of_box, const double* targs,
                    const int* perm, const double* vals, double* out, hipStream_t s);

}  // namespace fgt
