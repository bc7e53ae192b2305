// hbt_fast.h -- the fast pair kernel: a cheap conservative prefilter over
// every enumerated pair, per-wave compaction of the survivors into an LDS
// ring, and the exact cascade on full waves of survivors.
//
// Why: the reference's cascade exits early for ~98% of pairs
// (HBT_correlation.cpp:319-398).  On a 64-wide wave, lanes that exit early
// idle while any lane continues, so a direct port pays the whole cascade
// (sqrt, three to five divisions, cos) for almost every pair.  Here the
// work items' windows leave out most pairs unevaluated, every evaluated pair
// costs its share of three matrix-core products and 9 VALU operations, and only its
// survivors (~1.4% of the enumerated pairs on the bench workload) reach the
// exact cascade, 64 at a time with all lanes busy.
//
// Prefilter (all conservative: a pair the exact cascade accepts always
// passes; the margins exceed the rounding error of both computations):
//   T = |p1T + p2T|^2 = 4 K_perp^2           in [4 KT_min^2, 4 KT_max^2]
//   q_out^2 = dn^2 / T <= H^2                (q_out = (p1T - p2T).(p1T + p2T)
//        / |p1T + p2T| = dn / sqrt(T), dn = n1 - n2, n = |pT|^2)
//   q_side^2 = C^2 / T <= H^2                (q_side = (p1T - p2T)x(p1T + p2T)
//        / |p1T + p2T|, whose numerator is C = 2 (p1x p2y - p1y p2x))
//   |y1 - y2| <= (H/2) (1/m_T1 + 1/m_T2)     (y the rapidity, E = m_T cosh y, pz =
//        m_T sinh y: q_long M_t = E2 pz1 - E1 pz2 = m_T1 m_T2 sinh(y1 - y2) and
//        M_t <= (m_T1 + m_T2) / 2 cosh((y1 - y2) / 2), so |q_long| <= H needs
//        2 sinh(|y1 - y2| / 2) <= (H/2) (1/m_T1 + 1/m_T2); the test passes 1 % more
//        pairs than |q_long| <= H itself, 6 % fewer than the same in beta and E)
// with H = max(|q_lo_cut|, |q_hi_cut|).  The two q windows are one test,
// max(|dn|, |C|)^2 <= H^2 T.  T, dn and C are bilinear in the two particles'
// (px, py, n, 1), so the matrix cores form them.
// For mixed pairs the i particle is rotated by -theta instead of rotating
// every j by +theta (T, dn, C and y are rotation invariant); the exact
// cascade then uses the reference's rotated j (HBT_correlation.cpp:522-523).
#pragma once
#include <algorithm>

#include "hbt_device.h"
#include "hbt_f32.h"
#include "hbt_slab.h"
#include "host_items.h"

namespace hbt {

// Per-particle prefilter record: nrm = px^2+py^2 - mid/2 (so that
// n1 + n2 + 2 p1.p2 = T - mid), and blo, the lower end of the particle's
// longitudinal interval [y - cw, y + cw] (y the rapidity, or pz without the LCMS
// boost); the upper end bhi is kept beside the records.  The kernel reads the
// FP32 records, which pass every pair the exact cascade of either precision
// accepts; the FP64 ones state the same tests without FP32's rounding.
struct PfRec64 {
    double px, py, nrm, blo;
};
struct PfRec32 {
    float px, py, nrm, blo;
};

// Prefilter constants in the records' precision: X = s (T - mid) is formed
// with the scale s = H^2 (1 with the q_inv branch on, whose q test passes
// every pair); sh bounds |X| (the T window's half-width, scaled and rounded
// up; nsh2 = -sh^2), c0 = H^2 mid + c bounds max(|dn|, |C|)^2 - X, with the q
// margin c (infinite with the q_inv branch on).
// dn: 1/2, or 0 where |dn| is left out (q_inv bins: no bound on q_out); wide: 0,
// or infinity where the longitudinal intervals count for nothing.
template <typename Prec>
struct PfConst {
    Prec s, nsh2, c0;
    Prec dn = (Prec)0.5, wide = 0;
};

template <typename Prec>
__host__ __device__ __forceinline__ PfConst<Prec> pf_const(const DevParams &P) {
    constexpr bool f64 = std::is_same<Prec, double>::value;
    constexpr double eps = f64 ? 1.1102230246251565e-16 : 5.9604644775390625e-8;
    PfConst<Prec> k;
    k.s = (Prec)(P.qinv ? 1.0 : P.pf_h2);
    const double sh = (double)k.s * (f64 ? P.pf_half : (double)P.f_half);
    k.nsh2 = (Prec)(-sh * sh * (1.0 + 16.0 * eps));
    k.c0 = (Prec)(((double)k.s * P.pf_mid) * (1.0 + 4.0 * eps) -
                  (f64 ? P.pf_negc : (double)P.f_negc));
    return k;
}

// The prefilter's tests of one pair (for a mixed pair, i rotated by
// -theta): it passes where all four values are negative, that is, where the
// largest is.  K_T window: X^2 - (s half)^2; q_out and q_side: max(|dn|, |C|)^2 -
// X - (H^2 mid + c); q_long: |y_i - y_j| <= cw_i + cw_j as the overlap of the two
// longitudinal intervals, blo_i - bhi_j and blo_j - bhi_i.  The margins leave
// every pair the exact cascade accepts strictly inside.
__host__ __device__ __forceinline__ float pf_fma(float a, float b, float c) {
    return __builtin_fmaf(a, b, c);
}
__host__ __device__ __forceinline__ double pf_fma(double a, double b, double c) {
    return __builtin_fma(a, b, c);
}
__host__ __device__ __forceinline__ float pf_abs(float a) { return __builtin_fabsf(a); }
__host__ __device__ __forceinline__ double pf_abs(double a) { return __builtin_fabs(a); }
__host__ __device__ __forceinline__ float pf_max(float a, float b) { return __builtin_fmaxf(a, b); }
__host__ __device__ __forceinline__ double pf_max(double a, double b) {
    return __builtin_fmax(a, b);
}

// Operands of one i particle, component 0..3, against a j particle's (px, py, n,
// 1): X = s (T - mid), and P = (dn + C) / 2, M = (dn - C) / 2 with dn = in - jn
// and C = 2 (ix jy - iy jx), so that max(|dn|, |C|) = |P| + |M| is one addition (a
// maximum would first quiet both operands).
template <typename Prec>
struct PfBlock {
    Prec X, P, M;
};
template <typename Prec>
__host__ __device__ __forceinline__ PfBlock<Prec> pf_block(const PfConst<Prec> &k, int comp, Prec x,
                                                           Prec y, Prec n) {
    PfBlock<Prec> o;
    const Prec s2 = (Prec)2 * k.s;
    o.X = comp == 0 ? s2 * x : comp == 1 ? s2 * y : comp == 2 ? k.s : k.s * n;
    const Prec c = comp == 0 ? -y : comp == 1 ? x : (Prec)0;
    const Prec d = comp == 2 ? -k.dn : comp == 3 ? k.dn * n : (Prec)0;
    o.P = d + c;
    o.M = d - c;
    return o;
}

// The largest of a pair's tests, from the products X, P and M and the two
// longitudinal intervals (i's widened by k.wide).
template <typename Prec>
__host__ __device__ __forceinline__ Prec pf_test(Prec X, Prec P, Prec M, Prec ilo, Prec ihi,
                                                 Prec jlo, Prec jhi, const PfConst<Prec> &k) {
    const Prec e = pf_abs(P) + pf_abs(M);
    return pf_max(pf_max(pf_fma(e, e, -X) - k.c0, pf_fma(X, X, k.nsh2)),
                  pf_max(ilo - jhi, jlo - ihi));
}

// A pair's test on the host, for the check of the margins: the kernel's operands
// and test, the four products added in order (the matrix cores' order is not
// known; the margins cover any).
template <typename Prec>
struct PfTerms {
    Prec m;
};
template <typename Prec>
__host__ __device__ __forceinline__ PfTerms<Prec> pf_terms(Prec ix, Prec iy, Prec in, Prec ilo,
                                                           Prec ihi, Prec jx, Prec jy, Prec jn,
                                                           Prec jlo, Prec jhi,
                                                           const PfConst<Prec> &k) {
    const Prec j[4] = {jx, jy, jn, (Prec)1};
    Prec X = 0, P = 0, M = 0;
    for (int c = 0; c < 4; c++) {
        const PfBlock<Prec> b = pf_block(k, c, ix, iy, in);
        X = pf_fma(j[c], b.X, X);
        P = pf_fma(j[c], b.P, P);
        M = pf_fma(j[c], b.M, M);
    }
    return PfTerms<Prec>{pf_test(X, P, M, ilo - k.wide, ihi + k.wide, jlo, jhi, k)};
}

template <typename Prec>
__host__ __device__ __forceinline__ bool pf_pass(const PfTerms<Prec> &t) {
    return t.m < 0;
}

// What a particle's prefilter record needs beside its momentum: the window
// centre, the longitudinal half-width's numerator H/2, the largest |beta| of the
// list (|pz| without the LCMS boost; margins), and the analysis' boost and q_inv switches.
struct PfMake {
    double mid, c_beta, bm;
    int boost, qinv;
};

// The neighbouring float below (up = false) or above; infinities and NaN stay.
__host__ __device__ __forceinline__ float next_float(float x, bool up) {
    if (!(fabsf(x) < INFINITY)) return x;
    if (x == 0.0f) return up ? 1.401298464e-45f : -1.401298464e-45f;
    const int b = __builtin_bit_cast(int, x);
    return __builtin_bit_cast(float, b + ((x > 0.0f) == up ? 1 : -1));
}

// Where a particle's longitudinal interval [y - cw, y + cw] lies: y its rapidity
// and cw = (H/2) / m_T (or pz and H/2 without the LCMS boost; no window with the
// q_inv branch on, or for E <= 0).  eps: the rounding unit of the interval's
// ends.  cw also covers the rounding of y and of cw: with |beta| <= bm over the
// list, cosh^2 y <= 1 / (1 - bm^2) scales beta's own rounding.
struct LongWindow {
    double y, cw;
};
__host__ __device__ __forceinline__ LongWindow long_window(const PfMake &m, double pz, double E,
                                                           double eps) {
    if (m.qinv || !(E > 0.0)) return LongWindow{0.0, INFINITY};
    if (!m.boost) return LongWindow{pz, m.c_beta * (1.0 + 8 * eps) + 4 * eps * fmax(1.0, m.bm)};
    const double g = 8.9e-16 / (1.0 - m.bm * m.bm);
    if (!(g >= 0.0 && g < 1.0)) return LongWindow{0.0, INFINITY};
    return LongWindow{atanh(pz / E), m.c_beta / sqrt((E - pz) * (E + pz)) * (1.0 + 8 * eps + g) +
                                         4 * eps * fmax(1.0, atanh(m.bm)) + g};
}

// FP32 record of one particle; the interval's ends are rounded to nearest, then
// one FP32 ulp outward.
__host__ __device__ __forceinline__ void pf_make(const PfMake &m, double px, double py, double pz,
                                                 double E, PfRec32 &r, float &bhi) {
    const LongWindow w = long_window(m, pz, E, 5.9604644775390625e-8);
    r = PfRec32{(float)px, (float)py, (float)(px * px + py * py - 0.5 * m.mid),
                next_float((float)(w.y - w.cw), false)};
    bhi = next_float((float)(w.y + w.cw), true);
}

// A particle as the kernel's matrix-core operand, and its longitudinal interval.
struct __align__(16) PfOp {
    float px, py, nrm, one;
};
struct __align__(8) PfBeta {
    float lo, hi;
};
// Entries past a list's end that the kernel may read (and ignore): its j
// tiles come in pairs of 16.
constexpr int kPfPad = 32;

// Same-event pair orientation: for a position in the cell-sorted list, the
// particle's index in the fast list and its rank in gather order (the
// reference's particle 1 is the earlier of the two in gather order).
struct OrigRank {
    int idx;
    int rank;
};

// One analysis resident in HBM: its particles, mixing plan and histograms.
// A launch may carry items of many analyses (the request server batches
// them); every index in a WorkItem is relative to its own View.  The
// particle lists are the fast lists: per event, the particles whose |pT|
// can reach a K_T bin, sorted by |pT|.
struct View {
    DevHist H;
    const PartRec *A;    // same-event fast list, 64 B per particle
    const PartRec *B;    // mixed fast list (separate, or an alias of A)
    const PfOp *pfA;     // prefilter operands of A, of B,
    const PfOp *pfB;
    const PfOp *pfS;     // and of the same-event fast list sorted by (px cell, py) per group
    const PfBeta *bwA;   // their longitudinal intervals
    const PfBeta *bwB;
    const PfBeta *bwS;
    const OrigRank *origS;     // cell-sorted position -> fast-list index and gather rank
    const PartRec *AS;         // records of the same-event fast list in the cell-sorted order
    const JWin *mwin;          // partner windows of the mixed items
    const double *plan_cs;     // cos, sin of each plan row's rotation
    const double *psi;         // psi_ref per group
    // the analysis' grid constants, for the exact stage: read from the view
    // table (constant address space) where they are used, so the kernel
    // neither holds them in SGPRs nor reloads spilled copies with VALU
    // instructions
    DevParams P;
};

// The fast lists on the device, from the uploaded records A (per event,
// |pT|-sorted) and the cell-sorted order: the prefilter operands and
// longitudinal intervals of both orders, and the cell-sorted copy of the records, AS[q] =
// A[orr[q].idx].
static __global__ __launch_bounds__(256) void k_build_lists(PfMake m, const PartRec *__restrict__ A,
                                                            const OrigRank *__restrict__ orr,
                                                            PartRec *__restrict__ AS,
                                                            PfOp *__restrict__ pfA,
                                                            PfBeta *__restrict__ bwA,
                                                            PfOp *__restrict__ pfS,
                                                            PfBeta *__restrict__ bwS,
                                                            long long nf) {
    const long long q = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= nf) return;
    PfRec32 r;
    float hi;
    const PartRec a = A[q];
    pf_make(m, a.px, a.py, a.pz, a.E, r, hi);
    pfA[q] = PfOp{r.px, r.py, r.nrm, 1.0f};
    bwA[q] = PfBeta{r.blo, hi};
    const PartRec s = A[orr[q].idx];
    AS[q] = s;
    pf_make(m, s.px, s.py, s.pz, s.E, r, hi);
    pfS[q] = PfOp{r.px, r.py, r.nrm, 1.0f};
    bwS[q] = PfBeta{r.blo, hi};
}

static inline hipError_t build_lists(const PfMake &m, const PartRec *A, const OrigRank *orr,
                                     PartRec *AS, PfOp *pfA, PfBeta *bwA, PfOp *pfS, PfBeta *bwS,
                                     long long nf, hipStream_t st) {
    if (nf <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_build_lists, dim3((unsigned)((nf + 255) / 256)), dim3(256), 0, st, m, A,
                       orr, AS, pfA, bwA, pfS, bwS, nf);
    return hipGetLastError();
}

// Work queues of a launch: at most one per XCD.  Queue q holds items
// [qoff[q], qoff[q+1]); its counter is counter[kQueueStride * q].
constexpr int kMaxQueues = 8;
constexpr int kQueueStride = 16;  // ints: one 64-byte line per counter

struct FastArgs {
    DevParams P;
    const View *views;
    const WorkItem *items;
    int nitems;
    int nqueues;                   // 1, 2, 4 or 8
    int qoff[kMaxQueues + 1];
    int *counter;              // work counters, zeroed before launch
    unsigned long long *binned;  // [2]: binned same, mixed (for stats)
    int qinv_lds = 0;          // q_inv bins kept in LDS (one view only), or 0
    // slab binning (hbt_slab.h) of the common-case instances; vals == null:
    // every binned pair is added with device-scope atomics
    SlabArgs slab;
};

// Read-only, wave-uniform data (the view table, the kernel's arguments, work
// items, partner windows, rotations) is read through the constant address
// space: scalar loads into scalar registers.
#if defined(__HIP_DEVICE_COMPILE__)
#define HBT_AS4 __attribute__((address_space(4)))
#else
#define HBT_AS4
#endif
#define HBT_CONST(T, p) ((const HBT_AS4 T *)(p))
using CView = const HBT_AS4 View;
using CParams = const HBT_AS4 DevParams;
using CArgs = const HBT_AS4 FastArgs;

// p, hidden from the optimiser: loads through it stay where they are written
// instead of being hoisted out of the caller's loops and held (spilled) in
// scalar registers.  For the exact stage, which reads its grid constants and
// pointers where it uses them.
template <typename T>
__device__ __forceinline__ T *fresh(T *p) {
#if defined(__HIP_DEVICE_COMPILE__)
    __asm__ volatile("" : "+s"(p));
#endif
    return p;
}
// The view table entry k, and the kernel's arguments.
__device__ __forceinline__ CView *view_at(const View *views, int k) {
    return fresh(HBT_CONST(View, views) + __builtin_amdgcn_readfirstlane(k));
}
__device__ __forceinline__ CArgs *kernel_args() {
#if defined(__HIP_DEVICE_COMPILE__)
    return fresh((CArgs *)__builtin_amdgcn_kernarg_segment_ptr());
#else
    return nullptr;
#endif
}

// ------------------------------------------------------------ exact stage
// A wave's LDS.  The exact stage takes 64 scattered survivors at a time; read
// from memory, each of their 128-byte pairs of records would cost the vector
// cache eight accesses per lane (measured: its address and data units 88 and
// 96 % busy, k_fast 8.0 ms on the headline workload).  So the tile's 64 i
// records are staged here once per item, and the 32 j records of a pair of
// tiles while its prefilter runs, by loads that cover whole lines; two j
// buffers let the survivors of a pair that do not fill a wave wait for the
// next pair's.  Chunk c (16 bytes) of row r sits at chunk c ^ (r / 4) of its
// row, which spreads 64 random rows over all banks.
struct __align__(16) WaveLds {
    char irec[64 * sizeof(PartRec)];
    char jrec[2][32 * sizeof(PartRec)];
    double2 rot[2];            // (cos, sin) of the j buffers' rotations
    int irank[64], jrank[2][32];
    unsigned short ring[128];  // queued survivors: i slot | j row << 6 | j buffer << 11
};

// Staged record `row`: chunks 0 and 1 (momentum), 2 and 3 (space-time).
struct PartMom {
    double px, py, pz, E;
};
__device__ __forceinline__ unsigned lds_row(unsigned row) {
    return row * (unsigned)sizeof(PartRec) + ((row & 12u) << 2);
}
__device__ __forceinline__ PartMom lds_mom(const char *rec, unsigned at) {
    const double2 u = *(const double2 *)(rec + at), v = *(const double2 *)(rec + (at ^ 16u));
    return PartMom{u.x, u.y, v.x, v.y};
}
__device__ __forceinline__ PartRec lds_rec(const char *rec, unsigned at) {
    const PartMom m = lds_mom(rec, at), p = lds_mom(rec, at ^ 32u);
    return PartRec{m.px, m.py, m.pz, m.E, p.px, p.py, p.pz, p.E};
}
// The exact stage of one pair whose staged records lie at a and b of rec, in
// the reference's orientation (same-event: particle 1 is the earlier in gather
// order); mixed: c, s rotate the partner.
template <typename Prec, bool EXT>
struct Exact;

template <bool EXT>
struct Exact<double, EXT> {
    static __device__ __forceinline__ int same(CView *vp, double psi, const char *rec, unsigned a,
                                               unsigned b, SameRec &out, const QinvSink &q) {
        const DevParams P = vp->P;
        const DevHist H = vp->H;
        const PartRec p = lds_rec(rec, a), r = lds_rec(rec, b);
        return eval_same_f64<EXT>(P, H, psi, p.px, p.py, p.pz, p.E, p.x, p.y, p.z, p.t, r.px,
                                  r.py, r.pz, r.E, r.x, r.y, r.z, r.t, out, q);
    }
    static __device__ __forceinline__ int mixed(CView *vp, double psi, const char *rec, unsigned a,
                                                unsigned b, double2 cs, long &k,
                                                const QinvSink &q) {
        const DevParams P = vp->P;
        const DevHist H = vp->H;
        const PartMom p = lds_mom(rec, a), r = lds_mom(rec, b);
        return eval_mixed_f64<EXT>(P, H, psi, p.px, p.py, p.pz, p.E, r.px * cs.x - r.py * cs.y,
                                   r.px * cs.y + r.py * cs.x, r.pz, r.E, k, q);
    }
};

// The precision form: negative where a decision is ambiguous.
template <bool EXT>
struct Exact<float, EXT> {
    static __device__ __forceinline__ int same(CView *vp, double psi, const char *rec, unsigned a,
                                               unsigned b, SameRec &out, const QinvSink &) {
        const PartRec p = lds_rec(rec, a), r = lds_rec(rec, b);
        out.sure = true;
        return eval_same_fast<EXT>(vp->P, psi, p, r, out);
    }
    static __device__ __forceinline__ int mixed(CView *vp, double psi, const char *rec, unsigned a,
                                                unsigned b, double2 cs, long &k,
                                                const QinvSink &) {
        const PartMom p = lds_mom(rec, a), r = lds_mom(rec, b);
        return eval_mixed_fast<EXT>(vp->P, psi, p.px, p.py, p.pz, p.E, r.px * cs.x - r.py * cs.y,
                                    r.px * cs.y + r.py * cs.x, r.pz, r.E, k);
    }
};

// Records of one queued survivor: offsets in the wave's LDS, same-event pairs
// in the reference's orientation.
struct PairAt {
    unsigned a, b, buf;
};
template <bool RANKED>
__device__ __forceinline__ PairAt pair_at(const WaveLds &wl, unsigned ent, bool mixed) {
    const unsigned i = ent & 63u, j = ent >> 6 & 31u, buf = ent >> 11;
    const unsigned ai = lds_row(i);
    const unsigned aj = (unsigned)offsetof(WaveLds, jrec) + buf * 2048u + lds_row(j);
    const bool swap = RANKED && !mixed && wl.irank[i] > wl.jrank[buf][j];
    return PairAt{swap ? aj : ai, swap ? ai : aj, buf};
}

// One same-event pair added directly.  With slab binning the precision
// form's per-pair values are FP32 on either path (its records hold FP32
// values), so the path a pair takes does not change what it adds; without it
// they stay FP64.
template <typename Prec>
__device__ __forceinline__ void add_same_slabwise(double *bins, SameRec rec, bool slab) {
    if (std::is_same<Prec, float>::value && slab) {
        rec.qo = (double)(float)rec.qo;
        rec.qs = (double)(float)rec.qs;
        rec.ql = (double)(float)rec.ql;
        rec.c = (double)(float)rec.c;
    }
    add_same_direct(bins, rec);
}

// Lane l's part of staging 64 / n rows from src (rows past `last` repeat it):
// chunk l % n of row r0 + l / n, n = 4 chunks, or 2 where only the momentum is
// wanted.
template <int N>
__device__ __forceinline__ double2 stage_load(const PartRec *src, int lane, int r0, int last) {
    const int row = min(r0 + lane / N, last);
    return *(const double2 *)((const char *)src + (unsigned)(row * 64 + (lane & (N - 1)) * 16));
}
template <int N>
__device__ __forceinline__ void stage_store(char *rec, int lane, int r0, double2 v) {
    const unsigned row = (unsigned)(r0 + lane / N), c = (unsigned)lane & (N - 1);
    *(double2 *)(rec + (lds_row(row) ^ (c << 4))) = v;
}

// Per-wave LDS staging of binned same-event pairs for the cooperative
// scatter: bin index and the four sums of up to 24 pairs (two instructions'
// worth; more would cost the fourth block per CU its LDS).
constexpr int kStage = 24;
struct Stage {
    long k[kStage];
    double v[kStage][4];
};

// Each lane with lane < cnt takes one queued survivor and runs the exact
// cascade.
// Binned same-event pairs are added cooperatively: they are staged in LDS,
// then groups of 5 lanes add one pair's count and four sums, so one atomic
// instruction touches 12 bins (12 cache lines) instead of 64.  Atomic
// throughput on this part is set by (instruction, cache line) accesses,
// about 2.4e10 per second whatever the histogram's size or placement, so
// the count is an FP64 add in the same instruction as the sums: one access
// per binned pair.
// unsure: the lanes whose pair the precision form could not decide, cos64 those
// of them that miss only their K_phi bin.
template <typename Prec, bool EXT, bool RANKED>
__device__ __forceinline__ int drain(CView *vp, CArgs *ka, const WaveLds &wl, Stage &stg,
                                     unsigned head, int cnt, bool mixed, double psi,
                                     unsigned *next, const unsigned *lim, double *qlds,
                                     unsigned long long &direct_n, unsigned long long &unsure,
                                     unsigned long long &cos64) {
    const int lane = __lane_id();
    int st = 0;
    SameRec rec;
    long kmix = 0;
    const QinvSink qs =
        EXT && std::is_same<Prec, double>::value ? QinvSink{qlds, ka->qinv_lds} : QinvSink();
    if (lane < cnt) {
        const PairAt pr = pair_at<RANKED>(wl, wl.ring[(head + lane) & 127u], mixed);
        const char *base = (const char *)&wl;
        if (mixed)
            st = Exact<Prec, EXT>::mixed(vp, psi, base, pr.a, pr.b, wl.rot[pr.buf], kmix, qs);
        else
            st = Exact<Prec, EXT>::same(vp, psi, base, pr.a, pr.b, rec, qs);
    }
    if (std::is_same<Prec, float>::value) {
        unsure = __ballot(st < 0);
        if (EXT) cos64 = __ballot(st == -2);
    }
    const bool binned = st > 0 && (st & ST_BIN) != 0;
    const int nbinned = __popcll(__ballot(binned));
    // slab binning: a same-event pair becomes a record of its (block, slab)
    // region; a full region, or stored values that would land in another
    // bin, send it down the direct path.  Mixed pairs are always direct.
    // (The host turns slab binning off for q_inv analyses.)
    const bool slab = ka->slab.vals != nullptr;
    if (mixed) {
        if (binned) add_mixed_direct(vp->H.bins, kmix);
        return nbinned;
    }
    bool direct = binned;
    if (slab && binned) direct = !slab_put_same<Prec>(ka->slab, next, lim, rec);
    const unsigned long long m = __ballot(direct);
    const int nb = __popcll(m);
    if (nb == 0) return nbinned;
    double *bins = vp->H.bins;
    if (slab) {  // few
        direct_n += nb;
        if (direct) add_same_slabwise<Prec>(bins, rec, true);
        return nbinned;
    }
    const unsigned idx = __builtin_amdgcn_mbcnt_hi((unsigned)(m >> 32),
                                                   __builtin_amdgcn_mbcnt_lo((unsigned)m, 0u));
    // lane sub of a group adds field sub of its pair's bin: the count (an
    // exact FP64 integer) and the four sums go out as one FP64 atomic
    // instruction, one cache line per pair
    const int grp = lane / 5, sub = lane - 5 * grp;
    for (int b0 = 0; b0 < nb; b0 += kStage) {
        __builtin_amdgcn_wave_barrier();
        if (direct && idx - b0 < (unsigned)kStage) {
            stg.k[idx - b0] = rec.k;
            stg.v[idx - b0][0] = rec.qo;
            stg.v[idx - b0][1] = rec.qs;
            stg.v[idx - b0][2] = rec.ql;
            stg.v[idx - b0][3] = rec.c;
        }
        __builtin_amdgcn_wave_barrier();
        const int n = min(kStage, nb - b0);
        for (int base = 0; base < n; base += 12) {
            const int p = base + grp;
            if (lane < 60 && p < n)
                atomic_add_f64(bins + stg.k[p] * BIN_STRIDE + sub,
                               sub == 0 ? 1.0 : stg.v[p][max(sub - 1, 0)]);
        }
    }
    __builtin_amdgcn_wave_barrier();
    return nbinned;
}

// The pairs the precision form could not decide, by the literal cascade of
// the FP64 form, each added directly.  After the exact stage of its batch
// rather than inside it: the literal cascade's registers then do not add to
// the exact stage's.  cos stays the form's own (FP32), except for the lanes
// cos64 and for pairs on an edge (on_edge, asked here and not in the exact stage:
// there it cost 2 % of the headline batch's kernel).
template <bool EXT, bool RANKED>
__device__ __forceinline__ int drain_literal(CView *vp, CArgs *ka, const WaveLds &wl, unsigned head,
                                             unsigned long long lanes, unsigned long long cos64,
                                             bool mixed, double psi,
                                             unsigned long long &direct_n) {
    const int lane = __lane_id();
    bool binned = false;
    if (lanes >> lane & 1ull) {
        const PairAt pr = pair_at<RANKED>(wl, wl.ring[(head + lane) & 127u], mixed);
        const char *base = (const char *)&wl;
        if (mixed) {
            long k = 0;
            binned = (Exact<double, EXT>::mixed(vp, psi, base, pr.a, pr.b, wl.rot[pr.buf], k,
                                                QinvSink()) & ST_BIN) != 0;
            if (binned) add_mixed_direct(vp->H.bins, k);
        } else {
            SameRec rec;
            binned = (Exact<double, EXT>::same(vp, psi, base, pr.a, pr.b, rec, QinvSink()) &
                      ST_BIN) != 0;
            if (binned && !(cos64 >> lane & 1ull)) {
                const PartRec p = lds_rec(base, pr.a), r = lds_rec(base, pr.b);
                const double sx = p.px + r.px, sy = p.py + r.py;
                if (!on_edge(vp->P, sx * sx + sy * sy, rec)) rec.c = pair_cos_f32(vp->P, p, r);
            }
            if (binned) add_same_slabwise<float>(vp->H.bins, rec, ka->slab.vals != nullptr);
        }
    }
    const int n = __popcll(__ballot(binned));
    if (!mixed && ka->slab.vals) direct_n += n;
    return n;
}

// XCD of the executing wave (hardware register XCC_ID, bits 3:0).
__device__ __forceinline__ int xcc_id() {
    return (int)(__builtin_amdgcn_s_getreg((3 << 11) | (0 << 6) | 20) & 7u);
}

typedef float v4f __attribute__((ext_vector_type(4)));

// Bits (from the top: block b, row r at bit 15 - (4 b + r)) of the rows of a
// tile that are in range: the first n of this lane's four rows.
__device__ __forceinline__ unsigned rows_first(int n) {
    const int k = min(max(n, 0), 4);
    return ((0xfu << (4 - k)) & 0xfu) * 0x1111u;
}

// What a wave carries from item to item: totals of binned pairs (uniform), and
// the block's slab regions.
struct WaveTotals {
    unsigned long long same = 0, mixed = 0, direct = 0;
    unsigned *slab_next;
    const unsigned *slab_lim;
    double *qlds = nullptr;  // the block's q_inv histograms (QinvSink)
};

// ------------------------------------------------------------------ an item
// The wave holds the item's 64 i particles as four blocks of 16 matrix
// columns and walks its j segments (same-event: one range with j > i;
// mixed: one partner window, window(seg), per segment with the i particles
// rotated by -theta) in pairs of tiles of 16 j rows.  Three 16x16x4 FP32
// products per block and tile give X, P and M of 256 pairs, four per lane; 8
// VALU operations test a pair and a ninth shifts the outcome into the lane's
// bit word.  (The scalar form took 16, and 7 more to queue the survivors of
// each j; comparisons whose masks are combined in scalar registers take 7,
// but the hops between the two units leave the VALU idle: 8000 cycles per
// pair of tiles and wave against 6200.)  Then each lane with bits left queues
// one survivor per round, and whenever 64 are queued they are binned, one per
// lane; the last survivors of a pair of tiles wait for at most the next
// pair's (the exact cascade has a single call site).
// RANKED: a same-event pair is oriented by the gather ranks of its particles;
// otherwise by their places in the list.
// Views: the item's view, from the kernel's arguments (Views::at).
template <typename Prec, bool EXT, bool RANKED, typename Views, typename Window>
__device__ __forceinline__ void walk_item(const WorkItem &w, CView *vp, double psi,
                                          const PfConst<float> &pk, WaveLds &wl, Stage &stg,
                                          WaveTotals &tot, Window window) {
    const bool mixed = w.kind != 0;
    const int lane = __lane_id();
    const int col = lane & 15, comp = lane >> 4, row0 = 4 * comp;
    // same-event tiles run over the cell-sorted list, mixed ones over the
    // |pT|-sorted fast lists
    const PfOp *pfi = (mixed ? vp->pfA : vp->pfS) + w.i0;
    const PfBeta *bwi = (mixed ? vp->bwA : vp->bwS) + w.i0;
    const PfOp *pfj = mixed ? vp->pfB : vp->pfS;
    const PfBeta *bwj = mixed ? vp->bwB : vp->bwS;
    const PartRec *recj = mixed ? vp->B : vp->AS;
    {
        const PartRec *reci = (mixed ? vp->A : vp->AS) + w.i0;
        const int last = w.ni - 1;
        const double2 v0 = stage_load<4>(reci, lane, 0, last);
        const double2 v1 = stage_load<4>(reci, lane, 16, last);
        const double2 v2 = stage_load<4>(reci, lane, 32, last);
        const double2 v3 = stage_load<4>(reci, lane, 48, last);
        __builtin_amdgcn_wave_barrier();
        stage_store<4>(wl.irec, lane, 0, v0);
        stage_store<4>(wl.irec, lane, 16, v1);
        stage_store<4>(wl.irec, lane, 32, v2);
        stage_store<4>(wl.irec, lane, 48, v3);
        if (RANKED && !mixed) wl.irank[lane] = vp->origS[w.i0 + min(lane, last)].rank;
    }
    float ilo[4], ihi[4];
    PfBlock<float> blk[4];
    // The i blocks, rotated by -theta for a mixed segment, one value per lane: lane
    // l holds component l / 16 of particle l % 16 (columns past the tile's end
    // repeat its last particle; `cols` masks them).
    auto load_blocks = [&](double c, double s) {
#pragma unroll
        for (int b = 0; b < 4; b++) {
            const PfOp p = pfi[min(16 * b + col, w.ni - 1)];
            float x = p.px, y = p.py;
            if (mixed) {
                x = (float)((double)p.px * c + (double)p.py * s);
                y = (float)((double)p.py * c - (double)p.px * s);
            }
            blk[b] = pf_block(pk, comp, x, y, p.nrm);
        }
    };
#pragma unroll
    for (int b = 0; b < 4; b++) {
        const PfBeta r = bwi[min(16 * b + col, w.ni - 1)];
        ilo[b] = r.lo - pk.wide;
        ihi[b] = r.hi + pk.wide;
    }
    unsigned cols = 0;  // the bits of the blocks' columns inside the tile
#pragma unroll
    for (int b = 0; b < 4; b++) cols = cols << 4 | (16 * b + col < w.ni ? 0xfu : 0u);
    cols |= cols << 16;
    const int nseg = mixed ? w.nj : 1;
    int seg = -1, jc = 0, je = 0;  // the segment, its next j and its end
    unsigned head = 0, tail = 0, buf = 0;
    double2 rot = {1.0, 0.0};
    for (;;) {
        while (jc >= je && ++seg < nseg) {  // the next segment
            if (mixed) {
                const JWin jw = window(seg);
                jc = jw.b;
                je = jw.e;
                rot.x = HBT_CONST(double, vp->plan_cs)[2 * jw.row];
                rot.y = HBT_CONST(double, vp->plan_cs)[2 * jw.row + 1];
            } else {
                jc = (int)w.j0;
                je = (int)w.j0 + w.nj;
            }
            load_blocks(rot.x, rot.y);
        }
        const bool end = jc >= je;
        const unsigned mark = tail;  // survivors of earlier pairs
        unsigned bits = 0, ent = 0;
        if (!end) {
            // 32 j's, two tiles (the lane's share as a 32-bit offset from
            // a uniform base)
            const int cnt = min(32, je - jc);
            const char *pa = (const char *)(pfj + jc), *pb = (const char *)(bwj + jc);
            float A[2];
            PfBeta jw[2][4];
#pragma unroll
            for (int t = 0; t < 2; t++) {
                A[t] = *(const float *)(pa + (unsigned)(256 * t + 16 * col + 4 * comp));
#pragma unroll
                for (int r = 0; r < 4; r++)
                    jw[t][r] = *(const PfBeta *)(pb + (unsigned)(128 * t + 8 * (row0 + r)));
            }
            double2 s0, s1 = {0.0, 0.0};
            int rank = 0;
            if (mixed) {
                s0 = stage_load<2>(recj + jc, lane, 0, 31);
            } else {
                s0 = stage_load<4>(recj + jc, lane, 0, 31);
                s1 = stage_load<4>(recj + jc, lane, 16, 31);
                if (RANKED) rank = vp->origS[jc + (lane & 31)].rank;
            }
#pragma unroll
            for (int t = 0; t < 2; t++) {
                if (16 * t >= cnt) {
                    bits <<= 16;
                    continue;
                }
#pragma unroll
                for (int b = 0; b < 4; b++) {
                    const v4f o = {0.0f, 0.0f, 0.0f, 0.0f};
                    const v4f X =
                        __builtin_amdgcn_mfma_f32_16x16x4f32(A[t], blk[b].X, o, 0, 0, 0);
                    const v4f U =
                        __builtin_amdgcn_mfma_f32_16x16x4f32(A[t], blk[b].P, o, 0, 0, 0);
                    const v4f V =
                        __builtin_amdgcn_mfma_f32_16x16x4f32(A[t], blk[b].M, o, 0, 0, 0);
#pragma unroll
                    for (int r = 0; r < 4; r++) {
                        const float m = pf_test(X[r], U[r], V[r], ilo[b], ihi[b], jw[t][r].lo,
                                                jw[t][r].hi, pk);
                        // bits << 1 | sign of m
                        bits = __builtin_amdgcn_alignbit(bits, __builtin_bit_cast(unsigned, m),
                                                         31);
                    }
                }
            }
            bits &= cols;
            if (cnt < 32)  // rows past the segment's end
                bits &= rows_first(cnt - row0) << 16 | rows_first(cnt - 16 - row0);
            if (!mixed && jc < (int)w.i0 + 64) {
                // the tile's own particles: only j > i
                const int d0 = (int)w.i0 - jc + col - row0 + 1;
                unsigned keep = 0;
#pragma unroll
                for (int t = 0; t < 2; t++)
#pragma unroll
                    for (int b = 0; b < 4; b++)
                        keep = keep << 4 | 0xfu >> min(max(d0 + 16 * b - 16 * t, 0), 4);
                bits &= keep;
            }
            buf ^= 1u;
            ent = buf << 11 | (unsigned)row0 << 6 | (unsigned)col;
            __builtin_amdgcn_wave_barrier();
            if (mixed) {
                stage_store<2>(wl.jrec[buf], lane, 0, s0);
                if (lane == 0) wl.rot[buf] = rot;
            } else {
                stage_store<4>(wl.jrec[buf], lane, 0, s0);
                stage_store<4>(wl.jrec[buf], lane, 16, s1);
                if (RANKED && lane < 32) wl.jrank[buf][lane] = rank;
            }
            jc += 32;
        }
        for (;;) {
            // queue one survivor of each lane that has any
            unsigned long long m;
            while ((m = __ballot(bits != 0u)) != 0ull && tail - head < 64u) {
                const unsigned pos = __builtin_amdgcn_mbcnt_hi(
                    (unsigned)(m >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)m, tail));
                if (bits != 0u) {
                    const unsigned p = (unsigned)__builtin_clz(bits);  // 16 t + 4 b + r
                    bits &= ~(0x80000000u >> p);
                    wl.ring[pos & 127u] = (unsigned short)(ent + (((p & 16u) | (p & 3u)) << 6) +
                                                           ((p & 12u) << 2));
                }
                tail += (unsigned)__popcll(m);
            }
            // a full wave; or, with nothing left to queue, the survivors
            // whose j buffer the next pair takes (at the end: all)
            const unsigned n = tail - head;
            if (n < 64u && (m != 0ull || (end ? n == 0u : (int)(mark - head) <= 0))) break;
            const int take = (int)min(64u, n);
            __builtin_amdgcn_wave_barrier();
            CArgs *kd = kernel_args();
            unsigned long long unsure = 0, cos64 = 0;
            int nb = drain<Prec, EXT, RANKED>(Views::at(kd, w.view), kd, wl, stg, head, take, mixed,
                                              psi, tot.slab_next, tot.slab_lim, tot.qlds, tot.direct,
                                              unsure, cos64);
            if (std::is_same<Prec, float>::value && __builtin_expect(unsure != 0ull, 0)) {
                kd = kernel_args();
                nb += drain_literal<EXT, RANKED>(Views::at(kd, w.view), kd, wl, head, unsure,
                                                 cos64, mixed, psi, tot.direct);
            }
            if (mixed)
                tot.mixed += nb;
            else
                tot.same += nb;
            head += take;
        }
        if (end) break;
    }
    __builtin_amdgcn_wave_barrier();
}

// ---------------------------------------------------------------- kernel
// Persistent: each wave pulls work items from the queue of its XCD (the host
// puts all items of a group in one queue, so a group's particles stay in one
// XCD's L2), then from the next queues in turn, until all are empty.
// Occupancy: four blocks' LDS fill the CU's 160 KB, so four waves per SIMD
// (128 VGPRs, no spills in the hot path); the K_phi / q_inv instance of the
// FP64 form, whose main path is the literal cascade with atan2 and the
// host-defer path, runs at three.
// Headline workload (2.5e10 pairs, 4.8e9 evaluated): 5.4 ms in the precision
// form, of which the prefilter alone 2.6 and the mixed adds' atomic floor 3.3;
// 8.0 ms with scalar tests and records fetched by scattered loads.  Bound by
// vector instructions: 9 a tested pair, some 230 a batch of 64 survivors.
struct TableViews {
    static __device__ __forceinline__ CView *at(CArgs *ka, int view) {
        return view_at(ka->views, view);
    }
};

template <typename Prec, bool EXT>
constexpr int fast_waves_per_eu() {
    return EXT && std::is_same<Prec, double>::value ? 3 : 4;
}

// Dynamic LDS: with slab binning each slab's next record in this block's
// region and (common case) the regions' ends; without it the waves' Stages.
// q_inv histograms of up to kMaxQinvLds bins follow the Stages: three blocks
// with them fill a CU's LDS.
constexpr int kMaxQinvLds = 560;
constexpr size_t kQinvBytes = 24;  // two sums and two counts a bin
inline int qinv_lds_bins(const DevParams &P) {
    const int nq = P.n_KT * P.qnpts;
    return P.qinv && nq <= kMaxQinvLds ? nq : 0;
}
// slabs: of a slab-binned launch, else 0.
inline size_t fast_dynamic_lds(int slabs, bool ext, int qinv_lds) {
    return qinv_lds ? 4 * sizeof(Stage) + kQinvBytes * qinv_lds
           : slabs  ? (size_t)slabs * sizeof(unsigned) * (ext ? 1 : 2) : 4 * sizeof(Stage);
}
// Blocks of an instance that a CU holds at once: as many as its registers
// leave room for (a block has one wave on each of the four SIMDs), and its LDS,
// which is handed out in steps of 1280 bytes.
constexpr size_t kCuLds = 160 * 1024, kLdsStep = 1280;
inline int fast_resident_blocks(bool f32, bool ext, size_t dynamic_lds) {
    const size_t steps = (4 * sizeof(WaveLds) + dynamic_lds + kLdsStep - 1) / kLdsStep;
    const int waves = f32 ? fast_waves_per_eu<float, true>()
                      : ext ? fast_waves_per_eu<double, true>() : fast_waves_per_eu<double, false>();
    return std::min(waves, (int)(kCuLds / kLdsStep / steps));
}

// The block's q_inv histograms: cleared at the kernel's start (null: none), and
// added to the view's at its end.
template <typename Prec, bool EXT>
__device__ __forceinline__ double *qinv_begin(char *dyn_lds, int nq) {
    if (!EXT || !std::is_same<Prec, double>::value || nq == 0) return nullptr;
    double *q = (double *)(dyn_lds + 4 * sizeof(Stage));
    for (int k = threadIdx.x; k < 3 * nq; k += blockDim.x) q[k] = 0.0;
    __syncthreads();
    return q;
}
template <typename Prec, bool EXT>
__device__ __forceinline__ void qinv_end(CView *vp, const double *q, int nq) {
    if (!EXT || !std::is_same<Prec, double>::value || nq == 0) return;
    __syncthreads();
    const unsigned *cnt = (const unsigned *)(q + 2 * nq);
    for (int k = threadIdx.x; k < nq; k += blockDim.x) {
        if (cnt[k]) atomic_add_u64(&vp->H.qinv_count[k], cnt[k]);
        // (not by the count: one that has wrapped may be 0)
        if (q[k] != 0.0) atomic_add_f64(&vp->H.qinv_sum[k], q[k]);
        if (q[nq + k] != 0.0) atomic_add_f64(&vp->H.qinv_num[k], q[nq + k]);
        if (cnt[nq + k]) atomic_add_u64(&vp->H.qinv_den[k], cnt[nq + k]);
    }
}

template <typename Prec, bool EXT>
__global__ __launch_bounds__(256)
__attribute__((amdgpu_waves_per_eu(fast_waves_per_eu<Prec, EXT>()))) void k_fast(FastArgs a) {
    __shared__ WaveLds wave_lds[4];
    extern __shared__ __align__(16) char dyn_lds[];
    unsigned *const slab_next = (unsigned *)dyn_lds;
    unsigned *const slab_lim = EXT ? nullptr : slab_next + a.slab.S;
    const bool slab = a.slab.vals != nullptr;
    if (slab) {
        for (int k = threadIdx.x; k < a.slab.S; k += blockDim.x) {
            slab_next[k] = slab_first(a.slab, k, blockIdx.x);
            if (!EXT) slab_lim[k] = slab_first(a.slab, k, blockIdx.x + 1);
        }
        __syncthreads();
    }
    WaveTotals tot;
    tot.slab_next = slab_next;
    tot.slab_lim = slab_lim;
    const int lane = __lane_id();
    WaveLds &wl = wave_lds[threadIdx.x >> 6];
    Stage &stg = ((Stage *)dyn_lds)[threadIdx.x >> 6];
    const PfConst<float> pk = pf_const<float>(a.P);
    tot.qlds = qinv_begin<Prec, EXT>(dyn_lds, a.qinv_lds);

    const int nq = a.nqueues;
    int wq = xcc_id() & (nq - 1);  // nq is a power of two
    int queues_left = nq;
    for (;;) {
        int it = 0;
        CArgs *ka = kernel_args();
        if (lane == 0) it = atomicAdd(ka->counter + kQueueStride * wq, 1);
        it = __builtin_amdgcn_readfirstlane(__shfl(it, 0));
        const int q0 = ka->qoff[wq];
        if (it >= ka->qoff[wq + 1] - q0) {  // this queue is empty: the next one
            if (--queues_left == 0) break;
            wq = (wq + 1) & (nq - 1);
            continue;
        }
        const WorkItem w = HBT_CONST(WorkItem, ka->items)[q0 + it];
        CView *vp = view_at(ka->views, w.view);
        const double psi = HBT_CONST(double, vp->psi)[w.grp];
        walk_item<Prec, EXT, true, TableViews>(w, vp, psi, pk, wl, stg, tot, [&](int seg) {
            return HBT_CONST(JWin, vp->mwin)[w.j0 + seg];
        });
    }
    // per-wave totals of binned pairs
    CArgs *ka = kernel_args();
    if (lane == 0) {
        if (tot.same) atomic_add_u64(&ka->binned[0], tot.same);
        if (tot.mixed) atomic_add_u64(&ka->binned[1], tot.mixed);
    }
    qinv_end<Prec, EXT>(view_at(ka->views, 0), tot.qlds, ka->qinv_lds);
    if (slab) {
        // the block's demand per slab, for k_slab_bin (which clamps it to the
        // regions' capacity) and for sizing later launches
        if (lane == 0 && tot.direct) atomic_add_u64(&ka->slab.stats[ka->slab.S], tot.direct);
        __syncthreads();
        for (int k = threadIdx.x; k < ka->slab.S; k += blockDim.x)
            ka->slab.sfill[(long long)blockIdx.x * ka->slab.S + k] =
                slab_next[k] - slab_first(ka->slab, k, blockIdx.x);
    }
}

}  // namespace hbt
