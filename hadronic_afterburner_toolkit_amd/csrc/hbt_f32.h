// hbt_f32.h -- exact stage of the precision form (HBT_PREC_FP32C).
//
// On CDNA4 an unpacked FP32 add/mul/fma issues at the same rate as its FP64
// form, so FP32 only pays where FP64 needs a multi-instruction sequence:
// division, square root and cos.  The precision form therefore keeps the
// pair's momentum sums/differences and products in FP64, takes reciprocal
// square roots from v_rsq_f64 (one instruction, ~2^-23) refined by one Newton
// step in FP64, and evaluates cos on the FP32 unit after an FP64 Cody-Waite
// reduction to [-pi, pi].  All survivors of the FP32 prefilter come here, and
// nearly all of them are binned, so the cascade has no early exits: every
// lane computes its four bin coordinates, one test says whether any lies too
// near an edge, one whether all are in range.
//
// Bit-identical counts: every bin coordinate (K_T index, bin indices) is
// within 1e-9 bins of the reference's, q_long within 1e-8 GeV besides; a pair
// with a coordinate within the guard (DevParams::guard, which also covers the
// 1e-8 GeV between the windows' cuts and the outer bin edges and the FP32
// rounding of a record's values) of an edge, or of lists with particles of
// larger boosts (boost_guard), is re-run through the literal FP64 cascade
// (eval_*_f64), so bins and counts equal the reference's exactly.  The
// accumulated q values carry ~1e-13 relative error, cos ~1e-7 absolute (FP32
// in slab records); sums are accumulated in FP64 (atomics) or exact fixed
// point (slab binning).
#pragma once
#include "hbt_device.h"

namespace hbt {

// 1/sqrt(a) from v_rsq_f64 (relative error e <= 2^-22) and one Newton step
// in FP64: relative error ~1.5 e^2 < 1e-13, far inside the guard.
__device__ __forceinline__ double rsqrt_refined(double a) {
    const double r = __builtin_amdgcn_rsq(a);
    return r * fma(-0.5 * a * r, r, 1.5);
}

// cos(x): argument reduced to [-pi, pi] in FP64, then split r = rh + rl
// with rh in FP32; cos and sin of rh on FP32 and the first-order
// compensation cos(rh + rl) = cos(rh) - rl sin(rh) (|rl| < 2^-22, so the
// dropped term rl^2/2 is below 1e-13).  Error ~1 FP32 ulp of the result.
template <typename Params>
__device__ __forceinline__ double cos_reduced_f32(const Params &P, double x) {
    const double k = rint(x * P.inv_two_pi);
    const double r = fma(-k, P.two_pi_lo, fma(-k, P.two_pi_hi, x));
    const float rh = (float)r;
    const float rl = (float)(r - (double)rh);
    float s, c;
    sincosf(rh, &s, &c);
    return fma(-(double)rl, (double)s, (double)c);
}

// cos of the pair's phase q.dx (HBT_correlation.cpp:431-436).
template <typename Params>
__device__ __forceinline__ double pair_cos_f32(const Params &P, const PartRec &p1,
                                               const PartRec &p2) {
    const double q_x = p1.px - p2.px, q_y = p1.py - p2.py, q_z = p1.pz - p2.pz;
    const double q_E = p1.E - p2.E;
    return cos_reduced_f32(P, P.hbarC_inv * (q_E * (p1.t - p2.t) - q_x * (p1.x - p2.x) -
                                             q_y * (p1.y - p2.y) - q_z * (p1.z - p2.z)));
}

constexpr double GUARD_PHI = 4e-6;   // radians, around K_phi bin edges

// Whether a pair's coordinates (literal, of a binned pair; T = 4 K_perp^2) lie on
// a bin edge or a window's cut to within 1e-9 bins: its cos is then FP64's.
template <typename Params>
__device__ __forceinline__ bool on_edge(const Params &P, double T, const SameRec &r) {
    const double w[4] = {fma(sqrt(T), P.kt_scale, P.kt_off), fma(r.qo, P.inv_dq, P.q_off),
                         fma(r.qs, P.inv_dq, P.q_off), fma(r.ql, P.inv_dq, P.q_off)};
    bool on = false;
    for (int k = 0; k < 4; k++) {
        const double d = fabs(w[k] - rint(w[k]));
        on = on || d < 1e-9 || (k > 0 && fabs(d - 1e-8 * P.inv_dq) < 1e-9);
    }
    return on;
}

// A bin coordinate raised by one: its integer part, and its distance to the
// nearest integer folded into the smallest so far.
__device__ __forceinline__ int bin_coord(double w, double &nearest) {
    nearest = fmin(nearest, fabs(w - rint(w)));
    return (int)w - 1;
}

// K_phi bin of the precision form (the reference's wrap loops,
// HBT_correlation.cpp:408-423): atan2 on the FP32 unit (error below 1e-6
// rad); an angle within GUARD_PHI of a bin edge, 0 or 2 pi returns -2 and
// the pair is re-run through the literal cascade.
template <typename Params>
__device__ __forceinline__ int kphi_index_fast(const Params &P, double K_x, double K_y,
                                               double psi_ref) {
    double delta = (double)atan2f((float)K_y, (float)K_x) - psi_ref;
    while (delta < 0.) delta += P.two_pi;
    while (delta > P.two_pi) delta -= P.two_pi;
    const double w = delta * P.inv_dKphi;
    const double n = rint(w);
    if (fabs(w - n) * P.dKphi < GUARD_PHI) return -2;
    const int idx = (int)w;
    return (idx < 0 || idx >= P.n_Kphi) ? -2 : idx;
}

// The K/q cascade of the precision form.  Returns ST_BIN with the bins in b,
// 0, or -1 or -2 when a decision is ambiguous (-2: only the K_phi bin is).
// Works on 2K (the reference's K times a power of two: its products round alike).
template <bool EXT = false, typename Params>
__device__ __forceinline__ int cascade_fast(const Params &P, double p1x, double p1y,
                                            double p1z, double p1E, double p2x, double p2y,
                                            double p2z, double p2E, double psi_ref,
                                            PairBins &b) {
    const double sx = p1x + p2x, sy = p1y + p2y, sz = p1z + p2z, sE = p1E + p2E;
    b.q_x = p1x - p2x;
    b.q_y = p1y - p2y;
    b.q_z = p1z - p2z;
    b.q_E = p1E - p2E;
    const double T = sx * sx + sy * sy;  // 4 K_perp^2
    const double rK = rsqrt_refined(T);
    double near = 1.0;
    b.kt = bin_coord(fma(T * rK, P.kt_scale, P.kt_off), near);
    b.q_out = fma(b.q_x, sx, b.q_y * sy) * rK;
    b.q_side = fma(b.q_y, sx, -(b.q_x * sy)) * rK;
    b.q_long = b.q_z;
    if (P.boost) {  // gamma (q_z - beta q_E) = (K_E q_z - K_z q_E) / M_t
        const double rM = rsqrt_refined(fma(sE, sE, -(sz * sz)));
        b.q_long = fma(sE, b.q_z, -(sz * b.q_E)) * rM;
    }
    b.io = bin_coord(fma(b.q_out, P.inv_dq, P.q_off), near);
    b.is = bin_coord(fma(b.q_side, P.inv_dq, P.q_off), near);
    b.il = bin_coord(fma(b.q_long, P.inv_dq, P.q_off), near);
    if (near < P.guard) return -1;
    const unsigned q = max(max((unsigned)b.io, (unsigned)b.is), (unsigned)b.il);
    // (the last K_T index, n_KT - 1, holds only K_perp = KT_max: near an edge)
    if (q >= (unsigned)P.qnpts || (unsigned)b.kt >= (unsigned)(P.n_KT - 1)) return 0;
    b.kphi = 0;
    if (EXT && P.azimuthal) {
        b.kphi = kphi_index_fast(P, sx, sy, psi_ref);
        if (b.kphi < 0) return -2;
    }
    return ST_BIN;
}

// Same-event pair (p1, p2) in the precision form (see eval_same_f64 for the
// contract); negative: ambiguous, the caller takes the literal cascade.
template <bool EXT = true, typename Params>
__device__ __forceinline__ int eval_same_fast(const Params &P, double psi, const PartRec &p1,
                                              const PartRec &p2, SameRec &rec) {
    PairBins b;
    const int st = cascade_fast<EXT>(P, p1.px, p1.py, p1.pz, p1.E, p2.px, p2.py, p2.pz, p2.E, psi,
                                     b);
    if (st != ST_BIN) return st;
    rec.k = bin_index(P, b.kt, b.kphi, b.io, b.is, b.il);
    rec.s = (b.kt * P.nphi + b.kphi) * P.qnpts + b.io;
    rec.is = b.is;
    rec.il = b.il;
    rec.qo = b.q_out;
    rec.qs = b.q_side;
    rec.ql = b.q_long;
    rec.c = pair_cos_f32(P, p1, p2);
    return st;
}

// Mixed pair in the precision form; p2x, p2y are the partner's momentum
// already rotated as the reference does (HBT_correlation.cpp:522-523).  Mixed
// windows are half-open: v < hi (HBT_correlation.cpp:613); the guard around
// the cut sends v == hi to the literal cascade (negative).
template <bool EXT = true, typename Params>
__device__ __forceinline__ int eval_mixed_fast(const Params &P, double psi, double p1x,
                                               double p1y, double p1z, double p1E, double p2x,
                                               double p2y, double p2z, double p2E, long &k) {
    PairBins b;
    const int st = cascade_fast<EXT>(P, p1x, p1y, p1z, p1E, p2x, p2y, p2z, p2E, psi, b);
    if (st == ST_BIN) k = bin_index(P, b.kt, b.kphi, b.io, b.is, b.il);
    return st;
}

}  // namespace hbt
