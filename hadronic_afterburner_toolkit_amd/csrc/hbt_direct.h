// hbt_direct.h -- pairs of one buffer without host-built lists: a gather on the
// device and a pair kernel whose work items follow from the kept offsets.
// Used by the allocation-free entry point and by the engine's one-buffer path.
//
// The gather keeps the particles a binned pair can contain (rapidity cut, and
// |pT| within reach of a K_T bin), in order, as the fast kernel's records and
// prefilter operands.  The pair kernel walks them like k_fast, in items of 64
// i particles: every pair takes the matrix-core prefilter, its survivors the
// exact cascade, 64 at a time.  There are no momentum windows, so it tests
// about five times the pairs that k_fast does on sorted lists, at 0.3 ps each:
// the kernel by itself is the slower one at a narrow q window or from some 3e8
// pairs on (20 events of 600 particles, 1.5e8 pairs, q_max 0.15: 160 us against
// k_fast's 167; 50 of 600, 9e8: 732 against 696, and 464 against 233 at 0.05),
// but sorting, windows and items on the host cost several times the kernel.
#pragma once
#include "hbt_fast.h"
#include "hbt_internal.h"

namespace hbt {

constexpr int kGatherSmall = 2048;  // particles gathered by one block in one launch

// With q_inv bins: the room, relative to H^2, that the prefilter's windows leave
// for particles off one mass shell (pair_consts).
constexpr double kQinvRoom = 1e-3;
__host__ __device__ inline double qinv_h2(double H) {
    const double Hm = H * (1.0 + 1e-9) + 1e-12;
    return Hm * Hm * (1.0 + kQinvRoom) + 1e-12;
}

// The scales of a gathered list, or of one event of it: largest |pT|^2 and
// |beta|, smallest and largest E^2 - p^2, and the number of particles.
struct ListStat {
    double pmax2, bmax, m2lo, m2hi;
    int n;
};

__host__ __device__ __forceinline__ ListStat stat_none() {
    return ListStat{0.0, 0.0, INFINITY, -INFINITY, 0};
}
__host__ __device__ __forceinline__ ListStat stat_join(const ListStat &a, const ListStat &b) {
    return ListStat{fmax(a.pmax2, b.pmax2), fmax(a.bmax, b.bmax), fmin(a.m2lo, b.m2lo),
                    fmax(a.m2hi, b.m2hi), a.n + b.n};
}

// The prefilter's constants for two lists' scales.  With q_inv bins a pair
// that bins in either kind of histogram has |q_side| and |q_long| within
// sqrt(1 + kQinvRoom) H, but no bound on q_out, so the kernel tests
// C^2 <= H^2 T alone (dn = 0).  For q_inv: in the LCMS q_E M_t = K_T q_out + d
// with d = (m1^2 - m2^2) / 2, so q_inv^2 = q_side^2 + q_long^2 +
// q_out^2 - q_E^2 and the smallest value of the last two, over all q_out, is
// -d^2 / K^2 with K^2 = (m1^2 + m2^2) / 2 + q_inv^2 / 4 at least the lists'
// smallest m^2.  Where the lists' m^2 = E^2 - p^2 differ too much for the room,
// every pair in the K_T window takes the cascade, as all did before: 435 us for
// 20 events of 200 particles, 105 with the windows.
__host__ __device__ __forceinline__ PfConst<float> pair_consts(DevParams P, const ListStat &st) {
    if (!P.qinv) {
        prefilter_margins(st.pmax2, P);
        return pf_const<float>(P);
    }
    const double d = 0.5 * (st.m2hi - st.m2lo), H = fmax(fabs(P.q_lo_cut), fabs(P.q_hi_cut));
    const bool windows = st.m2lo > 0.0 && d * d <= 0.5 * kQinvRoom * H * H * st.m2lo;
    if (windows) {
        P.qinv = 0;
        P.pf_h2 = qinv_h2(H);
        prefilter_margins(st.pmax2, P);
        PfConst<float> k = pf_const<float>(P);
        k.dn = 0.0f;
        return k;
    }
    prefilter_margins(st.pmax2, P);
    PfConst<float> k = pf_const<float>(P);
    k.wide = INFINITY;
    return k;
}

// A gathered list: event e is [koff[e], koff[e + 1]).  rec, pf and bw have
// kPfPad entries past cap; stat is per event.
struct List {
    ListStat *head;
    int *koff;
    ListStat *stat;
    PartRec *rec;
    PfOp *pf;
    PfBeta *bw;
    int cap;
};

struct GatherArgs {
    const long long *ev_off;
    DevSoA in;
    double cut_min, cut_max;  // tanh of the rapidity bounds
    PtRange pt;
    double mid, c_beta;
    int boost, qinv;
    int nev;
    List out;
};

// Item k < nsame: i tile k / nchunk against its chunk k % nchunk of the list's
// j's; then the mixed items: event, i tile of it, and a run of at most `rows`
// of its M plan rows.
struct PairArgs {
    FastArgs f;  // first (kernel_args): the binned counters, no slabs
    View v;      // the lists A and B, the histograms and the grid constants
    const ListStat *ha, *hb;
    const int *koff_a, *koff_b;
    const int *ids;  // partner of each plan row; outside [0, nev_b): no pairs
    double psi;
    int nev_b, M;
    int jchunk, nchunk;     // same-event: j's per item, items per i tile
    int tiles, rows, runs;  // mixed: i tiles per event, rows per item, items per tile
    long long nsame, nitems;
};

// The grid-dependent part of GatherArgs.
inline void gather_setup(const Derived &d, const hbt_config &k, GatherArgs &g) {
    g.cut_min = std::tanh(k.HBTrap_min);
    g.cut_max = std::tanh(k.HBTrap_max);
    g.pt = fast_pt_range(d);
    g.mid = d.P.pf_mid;
    g.boost = d.P.boost;
    g.qinv = d.P.qinv;
    g.c_beta = d.P.qinv ? 0.5 * std::sqrt(qinv_h2(d.H)) * (1.0 + 1e-9) : d.c_beta;
}

// The lists and histograms of a pair launch.
inline void pair_lists(PairArgs &p, const List &a, const List &b) {
    p.v.A = p.v.AS = a.rec;
    p.v.pfA = p.v.pfS = a.pf;
    p.v.bwA = p.v.bwS = a.bw;
    p.v.B = b.rec;
    p.v.pfB = b.pf;
    p.v.bwB = b.bw;
    p.ha = a.head;
    p.hb = b.head;
    p.koff_a = a.koff;
    p.koff_b = b.koff;
}

// The items of n particles in nev events of at most max_event, M plan rows an
// event (0: no mixed items).
void pair_items(PairArgs &p, long long n, long long nev, long long max_event, bool same, int M);

// Kernel launches on st only (they can be captured).  n: particles passed in.
hipError_t launch_gather(const GatherArgs &g, long long n, hipStream_t st);
hipError_t launch_pairs(const PairArgs &p, bool f32, bool ext, hipStream_t st);

}  // namespace hbt
