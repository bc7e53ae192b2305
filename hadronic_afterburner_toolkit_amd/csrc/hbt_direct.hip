// hbt_direct.hip -- the gather and pair kernels of hbt_direct.h.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstddef>

#include "hbt_direct.h"

namespace {

using namespace hbt;

constexpr long long kWaves = 4096;  // the pair kernel's resident waves (256 CUs x 16)

// A particle of the list: tanh(HBTrap_min) < pz/E < tanh(HBTrap_max)
// (HBT_correlation.cpp:255-266), and |pT| as a binnable pair needs it.
__device__ __forceinline__ bool list_kept(const GatherArgs &g, long long i, ListStat &st) {
    const double px = g.in.px[i], py = g.in.py[i], pz = g.in.pz[i], E = g.in.E[i], r = pz / E;
    const double p2 = px * px + py * py, pt = sqrt(p2), m2 = E * E - p2 - pz * pz;
    const bool keep = r > g.cut_min && r < g.cut_max && pt >= g.pt.lo && pt <= g.pt.hi;
    if (keep) st = stat_join(st, ListStat{p2, fabs(g.boost ? r : pz), m2, m2, 1});
    return keep;
}

__device__ __forceinline__ void list_store(const GatherArgs &g, double bmax, long long i, int o) {
    const PartRec p{g.in.px[i], g.in.py[i], g.in.pz[i], g.in.E[i],
                    g.in.x[i],  g.in.y[i],  g.in.z[i],  g.in.t[i]};
    g.out.rec[o] = p;
    PfRec32 r;
    float hi;
    pf_make(PfMake{g.mid, g.c_beta, bmax, g.boost, 0}, p.px, p.py, p.pz, p.E, r, hi);
    g.out.pf[o] = PfOp{r.px, r.py, r.nrm, 1.0f};
    // (with q_inv bins and no LCMS boost q_long is not the LCMS one: no window)
    g.out.bw[o] = !g.qinv || g.boost ? PfBeta{r.blo, hi} : PfBeta{-INFINITY, INFINITY};
}

// The block's join of its threads' statistics (in every thread).
template <int N>
__device__ __forceinline__ ListStat block_stat(ListStat v) {
    __shared__ ListStat part[N / 64];
    for (int off = 32; off > 0; off >>= 1)
        v = stat_join(v, ListStat{__shfl_down(v.pmax2, off), __shfl_down(v.bmax, off),
                                  __shfl_down(v.m2lo, off), __shfl_down(v.m2hi, off),
                                  __shfl_down(v.n, off)});
    __syncthreads();
    if (__lane_id() == 0) part[threadIdx.x >> 6] = v;
    __syncthreads();
    v = part[0];
    for (int k = 1; k < N / 64; k++) v = stat_join(v, part[k]);
    return v;
}

// Kept particles per event, and the scales: one block per event.
__global__ __launch_bounds__(256) void k_gather_count(GatherArgs g) {
    const int e = blockIdx.x;
    const long long b = g.ev_off[e], n = g.ev_off[e + 1] - b;
    ListStat st = stat_none();
    for (long long i = threadIdx.x; i < n; i += blockDim.x) list_kept(g, b + i, st);
    st = block_stat<256>(st);
    if (threadIdx.x == 0) g.out.stat[e] = st;
}

// Inclusive scan over the 1024 threads of a block.
__device__ __forceinline__ int block_scan(int v, int *s) {
    const int t = threadIdx.x;
    s[t] = v;
    __syncthreads();
    for (int off = 1; off < 1024; off <<= 1) {  // Hillis-Steele
        const int x = t >= off ? s[t - off] : 0;
        __syncthreads();
        s[t] += x;
        __syncthreads();
    }
    return s[t];
}

// Exclusive scan of the kept counts into event offsets, and the head: one
// block of 1024 threads, each summing a run of ceil(nev/1024) events.
// (Offsets are clamped to the list's capacity, so a caller whose n_particles
// understates its events cannot make a kernel reach past it.)
__global__ __launch_bounds__(1024) void k_gather_scan(GatherArgs g) {
    __shared__ int sc[1024];
    const int t = threadIdx.x, nev = g.nev, cap = g.out.cap;
    const int per = (nev + 1023) / 1024;
    const int a = min(nev, t * per), b = min(nev, a + per);
    ListStat st = stat_none();
    for (int e = a; e < b; e++) {
        ListStat x = g.out.stat[e];
        x.n = min(x.n, cap - st.n);
        st = stat_join(st, x);
    }
    const int incl = block_scan(st.n, sc);  // (1024 runs of at most 2^20 stay below 2^31)
    int run = incl - st.n;
    for (int e = a; e < b; e++) {
        g.out.koff[e] = min(run, cap);
        run = min(run + g.out.stat[e].n, cap);
    }
    st = block_stat<1024>(st);
    if (t == 1023) {
        st.n = min(incl, cap);
        g.out.koff[nev] = st.n;
        *g.out.head = st;
    }
}

// Order-preserving compaction of each event's kept particles to its kept
// offset (the reference's gather order: event by event, particle order).
// SCAN: each block sums the counts before its event itself, which spares up
// to kScanEvents events the launch of the scan; the list's length and scales
// are the last event's block's to write.
constexpr int kScanEvents = 1024;
template <bool SCAN>
__global__ __launch_bounds__(256) void k_gather_compact(GatherArgs g) {
    const int e = blockIdx.x, cap = g.out.cap;
    const long long b = g.ev_off[e], n = g.ev_off[e + 1] - b;
    __shared__ int wsum[4];
    int base;
    double bmax;
    if (SCAN) {
        ListStat st = stat_none(), mine = st;
        for (int k = threadIdx.x; k < g.nev; k += 256) {
            ListStat x = g.out.stat[k];
            x.n = min(x.n, cap);  // (1024 of at most 2^20 stay below 2^31)
            if (k < e) mine.n += x.n;
            st = stat_join(st, x);
        }
        const int before = block_stat<256>(mine).n;
        st = block_stat<256>(st);
        st.n = min(st.n, cap);
        base = min(before, cap);
        bmax = st.bmax;
        if (threadIdx.x == 0) {
            g.out.koff[e] = base;
            if (e == g.nev - 1) {
                g.out.koff[g.nev] = st.n;
                *g.out.head = st;
            }
        }
    } else {
        base = g.out.koff[e];
        bmax = g.out.head->bmax;
    }
    const int w = threadIdx.x >> 6;
    for (long long c0 = 0; c0 < n; c0 += 256) {
        const long long i = c0 + threadIdx.x;
        ListStat st = stat_none();
        const bool keep = i < n && list_kept(g, b + i, st);
        const unsigned long long mk = __ballot(keep);
        const int rank = __builtin_amdgcn_mbcnt_hi((unsigned)(mk >> 32),
                                                   __builtin_amdgcn_mbcnt_lo((unsigned)mk, 0u));
        if (__lane_id() == 0) wsum[w] = __popcll(mk);
        __syncthreads();
        int before = 0, total = 0;
        for (int k = 0; k < 4; k++) {
            before += k < w ? wsum[k] : 0;
            total += wsum[k];
        }
        const int o = base + before + rank;
        if (keep && o < cap) list_store(g, bmax, b + i, o);
        base = min(base + total, cap);
        __syncthreads();  // wsum is rewritten by the next chunk
    }
}

// The same in one launch for a small buffer: one block, each thread a run of
// consecutive particles (630 particles: a call of 35 us, of which a second
// launch would be a large part; 4000: 33 us against 18 with a block per event).
__global__ __launch_bounds__(1024) void k_gather_small(GatherArgs g) {
    __shared__ int sc[1024];
    __shared__ int koff[kGatherSmall + 1];  // kept before each particle
    const int t = threadIdx.x;
    const long long b = g.ev_off[0];
    const int n = (int)min(g.ev_off[g.nev] - b, (long long)kGatherSmall);
    const int per = (n + 1023) / 1024, i0 = min(n, t * per), i1 = min(n, i0 + per);
    unsigned keep = 0;  // per <= 2
    ListStat st = stat_none();
    for (int i = i0; i < i1; i++)
        if (list_kept(g, b + i, st)) keep |= 1u << (i - i0);
    const int c = __popc(keep), incl = block_scan(c, sc);
    st = block_stat<1024>(st);
    int run = incl - c;
    for (int i = i0; i < i1; i++) {
        koff[i] = run;
        run += keep >> (i - i0) & 1u;
    }
    if (t == 1023) koff[n] = incl;
    for (int i = i0, o = incl - c; i < i1; i++)
        if (keep >> (i - i0) & 1u) list_store(g, st.bmax, b + i, o++);
    __syncthreads();
    for (int e = t; e <= g.nev; e += 1024)
        g.out.koff[e] = koff[(int)max(0ll, min(g.ev_off[e] - b, (long long)n))];
    if (t == 1023) *g.out.head = st;
}

// The pair kernel's view: its own argument.
struct ArgView {
    static __device__ __forceinline__ CView *at(CArgs *ka, int) {
        return (CView *)((const HBT_AS4 char *)ka + offsetof(PairArgs, v));
    }
};

// Bound by the adds' atomics (2.35e10 binned same-event and 2.68e10 mixed pairs
// per second, memory side) where more than a percent of the pairs bins, else
// by the prefilter's vector operations.
template <typename Prec, bool EXT>
__global__ __launch_bounds__(256)
__attribute__((amdgpu_waves_per_eu(fast_waves_per_eu<Prec, EXT>()))) void k_pairs(PairArgs g) {
    __shared__ WaveLds wave_lds[4];
    extern __shared__ __align__(16) char dyn_lds[];
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    WaveLds &wl = wave_lds[wv];
    Stage &stg = ((Stage *)dyn_lds)[wv];
    WaveTotals tot;
    tot.slab_next = nullptr;
    tot.slab_lim = nullptr;
    CView *vp = ArgView::at(kernel_args(), 0);
    const int n = HBT_CONST(ListStat, g.ha)->n;
    const HBT_AS4 int *ka = HBT_CONST(int, g.koff_a), *kb = HBT_CONST(int, g.koff_b);
    const PfConst<float> pk = pair_consts(
        g.v.P, stat_join(*(const ListStat *)g.ha, *(const ListStat *)g.hb));
    const double psi = g.psi;
    tot.qlds = qinv_begin<Prec, EXT>(dyn_lds, g.f.qinv_lds);
    for (long long it = (long long)blockIdx.x * 4 + wv; it < g.nitems;
         it += (long long)gridDim.x * 4) {
        WorkItem w{};
        if (it < g.nsame) {
            const int i0 = (int)(it / g.nchunk) * 64;
            const int j0 = i0 + (int)(it % g.nchunk) * g.jchunk;
            w.ni = min(64, n - i0);
            w.nj = min(g.jchunk, n - j0);
            if (w.ni <= 0 || w.nj <= 0) continue;
            w.i0 = i0;
            w.j0 = j0;
        } else {
            const long long k = it - g.nsame;
            const int r = (int)(k % g.runs) * g.rows, tile = (int)(k / g.runs % g.tiles);
            const int e = (int)(k / g.runs / g.tiles);
            w.kind = 1;
            w.i0 = ka[e] + tile * 64;
            w.ni = min(64, ka[e + 1] - (int)w.i0);
            w.nj = min(g.rows, g.M - r);
            if (w.ni <= 0 || w.nj <= 0) continue;
            w.j0 = (long long)e * g.M + r;  // its first plan row
        }
        walk_item<Prec, EXT, false, ArgView>(w, vp, psi, pk, wl, stg, tot, [&](int seg) {
            const int row = (int)w.j0 + seg;
            const int pid = HBT_CONST(int, g.ids)[row];
            const bool ok = pid >= 0 && pid < g.nev_b;
            return JWin{ok ? kb[pid] : 0, ok ? kb[pid + 1] : 0, row, 0};
        });
    }
    if (g.f.binned && __lane_id() == 0) {
        if (tot.same) atomic_add_u64(&g.f.binned[0], tot.same);
        if (tot.mixed) atomic_add_u64(&g.f.binned[1], tot.mixed);
    }
    qinv_end<Prec, EXT>(vp, tot.qlds, g.f.qinv_lds);
}

}  // namespace

namespace hbt {

void pair_items(PairArgs &p, long long n, long long nev, long long max_event, bool same, int M) {
    // 64 i's against about 1024 j's (a chunk of the list, or several plan
    // rows' partners), where an item's own cost, some 750 cycles, is below a
    // tenth of its pairs'; finer, down to 64 j's or one row, while that leaves
    // waves of the chip idle.
    const long long tiles = (n + 63) / 64;
    p.jchunk = 1024;
    while (p.jchunk > 64 && tiles * ((n + p.jchunk - 1) / p.jchunk) < 2 * kWaves) p.jchunk /= 2;
    p.nchunk = (int)std::max(1ll, (n + p.jchunk - 1) / p.jchunk);
    p.nsame = same ? tiles * p.nchunk : 0;
    p.M = M;
    p.tiles = p.rows = p.runs = 1;
    p.nitems = p.nsame;
    if (M <= 0 || max_event <= 0) return;
    p.tiles = (int)((max_event + 63) / 64);
    p.rows = (int)std::max(1ll, std::min<long long>(M, 1024 / max_event));
    const long long ev_tiles = nev * p.tiles;
    while (p.rows > 1 && ev_tiles * ((M + p.rows - 1) / p.rows) < 2 * kWaves) p.rows /= 2;
    p.runs = (M + p.rows - 1) / p.rows;
    p.nitems += ev_tiles * p.runs;
}

hipError_t launch_gather(const GatherArgs &g, long long n, hipStream_t st) {
    if (n <= kGatherSmall) {
        hipLaunchKernelGGL(k_gather_small, dim3(1), dim3(1024), 0, st, g);
    } else {
        hipLaunchKernelGGL(k_gather_count, dim3(g.nev), dim3(256), 0, st, g);
        if (g.nev <= kScanEvents) {
            hipLaunchKernelGGL(k_gather_compact<true>, dim3(g.nev), dim3(256), 0, st, g);
        } else {
            hipLaunchKernelGGL(k_gather_scan, dim3(1), dim3(1024), 0, st, g);
            hipLaunchKernelGGL(k_gather_compact<false>, dim3(g.nev), dim3(256), 0, st, g);
        }
    }
    return hipGetLastError();
}

hipError_t launch_pairs(const PairArgs &p, bool f32, bool ext, hipStream_t st) {
    if (p.nitems <= 0) return hipSuccess;
    const dim3 blocks((unsigned)std::min<long long>((p.nitems + 3) / 4, 2 * kWaves / 4));
    const size_t dyn = fast_dynamic_lds(0, ext, p.f.qinv_lds);
    // (with the q_inv branch on every pair takes the literal cascade)
    f32 = f32 && !p.v.P.qinv;
    if (f32 && ext) hipLaunchKernelGGL((k_pairs<float, true>), blocks, dim3(256), dyn, st, p);
    if (f32 && !ext) hipLaunchKernelGGL((k_pairs<float, false>), blocks, dim3(256), dyn, st, p);
    if (!f32 && ext) hipLaunchKernelGGL((k_pairs<double, true>), blocks, dim3(256), dyn, st, p);
    if (!f32 && !ext) hipLaunchKernelGGL((k_pairs<double, false>), blocks, dim3(256), dyn, st, p);
    return hipGetLastError();
}

}  // namespace hbt
