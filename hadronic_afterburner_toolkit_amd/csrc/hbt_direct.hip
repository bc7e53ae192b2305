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
struct Kept {
    bool keep;
    double p2, beta;
};
__device__ __forceinline__ Kept list_kept(const GatherArgs &g, long long i) {
    const double px = g.in.px[i], py = g.in.py[i], pz = g.in.pz[i], r = pz / g.in.E[i];
    const double p2 = px * px + py * py, pt = sqrt(p2);
    return Kept{r > g.cut_min && r < g.cut_max && pt >= g.pt.lo && pt <= g.pt.hi, p2,
                fabs(g.boost ? r : pz)};
}

__device__ __forceinline__ void list_store(const GatherArgs &g, double bmax, long long i, int o) {
    const PartRec p{g.in.px[i], g.in.py[i], g.in.pz[i], g.in.E[i],
                    g.in.x[i],  g.in.y[i],  g.in.z[i],  g.in.t[i]};
    g.out.rec[o] = p;
    PfRec32 r;
    float hi;
    pf_make(PfMake{g.mid, g.c_beta, bmax, g.boost, g.qinv}, p.px, p.py, p.pz, p.E, r, hi);
    g.out.pf[o] = PfOp{r.px, r.py, r.nrm, 1.0f};
    // (the beta window holds for E > 0; other particles take the cascade's word)
    g.out.bw[o] = p.E > 0.0 ? PfBeta{r.blo, hi} : PfBeta{-INFINITY, INFINITY};
}

__device__ __forceinline__ double wave_max(double v) {
    for (int off = 32; off > 0; off >>= 1) v = fmax(v, __shfl_down(v, off));
    return v;
}

// Kept particles per event, and the scales: one block per event.
__global__ __launch_bounds__(256) void k_gather_count(GatherArgs g) {
    const int e = blockIdx.x;
    const long long b = g.ev_off[e], n = g.ev_off[e + 1] - b;
    int c = 0;
    double p2 = 0.0, be = 0.0;
    for (long long i = threadIdx.x; i < n; i += blockDim.x) {
        const Kept k = list_kept(g, b + i);
        if (!k.keep) continue;
        c++;
        p2 = fmax(p2, k.p2);
        be = fmax(be, k.beta);
    }
    for (int off = 32; off > 0; off >>= 1) c += __shfl_down(c, off);
    p2 = wave_max(p2);
    be = wave_max(be);
    __shared__ int pc[4];
    __shared__ double pp[4], pb[4];
    const int w = threadIdx.x >> 6;
    if (__lane_id() == 0) pc[w] = c, pp[w] = p2, pb[w] = be;
    __syncthreads();
    if (threadIdx.x == 0) {
        g.out.cnt[e] = pc[0] + pc[1] + pc[2] + pc[3];
        g.out.pmax2[e] = fmax(fmax(pp[0], pp[1]), fmax(pp[2], pp[3]));
        g.out.bmax[e] = fmax(fmax(pb[0], pb[1]), fmax(pb[2], pb[3]));
    }
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
__device__ __forceinline__ double block_max(double v, double *s) {
    v = wave_max(v);
    __syncthreads();
    if (__lane_id() == 0) s[threadIdx.x >> 6] = v;
    __syncthreads();
    double m = 0.0;
    for (int k = 0; k < (int)(blockDim.x >> 6); k++) m = fmax(m, s[k]);
    return m;
}

// Exclusive scan of the kept counts into event offsets, and the head: one
// block of 1024 threads, each summing a run of ceil(nev/1024) events.
// (Offsets are clamped to the list's capacity, so a caller whose n_particles
// understates its events cannot make a kernel reach past it.)
__global__ __launch_bounds__(1024) void k_gather_scan(GatherArgs g) {
    __shared__ int sc[1024];
    __shared__ double sm[16];
    const int t = threadIdx.x, nev = g.nev;
    const int per = (nev + 1023) / 1024;
    const int a = min(nev, t * per), b = min(nev, a + per);
    long long sum = 0;
    double p2 = 0.0, be = 0.0;
    for (int e = a; e < b; e++) {
        sum = min(sum + g.out.cnt[e], (long long)g.out.cap);
        p2 = fmax(p2, g.out.pmax2[e]);
        be = fmax(be, g.out.bmax[e]);
    }
    const int cap = g.out.cap;  // (1024 runs of at most 2^20 stay below 2^31)
    const int incl = block_scan((int)sum, sc);
    int run = incl - (int)sum;
    for (int e = a; e < b; e++) {
        g.out.koff[e] = min(run, cap);
        run = min(run + g.out.cnt[e], cap);
    }
    p2 = block_max(p2, sm);
    be = block_max(be, sm);
    if (t == 1023) {
        const int n = min(incl, cap);
        g.out.koff[nev] = n;
        *g.out.head = ListHead{p2, be, n, 0};
    }
}

// Order-preserving compaction of each event's kept particles to its kept
// offset (the reference's gather order: event by event, particle order).
__global__ __launch_bounds__(256) void k_gather_compact(GatherArgs g) {
    const int e = blockIdx.x;
    const long long b = g.ev_off[e], n = g.ev_off[e + 1] - b;
    __shared__ int wsum[4];
    int base = g.out.koff[e];
    const double bmax = g.out.head->bmax;
    const int w = threadIdx.x >> 6;
    for (long long c0 = 0; c0 < n; c0 += 256) {
        const long long i = c0 + threadIdx.x;
        const bool keep = i < n && list_kept(g, b + i).keep;
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
        if (keep && o < g.out.cap) list_store(g, bmax, b + i, o);
        base = min(base + total, g.out.cap);
        __syncthreads();  // wsum is rewritten by the next chunk
    }
}

// The same in one launch for a small buffer: one block, each thread a run of
// consecutive particles (of a call of 32 us with two launches, a third and a
// fourth would be a large part).
__global__ __launch_bounds__(1024) void k_gather_small(GatherArgs g) {
    __shared__ int sc[1024];
    __shared__ double sm[16];
    __shared__ int koff[kGatherSmall + 1];  // kept before each particle
    const int t = threadIdx.x;
    const long long b = g.ev_off[0];
    const int n = (int)min(g.ev_off[g.nev] - b, (long long)kGatherSmall);
    const int per = (n + 1023) / 1024, i0 = min(n, t * per), i1 = min(n, i0 + per);
    unsigned keep = 0;  // per <= 8
    double p2 = 0.0, be = 0.0;
    for (int i = i0; i < i1; i++) {
        const Kept k = list_kept(g, b + i);
        if (!k.keep) continue;
        keep |= 1u << (i - i0);
        p2 = fmax(p2, k.p2);
        be = fmax(be, k.beta);
    }
    const int c = __popc(keep), incl = block_scan(c, sc);
    p2 = block_max(p2, sm);
    be = block_max(be, sm);
    int run = incl - c;
    for (int i = i0; i < i1; i++) {
        koff[i] = run;
        run += keep >> (i - i0) & 1u;
    }
    if (t == 1023) koff[n] = incl;
    for (int i = i0, o = incl - c; i < i1; i++)
        if (keep >> (i - i0) & 1u) list_store(g, be, b + i, o++);
    __syncthreads();
    for (int e = t; e <= g.nev; e += 1024)
        g.out.koff[e] = koff[(int)max(0ll, min(g.ev_off[e] - b, (long long)n))];
    if (t == 1023) *g.out.head = ListHead{p2, be, incl, 0};
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
    const int n = HBT_CONST(ListHead, g.ha)->n;
    const HBT_AS4 int *ka = HBT_CONST(int, g.koff_a), *kb = HBT_CONST(int, g.koff_b);
    DevParams P = g.v.P;
    prefilter_margins(fmax(HBT_CONST(ListHead, g.ha)->pmax2, HBT_CONST(ListHead, g.hb)->pmax2), P);
    const PfConst<float> pk = pf_const<float>(P);
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
        hipLaunchKernelGGL(k_gather_scan, dim3(1), dim3(1024), 0, st, g);
        hipLaunchKernelGGL(k_gather_compact, dim3(g.nev), dim3(256), 0, st, g);
    }
    return hipGetLastError();
}

hipError_t launch_pairs(const PairArgs &p, bool f32, bool ext, hipStream_t st) {
    if (p.nitems <= 0) return hipSuccess;
    const dim3 blocks((unsigned)std::min<long long>((p.nitems + 3) / 4, 2 * kWaves / 4));
    const size_t dyn = fast_dynamic_lds(p.f.slab, ext, p.f.qinv_lds);
    // (with the q_inv branch on every pair takes the literal cascade)
    f32 = f32 && !p.v.P.qinv;
    if (f32 && ext) hipLaunchKernelGGL((k_pairs<float, true>), blocks, dim3(256), dyn, st, p);
    if (f32 && !ext) hipLaunchKernelGGL((k_pairs<float, false>), blocks, dim3(256), dyn, st, p);
    if (!f32 && ext) hipLaunchKernelGGL((k_pairs<double, true>), blocks, dim3(256), dyn, st, p);
    if (!f32 && !ext) hipLaunchKernelGGL((k_pairs<double, false>), blocks, dim3(256), dyn, st, p);
    return hipGetLastError();
}

}  // namespace hbt
