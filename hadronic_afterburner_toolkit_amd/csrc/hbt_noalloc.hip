// hbt_noalloc.hip -- hbt_calculate_noalloc: the pair loops of one buffer (what
// hbt_upload + hbt_run_same + hbt_run_mixed do, in FP64) for callers that
// cannot allocate device memory: code under HIP graph capture, tight serving
// loops.  The caller passes the particles, the mixing plan and the histogram
// in device memory; the kept particles and all that is derived from them live
// in `scratch`, a file-scope device array of fixed size that each GPU holds
// until the process ends.  No hipMalloc, hipFree or other allocating call is
// made; every launch goes on the caller's stream.
//
// Two steps.  The gather keeps the particles a binned pair can contain
// (rapidity cut, and |pT| within reach of a K_T bin), in order, as the fast
// kernel's records and prefilter operands.  The pair kernel walks them in
// items of 64 i particles like k_fast: every pair takes the matrix-core
// prefilter, its survivors the literal cascade, 64 at a time.  Nothing is
// known of the data on the host, so the items are worked out from the kept
// offsets on the device and there are no momentum windows.
// One literal cascade per enumerated pair, one thread per i particle (the
// form before), cost 1420 us for 20 events of 600 particles (1.5e8 pairs) and
// 335 us for 7 of 90, whose few threads each walked hundreds of pairs one
// after the other; this form takes 168 (140 of them the pair kernel) and 32.
//
// Calls on one GPU share its scratch array: calls that overlap on one GPU
// (two streams, two host threads) race and must be serialized by the caller.
#include <hip/hip_runtime.h>

#include <mutex>
#include <string>

#include "../../include/hbt_hip.h"
#include "hbt_device.h"
#include "hbt_internal.h"

using namespace hbt;

namespace {

constexpr long long kMaxParticles = HBT_NOALLOC_MAX_PARTICLES;
constexpr int kMaxEvents = HBT_NOALLOC_MAX_EVENTS;
constexpr long long kWaves = 4096;     // the pair kernel's resident waves (256 CUs x 16)
constexpr int kSmallParticles = 8192;  // gathered by one block in one launch

// What the gather leaves for the pair kernel, beside the lists.
struct Head {
    View v;                  // the lists and the grid constants (with margins)
    PfMake make;
    double psi;              // 0 (no K_phi bins)
    int n;                   // kept particles
    int koff[kMaxEvents + 1];
};

struct Scratch {
    Head head;
    int cnt[kMaxEvents];     // kept per event, largest |pT|^2 and |beta|
    double pmax2[kMaxEvents], bmax[kMaxEvents];
    alignas(256) PartRec rec[kMaxParticles + kPfPad];
    alignas(256) PfOp pf[kMaxParticles + kPfPad];
    alignas(256) PfBeta bw[kMaxParticles + kPfPad];
};

static __device__ __align__(256) unsigned char scratch[sizeof(Scratch)];

constexpr int kMaxDevices = 64;
std::mutex g_mu;
unsigned char *g_ptr[kMaxDevices] = {};  // device address of scratch, per device
std::string g_err;

int fail(int code, const char *msg) {
    std::lock_guard<std::mutex> lk(g_mu);
    g_err = msg;
    return code;
}

// The device address of this GPU's scratch array, looked up once per device
// with that device current.  The symbol's host-side name is only a handle:
// kernels and copies take this address.
int scratch_ptr(int dev, unsigned char **out) {
    std::lock_guard<std::mutex> lk(g_mu);
    if (!g_ptr[dev]) {
        void *p = nullptr;
        if (hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)) != hipSuccess || !p) {
            g_err = "hipGetSymbolAddress(scratch) failed";
            return HBT_ERR_HIP;
        }
        g_ptr[dev] = (unsigned char *)p;
    }
    *out = g_ptr[dev];
    return HBT_OK;
}

struct GatherArgs {
    const long long *ev_off;
    DevSoA in;
    double cut_min, cut_max;  // tanh of the rapidity bounds
    PtRange pt;
    DevParams P;
    double c_beta;
    double *bins;
    const double *plan_cs;
    int nev;
};

// A particle of the list: tanh(HBTrap_min) < pz/E < tanh(HBTrap_max)
// (HBT_correlation.cpp:255-266), and |pT| as a binnable pair needs it.
struct Kept {
    bool keep;
    double p2, beta;
};
__device__ __forceinline__ Kept na_kept(const GatherArgs &g, long long i) {
    const double px = g.in.px[i], py = g.in.py[i], pz = g.in.pz[i], r = pz / g.in.E[i];
    const double p2 = px * px + py * py, pt = sqrt(p2);
    return Kept{r > g.cut_min && r < g.cut_max && pt >= g.pt.lo && pt <= g.pt.hi, p2,
                fabs(g.P.boost ? r : pz)};
}

__device__ __forceinline__ void na_store(const GatherArgs &g, const PfMake &m, Scratch *s,
                                         long long i, int o) {
    const PartRec p{g.in.px[i], g.in.py[i], g.in.pz[i], g.in.E[i],
                    g.in.x[i],  g.in.y[i],  g.in.z[i],  g.in.t[i]};
    s->rec[o] = p;
    PfRec32 r;
    float hi;
    pf_make(m, p.px, p.py, p.pz, p.E, r, hi);
    s->pf[o] = PfOp{r.px, r.py, r.nrm, 1.0f};
    // (the beta window holds for E > 0; other particles take the cascade's word)
    s->bw[o] = p.E > 0.0 ? PfBeta{r.blo, hi} : PfBeta{-INFINITY, INFINITY};
}

// The head, once the kept count and the momentum scales are known.
__device__ __forceinline__ void na_head(const GatherArgs &g, Scratch *s, int n, double pmax2,
                                        double bmax) {
    Head &h = s->head;
    View v{};
    v.P = g.P;
    prefilter_margins(pmax2, v.P);
    v.H.bins = g.bins;
    v.A = v.B = v.AS = s->rec;
    v.pfA = v.pfB = v.pfS = s->pf;
    v.bwA = v.bwB = v.bwS = s->bw;
    v.plan_cs = g.plan_cs;
    v.psi = &h.psi;
    h.v = v;
    h.make = PfMake{g.P.pf_mid, g.c_beta, bmax, g.P.boost, 0};
    h.psi = 0.0;
    h.n = n;
}

__device__ __forceinline__ double wave_max(double v) {
    for (int off = 32; off > 0; off >>= 1) v = fmax(v, __shfl_down(v, off));
    return v;
}

// Kept particles per event, and the scales: one block per event.
__global__ __launch_bounds__(256) void k_na_count(GatherArgs g, Scratch *s) {
    const int e = blockIdx.x;
    const long long b = g.ev_off[e], n = g.ev_off[e + 1] - b;
    int c = 0;
    double p2 = 0.0, be = 0.0;
    for (long long i = threadIdx.x; i < n; i += blockDim.x) {
        const Kept k = na_kept(g, b + i);
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
        s->cnt[e] = pc[0] + pc[1] + pc[2] + pc[3];
        s->pmax2[e] = fmax(fmax(pp[0], pp[1]), fmax(pp[2], pp[3]));
        s->bmax[e] = fmax(fmax(pb[0], pb[1]), fmax(pb[2], pb[3]));
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
__global__ __launch_bounds__(1024) void k_na_scan(GatherArgs g, Scratch *s) {
    __shared__ int sc[1024];
    __shared__ double sm[16];
    const int t = threadIdx.x, nev = g.nev;
    const int per = (nev + 1023) / 1024;
    const int a = min(nev, t * per), b = min(nev, a + per);
    long long sum = 0;
    double p2 = 0.0, be = 0.0;
    for (int e = a; e < b; e++) {
        sum = min(sum + s->cnt[e], kMaxParticles);
        p2 = fmax(p2, s->pmax2[e]);
        be = fmax(be, s->bmax[e]);
    }
    const int cap = (int)kMaxParticles;
    // (1024 runs of at most 2^18 stay below 2^31)
    const int incl = block_scan((int)sum, sc);
    int run = incl - (int)sum;
    for (int e = a; e < b; e++) {
        s->head.koff[e] = min(run, cap);
        run = min(run + s->cnt[e], cap);
    }
    p2 = block_max(p2, sm);
    be = block_max(be, sm);
    if (t == 1023) {
        const int n = min(incl, cap);
        s->head.koff[nev] = n;
        na_head(g, s, n, p2, be);
    }
}

// Order-preserving compaction of each event's kept particles to its kept
// offset (the reference's gather order: event by event, particle order).
__global__ __launch_bounds__(256) void k_na_compact(GatherArgs g, Scratch *s) {
    const int e = blockIdx.x;
    const long long b = g.ev_off[e], n = g.ev_off[e + 1] - b;
    __shared__ int wsum[4];
    int base = s->head.koff[e];
    const PfMake m = s->head.make;
    const int w = threadIdx.x >> 6;
    for (long long c0 = 0; c0 < n; c0 += 256) {
        const long long i = c0 + threadIdx.x;
        const bool keep = i < n && na_kept(g, b + i).keep;
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
        if (keep && o < (int)kMaxParticles) na_store(g, m, s, b + i, o);
        base = min(base + total, (int)kMaxParticles);
        __syncthreads();  // wsum is rewritten by the next chunk
    }
}

// The same in one launch for a small buffer: one block, each thread a run of
// consecutive particles (of a call of 32 us with two launches, a third and a
// fourth would be a large part).
__global__ __launch_bounds__(1024) void k_na_gather_small(GatherArgs g, Scratch *s) {
    __shared__ int sc[1024];
    __shared__ double sm[16];
    __shared__ int koff[kSmallParticles + 1];  // kept before each particle
    const int t = threadIdx.x;
    const long long b = g.ev_off[0];
    const int n = (int)min(g.ev_off[g.nev] - b, (long long)kSmallParticles);
    const int per = (n + 1023) / 1024, i0 = min(n, t * per), i1 = min(n, i0 + per);
    unsigned keep = 0;  // per <= 8
    double p2 = 0.0, be = 0.0;
    for (int i = i0; i < i1; i++) {
        const Kept k = na_kept(g, b + i);
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
    const PfMake m{g.P.pf_mid, g.c_beta, be, g.P.boost, 0};
    for (int i = i0, o = incl - c; i < i1; i++)
        if (keep >> (i - i0) & 1u) na_store(g, m, s, b + i, o++);
    __syncthreads();
    for (int e = t; e <= g.nev; e += 1024)
        s->head.koff[e] = koff[(int)max(0ll, min(g.ev_off[e] - b, (long long)n))];
    if (t == 1023) na_head(g, s, incl, p2, be);
}

// The pair kernel.  Item k < nsame: i tile k / nchunk against its chunk
// k % nchunk of the list's j's; then the mixed items: event, i tile of it,
// and a run of at most `rows` of its M plan rows.
struct PairArgs {
    const Head *head;
    const int *ids;
    int nev, M;
    int jchunk, nchunk;  // same-event: j's per item, items per i tile
    int tiles, rows, runs;  // mixed: i tiles per event, rows per item, items per tile
    long long nsame, nitems;
};

__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4))) void k_na_pairs(
    FastArgs a, PairArgs g) {
    __shared__ WaveLds wave_lds[4];
    extern __shared__ __align__(16) char dyn_lds[];
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    WaveLds &wl = wave_lds[wv];
    Stage &stg = ((Stage *)dyn_lds)[wv];
    WaveTotals tot;
    tot.slab_next = nullptr;
    tot.slab_lim = nullptr;
    CView *vp = HBT_CONST(View, a.views);
    const int n = HBT_CONST(Head, g.head)->n;
    const HBT_AS4 int *koff = HBT_CONST(int, g.head->koff);
    const PfConst<float> pk = pf_const<float>(vp->P);
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
            walk_item<double, false, false>(w, vp, 0.0, pk, wl, stg, tot,
                                            [](int) { return JWin{0, 0, 0, 0}; });
            continue;
        }
        const long long k = it - g.nsame;
        const int r = (int)(k % g.runs), tile = (int)(k / g.runs % g.tiles);
        const int e = (int)(k / g.runs / g.tiles);
        const int ib = koff[e], ie = koff[e + 1];
        w.kind = 1;
        w.ni = min(64, ie - ib - tile * 64);
        w.nj = min(g.rows, g.M - r * g.rows);
        if (w.ni <= 0 || w.nj <= 0) continue;
        w.i0 = ib + tile * 64;
        const long long row0 = (long long)e * g.M + r * g.rows;
        walk_item<double, false, false>(w, vp, 0.0, pk, wl, stg, tot, [&](int seg) {
            const int pid = HBT_CONST(int, g.ids)[row0 + seg];
            const bool ok = pid >= 0 && pid < g.nev;  // other partners form no pairs
            return JWin{ok ? koff[pid] : 0, ok ? koff[pid + 1] : 0, (int)(row0 + seg), 0};
        });
    }
}

}  // namespace

extern "C" {

const char *hbt_noalloc_last_error(void) {
    std::lock_guard<std::mutex> lk(g_mu);
    return g_err.c_str();
}

int hbt_calculate_noalloc(const hbt_config *cfg, int32_t nev, int64_t n_particles,
                          int64_t max_event, const int64_t *ev_off, const double *const soa[8],
                          int32_t M, const int32_t *partner_ids, const double *cos_sin,
                          double *bins, void *stream) {
    if (!cfg || !soa || !bins || (nev > 0 && !ev_off)) return fail(HBT_ERR_ARG, "null argument");
    Derived D;
    std::string err;
    if (int rc = derive(*cfg, D, err)) return fail(rc, "invalid configuration");
    if (cfg->kernel != HBT_KERNEL_PLAIN || cfg->precision != HBT_PREC_FP64)
        return fail(HBT_ERR_ARG, "hbt_calculate_noalloc runs the plain FP64 kernel only");
    if (cfg->azimuthal_flag || cfg->invariant_radius_flag)
        return fail(HBT_ERR_ARG, "hbt_calculate_noalloc bins the 3D histogram only "
                                 "(azimuthal_flag = invariant_radius_flag = 0)");
    if (!(cfg->needed_number_of_pairs >= 1e18))
        return fail(HBT_ERR_ARG, "hbt_calculate_noalloc needs the pair cap off "
                                 "(needed_number_of_pairs >= 1e18)");
    if (nev < 0 || nev > kMaxEvents)
        return fail(HBT_ERR_CAPACITY, "more events than the scratch array holds "
                                      "(HBT_NOALLOC_MAX_EVENTS)");
    if (n_particles < 0 || n_particles > kMaxParticles)
        return fail(HBT_ERR_CAPACITY, "more particles than the scratch array holds "
                                      "(HBT_NOALLOC_MAX_PARTICLES)");
    if (max_event < 0 || max_event > n_particles)
        return fail(HBT_ERR_ARG, "max_event must lie in [0, n_particles]");
    if (M < 0 || M > 64 * 1024 || (M > 0 && nev > 0 && (!partner_ids || !cos_sin)))
        return fail(HBT_ERR_ARG, "bad mixing plan");
    for (int a = 0; a < 8; a++)
        if (!soa[a] && n_particles > 0) return fail(HBT_ERR_ARG, "null particle column");
    int ndev = 0, cur = 0;
    if (hipGetDeviceCount(&ndev) != hipSuccess || cfg->device < 0 || cfg->device >= ndev ||
        cfg->device >= kMaxDevices)
        return fail(HBT_ERR_NODEVICE, "bad device");
    if (hipGetDevice(&cur) != hipSuccess) return fail(HBT_ERR_HIP, "hipGetDevice failed");
    if (cur != cfg->device && hipSetDevice(cfg->device) != hipSuccess)
        return fail(HBT_ERR_NODEVICE, "hipSetDevice failed");
    int rc = HBT_OK;
    unsigned char *scr = nullptr;
    hipStream_t st = (hipStream_t)stream;
    do {
        if (nev == 0 || n_particles == 0) break;
        rc = scratch_ptr(cfg->device, &scr);
        if (rc) break;
        Scratch *s = (Scratch *)scr;
        GatherArgs g{};
        g.ev_off = (const long long *)ev_off;
        g.in = DevSoA{soa[0], soa[1], soa[2], soa[3], soa[4], soa[5], soa[6], soa[7]};
        g.cut_min = tanh(cfg->HBTrap_min);
        g.cut_max = tanh(cfg->HBTrap_max);
        g.pt = fast_pt_range(D);
        g.P = D.P;
        g.c_beta = D.c_beta;
        g.bins = bins;
        g.plan_cs = cos_sin;
        g.nev = (int)nev;
        if (n_particles <= kSmallParticles) {
            hipLaunchKernelGGL(k_na_gather_small, dim3(1), dim3(1024), 0, st, g, s);
        } else {
            hipLaunchKernelGGL(k_na_count, dim3(nev), dim3(256), 0, st, g, s);
            hipLaunchKernelGGL(k_na_scan, dim3(1), dim3(1024), 0, st, g, s);
            hipLaunchKernelGGL(k_na_compact, dim3(nev), dim3(256), 0, st, g, s);
        }
        PairArgs p{};
        p.head = &s->head;
        p.ids = partner_ids;
        p.nev = (int)nev;
        p.M = M;
        // Items: 64 i's against about 1024 j's (a chunk of the list, or
        // several plan rows' partners), where an item's own cost, some 750
        // cycles, is below a tenth of its pairs'; finer, down to 64 j's or one
        // row, while that leaves waves of the chip idle.
        const long long tiles = (n_particles + 63) / 64;
        p.jchunk = 1024;
        while (p.jchunk > 64 && tiles * ((n_particles + p.jchunk - 1) / p.jchunk) < 2 * kWaves)
            p.jchunk /= 2;
        p.nchunk = (int)((n_particles + p.jchunk - 1) / p.jchunk);
        p.nsame = tiles * p.nchunk;
        p.tiles = (int)((max_event + 63) / 64);
        p.rows = 1;
        if (M > 0 && p.tiles > 0) {
            const long long ev_tiles = (long long)nev * p.tiles;
            p.rows = (int)std::max(1ll, std::min<long long>(M, 1024 / std::max<long long>(1, max_event)));
            while (p.rows > 1 && ev_tiles * ((M + p.rows - 1) / p.rows) < 2 * kWaves) p.rows /= 2;
            p.runs = (M + p.rows - 1) / p.rows;
            p.nitems = p.nsame + ev_tiles * p.runs;
        } else {
            p.tiles = p.runs = 1;
            p.nitems = p.nsame;
        }
        FastArgs a{};
        a.views = &s->head.v;
        const long blocks = (long)std::min<long long>((p.nitems + 3) / 4, 2 * kWaves / 4);
        hipLaunchKernelGGL(k_na_pairs, dim3((unsigned)blocks), dim3(256), 4 * sizeof(Stage), st, a,
                           p);
        if (hipGetLastError() != hipSuccess) rc = fail(HBT_ERR_HIP, "kernel launch failed");
    } while (false);
    if (cur != cfg->device) hipSetDevice(cur);
    return rc;
}

}  // extern "C"
