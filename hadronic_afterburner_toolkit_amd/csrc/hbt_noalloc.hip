// hbt_noalloc.hip -- hbt_calculate_noalloc: the pair loops of one buffer (what
// hbt_upload + hbt_run_same + hbt_run_mixed do, in FP64) for callers that
// cannot allocate device memory: code under HIP graph capture, tight serving
// loops.  The caller passes the particles, the mixing plan and the histogram
// in device memory; the kept particles and all that is derived from them live
// in `scratch`, a file-scope device array of fixed size that each GPU holds
// until the process ends.  No hipMalloc, hipFree or other allocating call is
// made; every launch goes on the caller's stream.
//
// The gather and the pair kernel of hbt_direct.h.
// One literal cascade per enumerated pair, one thread per i particle (the
// form before), cost 1420 us for 20 events of 600 particles (1.5e8 pairs) and
// 335 us for 7 of 90, whose few threads each walked hundreds of pairs one
// after the other; this form takes 175 (151 of them the pair kernel) and 35.
//
// Calls on one GPU share its scratch array: calls that overlap on one GPU
// (two streams, two host threads) race and must be serialized by the caller.
#include <hip/hip_runtime.h>

#include <mutex>
#include <string>

#include "../../include/hbt_hip.h"
#include "hbt_direct.h"

using namespace hbt;

namespace {

constexpr long long kMaxParticles = HBT_NOALLOC_MAX_PARTICLES;
constexpr int kMaxEvents = HBT_NOALLOC_MAX_EVENTS;
// The kept particles.
struct Scratch {
    ListStat head;
    ListStat stat[kMaxEvents];
    int koff[kMaxEvents + 1];
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
        const List list{&s->head, s->koff, s->stat, s->rec, s->pf, s->bw, (int)kMaxParticles};
        GatherArgs g{};
        g.ev_off = (const long long *)ev_off;
        g.in = DevSoA{soa[0], soa[1], soa[2], soa[3], soa[4], soa[5], soa[6], soa[7]};
        gather_setup(D, *cfg, g);
        g.nev = (int)nev;
        g.out = list;
        PairArgs p{};
        p.v.P = D.P;
        p.v.H.bins = bins;
        p.v.plan_cs = cos_sin;
        pair_lists(p, list, list);
        p.ids = partner_ids;
        p.nev_b = (int)nev;
        pair_items(p, n_particles, nev, max_event, true, M);
        hipError_t e = launch_gather(g, n_particles, st);
        if (e == hipSuccess) e = launch_pairs(p, false, false, st);
        if (e != hipSuccess) rc = fail(HBT_ERR_HIP, "kernel launch failed");
    } while (false);
    if (cur != cfg->device) hipSetDevice(cur);
    return rc;
}

}  // extern "C"
