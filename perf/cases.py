"""Timing cases of the framework's public entry points.

Every case is a dict of plain values.  ``path`` names how a program drives
the framework:

  buffers  HBTCorrelation.calculate_HBT_correlation_function, buffer after
           buffer, then results(): the reference's own analysis loop;
  batch    all groups resident (upload_groups, prepare_batch), one
           launch_batch per analysis, then results();
  sides    run_same and run_mixed of one resident buffer, then results();
  noalloc  hbt_calculate_noalloc on the caller's device arrays and stream;
  balance  BalanceFunction.calculate_balance_function, then results();
  serve    HBTServer: requests submitted together, waited for and read.

Shared keys: nev events in all, per events in a buffer or group, mult mean
multiplicity (spread: log-uniform between mult/37 and 5.4 mult, else Poisson),
the q, K_T and rapidity grids, M rotations per event (0: the reference's
rule), nphi K_phi bins (0: none), qinv, boost, prec, binning, cap, and tune
(R, jchunk, kchunk, blocks per CU as a text; "": the default shape).
"""
import ctypes as C
import math

import numpy as np
import torch

from hadronic_afterburner_toolkit_amd import _lib, hbt, samples

FREE = 1e18  # pair cap off

_HBT = dict(qnpts=41, q_max=0.15, n_KT=6, KT_min=0.2, KT_max=0.7, rap=1.0, M=10, nphi=0,
            qinv=False, boost=True, prec="fp64", binning=0, cap=FREE, tune="", spread=False)
_DEFAULT_GRID = dict(qnpts=31, n_KT=5, KT_min=0.15, KT_max=0.55, rap=0.5, M=0, cap=3e7)


def _case(path, **kw):
    return dict(dict(_HBT, path=path), **kw)


def listed():
    return [
        # a first look at a small sample with the reference's default
        # parameters: latency of one call and of reading the histograms
        _case("buffers", name="buffer small", nev=10, per=10, mult=60.0, **_DEFAULT_GRID),
        # the reference's default parameters on an ordinary oversampled run,
        # its default pair cap (3e7 per K_T bin) on
        _case("buffers", name="buffers default", nev=200, per=50, mult=600.0, **_DEFAULT_GRID),
        # the same loop in the precision form, the cap off
        _case("buffers", name="buffers fp32c", nev=400, per=50, mult=600.0, prec="fp32c"),
        # the headline workload of bench.py, precision form, slab binning
        _case("batch", name="batch fp32c", nev=2000, per=50, mult=600.0, prec="fp32c", binning=1,
              tune="1 4096 4 8"),
        # half of it in FP64
        _case("batch", name="batch fp64", nev=1000, per=50, mult=600.0, binning=1,
              tune="1 4096 4 8"),
        # central to peripheral events in one batch, 16 K_phi bins
        _case("batch", name="batch uneven kphi", nev=512, per=20, mult=746.0, spread=True, nphi=16,
              M=0, prec="fp32c"),
        # one-dimensional radii: the invariant-q histograms beside the 3D ones
        _case("buffers", name="buffers qinv", nev=60, per=20, mult=200.0, qnpts=31, qinv=True, M=0),
        # fine grid and high multiplicity, the two sides run one by one
        _case("sides", name="sides fine grid", nev=10, per=10, mult=4000.0, qnpts=61, q_max=0.2,
              n_KT=9, KT_min=0.15, KT_max=1.0, M=5),
        # callers that hold everything on the device: a tight loop over small
        # buffers, and one ordinary buffer
        _case("noalloc", name="noalloc small", nev=7, per=7, mult=90.0, qnpts=21, M=0),
        _case("noalloc", name="noalloc group", nev=20, per=20, mult=600.0, M=0),
        # balance functions of charged pions with the reference's cuts
        dict(name="balance", path="balance", nev=500, mult=900.0, Bnpts=21, rap_type=1,
             kernel="fast"),
        # several users' analyses arriving together
        _case("serve", name="serve", nev=600, per=10, mult=500.0, requests=6, prec="fp32c"),
    ]


def _log(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def _pairs(c):
    """Same-event and mixed pairs of an HBT case (of its mean multiplicity; a
    log-uniform one has 2.9 times the mean square of a fixed one)."""
    per, kept = min(c["per"], c["nev"]), c["rap"] * c["mult"]
    sq = 2.9 if c["spread"] else 1.0
    same = 0.5 * c["nev"] / per * (per * (per + sq - 1) * kept ** 2)
    return same + c["nev"] * (c["M"] or per // 2 + 1) * kept ** 2


def draw(rng):
    path = rng.choice(["buffers", "buffers", "batch", "batch", "sides", "noalloc", "balance",
                       "serve"])
    if path == "balance":
        return dict(path=path, nev=int(_log(rng, 10, 500)), mult=_log(rng, 40, 900),
                    Bnpts=rng.choice([20, 21, 41]), rap_type=rng.choice([0, 1]),
                    kernel=rng.choice(["fast", "fast", "exact"]))
    c = _case(path, mult=_log(rng, 40, 1200), boost=rng.random() < 0.8,
              M=rng.choice([0, rng.randint(1, 12)]), qnpts=rng.randint(11, 45),
              n_KT=rng.randint(2, 8), rap=rng.choice([0.5, 1.0]),
              KT_min=rng.choice([0.15, 0.2]), KT_max=rng.uniform(0.5, 0.8),
              q_max=rng.uniform(0.08, 0.2))
    most = 2e8  # pairs: no drawn case costs more than the largest listed one
    if path == "noalloc":
        c["per"] = c["nev"] = int(_log(rng, 2, 30))
    else:
        c["prec"] = rng.choice(["fp64", "fp32c"])
        c["per"] = int(_log(rng, 5, 50))
        c["spread"] = rng.random() < 0.25
        c["nphi"] = rng.choice([0, 0, rng.randint(2, 16)])
    if path == "buffers":
        c["nev"] = c["per"] * rng.randint(1, 5) - rng.randint(0, 2)
        c["cap"] = rng.choice([FREE, 3e7, 3e7])
        c["qinv"] = rng.random() < 0.25
        most = 1e8 if c["qinv"] else 1e9
    elif path == "batch":
        c["nev"] = c["per"] * rng.randint(2, 24) - rng.randint(0, 2)
        c["binning"] = rng.choice([0, 1, 1])
        c["tune"] = rng.choice(["", "1 4096 4 8", "1 256 16 8", "2 1024 4 8"])
        most = 1e10
    elif path == "sides":
        c["nev"] = c["per"]
        c["qnpts"] = rng.randint(11, 61)
        most = 1e9
    elif path == "serve":
        c["requests"] = rng.randint(1, 8)
        c["nev"] = c["requests"] * rng.randint(10, 100)
        c["per"] = rng.choice([5, 10, 20])
        c["nphi"] = 0
        most = 1e9
    while _pairs(c) > most:
        c["mult"] *= 0.8
    return c


# ------------------------------------------------------------------ inputs

BF_SPECIES = ((211, 0.13957, 0.25, 3.0), (-211, 0.13957, 0.25, 3.0),
              (321, 0.49368, 0.30, 1.0), (-321, 0.49368, 0.30, 1.0))


def _params(c):
    return dict(qnpts=c["qnpts"], q_min=-c["q_max"], q_max=c["q_max"], n_KT=c["n_KT"],
                KT_min=c["KT_min"], KT_max=c["KT_max"], HBTrap_min=-c["rap"], HBTrap_max=c["rap"],
                needed_number_of_pairs=c["cap"], number_of_mixed_events=c["M"],
                long_comoving_boost=int(c["boost"]), azimuthal_flag=int(c["nphi"] > 0),
                n_Kphi=max(1, c["nphi"]), invariant_radius_flag=int(c["qinv"]),
                hbt_binning=c["binning"])


def _seed(seed):
    return int(seed) % (1 << 30)


def _sample(c, seed):
    """The whole sample of an HBT case."""
    m = c["mult"]
    mult = samples.log_uniform_mult(max(2.0, m / 37), 5.4 * m) if c["spread"] else m
    return samples.generate(_seed(seed), c["nev"], mult)


def _split(full, per):
    return [full.events(e, min(per, full.nev - e)) for e in range(0, full.nev, per)]


def _requests(c, full):
    """Requests of 1, 2, 3, ... parts of the sample's events."""
    k = c["requests"]
    at = [c["nev"] * i * (i + 1) // (k * (k + 1)) for i in range(k + 1)]
    return [full.events(a, b - a) for a, b in zip(at, at[1:]) if b > a]


def _bf_params(c):
    return dict(particle_alpha=211, particle_beta=211, BpT_min=0.2, BpT_max=3.0, Brap_max=2.0,
                Bnpts=c["Bnpts"], rap_type=c["rap_type"])


def _bf_sample(c, seed):
    return samples.generate(_seed(seed), c["nev"], c["mult"], species=BF_SPECIES)


def _plan(rng, nev, M):
    """A mixing plan: partners other than the event itself, rotations."""
    M = M or nev // 2 + 1
    ids = rng.integers(0, max(1, nev - 1), (nev, M))
    if nev > 1:
        ids += ids >= np.arange(nev)[:, None]
    th = rng.uniform(0, 2 * np.pi, nev * M)
    return M, ids.ravel().astype(np.int32), np.stack([np.cos(th), np.sin(th)], 1).ravel()


def prepare(case, seed):
    path = case["path"]
    s = dict(path=path, seed=_seed(seed))
    if path == "balance":
        s["buf"] = _bf_sample(case, seed)
        kern = _lib.HBT_BF_KERNEL_FAST if case["kernel"] == "fast" else _lib.HBT_BF_KERNEL_EXACT
        s["g"] = hbt.BalanceFunction(_bf_params(case), kernel=kern)
        return s
    full = _sample(case, seed)
    prec = _lib.HBT_PREC_FP32C if case["prec"] == "fp32c" else _lib.HBT_PREC_FP64
    rng = np.random.default_rng(_seed(seed) + 1)
    if path == "noalloc":
        M, ids, cs = _plan(rng, full.nev, case["M"])
        s["cfg"] = hbt.config_from_params(_params(case), kernel=_lib.HBT_KERNEL_PLAIN)
        s["cols"] = [torch.from_numpy(np.ascontiguousarray(a)).cuda() for a in full.soa()]
        s["soa"] = (C.c_void_p * 8)(*[a.data_ptr() for a in s["cols"]])
        s["off"] = torch.from_numpy(full.ev_off).cuda()
        s["ids"], s["cs"] = torch.from_numpy(ids).cuda(), torch.from_numpy(cs).cuda()
        s["size"] = (full.nev, full.n, int(np.diff(full.ev_off).max()), M)
        s["bins"] = torch.zeros(case["n_KT"] * case["qnpts"] ** 3, 8, dtype=torch.float64,
                                device="cuda")
        return s
    if path == "serve":
        s["reqs"] = _requests(case, full)
        s["per"] = case["per"]
        s["g"] = hbt.HBTServer(_params(case), precision=prec)
        return s
    s["bufs"] = _split(full, case["per"])
    g = s["g"] = hbt.HBTCorrelation(_params(case), precision=prec)
    if case["tune"]:
        g.set_tuning(*[int(v) for v in case["tune"].split()])
    if path == "batch":
        plans = [_plan(rng, b.nev, case["M"]) for b in s["bufs"]]
        g.upload_groups(s["bufs"])
        g.prepare_batch(np.array([p[0] for p in plans], np.int32),
                        np.concatenate([p[1] for p in plans]),
                        np.concatenate([p[2] for p in plans]))
    elif path == "sides":
        s["plan"] = _plan(rng, full.nev, case["M"])
        g.upload(s["bufs"][0])
    return s


# ------------------------------------------------------------------ one pass

def run(s):
    path, g = s["path"], s.get("g")
    if path == "noalloc":
        s["bins"].zero_()
        nev, n, most, M = s["size"]
        rc = _lib.load().hbt_calculate_noalloc(
            C.byref(s["cfg"]), nev, n, most, s["off"].data_ptr(), s["soa"], M,
            s["ids"].data_ptr(), s["cs"].data_ptr(), s["bins"].data_ptr(),
            torch.cuda.current_stream().cuda_stream)
        if rc:
            raise RuntimeError(_lib.load().hbt_noalloc_last_error().decode())
        b = s["bins"]  # count, four sums, denominator (an integer's bits) per bin
        return dict(count=b[:, 0], sums=b[:, 1:5], den=b[:, 5].view(torch.int64))
    if path == "serve":
        ids = [g.submit(b, s["per"], s["seed"] + k) for k, b in enumerate(s["reqs"])]
        out = []
        for r in ids:
            g.wait(r)
            res = vars(g.result(r))
            g.release(r)
            # a request's histograms (the pair counters are their sums)
            out.append({k: res[k] for k in ("num_count", "den", *_SUMS)})
        return out
    g.reset()
    if path == "balance":
        g.calculate_balance_function(s["buf"], hbt.Random(s["seed"]))
        return g.results()
    if path == "buffers":
        rng = hbt.Random(s["seed"])
        for b in s["bufs"]:
            g.calculate_HBT_correlation_function(b, rng)
    elif path == "batch":
        g.launch_batch()
        g.sync()
    else:
        g.run_same()
        g.run_mixed(*s["plan"])
    return dict(vars(g.results()))


# ------------------------------------------------------------------ work

def work(case):
    """Every particle read once (8 doubles; momentum, mass and species for the
    balance function), every histogram value written once, and the arithmetic
    of the pairs that are binned (about 58 operations each, 12 for the
    balance function's): pairs outside the windows need not be formed."""
    nev, m = case["nev"], case["mult"]
    if case["path"] == "balance":
        n = 0.375 * m
        return dict(bytes=44.0 * nev * m + 8.0 * 8 * case["Bnpts"] * 20, flops=12.0 * 8 * nev * n * n)
    frac = 0.012 * (case["q_max"] / 0.15) ** 3
    copies = case.get("requests", 1)
    nbins = case["n_KT"] * max(1, case["nphi"]) * case["qnpts"] ** 3
    return dict(bytes=64.0 * nev * m + 48.0 * nbins * copies, flops=58.0 * frac * _pairs(case))


# ------------------------------------------------------------------ 64-bit values

_SUMS = ("q_out_sum", "q_side_sum", "q_long_sum", "num")
_HBARC = 0.197327053


def _dev():
    return "cuda" if torch.cuda.is_available() else "cpu"


def _same_sums(case, bufs):
    """The same-event sums of the buffers, pair by pair in plain torch."""
    q, nkt, nphi = case["qnpts"], case["n_KT"], max(1, case["nphi"])
    dq = 2 * case["q_max"] / (q - 1)
    base = -case["q_max"] - dq / 2
    lo, hi = base + 1e-8, case["q_max"] + dq / 2 - 1e-8
    k0, k1 = case["KT_min"], case["KT_max"]
    dkt, dphi = (k1 - k0) / (nkt - 1), 2 * math.pi / nphi
    f8 = dict(dtype=torch.float64, device=_dev())
    acc = {k: torch.zeros(nkt * nphi * q ** 3, **f8) for k in _SUMS}
    inv = {k: torch.zeros(nkt * q, **f8) for k in ("qinv_sum", "qinv_num")}
    cut = math.tanh(case["rap"])
    for b in bufs:
        psi = 0.0
        if case["nphi"]:
            ph = 2 * np.arctan2(b.py, b.px)
            psi = math.atan2(float(np.sin(ph).sum()), float(np.cos(ph).sum())) / 2
        r = b.pz / b.E
        keep = (r > -cut) & (r < cut)
        p = torch.from_numpy(np.stack(b.soa())[:, keep]).to(_dev())
        n = p.shape[1]
        rows = max(1, (1 << 25) // max(1, n))
        for i0 in range(0, n - 1, rows):
            a, c = p[:, i0:min(n, i0 + rows)], p[:, i0 + 1:]
            kx, ky = 0.5 * (a[0][:, None] + c[0]), 0.5 * (a[1][:, None] + c[1])
            k2 = kx * kx + ky * ky
            ok = (k2 >= k0 * k0) & (k2 <= k1 * k1)
            if not case["qinv"]:  # |q_T| of a pair inside the windows is below sqrt(2) hi
                dx, dy = a[0][:, None] - c[0], a[1][:, None] - c[1]
                ok &= dx * dx + dy * dy <= 2.001 * hi * hi
            i, j = ok.triu_().nonzero(as_tuple=True)  # column j is particle i0 + 1 + j
            del kx, ky, k2, ok
            u, v = a[:, i], c[:, j]
            del i, j
            kx, ky, kz, ke = (0.5 * (u[f] + v[f]) for f in range(4))
            kp = torch.sqrt(kx * kx + ky * ky)
            kt = ((kp - k0) / dkt).to(torch.int64)
            qx, qy, qz, qe = (u[f] - v[f] for f in range(4))
            d = u[4:] - v[4:]
            cosq = torch.cos((1 / _HBARC) * (qe * d[3] - qx * d[0] - qy * d[1] - qz * d[2]))
            ok = (kt >= 0) & (kt < nkt)
            if case["qinv"]:
                qi = torch.sqrt(-(qe * qe - qx * qx - qy * qy - qz * qz))
                at = ((qi - base) / dq).to(torch.int64)
                w = ok & (qi > lo) & (qi < hi) & (at < q)
                inv["qinv_sum"].index_add_(0, (kt * q + at)[w], qi[w])
                inv["qinv_num"].index_add_(0, (kt * q + at)[w], cosq[w])
            ck, sk = kx / kp, ky / kp
            qs = [qx * ck + qy * sk, qy * ck - qx * sk, qz]
            if case["boost"]:
                qs[2] = ke / torch.sqrt(ke * ke - kz * kz) * (qz - kz / ke * qe)
            bins = kt * nphi
            if case["nphi"]:
                ph = torch.atan2(ky, kx) - psi
                ph = torch.where(ph < 0, ph + 2 * math.pi, ph)
                ph = torch.where(ph < 0, ph + 2 * math.pi, ph)
                ph = torch.where(ph > 2 * math.pi, ph - 2 * math.pi, ph)
                at = (ph / dphi).to(torch.int64)
                ok &= at < nphi
                bins = bins + at
            for x in qs:
                at = ((x - base) / dq).to(torch.int64)
                ok &= (x >= lo) & (x <= hi) & (at >= 0) & (at < q)
                bins = bins * q + at
            bins = bins[ok]
            for k, x in zip(_SUMS, (*qs, cosq)):
                acc[k].index_add_(0, bins, x[ok])
    return acc, inv


def _draws(seed, nev, count):
    """Partner and rotation of each event, `count` times: std::mt19937 as the
    standard library draws a non-negative int and a double in [0, 1)."""
    raw = np.random.RandomState(seed).randint(0, 1 << 32, size=(count, nev, 3), dtype=np.uint32)
    u = (raw[..., 1].astype(np.float64) + raw[..., 2].astype(np.float64) * 2.0 ** 32) / 2.0 ** 64
    return (raw[..., 0] >> 1).astype(np.int64) % nev, u * 2.0 * math.pi


def _balance_counts(case, seed):
    b = _bf_sample(case, seed)
    pt = np.sqrt(b.px * b.px + b.py * b.py)
    low = pt if case["rap_type"] == 0 else np.sqrt(pt * pt + b.mass * b.mass)
    phi, y = np.arctan2(b.py, b.px), np.arcsinh(b.pz / low)
    ok = (pt >= 0.2) & (pt <= 3.0)
    lists = {}
    for mon in (211, -211):
        lists[mon] = []
        for e in range(b.nev):
            sl = slice(int(b.ev_off[e]), int(b.ev_off[e + 1]))
            w = ok[sl] & (b.monval[sl] == mon)
            lists[mon].append(torch.from_numpy(np.stack([phi[sl][w], y[sl][w]])).to(_dev()))
    nb = case["Bnpts"]
    drap, dphi = 4.0 / (nb - 1), 2 * math.pi / 20
    ymin, pmin = -2.0 - 0.5 * drap, -math.pi / 2
    hist = torch.zeros(8, nb * 20, dtype=torch.float64, device=_dev())
    part, rot = _draws(_seed(seed), b.nev, 4)
    for k in range(8):
        one, two = (211, -211)[k & 1], (211, -211)[int(k & 3 in (1, 2))]
        for e in range(b.nev):
            f, r = (e, 0.0) if k < 4 else (int(part[k - 4, e]), float(rot[k - 4, e]))
            u, v = lists[one][e], lists[two][f]
            d, dy = u[0][:, None] - v[0] + r, u[1][:, None] - v[1]
            p = torch.floor((d - pmin) / dphi).to(torch.int64) % 20
            at = ((dy - ymin) / drap).to(torch.int64)
            w = (dy.abs() >= 1e-10) & (dy >= ymin) & (at >= 0) & (at < nb)
            at = (at * 20 + p)[w]
            hist[k].index_add_(0, at, torch.ones_like(at, dtype=torch.float64))
    return dict(hist=hist.reshape(8, nb, 20), N_b=None, N_bbar=None)


def exact(case, seed):
    if case["path"] == "balance":
        return _balance_counts(case, seed) if case["nev"] <= 700 else None
    full = _sample(case, seed)
    if case["path"] == "serve":
        out = []
        for r in _requests(case, full):
            acc, _ = _same_sums(case, _split(r, case["per"]))
            out.append(dict(acc, num_count=None, den=None))
        return out
    acc, inv = _same_sums(case, _split(full, case["per"]))
    if case["path"] == "noalloc":
        return dict(count=None, sums=torch.stack([acc[k] for k in _SUMS], 1), den=None)
    names = hbt.Results.__dataclass_fields__
    return {k: acc.get(k, inv.get(k)) for k in names}
