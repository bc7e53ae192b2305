"""The prefilter as the kernels evaluate it (pf_block's operands, pf_test, and for
q_inv bins pair_consts in csrc/hbt_direct.h) on the host, against the reference's
FP64 cascade (cascade_f64): a pair that bins in the 3D or in the q_inv histograms
passes, in both orders of the pair, with the four products of X, P and M added in
every order, fused and not (the matrix cores' own is not known).

q_inv: particles whose m^2 = E^2 - p^2 differ by as much as the windows allow
(d^2 = H^2 m^2 kQinvRoom / 2), at the q_out where q_side and q_long reach furthest,
q_inv just inside its window; with and without the LCMS boost.  Planted mistakes:
the room left out of the windows' H^2, and C taken with the wrong sign in one
operand; each must drop binnable pairs."""
import shutil
import subprocess
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parents[1] / "hadronic_afterburner_toolkit_amd" / "csrc"
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"

PROGRAM = r"""
#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <random>
#include <string>
#include <vector>
#include "hbt_internal.h"
#include "hbt_direct.h"
using namespace hbt;

struct P4 { double px, py, pz, E; };
static bool plant_room, plant_sign;

// Passes with the products in every order?
static bool passes(const PfConst<float> &k, const PfRec32 &i, float ihi, const PfRec32 &j, float jhi) {
    PfBlock<float> b[4];
    for (int c = 0; c < 4; c++) b[c] = pf_block(k, c, i.px, i.py, i.nrm);
    if (plant_sign) b[1].P = -b[1].P;
    const float jv[4] = {j.px, j.py, j.nrm, 1.0f};
    const float ilo = i.blo - k.wide;
    int o[4] = {0, 1, 2, 3};
    do {
        for (int fused = 0; fused < 2; fused++) {
            float X = 0, P = 0, M = 0;
            for (int c : o) {
                if (fused) {
                    X = pf_fma(jv[c], b[c].X, X);
                    P = pf_fma(jv[c], b[c].P, P);
                    M = pf_fma(jv[c], b[c].M, M);
                } else {
                    X = X + jv[c] * b[c].X;
                    P = P + jv[c] * b[c].P;
                    M = M + jv[c] * b[c].M;
                }
            }
            if (!pf_pass(PfTerms<float>{pf_test(X, P, M, ilo, ihi + k.wide, j.blo, jhi, k)}))
                return false;
        }
    } while (std::next_permutation(o, o + 4));
    return true;
}

int main(int argc, char **argv) {
    plant_room = argc > 1 && !std::strcmp(argv[1], "room");
    plant_sign = argc > 1 && !std::strcmp(argv[1], "sign");
    std::mt19937_64 rng(7);
    std::uniform_real_distribution<double> U(0.0, 1.0);
    long long binned3 = 0, binnedq = 0, dropped = 0;
    for (int qinv = 0; qinv < 2; qinv++)
        for (int boost = 0; boost < 2; boost++)
            for (double qmax : {0.03, 0.15, 0.3}) {
                hbt_config c{};
                c.qnpts = 21; c.q_min = qinv ? 0.0 : -qmax; c.q_max = qmax;
                c.n_KT = 5; c.KT_min = 0.1; c.KT_max = 1.0; c.n_Kphi = 1;
                c.long_comoving_boost = boost; c.invariant_radius_flag = qinv;
                c.HBTrap_min = -2; c.HBTrap_max = 2; c.needed_number_of_pairs = 1e18;
                c.number_of_mixed_events = 1; c.kernel = 1;
                Derived d;
                std::string err;
                if (derive(c, d, err)) return 2;
                const double H = d.H, m = 0.13957;
                // the two masses: m2lo = m^2, and m2hi at the edge of the room
                const double dd = qinv ? std::sqrt(0.5 * kQinvRoom * (1 - 1e-9)) * H * m : 0.0;
                const double m2[2] = {m * m, m * m + 2 * dd};
                std::vector<std::pair<P4, P4>> prs;
                for (int n = 0; n < 20000; n++) {
                    const int swap = (int)(rng() & 1);
                    const double ma = m2[swap], mb = m2[1 - swap];
                    const double kt = 0.11 + 0.85 * U(rng), phi = 2 * M_PI * U(rng);
                    const double Y = 2.4 * U(rng) - 1.2;
                    const double far = n % 3 == 0 ? 3.0 * (U(rng) - 0.5) : 0.0;
                    double al = 2 * M_PI * U(rng);
                    if (n % 5 == 0) al = M_PI / 2 * (int)(rng() % 4);
                    // scale of (q_side, q_long): q_inv (3D: the larger of them) just inside
                    const double want = (qinv ? d.P.q_hi_cut : H) *
                                        (1 - std::pow(10.0, -(4 + (int)(rng() % 9))));
                    P4 a, b;
                    auto make = [&](double s) {
                        const double qs = s * std::cos(al), ql = s * std::sin(al);
                        double qo = far * H;
                        if (!qinv) qo = std::max(-1.0, std::min(1.0, far)) * 0.999 * H;
                        for (int it = 0; it < (qinv && far == 0.0 ? 3 : 1); it++) {
                            const double ax = kt + qo / 2, bx = kt - qo / 2;
                            const double Ea = std::sqrt(ma + ax * ax + qs * qs / 4 + ql * ql / 4);
                            const double Eb = std::sqrt(mb + bx * bx + qs * qs / 4 + ql * ql / 4);
                            a = {ax, qs / 2, ql / 2, Ea};
                            b = {bx, -qs / 2, -ql / 2, Eb};
                            const double KE = 0.5 * (Ea + Eb);
                            if (qinv && far == 0.0)  // where q_out^2 - q_E^2 is smallest
                                qo = kt * 0.5 * (ma - mb) / (KE * KE - kt * kt);
                        }
                        const double qx = a.px - b.px, qy = a.py - b.py, qz = a.pz - b.pz, qe = a.E - b.E;
                        return qinv ? std::sqrt(std::max(0.0, qx * qx + qy * qy + qz * qz - qe * qe))
                                    : std::max(std::fabs(qs), std::fabs(ql));
                    };
                    double s0 = 0.0, s1 = 4 * H;
                    for (int it = 0; it < 60; it++) {
                        const double s = 0.5 * (s0 + s1);
                        (make(s) < want ? s0 : s1) = s;
                    }
                    make(s0);
                    const double cs = std::cos(phi), sn = std::sin(phi), ch = std::cosh(Y), sh = std::sinh(Y);
                    for (P4 *p : {&a, &b}) {
                        const P4 q = *p;
                        *p = {q.px * cs - q.py * sn, q.px * sn + q.py * cs, q.pz * ch + q.E * sh,
                              q.E * ch + q.pz * sh};
                    }
                    prs.push_back({a, b});
                }
                ListStat st = stat_none();
                for (auto &pr : prs)
                    for (const P4 *p : {&pr.first, &pr.second}) {
                        const double p2 = p->px * p->px + p->py * p->py;
                        const double mm = p->E * p->E - p2 - p->pz * p->pz;
                        st = stat_join(st, ListStat{p2, std::fabs(boost ? p->pz / p->E : p->pz), mm, mm, 1});
                    }
                // (the boosted energies' rounding must not switch the windows off)
                const double mid = 0.5 * (st.m2lo + st.m2hi), half = std::min(0.5 * (st.m2hi - st.m2lo), dd);
                st.m2lo = mid - half;
                st.m2hi = mid + half;
                PfConst<float> k = pair_consts(d.P, st);
                if (qinv && k.wide != 0.0f) return 3;
                GatherArgs g{};
                gather_setup(d, c, g);
                if (plant_room && qinv) {
                    DevParams P = d.P;
                    P.qinv = 0;
                    P.pf_h2 = d.h2;
                    prefilter_margins(st.pmax2, P);
                    k = pf_const<float>(P);
                    k.dn = 0.0f;
                    g.c_beta = d.c_beta;
                }
                for (auto &pr : prs) {
                    const P4 &a = pr.first, &b = pr.second;
                    PairBins bins;
                    double q;
                    int ok;
                    const int stg = cascade_f64<false, true>(d.P, a.px, a.py, a.pz, a.E, b.px, b.py,
                                                             b.pz, b.E, 0.0, bins, q, ok);
                    if (!(stg & ST_BIN) && !ok) continue;
                    binned3 += (stg & ST_BIN) != 0;
                    binnedq += ok != 0;
                    const PfMake mk{g.mid, g.c_beta, st.bmax, g.boost, 0};
                    PfRec32 ra, rb;
                    float ha, hb;
                    pf_make(mk, a.px, a.py, a.pz, a.E, ra, ha);
                    pf_make(mk, b.px, b.py, b.pz, b.E, rb, hb);
                    if (g.qinv && !g.boost) {  // list_store: no longitudinal window
                        ra.blo = rb.blo = -INFINITY;
                        ha = hb = INFINITY;
                    }
                    dropped += !passes(k, ra, ha, rb, hb);
                    dropped += !passes(k, rb, hb, ra, ha);
                }
            }
    std::printf("binned3 %lld binnedq %lld dropped %lld\n", binned3, binnedq, dropped);
    return 0;
}
"""


@pytest.mark.skipif(not Path(HIPCC).exists(), reason="needs hipcc")
def test_kernel_form_never_drops_a_binnable_pair(tmp_path):
    src = tmp_path / "po.cpp"
    src.write_text(PROGRAM)
    exe = tmp_path / "po"
    subprocess.run([HIPCC, "-O2", "-std=c++17", "-x", "hip", "--cuda-host-only", "-ffp-contract=off",
                    f"-I{CSRC}", str(src), "-o", str(exe)], check=True, timeout=300,
                   capture_output=True)

    def run(*args):
        r = subprocess.run([str(exe), *args], capture_output=True, text=True, timeout=300)
        assert r.returncode == 0, (r.returncode, r.stdout, r.stderr)
        f = r.stdout.split()
        return int(f[1]), int(f[3]), int(f[5])

    b3, bq, dropped = run()
    assert b3 > 50000 and bq > 50000 and dropped == 0
    for plant in ("room", "sign"):
        p3, pq, d = run(plant)
        assert (p3, pq) == (b3, bq) and d > 0
