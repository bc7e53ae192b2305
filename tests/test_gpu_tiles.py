"""The fast kernel at the edges of its tiles (blocks of 16, i tiles of 64,
pairs of j tiles of 32) against the oracle: groups of n particles whose
momenta lie so close together that every pair survives the prefilter (each
j tile fills the survivor queue many times over), or are spread so that few
do (survivors of one pair of tiles wait for the next), same-event and mixed,
in both precisions, with device-scope atomics, slab binning and K_phi bins.

Counts bit-exact; sums within 1e-12 (FP64) and 1e-6 (precision form) under
err = |S - S_ref| / max(|S_ref|, sum|.|_bin)."""
import numpy as np
import pytest

from hadronic_afterburner_toolkit_amd import _lib, hbt, samples

pytestmark = pytest.mark.gpu

SUMS = (("q_out_sum", "abs_q_out"), ("q_side_sum", "abs_q_side"), ("q_long_sum", "abs_q_long"),
        ("num", "abs_num"))


def cluster(rng, counts, spread):
    """Events of `counts` pions around (0.35, 0.2) GeV, |y| < 0.3."""
    n = int(sum(counts))
    px = 0.35 + spread * rng.uniform(-1, 1, n)
    py = 0.20 + spread * rng.uniform(-1, 1, n)
    mt = np.sqrt(px * px + py * py + 0.13957 ** 2)
    y = 0.3 * spread / 0.02 * rng.uniform(-1, 1, n) if spread < 0.02 else rng.uniform(-0.3, 0.3, n)
    x = rng.normal(0.0, 3.0, (3, n))
    return samples.Buffer(np.concatenate([[0], np.cumsum(counts)]).astype(np.int64), px, py,
                          mt * np.sinh(y), mt * np.cosh(y), *x, 8.0 + rng.exponential(2.0, n))


@pytest.mark.parametrize("binning,nphi", [(0, 0), (1, 0), (0, 3), (1, 3)])
@pytest.mark.parametrize("prec,tol", [(_lib.HBT_PREC_FP64, 1e-12), (_lib.HBT_PREC_FP32C, 1e-6)])
@pytest.mark.parametrize("spread", [0.01, 0.3])
def test_tile_edges(oracle_mod, prec, tol, spread, binning, nphi):
    params = dict(qnpts=21, q_min=-0.15, q_max=0.15, n_KT=4, KT_min=0.2, KT_max=0.7,
                  HBTrap_min=-1.0, HBTrap_max=1.0, needed_number_of_pairs=1e18,
                  number_of_mixed_events=2, azimuthal_flag=int(nphi > 0), n_Kphi=max(1, nphi),
                  hbt_binning=binning)
    rng = np.random.default_rng(17)
    # groups of one event and of several; sizes around 16, 32, 64 and their multiples
    groups = [cluster(rng, [n], spread) for n in (1, 2, 15, 16, 17, 31, 32, 33, 63, 64, 65, 129)]
    groups.append(cluster(rng, [64, 33, 1, 17, 95], spread))
    g = hbt.HBTCorrelation(params, precision=prec)
    g.calculate_groups(groups, hbt.Random(5))
    r = g.results()
    g.close()
    o = oracle_mod.Oracle(params)
    orng = oracle_mod.OracleRng(5)
    for b in groups:
        o.calculate_buffer(b, orng)
    a = o.arrays()
    assert a["num_count"].sum() > 1000 and a["den"].sum() > 1000
    assert np.array_equal(r.num_count, a["num_count"].astype(np.uint64))
    assert np.array_equal(r.den, a["den"].astype(np.uint64))
    for key, fl in SUMS:
        d = np.maximum(np.abs(a[key]), a[fl])
        err = np.abs(getattr(r, key) - a[key]) / np.where(d > 0, d, 1.0)
        assert float(err.max()) <= tol, key
