"""A capped batch whose pairs all lie on a K_phi bin edge (p_y = 0, unrotated
partners): each side leaves the host fewer than the 65536 pairs of the deferral
buffer, both sides together more.  The fast kernel against the plain one, which
takes the sides one after the other.

Counts bit-exact; sums within 1e-12 of max(|S|, the bin's count times the
window's edge for q, times 1 for cos): the same FP64 terms in another order."""
import numpy as np
import pytest

from hadronic_afterburner_toolkit_amd import _lib, hbt, samples

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("qinv", [0, 1])
@pytest.mark.parametrize("ngroups", [1, 2])
@pytest.mark.parametrize("prec", [_lib.HBT_PREC_FP64, _lib.HBT_PREC_FP32C])
def test_more_edge_pairs_than_the_deferral_buffer(prec, ngroups, qinv):
    rng = np.random.default_rng(4)
    nev, mult, M = 4, 70 if ngroups == 1 else 50, 2 if ngroups == 1 else 3

    def group():
        n = nev * mult
        px = 0.4 + 0.05 * rng.uniform(-1, 1, n)
        mt, y = np.sqrt(px * px + 0.13957 ** 2), 0.1 * rng.uniform(-1, 1, n)
        x = rng.normal(0.0, 3.0, (3, n))
        return samples.Buffer(np.arange(nev + 1, dtype=np.int64) * mult, px, np.zeros(n),
                              mt * np.sinh(y), mt * np.cosh(y), *x, 8.0 + rng.exponential(2.0, n))

    groups = [group() for _ in range(ngroups)]
    params = dict(qnpts=15, q_min=-0.15, q_max=0.15, n_KT=4, KT_min=0.2, KT_max=0.7,
                  HBTrap_min=-1.0, HBTrap_max=1.0, needed_number_of_pairs=9000,
                  azimuthal_flag=1, n_Kphi=3, invariant_radius_flag=qinv)
    ids = np.concatenate([(np.arange(nev)[:, None] + 1 + np.arange(M)).ravel() % nev] * ngroups)
    cs = np.tile([1.0, 0.0], ngroups * nev * M)
    out = []
    for kw in (dict(precision=prec), dict(precision=_lib.HBT_PREC_FP64,
                                          kernel=_lib.HBT_KERNEL_PLAIN)):
        g = hbt.HBTCorrelation(params, **kw)
        g.upload_groups(groups)
        g.prepare_batch([M] * ngroups, ids.astype(np.int32), cs)
        for _ in range(2):
            g.launch_batch()
        out.append((g.results(), g.deferred_pairs()))
        g.close()
    (a, na), (b, nb) = out
    assert na == nb and 65536 < na // 2 < 2 * 65536
    assert b.num_count.sum() > 0 and b.den.sum() > 0
    for key in ("num_count", "den", "qinv_count", "qinv_den", "cnt_num_ktphi", "cnt_den_ktphi"):
        assert np.array_equal(getattr(a, key), getattr(b, key)), key
    for cnt, keys in (("num_count", (("q_out_sum", .1575), ("q_side_sum", .1575),
                                     ("q_long_sum", .1575), ("num", 1.0))),
                      ("qinv_count", (("qinv_sum", .1575), ("qinv_num", 1.0)))):
        n = np.maximum(getattr(b, cnt).astype(np.float64), 1.0)
        for key, scale in keys:
            ref = getattr(b, key)
            err = np.abs(getattr(a, key) - ref) / np.maximum(np.abs(ref), n * scale)
            assert float(err.max()) <= 1e-12, key
