"""The fast kernel far from mid-rapidity, where the rounding of q_long (in any
form) grows as the square of the pair's longitudinal boost: counts of both
precisions bit-identical to the plain kernel's literal cascade, sums within
1e-12 (FP64) and 1e-6 (precision form) of max(|S|, the bin's count times the
window's edge for q, times 1 for cos): the same terms in another order, and
FP32's cos."""
import numpy as np
import pytest

from hadronic_afterburner_toolkit_amd import _lib, hbt, samples

pytestmark = pytest.mark.gpu


def events(rng, y0, counts):
    n = int(sum(counts))
    px, py = 0.35 + 0.2 * rng.uniform(-1, 1, n), 0.2 + 0.2 * rng.uniform(-1, 1, n)
    mt = np.sqrt(px * px + py * py + 0.13957 ** 2)
    y = y0 + 0.15 * rng.uniform(-1, 1, n)
    x = rng.normal(0.0, 3.0, (3, n))
    return samples.Buffer(np.concatenate([[0], np.cumsum(counts)]).astype(np.int64), px, py,
                          mt * np.sinh(y), mt * np.cosh(y), *x, 8.0 + rng.exponential(2.0, n))


@pytest.mark.parametrize("how", ["buffer", "batch"])
@pytest.mark.parametrize("prec,tol", [(_lib.HBT_PREC_FP64, 1e-12), (_lib.HBT_PREC_FP32C, 1e-6)])
@pytest.mark.parametrize("y0", [7.6, 10.0, -12.0, 13.0, 15.0])
def test_boosted_pairs(y0, prec, tol, how):
    rng = np.random.default_rng(int(abs(y0) * 10))
    bufs = [events(rng, y0, [400, 300, 500]), events(rng, y0, [250, 450])]
    params = dict(qnpts=41, q_min=-0.15, q_max=0.15, n_KT=6, KT_min=0.2, KT_max=0.7,
                  HBTrap_min=-17.0, HBTrap_max=17.0, needed_number_of_pairs=1e18,
                  number_of_mixed_events=2)
    out = []
    for kw in (dict(precision=prec), dict(kernel=_lib.HBT_KERNEL_PLAIN)):
        g = hbt.HBTCorrelation(params, **kw)
        draws = hbt.Random(2)
        if how == "buffer":
            for b in bufs:
                g.calculate_HBT_correlation_function(b, draws)
        else:
            g.calculate_groups(bufs, draws)
        out.append(g.results())
        g.close()
    a, b = out
    assert int(b.num_count.sum()) > 1e5 and int(b.den.sum()) > 1e4
    assert np.array_equal(a.num_count, b.num_count)
    assert np.array_equal(a.den, b.den)
    n = np.maximum(b.num_count.astype(np.float64), 1.0)
    for key, scale in (("q_out_sum", .1575), ("q_side_sum", .1575), ("q_long_sum", .1575),
                       ("num", 1.0)):
        ref = getattr(b, key)
        err = np.abs(getattr(a, key) - ref) / np.maximum(np.abs(ref), n * scale)
        assert float(err.max()) <= tol, key
