"""Calls in which a pair cap may bind, on the fast kernel: its launch is tried
first and the ordered passes run for the keys that passed the cap.  Against a
context of the plain kernel, which takes the ordered passes alone, over caps
from zero (every key full at once), through ones passed by some K_T bins in
some buffers, to one that no counter reaches, per buffer, batched and side by
side, with and without q_inv and K_phi bins, in both precisions (a capped call
computes in FP64 in either).

Counts bit-exact.  Sums within 1e-12 of max(|S|, the bin's count times the
window's edge for q, times 1 for cos): the same FP64 terms in another order,
fewer than 1e4 per bin."""
import numpy as np
import pytest

from hadronic_afterburner_toolkit_amd import _lib, hbt, samples

pytestmark = pytest.mark.gpu


def config(cap, qinv, nphi):
    return dict(qnpts=11, q_min=-0.15, q_max=0.15, n_KT=4, KT_min=0.2, KT_max=0.7,
                HBTrap_min=-1.0, HBTrap_max=1.0, needed_number_of_pairs=cap,
                number_of_mixed_events=2, azimuthal_flag=int(nphi > 0), n_Kphi=max(1, nphi),
                invariant_radius_flag=qinv)


def run(params, bufs, how, **kw):
    g = hbt.HBTCorrelation(params, **kw)
    rng = hbt.Random(3)
    if how == "buffers":
        for b in bufs:
            g.calculate_HBT_correlation_function(b, rng)
    elif how == "batch":
        g.calculate_groups(bufs, rng)
        g.calculate_groups(bufs[::-1], rng)
    else:
        for b in bufs:
            g.upload(b)
            g.run_same()
            M, ids, cs = rng.draw_plan(b.nev, b.nev, 2)
            g.run_mixed(M, ids, cs)
    r = g.results()
    nd = g.deferred_pairs() if hasattr(g, "deferred_pairs") else 0
    g.close()
    return r, nd


@pytest.mark.parametrize("how", ["buffers", "batch", "sides"])
@pytest.mark.parametrize("qinv,nphi", [(0, 0), (1, 0), (0, 3)])
@pytest.mark.parametrize("prec", [_lib.HBT_PREC_FP64, _lib.HBT_PREC_FP32C])
@pytest.mark.parametrize("cap", [0, 40, 700, 4000, 60000])
def test_trial_equals_ordered(cap, prec, qinv, nphi, how):
    full = samples.generate(91, 12, 110.0)
    bufs = [full.events(0, 5), full.events(5, 4), full.events(9, 3)]
    params = config(cap, qinv, nphi)
    a, na = run(params, bufs, how, precision=prec)
    b, nb = run(params, bufs, how, precision=_lib.HBT_PREC_FP64, kernel=_lib.HBT_KERNEL_PLAIN)
    assert na == nb
    assert cap == 0 or b.num_count.sum() > 0
    for key in ("num_count", "den", "qinv_count", "qinv_den"):
        if getattr(b, key, None) is not None:
            assert np.array_equal(getattr(a, key), getattr(b, key)), key
    if prec == _lib.HBT_PREC_FP32C and cap == 60000:
        return  # the first calls are too small for it and add the precision form's sums
    n = b.num_count.astype(np.float64)
    for key, scale in (("q_out_sum", 0.1575), ("q_side_sum", 0.1575), ("q_long_sum", 0.1575),
                       ("num", 1.0)):
        ref = getattr(b, key)
        err = np.abs(getattr(a, key) - ref) / np.maximum(np.abs(ref), np.maximum(n, 1.0) * scale)
        assert float(err.max()) <= 1e-12, key
    n = b.qinv_count.astype(np.float64)
    for key, scale in (("qinv_sum", 0.1575), ("qinv_num", 1.0)):
        ref = getattr(b, key)
        err = np.abs(getattr(a, key) - ref) / np.maximum(np.abs(ref), np.maximum(n, 1.0) * scale)
        assert float(err.max()) <= 1e-12, key
