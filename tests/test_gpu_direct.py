"""One buffer gathered on the device and walked without windows (the per-buffer
and the side-by-side entry points) against the host's sorted lists and windowed
items (hbt_prepare_batch takes them for the same upload): event sizes around 16,
32 and 64, empty events, one block's gather (up to 8192 particles) and a block
per event, a mixed-event buffer of its own, q_inv and K_phi bins, both
precisions; and the entry points that go from one form to the other on a
prepared call.

Counts bit-exact.  Sums within 1e-12 of max(|S|, the bin's count times the
window's edge for q, times 1 for cos): the same terms in another order, fewer
than 1e4 per bin."""
import numpy as np
import pytest

from hadronic_afterburner_toolkit_amd import _lib, hbt, samples

pytestmark = pytest.mark.gpu


def events(rng, counts, spread):
    n = int(sum(counts))
    px = 0.35 + spread * rng.uniform(-1, 1, n)
    py = 0.20 + spread * rng.uniform(-1, 1, n)
    mt = np.sqrt(px * px + py * py + 0.13957 ** 2)
    y = rng.uniform(-1.2, 1.2, n)
    x = rng.normal(0.0, 3.0, (3, n))
    return samples.Buffer(np.concatenate([[0], np.cumsum(counts)]).astype(np.int64), px, py,
                          mt * np.sinh(y), mt * np.cosh(y), *x, 8.0 + rng.exponential(2.0, n))


def config(qinv=0, nphi=0):
    return dict(qnpts=15, q_min=-0.15, q_max=0.15, n_KT=4, KT_min=0.2, KT_max=0.7,
                HBTrap_min=-1.0, HBTrap_max=1.0, needed_number_of_pairs=1e18,
                number_of_mixed_events=2, azimuthal_flag=int(nphi > 0), n_Kphi=max(1, nphi),
                invariant_radius_flag=qinv)


def same(a, b):
    for key in ("num_count", "den", "qinv_count", "qinv_den"):
        assert np.array_equal(getattr(a, key), getattr(b, key)), key
    for cnt, keys in (("num_count", (("q_out_sum", .1575), ("q_side_sum", .1575),
                                     ("q_long_sum", .1575), ("num", 1.0))),
                      ("qinv_count", (("qinv_sum", .1575), ("qinv_num", 1.0)))):
        n = getattr(b, cnt).astype(np.float64)
        for key, scale in keys:
            ref = getattr(b, key)
            err = np.abs(getattr(a, key) - ref)
            err /= np.maximum(np.abs(ref), np.maximum(n, 1.0) * scale)
            assert float(err.max()) <= 1e-12, key


SIZES = [([1], 0.02), ([15, 16, 17, 0, 31, 32, 33], 0.1), ([63, 64, 65, 0, 1], 0.3),
         ([900, 0, 1025, 6267], 0.6), ([900, 0, 1026, 6267], 0.6), ([300] * 60, 0.8)]


@pytest.mark.parametrize("how", ["buffer", "mixed buffer", "sides"])
@pytest.mark.parametrize("qinv,nphi", [(0, 0), (1, 0), (0, 3)])
@pytest.mark.parametrize("prec", [_lib.HBT_PREC_FP64, _lib.HBT_PREC_FP32C])
@pytest.mark.parametrize("counts,spread", SIZES)
def test_direct_equals_lists(counts, spread, prec, qinv, nphi, how):
    if how == "sides" and sum(counts) > 9000 and qinv:
        pytest.skip("every pair takes the literal cascade: the same kernel as 'buffer'")
    rng = np.random.default_rng(sum(counts))
    buf = events(rng, counts, spread)
    other = events(rng, counts[::-1] + [40], spread) if how == "mixed buffer" else None
    nm = (other or buf).nev
    M, ids, cs = hbt.Random(7).draw_plan(buf.nev, nm, 2)
    g = hbt.HBTCorrelation(config(qinv, nphi), precision=prec)

    def upload():
        g.upload(buf)
        if other is not None:
            g.upload(other, 1)

    upload()
    if how == "sides":
        g.run_same()
        g.run_mixed(M, ids, cs)
    else:
        g.calculate_HBT_correlation_function(buf, hbt.Random(7), other)
    a = g.results()
    na, sa = g.deferred_pairs(), g.stage_counts()
    g.reset()
    upload()
    g.prepare_batch([M], ids, cs)
    g.launch_batch()
    b = g.results()
    assert g.deferred_pairs() - na == na
    for x, y in zip(sa, g.stage_counts()):
        assert list(x) == list(y)
    g.close()
    if sum(counts) > 100:
        assert b.num_count.sum() > 0 and b.den.sum() > 0
    same(a, b)


def test_direct_call_goes_on_as_a_batch():
    rng = np.random.default_rng(5)
    bufs = [events(rng, [200] * 20, 0.5), events(rng, [90] * 7, 0.5)]
    g = hbt.HBTCorrelation(config(), precision=_lib.HBT_PREC_FP64)
    r1 = hbt.Random(3)
    for b in bufs:
        g.calculate_HBT_correlation_function(b, r1)
    g.launch_batch()          # the last buffer once more, on the device's lists
    g.set_tuning(1, 256, 4, 8)
    g.launch_batch()          # and on the host's
    a = g.results()
    g.reset()
    r2 = hbt.Random(3)
    g.calculate_HBT_correlation_function(bufs[0], r2)
    M, ids, cs = r2.draw_plan(7, 7, 2)
    g.upload(bufs[1])
    g.prepare_batch([M], ids, cs)
    for _ in range(3):
        g.launch_batch()
    same(a, g.results())
    g.close()


@pytest.mark.parametrize("boost", [0, 1])
@pytest.mark.parametrize("shell", ["on", "rounded", "two masses", "massless"])
def test_qinv_windows(shell, boost):
    """q_inv bins: particles on one mass shell, within the room of it (energies
    rounded to seven digits), of two masses, and massless (the last two leave
    every pair to the cascade); wide momenta, so that q_out far outside the 3D
    windows bins in q_inv."""
    rng = np.random.default_rng(11)
    buf = events(rng, [150] * 20, 1.2)
    if shell == "rounded":
        buf.E[:] = np.array([float("%.6e" % e) for e in buf.E])
    elif shell == "two masses":
        p2 = buf.px ** 2 + buf.py ** 2 + buf.pz ** 2
        buf.E[::3] = np.sqrt(p2[::3] + 0.494 ** 2)
    elif shell == "massless":
        buf.E[:] = np.sqrt(buf.px ** 2 + buf.py ** 2 + buf.pz ** 2)
    params = dict(config(qinv=1), long_comoving_boost=boost, KT_max=1.5)
    M, ids, cs = hbt.Random(7).draw_plan(buf.nev, buf.nev, 4)
    g = hbt.HBTCorrelation(params, precision=_lib.HBT_PREC_FP64)
    g.upload(buf)
    g.run_same()
    g.run_mixed(M, ids, cs)
    a = g.results()
    g.reset()
    g.upload(buf)
    g.prepare_batch([M], ids, cs)
    g.launch_batch()
    b = g.results()
    g.close()
    assert b.qinv_count.sum() > 5000 and b.qinv_den.sum() > 5000
    same(a, b)
