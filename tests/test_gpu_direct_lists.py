"""One buffer's upload sends the device only what the calls on it read: the
lists that the device gathers, the host's sorted lists, or the columns of the
ordered passes.  The device memory a context takes for each, and the paths from
one to the other (prepared batch, side by side, capped) against the plain kernel.

Counts bit-exact; sums within 1e-12 of max(|S|, the bin's count times the
window's edge for q, times 1 for cos): the same FP64 terms in another order."""
import ctypes

import numpy as np
import pytest

from hadronic_afterburner_toolkit_amd import _lib, hbt, samples

pytestmark = pytest.mark.gpu


def config(cap=1e18):
    return dict(qnpts=15, q_min=-0.15, q_max=0.15, n_KT=4, KT_min=0.2, KT_max=0.7,
                HBTrap_min=-1.0, HBTrap_max=1.0, needed_number_of_pairs=cap,
                number_of_mixed_events=2)


def test_memory_follows_the_calls():
    hip = ctypes.CDLL("libamdhip64.so")

    def used():
        free, total = ctypes.c_size_t(), ctypes.c_size_t()
        assert hip.hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
        return total.value - free.value

    buf = samples.generate(3, 10, 6000.0)
    plan = hbt.Random(1).draw_plan(10, 10, 2)
    taken = {}
    for how in ("lists", "gathered"):
        g = hbt.HBTCorrelation(config())
        small = samples.generate(4, 2, 30.0)  # what a context takes at any rate
        g.upload(small)
        g.run_same()
        g.prepare_batch([1], np.zeros(2, np.int32), np.tile([1.0, 0.0], 2))
        g.launch_batch()
        g.sync()
        before = used()
        g.upload(buf)
        if how == "lists":
            g.prepare_batch([plan[0]], plan[1], plan[2])
            g.launch_batch()
            g.sync()
        else:
            g.run_same()
        taken[how] = used() - before
        g.close()
    # bytes a particle, and 8 MB for the items, the plan and rounding
    assert taken["lists"] <= 184 * 1.05 * buf.n + 4 * (2 << 20), taken
    assert taken["gathered"] <= (64 + 88) * 1.05 * buf.n + 4 * (2 << 20), taken


@pytest.mark.parametrize("cap", [0, 300, 5000, 1e18])
@pytest.mark.parametrize("own_mixed", [False, True])
def test_paths_of_one_upload(own_mixed, cap):
    full = samples.generate(17, 14, 130.0)
    a, b, other = full.events(0, 5), full.events(5, 3), full.events(8, 6)
    out = []
    for kernel in (_lib.HBT_KERNEL_FAST, _lib.HBT_KERNEL_PLAIN):
        g = hbt.HBTCorrelation(config(cap), kernel=kernel)
        draws = hbt.Random(9)
        if own_mixed:
            g.upload(other, 1)
        for buf in (a, b, a):
            g.upload(buf)
            plan = draws.draw_plan(buf.nev, 6 if own_mixed else buf.nev, 2)
            g.prepare_batch([plan[0]], plan[1], plan[2])
            g.launch_batch()
            g.run_same()
            g.run_mixed(*plan)
            g.calculate_HBT_correlation_function(buf, draws)
            g.prepare_batch([plan[0]], plan[1], plan[2])
            g.launch_batch()
            g.launch_batch()
        out.append(g.results())
        g.close()
    x, y = out
    assert cap == 0 or (y.num_count.sum() > 0 and y.den.sum() > 0)
    assert np.array_equal(x.num_count, y.num_count) and np.array_equal(x.den, y.den)
    n = np.maximum(y.num_count.astype(np.float64), 1.0)
    for key, scale in (("q_out_sum", .1575), ("q_side_sum", .1575), ("q_long_sum", .1575),
                       ("num", 1.0)):
        ref = getattr(y, key)
        err = np.abs(getattr(x, key) - ref) / np.maximum(np.abs(ref), n * scale)
        assert float(err.max()) <= 1e-12, key


def times(a, b, k):
    """a's histograms are k times b's (counts exactly)."""
    assert np.array_equal(a.num_count, b.num_count * np.uint64(k))
    assert np.array_equal(a.den, b.den * np.uint64(k))
    n = np.maximum(b.num_count.astype(np.float64), 1.0)
    for key, scale in (("q_out_sum", .0525), ("q_side_sum", .0525), ("q_long_sum", .0525),
                       ("num", 1.0)):
        ref = getattr(b, key)
        err = np.abs(getattr(a, key) / k - ref) / np.maximum(np.abs(ref), n * scale)
        assert float(err.max()) <= 1e-12, key


@pytest.mark.parametrize("mult,lists", [(100.0, False), (900.0, True)])
def test_a_large_narrow_batch_launched_again_takes_the_lists(mult, lists):
    """hbt_batch_graph tells the form: the walk without windows is no graph."""
    params = dict(config(), q_min=-0.05, q_max=0.05, number_of_mixed_events=0)
    buf = samples.generate(5, 20, mult)
    g = hbt.HBTCorrelation(params)
    g.calculate_HBT_correlation_function(buf, hbt.Random(1))
    assert (sum(g.batch_info()[:2]) > 250000000) == lists
    one = g.results()
    assert not g.batch_graph()
    for _ in range(2):
        g.launch_batch()
    assert g.batch_graph() == lists
    times(g.results(), one, 3)
    g.close()


@pytest.mark.parametrize("nev,mult", [(20, 100.0), (6, 8000.0)])
def test_a_side_run_again(nev, mult):
    params = dict(config(), q_min=-0.03, q_max=0.03)
    buf = samples.generate(6, nev, mult)
    plan = hbt.Random(1).draw_plan(nev, nev, 3)
    g = hbt.HBTCorrelation(params)
    g.upload(buf)
    g.run_same()
    g.run_mixed(*plan)
    one = g.results()
    for _ in range(2):
        g.run_same()
        g.run_mixed(*plan)
    times(g.results(), one, 3)
    g.close()
