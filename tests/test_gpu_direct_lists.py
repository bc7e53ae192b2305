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
