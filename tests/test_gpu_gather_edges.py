"""The device's gathers at the edges of their launches: one block up to 2048
particles (1024, 1025: one and two particles a thread; 2048, 2049: its list full,
and a block per event), one scan fewer up to 1024 events (1024, 1025), with empty
events first, between and last.  The per-buffer and the side-by-side entry points
against the host's lists, hbt_calculate_noalloc against the plain kernel; same
bounds as in the tests of those entry points.  And the side runs of q_inv analyses
above 9000 particles."""
import numpy as np
import pytest

import test_gpu_direct as direct
import test_zz_no_alloc_edges as noalloc
from hadronic_afterburner_toolkit_amd import _lib, hbt

pytestmark = pytest.mark.gpu

SIZES = {
    "1023": [0, 500, 0, 523], "1024": [0, 500, 0, 524, 0], "1025": [500, 0, 525],
    "2047": [1000, 0, 1047], "2048": [0, 1024, 0, 1023, 1], "2049": [0, 1024, 0, 1024, 1, 0],
    "1024 events": [0] + [7] * 1022 + [0], "1025 events": [7] * 1023 + [0, 5],
}


@pytest.mark.parametrize("size", list(SIZES))
@pytest.mark.parametrize("how", ["buffer", "sides", "mixed buffer"])
@pytest.mark.parametrize("qinv", [0, 1])
def test_gathered_lists(size, how, qinv):
    counts = SIZES[size]
    direct.test_direct_equals_lists(counts, 0.5, _lib.HBT_PREC_FP64, qinv, 0, how)


@pytest.mark.parametrize("size", list(SIZES))
def test_noalloc(size):
    noalloc.test_noalloc_edges(SIZES[size], 2, 0.5, False)


@pytest.mark.parametrize("counts", [[300] * 60, [900, 0, 1026, 8000]])
def test_qinv_sides_of_many_particles(counts):
    rng = np.random.default_rng(sum(counts))
    buf = direct.events(rng, counts, 0.8)
    M, ids, cs = hbt.Random(7).draw_plan(buf.nev, buf.nev, 2)
    g = hbt.HBTCorrelation(direct.config(qinv=1))
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
    assert b.qinv_count.sum() > 10000
    direct.same(a, b)
