"""hbt_calculate_noalloc at the edges of its tiles and of its two gathers
(one block up to 8192 particles, a block per event beyond): event sizes around
16, 32 and 64 and the chunk of 1024, empty events, no plan rows, several rows
per work item, partner ids outside the buffer (no pairs: the reference names an
empty event instead), and particles with E < 0.  Against the plain FP64 kernel
of a context on the same buffer and plan, every pair evaluated there.

Counts bit-exact; sums within 1e-12 of max(|S|, the bin's count times the
window's edge for q, times 1 for cos) (both are the same FP64 terms in another
order: a bin of n <= 1e4 terms differs by at most n 2^-53 of that)."""
import numpy as np
import pytest

import test_zz_no_alloc as na
from hadronic_afterburner_toolkit_amd import samples

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


CASES = [
    ([1, 0, 2], 2, 0.02, False),
    ([15, 16, 17, 0, 31, 32, 33], 3, 0.1, False),
    ([63, 64, 65, 0, 1], 5, 0.3, True),
    ([90] * 7 + [0], 0, 0.5, False),
    ([1024, 0, 1025, 6143], 2, 0.5, False),   # 8192 particles: one block gathers
    ([1023, 1, 1026, 0, 6143], 2, 0.5, True),  # 8193: a block per event
    ([300] * 60 + [0], 3, 0.8, False),
    ([8] * 1300 + [0], 20, 0.8, False),        # more events than the scan's threads
]


@pytest.mark.parametrize("counts,M,spread,neg", CASES)
def test_noalloc_edges(counts, M, spread, neg):
    rng = np.random.default_rng(len(counts) + M)
    buf = events(rng, counts, spread)
    if neg:
        buf.E[::7] *= -1.0
        buf.pz[::7] *= -1.0
    nev = buf.nev
    empty = int(np.flatnonzero(np.diff(buf.ev_off) == 0)[0]) if 0 in counts else 0
    ids = rng.integers(0, nev, (nev, M)).astype(np.int32)
    th = rng.uniform(-np.pi, np.pi, (nev, M))
    cs = np.stack([np.cos(th), np.sin(th)], axis=-1)
    out = ids.copy()
    if M > 1:
        ids[::2, 1] = empty
        out[::4, 1] = -1
        out[2::4, 1] = nev
    if M == 0:
        r = na.existing_entry(buf, 1, np.full((nev, 1), empty, np.int32), np.ones((nev, 1, 2)))
    else:
        r = na.existing_entry(buf, M, ids, cs)
    hip = na.Hip()
    stream = hip.stream()
    bins = na.noalloc_entry(hip, buf, M, out, cs, stream)
    hip.h.hipStreamDestroy(stream)
    n = r.num_count.astype(np.float64)
    if buf.n > 100:  # enough particles for pairs in every window
        assert n.sum() > 0 and (M == 0 or r.den.sum() > 0)
    assert np.array_equal(bins[:, 0], n)
    assert np.array_equal(bins[:, 5].view(np.uint64), r.den)
    for col, key, scale in ((1, "q_out_sum", 0.1575), (2, "q_side_sum", 0.1575),
                            (3, "q_long_sum", 0.1575), (4, "num", 1.0)):
        ref = getattr(r, key)
        err = np.abs(bins[:, col] - ref) / np.maximum(np.abs(ref), np.maximum(n, 1.0) * scale)
        assert float(err.max()) <= 1e-12, key
