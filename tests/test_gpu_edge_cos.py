"""Pairs on a bin edge or on a window's cut (to within 1e-9 bins) in the
precision form: decided by the literal cascade, whose FP64 cos they keep.  Groups
of two particles, so that a bin holds a few pairs; counts equal to the FP64
form's, sums within 1e-12 of max(|S|, the bin's count times the window's edge for
q, times 1 for cos) -- FP32's cos would differ by some 1e-8."""
import numpy as np
import pytest

from hadronic_afterburner_toolkit_amd import _lib, hbt, samples

pytestmark = pytest.mark.gpu

Q, QMAX, NKT, K0, K1 = 21, 0.1, 5, 0.2, 0.6
DQ, DK = 2 * QMAX / (Q - 1), (K1 - K0) / (NKT - 1)


@pytest.mark.parametrize("at", ["q_long", "q_out", "q_side", "cut", "K_T"])
@pytest.mark.parametrize("binning", [0, 1])
def test_edge_pairs_keep_fp64_cos(at, binning):
    rng = np.random.default_rng(3)
    n = 600
    q = {k: rng.uniform(-0.9 * QMAX, 0.9 * QMAX, n) for k in ("q_out", "q_side", "q_long")}
    K = rng.uniform(K0 + 0.02, K1 - 0.02, n)
    if at == "K_T":
        K = K0 + DK * rng.integers(1, NKT - 1, n)
    elif at == "cut":
        q["q_long"] = rng.choice([-1, 1], n) * (QMAX + DQ / 2 - 1e-8) * (1 - 1e-14)
    else:
        q[at] = DQ * (rng.integers(-8, 9, n) + 0.5)
    # K along x, no boost: q_out, q_side, q_long are the differences in x, y, z
    kz = rng.uniform(-0.1, 0.1, n)
    p1 = np.stack([K + q["q_out"] / 2, q["q_side"] / 2, kz + q["q_long"] / 2])
    p2 = np.stack([K - q["q_out"] / 2, -q["q_side"] / 2, kz - q["q_long"] / 2])
    p = np.stack([p1, p2], axis=2).reshape(3, 2 * n)  # 1, 2, 1, 2, ...
    E = np.sqrt(0.13957 ** 2 + (p * p).sum(0))
    x = rng.normal(0.0, 3.0, (3, 2 * n))
    buf = samples.Buffer(np.arange(0, 2 * n + 1, 2), *p, E, *x, 8.0 + rng.exponential(2.0, 2 * n))
    groups = [buf.events(k, 1) for k in range(n)]
    params = dict(qnpts=Q, q_min=-QMAX, q_max=QMAX, n_KT=NKT, KT_min=K0, KT_max=K1,
                  HBTrap_min=-3.0, HBTrap_max=3.0, needed_number_of_pairs=1e18,
                  long_comoving_boost=0, hbt_binning=binning)
    out = []
    for prec in (_lib.HBT_PREC_FP64, _lib.HBT_PREC_FP32C):
        g = hbt.HBTCorrelation(params, precision=prec)
        g.upload_groups(groups)
        g.prepare_batch([0] * n, np.zeros(0, np.int32), np.zeros(0))
        g.launch_batch()
        out.append(g.results())
        g.close()
    b, a = out
    assert b.num_count.sum() > n // 4
    assert np.array_equal(a.num_count, b.num_count)
    count = np.maximum(b.num_count.astype(np.float64), 1.0)
    sums = (("num", 1.0),) if binning else (("q_out_sum", .105), ("q_side_sum", .105),
                                            ("q_long_sum", .105), ("num", 1.0))
    tol = 2.0 ** -23 if binning else 1e-12  # slab binning's values are FP32 on either path
    for key, scale in sums:
        ref = getattr(b, key)
        err = np.abs(getattr(a, key) - ref) / np.maximum(np.abs(ref), count * scale)
        assert float(err.max()) <= tol, key
