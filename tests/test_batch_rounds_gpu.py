"""Batches where their loops end otherwise than in the common case: items with
more segments than mode 2 stages in LDS at once, and right-hand sides that are
all zero.

Tolerance of the products: sums of up to 50,000 terms in another order stay
within 2^-53 sqrt(50000) = 2.5e-14 of the result's norm in FP64, 1e-13 asked;
FP32 operands and results with FP64 sums round to a few 2^-24, 1e-6 asked.
"""
import numpy as np
import pytest

from conftest import rel

pytestmark = pytest.mark.gpu

MAX_SLICES = 64  # of a problem's rows
# every launch shape of mode 2
SHAPES2 = [dict(rows_per_wave=4, nnz_per_lane=4, block_rows=256, block_cols=c, gather_kib=k)
           for c in (128, 256, 512) for k in (32, 64)]


@pytest.mark.parametrize("rhs,rays", [(1, 1100000), (2, 550000), (3, 300000), (4, 300000)])
def test_mode2_in_rounds_matches_oracle(P, O, gpu_available, rhs, rays):
    """All rays cross the one brick, so an item of at most 64 slices has
    rays / 64 segments on average, more than the largest staging capacity."""
    print(f"batch rounds: {rays} rays through one brick, {rhs} right-hand sides", flush=True)
    s = P.generate(4, 4, 8, rays, P.GEOM_OPPOSITE_FACES, 3, 0.02, 0.1)
    assert np.unique(s.k_row_idx).size == rays
    width = 4 if rhs == 3 else rhs
    assert rays / MAX_SLICES > 64 * 1024 // (4 * width), "FP32 in 64 KiB holds the most segments"
    orc = O.Oracle(s)
    rng = np.random.default_rng(rhs)
    X, Y = rng.standard_normal((rhs, s.n)), rng.standard_normal((rhs, s.m_k + s.m_d))
    want = X.copy()
    for k in range(rhs):
        orc.aprod(2, want[k], Y[k].copy())
    with P.Batch([s], rhs, flags=P.BATCH_NO_TUNE) as bt:
        for shape in SHAPES2:
            for precision, bar in ((P.PREC_FP64, 1e-13), (P.PREC_MIXED, 1e-6)):
                bt.set_tuning(precision, **shape)
                xg, _ = bt.aprod(2, [X.copy()], [Y], precision)
                for k in range(rhs):
                    assert rel(xg[0][k], want[k]) < bar, (shape, precision, k, rel(xg[0][k], want[k]))


@pytest.mark.parametrize("itn", [8, 9, 400])
def test_zero_right_hand_sides_end_after_one_launch(P, gpu_available, itn):
    """No state starts, so x stays zero and the solve costs about what one
    iteration on zeros costs, however many are asked for beyond eight (eight
    launches cost 2 to 3 times as much)."""
    print(f"zero right-hand sides, {itn} iterations", flush=True)
    systems = [P.generate(e, e, e, 8 * e ** 3, P.GEOM_OPPOSITE_FACES, e, 0.02, 0.1) for e in (40, 30)]
    zero = [np.zeros((4, s.m_k)) for s in systems]
    some = [np.zeros((4, s.m_k)) for s in systems]
    some[1][2] = 1.0
    with P.Batch(systems, 4, flags=P.BATCH_NO_TUNE) as bt:
        def best(n):
            return min(bt.solve(zero, n)[2] for _ in range(8))
        X, infos, _ = bt.solve(zero, itn)
        assert not any(x.any() for x in X) and all(i["itn"] == 0 for row in infos for i in row)
        one, many = best(1), best(itn)
        print(f"1 iteration {one * 1e3:.1f} us, {itn} {many * 1e3:.1f} us", flush=True)
        if itn > 8:
            assert many < 1.3 * one, (many, one)
        # one live state keeps the others' launches going
        X, infos, _ = bt.solve(some, itn)
        assert [i["itn"] for row in infos for i in row] == [0] * 6 + [itn, 0]
        assert X[1][2].any() and not X[0].any() and not X[1][[0, 1, 3]].any()
