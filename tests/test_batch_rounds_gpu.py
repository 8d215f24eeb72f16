"""Batches at the ends of their iteration loop: right-hand sides that are all zero."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


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
