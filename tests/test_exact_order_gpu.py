"""The exact-order kernels bit for bit against the oracle where they can go
wrong: vector lengths around the 64-element groups and 512-element tiles of
the sequential norms, elements that raise the norm's scale in every position,
and segments longer and shorter than a staging round.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def right_hand_side(kind, m, rng):
    b = rng.standard_normal(m)
    if kind == "ascending":      # every element is a new scale
        b = np.arange(1, m + 1) * 1.7
    elif kind == "zeros":        # leading, trailing and scattered zeros
        b[rng.random(m) < 0.6] = 0.0
        b[: m // 3] = 0.0
        b[m // 2] = -3.0
    elif kind == "last":         # the scale rises in the last element
        b *= 1e-3
        b[-1] = 1e3
    elif kind == "range":        # many orders of magnitude
        b *= 10.0 ** rng.integers(-12, 12, m)
    return b


@pytest.mark.parametrize("m_k", [1, 2, 63, 64, 65, 511, 512, 513, 1024, 1600])
def test_exact_order_solves_are_bitwise_the_oracle(P, O, gpu_available, m_k):
    s = P.generate(5, 4, 3, m_k, P.GEOM_OPPOSITE_FACES, 7, 0.01, 0.1)
    orc = O.Oracle(s)
    rng = np.random.default_rng(m_k)
    with P.Operator(s, P.OP_EXACT_ORDER) as op:
        for kind in ("normal", "ascending", "zeros", "last", "range"):
            print(f"exact order: {m_k} rays, b {kind}", flush=True)
            b = right_hand_side(kind, m_k, rng)
            x, info = op.lsqr(b, 4)
            xo, out, _ = orc.lsqr(b, 4)
            assert np.array_equal(x, xo), (kind, np.abs(x - xo).max())
            assert info["bnorm"] == out["bnorm"] and info["rnorm"] == out["rnorm"], kind


# (grid, rays): mean row / column lengths on both sides of the segment widths
# (64, 16, 4 per wavefront) and of a 512-entry round
@pytest.mark.parametrize("grid,rays", [((3, 3, 3), 9001), ((4, 4, 4), 65), ((40, 3, 3), 301), ((90, 4, 3), 517),
                                       ((9, 8, 7), 3)])
def test_exact_order_products_are_bitwise_the_oracle(P, O, gpu_available, grid, rays):
    print(f"exact order products: grid {grid}, {rays} rays", flush=True)
    s = P.generate(*grid, rays, P.GEOM_OPPOSITE_FACES, 11, 0.01, 0.1)
    orc = O.Oracle(s)
    rng = np.random.default_rng(5)
    x, y = rng.standard_normal(s.n), rng.standard_normal(s.m_k + s.m_d)
    with P.Operator(s, P.OP_EXACT_ORDER) as op:
        for mode in (1, 2):
            xg, yg, xo, yo = x.copy(), y.copy(), x.copy(), y.copy()
            op.aprod(mode, xg, yg)
            orc.aprod(mode, xo, yo)
            assert np.array_equal(xg, xo) and np.array_equal(yg, yo), mode
