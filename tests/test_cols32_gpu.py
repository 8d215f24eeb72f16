"""FP32 mode 2 on both workgroup sizes (few items: 1024 threads, many: 512), one
and several LDS rounds per item, against the FP64 oracle.

FP32 values, u and results with FP64 sums: the rounding of values and result
bounds the difference by a few 1e-8 of the result; the bar is 1e-6.
"""
import numpy as np
import pytest

from conftest import rel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("grid,rays", [((40, 48, 48), 9001),   # 2880 items
                                       ((13, 17, 11), 6007),   # few items, ragged bricks
                                       ((4, 8, 8), 80000),     # one brick, two rounds of segments per item
                                       ((5, 9, 3), 70)])       # one row slice
def test_fp32_products_on_both_workgroup_sizes(P, O, gpu_available, grid, rays):
    print(f"fp32 products: grid {grid}, {rays} rays", flush=True)
    s = P.generate(*grid, rays, P.GEOM_OPPOSITE_FACES, 23, 0.01, 0.1)
    orc = O.Oracle(s)
    rng = np.random.default_rng(3)
    x = rng.standard_normal(s.n).astype(np.float32)
    y = rng.standard_normal(s.m_k + s.m_d).astype(np.float32)
    with P.Operator(s) as op:
        for mode in (1, 2):
            xg, yg, xo, yo = x.copy(), y.copy(), x.astype(np.float64), y.astype(np.float64)
            op.aprod_f32(mode, xg, yg)
            orc.aprod(mode, xo, yo)
            got, want = (yg, yo) if mode == 1 else (xg, xo)
            assert rel(got.astype(np.float64), want) < 1e-6, (mode, rel(got.astype(np.float64), want))
