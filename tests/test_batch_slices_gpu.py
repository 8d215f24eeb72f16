"""Batched products where the row-slice rule reaches its limits: fewer rows than
slices, the 64-slice cap on one tile, systems without a grid, one next to a
larger one, for every right-hand-side width, against the oracle.

Tolerance: sums of at most a few thousand terms in another order, 1e-13
relative in FP64; FP32 values and results, 1e-6.
"""
import numpy as np
import pytest

from conftest import rel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rhs", [1, 2, 3, 4])
def test_batch_products_on_uneven_slices(P, O, gpu_available, rhs):
    print(f"batch slices: {rhs} right-hand sides", flush=True)
    shapes = [((3, 3, 3), 20000), ((5, 4, 3), 3), ((17, 9, 11), 4000), ((4, 8, 9), 129)]
    systems = [P.generate(*g, r, P.GEOM_OPPOSITE_FACES, 31 + i, 0.01, 0.1) for i, (g, r) in enumerate(shapes)]
    grids = [s.grid for s in systems]
    grids[3] = None
    rng = np.random.default_rng(rhs)
    X = [rng.standard_normal((rhs, s.n)) for s in systems]
    Y = [rng.standard_normal((rhs, s.m_k + s.m_d)) for s in systems]
    with P.Batch(systems, rhs, grids=grids, flags=P.BATCH_NO_TUNE) as bt:
        for precision, bar in ((P.PREC_FP64, 1e-13), (P.PREC_MIXED, 1e-6)):
            for mode in (1, 2):
                xg, yg = bt.aprod(mode, X, Y, precision)
                for p, s in enumerate(systems):
                    orc = O.Oracle(s)
                    for k in range(rhs):
                        x, y = X[p][k].copy(), Y[p][k].copy()
                        orc.aprod(mode, x, y)
                        got, want = (yg[p][k], y) if mode == 1 else (xg[p][k], x)
                        assert rel(got, want) < bar, (precision, mode, p, k, rel(got, want))
