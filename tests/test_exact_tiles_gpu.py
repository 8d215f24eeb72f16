"""The exact order's sequential norms on vectors around the line between short
(64) and long (512) tiles, bit for bit against the oracle: u with 127 to 257 rays
and fewer or more damping rows, v of 63 to 261 columns, a scale that rises late."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("grid", [(3, 3, 3), (7, 3, 3), (4, 4, 4), (13, 5, 3), (16, 4, 4), (29, 3, 3)])
@pytest.mark.parametrize("rays", [127, 128, 129, 255, 256, 257])
def test_norms_on_short_and_long_tiles(P, O, gpu_available, grid, rays):
    print(f"exact order tiles: grid {grid}, {rays} rays", flush=True)
    s = P.generate(*grid, rays, P.GEOM_OPPOSITE_FACES, 7, 0.01, 0.1)
    orc = O.Oracle(s)
    rng = np.random.default_rng(rays)
    with P.Operator(s, P.OP_EXACT_ORDER) as op:
        for late in (False, True):
            b = rng.standard_normal(rays)
            if late:
                b[-2:] = 1e3, -2e3
            x, info = op.lsqr(b, 4)
            xo, out, _ = orc.lsqr(b, 4)
            assert np.array_equal(x, xo), np.abs(x - xo).max()
            assert info["bnorm"] == out["bnorm"] and info["rnorm"] == out["rnorm"]
