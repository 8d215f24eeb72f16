"""Products on vectors in the caller's order where the output is updated in place
and where it is reordered, before and after, around the product (mode 1 above
PLSQR_IN_PLACE_ROWS rows): both against the oracle and bit for bit alike.

FP64: sums in another order, 1e-13.  FP32 values, operands and results with
FP64 sums: a few 2^-24, 1e-6.
"""
import numpy as np
import pytest

from conftest import rel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("grid", ["auto", None])
@pytest.mark.parametrize("shape,rays", [((13, 17, 11), 6007), ((5, 9, 3), 70)])
def test_outputs_in_place_and_reordered(P, O, gpu_available, monkeypatch, shape, rays, grid):
    import torch
    print(f"caller order: {shape}, {rays} rays, grid {grid}", flush=True)
    s = P.generate(*shape, rays, P.GEOM_TOP_SOURCES, 5, 0.01, 0.1)
    orc = O.Oracle(s)
    rng = np.random.default_rng(6)
    x, y = rng.standard_normal(s.n), rng.standard_normal(s.m_k + s.m_d)
    x32, y32 = x.astype(np.float32), y.astype(np.float32)
    res = {}
    for limit in ("0", "1000000"):
        monkeypatch.setenv("PLSQR_IN_PLACE_ROWS", limit)
        out = []
        with P.Operator(s, grid=grid) as op:
            for mode in (1, 2):
                a, b = x.copy(), y.copy()
                op.aprod(mode, a, b)
                out.append(b if mode == 1 else a)
                a, b = torch.from_numpy(x).cuda(), torch.from_numpy(y).cuda()
                torch.cuda.synchronize()
                op.aprod_device(mode, a.data_ptr(), b.data_ptr())
                torch.cuda.synchronize()
                got, kept, was = (b, a, x) if mode == 1 else (a, b, y)
                assert np.array_equal(out[-1], got.cpu().numpy()) and np.array_equal(kept.cpu().numpy(), was)
                a, b = x32.copy(), y32.copy()
                op.aprod_f32(mode, a, b)
                out.append(b if mode == 1 else a)
        res[limit] = out
    for a, b in zip(*res.values()):
        assert np.array_equal(a, b)
    for i, mode in ((0, 1), (2, 2)):
        a, b = x.copy(), y.copy()
        orc.aprod(mode, a, b)
        assert rel(res["0"][i], b if mode == 1 else a) < 1e-13
        a, b = x32.astype(np.float64), y32.astype(np.float64)
        orc.aprod(mode, a, b)
        assert rel(res["0"][i + 1], b if mode == 1 else a) < 1e-6
