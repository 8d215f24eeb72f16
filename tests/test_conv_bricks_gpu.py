"""The convolution kernel at the edges of its 8 x 8 x 8 bricks, on operands that
are not 16-byte aligned and in place, against the oracle's exact sums of the
same bf16 operands.

Tolerance: 864 products are added in FP32; each of the 55 additions of a
16-term step rounds to 2^-24 of a partial sum, so the 2-norm of the error stays
below 1e-5 of the result's.
"""
import ctypes as C
import os
import sys

import numpy as np
import pytest

from conftest import ROOT, rel

sys.path.insert(0, os.path.join(ROOT, "oracle"))
import cnn_oracle as K  # noqa: E402

pytestmark = pytest.mark.gpu


def operands(grid, batch, seed):
    rng = np.random.default_rng(seed)
    x = rng.standard_normal((batch, grid[0] * grid[1] * grid[2], 32)).astype(np.float32)
    w = (rng.standard_normal((27, 32, 32)) * 0.1).astype(np.float32)
    return x, w, rng.standard_normal(32).astype(np.float32), rng.standard_normal(x.shape).astype(np.float32)


@pytest.mark.parametrize("grid,batch", [((1, 1, 1), 1), ((8, 8, 8), 2), ((7, 9, 8), 1), ((9, 4, 17), 3), ((17, 5, 1), 2),
                                        ((2, 33, 3), 1)])
def test_conv_layer_on_ragged_bricks(P, gpu_available, grid, batch):
    print(f"conv layer: grid {grid}, batch {batch}", flush=True)
    x, w, b, d = operands(grid, batch, 3)
    for relu in (False, True):
        got = P.conv_forward(grid, x, w, b, relu=relu)
        assert rel(got, K.conv_forward(grid, K.bf16(x), K.bf16(w), b, relu=relu)) < 1e-5
    din, dw, db = P.conv_backward(grid, x, w, d)
    rdin, rdw, rdb = K.conv_backward(grid, K.bf16(x), K.bf16(w), K.bf16(d))
    assert rel(din, rdin) < 1e-5 and rel(dw, rdw) < 1e-5 and rel(db, rdb) < 1e-5


@pytest.mark.parametrize("how", ["offset", "in place"])
def test_conv_noalloc_takes_any_float_pointers(P, gpu_available, how):
    import torch
    print(f"noalloc conv forward, operands {how}", flush=True)
    lib = P.load()
    grid, batch = (9, 10, 11), 2
    x, w, b, _ = operands(grid, batch, 4)
    want = P.conv_forward(grid, x, w, b, relu=True)
    off = 1 if how == "offset" else 0  # floats past a 16-byte boundary

    def on_gpu(a):
        t = torch.zeros(a.size + off, dtype=torch.float32, device="cuda")
        t[off:] = torch.from_numpy(a.ravel()).cuda()
        return t

    x_d, w_d, b_d = on_gpu(x), on_gpu(w), on_gpu(b)
    out = x_d if how == "in place" else torch.zeros_like(x_d)
    ptr = [C.c_void_p(t.data_ptr() + 4 * off) for t in (x_d, w_d, b_d, out)]
    rc = lib.plsqr_cnn_conv_forward_noalloc(*grid, batch, ptr[0], ptr[1], ptr[2], 1, ptr[3],
                                            C.c_void_p(torch.cuda.current_stream().cuda_stream))
    assert rc == 0, lib.plsqr_cnn_last_error(None)
    torch.cuda.synchronize()
    assert np.array_equal(out[off:].cpu().numpy().reshape(x.shape), want)


# three taps per workgroup on short, long and single-voxel lines, and enough
# chunks of 4096 rows for nine, up to the longest line that takes them (191);
# ragged last chunks.  Each weight is a sum of up to 724k products in chains of
# 128 steps and 177 chunks: 2^-24 sqrt(300) of the result, well below 1e-5.
@pytest.mark.parametrize("grid,batch", [((260, 3, 3), 1), ((410, 3, 2), 2), ((600, 2, 2), 1), ((1, 70, 1), 2),
                                        ((20, 200, 181), 1), ((191, 61, 62), 1)])
def test_weight_gradient_layouts(P, gpu_available, grid, batch):
    print(f"weight gradient: grid {grid}, batch {batch}", flush=True)
    x, w, _, d = operands(grid, batch, 8)
    _, dw, db = P.conv_backward(grid, x, w, d)
    _, rdw, rdb = K.conv_backward(grid, K.bf16(x), K.bf16(w), K.bf16(d))
    assert rel(dw, rdw) < 1e-5 and rel(db, rdb) < 1e-5, (rel(dw, rdw), rel(db, rdb))
