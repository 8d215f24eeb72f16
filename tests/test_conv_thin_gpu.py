"""Layers on grids that fill 8 x 8 x 8 bricks badly (thin, tiny, just past a
brick), which are computed by rows: against the oracle's exact sums of the same
bf16 operands, bit for bit against the brick kernel, inside the network, and in
time.

Tolerance of a layer as in test_conv_bricks_gpu.py: 864 products added in FP32,
1e-5 of the result's 2-norm.  Gradient of the network as in test_cnn_gpu.py: a
bf16 activation may round the other way after another FP32 order, 2e-2.
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


# three rounds of bricks over 256 CUs each, 1 to 91 voxels per brick; totals that
# end inside a wavefront's 32 rows and inside a workgroup's 256
SHAPES = [((1, 1, 1), 701), ((1, 1, 4201), 1), ((4201, 1, 1), 1), ((3, 2, 5), 700), ((9, 9, 9), 70), ((2, 9, 17), 90),
          ((4, 5, 3), 601)]


@pytest.mark.parametrize("grid,batch", SHAPES)
def test_layer_by_rows(P, gpu_available, grid, batch):
    print(f"layer by rows: grid {grid}, batch {batch}", flush=True)
    x, w, b, d = operands(grid, batch, 12)
    got = P.conv_forward(grid, x, w, b, relu=True)
    assert rel(got, K.conv_forward(grid, K.bf16(x), K.bf16(w), b, relu=True)) < 1e-5
    din, dw, db = P.conv_backward(grid, x, w, d)
    rdin, rdw, rdb = K.conv_backward(grid, K.bf16(x), K.bf16(w), K.bf16(d))
    assert rel(din, rdin) < 1e-5 and rel(dw, rdw) < 1e-5 and rel(db, rdb) < 1e-5
    if batch > 1:  # few samples at a time fit one brick per CU
        n = 8
        parts = [P.conv_forward(grid, x[k:k + n], w, b, relu=True) for k in range(0, batch, n)]
        assert np.array_equal(got, np.concatenate(parts)), "rows and bricks differ"


@pytest.mark.parametrize("off", [0, 1])
def test_layer_by_rows_on_any_float_pointer(P, gpu_available, off):
    import torch
    print(f"layer by rows, {off} floats past a 16-byte boundary", flush=True)
    lib = P.load()
    grid, batch = (2, 9, 17), 90
    x, w, b, _ = operands(grid, batch, 4)
    x[0, 0, 0], x[3, 7, 5] = np.inf, np.nan
    want = P.conv_forward(grid, x, w, b)

    def on_gpu(a):
        t = torch.zeros(a.size + off, dtype=torch.float32, device="cuda")
        t[off:] = torch.from_numpy(a.ravel()).cuda()
        return t

    x_d, w_d, b_d = on_gpu(x), on_gpu(w), on_gpu(b)
    for out in (torch.zeros_like(x_d), x_d):  # the second call in place
        ptr = [C.c_void_p(t.data_ptr() + 4 * off) for t in (x_d, w_d, b_d, out)]
        rc = lib.plsqr_cnn_conv_forward_noalloc(*grid, batch, ptr[0], ptr[1], ptr[2], 0, ptr[3],
                                                C.c_void_p(torch.cuda.current_stream().cuda_stream))
        assert rc == 0, lib.plsqr_cnn_last_error(None)
        torch.cuda.synchronize()
        assert np.array_equal(out[off:].cpu().numpy().reshape(x.shape), want, equal_nan=True)


@pytest.mark.parametrize("grid,batch", [((1, 3, 500), 9), ((2, 2, 2), 600)])
def test_network_by_rows(P, gpu_available, grid, batch):
    print(f"network by rows: grid {grid}, batch {batch}", flush=True)
    V = grid[0] * grid[1] * grid[2]
    rng = np.random.default_rng(7)
    atb, xs = rng.standard_normal((batch, V)) * 3.0, rng.standard_normal((batch, V))
    with P.WarmStartNet(grid, max_batch=batch, seed=11) as net, P.WarmStartNet(grid, max_batch=1, seed=11) as one:
        params = net.get_params()
        loss, g = net.gradient(atb, xs)
        assert np.array_equal(net.predict(atb), one.predict(atb)), "rows and bricks differ"
    ref = K.network(grid, params, atb, xs)
    assert abs(loss - ref["loss"]) < 1e-4 * ref["loss"], (loss, ref["loss"])
    lsz = 27 * 32 * 32 + 32
    for l in range(4):
        a, b = g[l * lsz:(l + 1) * lsz], ref["grads"][l * lsz:(l + 1) * lsz]
        assert rel(a, b) < 2e-2, (l, rel(a, b))


@pytest.mark.parametrize("grid,batch", [((1, 1, 1), 131072), ((1, 1, 131072), 1), ((2, 2, 2), 16384), ((1, 4, 32768), 1)])
def test_layer_time_follows_the_voxels(P, gpu_available, grid, batch):
    """131072 voxels take about as long whatever grid they lie on: by bricks of
    8^3 these took 3 to 60 times as long as 50^3."""
    import torch
    lib = P.load()

    def time_us(grid, batch):
        n = batch * grid[0] * grid[1] * grid[2] * 32
        x, w, b = torch.ones(n, device="cuda"), torch.ones(27 * 1024, device="cuda"), torch.ones(32, device="cuda")
        out = torch.empty_like(x)
        st = torch.cuda.current_stream().cuda_stream

        def call():
            assert lib.plsqr_cnn_conv_forward_noalloc(*grid, batch, *(C.c_void_p(t.data_ptr()) for t in (x, w, b)), 1,
                                                      C.c_void_p(out.data_ptr()), C.c_void_p(st)) == 0
        call()
        best = float("inf")
        for _ in range(5):
            e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            e0.record()
            for _ in range(10):
                call()
            e1.record()
            torch.cuda.synchronize()
            best = min(best, e0.elapsed_time(e1) * 100.0)
        return best

    full, thin = time_us((50, 50, 50), 1), time_us(grid, batch)
    print(f"50^3 {full:.1f} us, {grid} x {batch} {thin:.1f} us", flush=True)
    assert thin < 2 * full, (thin, full)
