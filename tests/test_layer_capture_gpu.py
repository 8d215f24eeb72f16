"""The allocation-free layer inside a captured HIP graph, by bricks, by rows and in
place: every replay against the eager calls, with eager work and synchronizations
between the replays."""
import ctypes as C

import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("grid,batch", [((9, 10, 11), 2), ((2, 9, 17), 90)])
@pytest.mark.parametrize("in_place", [False, True])
def test_captured_layer_replays(P, gpu_available, grid, batch, in_place):
    import torch
    print(f"captured layer: grid {grid}, batch {batch}, in place {in_place}", flush=True)
    lib = P.load()
    n = batch * grid[0] * grid[1] * grid[2] * 32
    gen = torch.Generator(device="cuda").manual_seed(3)
    w, bias = torch.randn(27 * 1024, generator=gen, device="cuda") * 0.03, torch.randn(32, generator=gen, device="cuda") * 0.1

    def layer(src, dst):
        rc = lib.plsqr_cnn_conv_forward_noalloc(*grid, batch, *(C.c_void_p(t.data_ptr()) for t in (src, w, bias)), 1,
                                                C.c_void_p(dst.data_ptr()), C.c_void_p(torch.cuda.current_stream().cuda_stream))
        assert rc == 0, lib.plsqr_cnn_last_error(None)

    x = torch.zeros(n, device="cuda")
    out = x if in_place else torch.zeros(n, device="cuda")
    layer(x, out)  # looks the device up before the capture
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        layer(x, out)
    for replay in range(4):
        fresh = torch.randn(n, generator=gen, device="cuda")
        want = torch.zeros(n, device="cuda")
        layer(fresh, want)
        x.copy_(fresh)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want), replay
