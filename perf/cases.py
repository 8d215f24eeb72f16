"""The workloads this library's speed is judged by.

Each case is one call (or one short sequence of calls) that a program makes
through the public entry points with everything it keeps between calls already
in hand: the operator of a system, a batch handle, a network.  The kinds:

  lsqr     Operator.lsqr_device, FP64 or the checked mixed solve on A D
  exact    the same on an exact-order operator (the reference's own order)
  aprod    y += A x and x += A^T y on device vectors in the caller's order
  batch    Batch.solve_device: uneven systems with several right-hand sides
  conv     one 32 -> 32 layer on device tensors (the allocation-free entry)
  convback the data, weight and bias gradients of one layer (host arrays)
  predict  WarmStartNet.predict: network inputs to starting points
  train    WarmStartNet.train: Adam steps, then the updated parameters

Systems are seeded straight-ray tomography problems.  Iteration counts are
chosen so that x is a well-conditioned function of the inputs: either a few
iterations, before rounding differences grow, or a run to convergence.
"""
import ctypes
import importlib.util
import math
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(ROOT, "plsqr3.2013.09_amd")
WEIGHTS = os.path.join(PKG, "weights", "warmstart_grid67_rays2m.npy")
TAPS, CH, LAYERS = 27, 32, 4
LAYER = TAPS * CH * CH + CH  # parameters of one layer: weights [tap][out][in], bias


def _pkg():
    name = "plsqr_amd"
    if name not in sys.modules:
        spec = importlib.util.spec_from_file_location(name, os.path.join(PKG, "__init__.py"),
                                                      submodule_search_locations=[PKG])
        mod = importlib.util.module_from_spec(spec)
        sys.modules[name] = mod
        spec.loader.exec_module(mod)
    return sys.modules[name]


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------
def listed():
    return [
        # the headline system: the FP64 iteration loop of a time-to-tol solve
        dict(name="lsqr_grid67_rays2m", kind="lsqr", nx=67, ny=67, nz=67, rays=2000000, top=True, lam=0.05, itn=10,
             mixed=False),
        # the smallest configuration: a whole solve of a small system, run to convergence
        dict(name="lsqr_grid16_rays20k", kind="lsqr", nx=16, ny=16, nz=16, rays=20000, top=False, lam=0.1, itn=200,
             mixed=False),
        # mixed precision on A D with adaptive FP64 checks, solved to test2 <= 1e-9
        dict(name="lsqr_mixed_grid32", kind="lsqr", nx=32, ny=32, nz=32, rays=262144, top=False, lam=0.1, itn=600,
             mixed=True),
        # a solve that has to reproduce the reference's x bit for bit
        dict(name="exact_grid24_rays60k", kind="exact", nx=24, ny=24, nz=24, rays=60000, top=True, lam=0.05, itn=10,
             mixed=False),
        # a caller's own iteration: FP64 products on a ragged grid
        dict(name="aprod_f64_37x29x41", kind="aprod", nx=37, ny=29, nz=41, rays=351000, top=False, lam=0.1, f32=False),
        # the FP32 operator on a mid-size top-face system
        dict(name="aprod_f32_grid48", kind="aprod", nx=48, ny=48, nz=48, rays=700000, top=True, lam=0.05, f32=True),
        # the smallest products: launch latency
        dict(name="aprod_f64_12x10x9", kind="aprod", nx=12, ny=10, nz=9, rays=3000, top=False, lam=0.1, f32=False),
        # several small surveys with four right-hand sides each, run to convergence
        dict(name="batch6_grid12to24_rhs4", kind="batch", problems=6, lo=12, hi=24, per_col=8, rhs=4, itn=250),
        # one network layer in a serving loop
        dict(name="conv_48x48x48", kind="conv", nx=48, ny=48, nz=48, batch=1, relu=True),
        # one layer's gradients on a ragged grid
        dict(name="convback_31x27x35_b2", kind="convback", nx=31, ny=27, nz=35, batch=2),
        # a starting point for one new right-hand side of the headline grid
        dict(name="predict_grid67", kind="predict", nx=67, ny=67, nz=67, count=1, max_batch=4),
        # training steps on the headline grid at the pipeline's batch size
        dict(name="train_grid67_b4", kind="train", nx=67, ny=67, nz=67, batch=4, samples=8, steps=2),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _grid(rng, lo, hi):
    """Edges around one size, each odd or even: ragged bricks are the rule."""
    e = _log(rng, lo, hi)
    return tuple(max(lo, min(hi, e + rng.randint(-e // 6, e // 6))) for _ in range(3))


def draw(rng):
    kind = rng.choice(["lsqr", "lsqr", "mixed", "exact", "aprod", "aprod", "aprod", "batch", "conv", "conv",
                       "convback", "predict", "train"])
    if kind == "lsqr" and rng.random() < 0.5:  # the first iterations of a larger system
        nx, ny, nz = _grid(rng, 28, 64)
        return dict(kind="lsqr", nx=nx, ny=ny, nz=nz, rays=int(nx * ny * nz * rng.uniform(3.0, 6.5)),
                    top=rng.random() < 0.5, lam=0.05, itn=rng.randint(6, 10), mixed=False)
    if kind in ("lsqr", "mixed"):  # a small or middle system to convergence
        nx, ny, nz = _grid(rng, 9, 32)
        rays = int(nx * ny * nz * rng.uniform(4.0, 8.0))
        return dict(kind="lsqr", nx=nx, ny=ny, nz=nz, rays=rays, top=False, lam=0.1,
                    itn=600 if kind == "mixed" else 300, mixed=kind == "mixed")
    if kind == "exact":
        nx, ny, nz = _grid(rng, 8, 26)
        return dict(kind="exact", nx=nx, ny=ny, nz=nz, rays=int(nx * ny * nz * rng.uniform(2.0, 5.0)),
                    top=rng.random() < 0.5, lam=0.05, itn=rng.randint(4, 10), mixed=False)
    if kind == "aprod":
        nx, ny, nz = _grid(rng, 8, 52)
        return dict(kind="aprod", nx=nx, ny=ny, nz=nz, rays=int(nx * ny * nz * rng.uniform(2.5, 7.0)),
                    top=rng.random() < 0.5, lam=0.1, f32=rng.random() < 0.4)
    if kind == "batch":
        lo = rng.randint(9, 16)
        return dict(kind="batch", problems=rng.randint(2, 6), lo=lo, hi=rng.randint(lo + 2, 24),
                    per_col=rng.randint(5, 8), rhs=rng.randint(1, 4), itn=250)
    nx, ny, nz = _grid(rng, 8, 58 if kind in ("predict", "train") else 40)
    if kind == "conv":
        return dict(kind="conv", nx=nx, ny=ny, nz=nz, batch=rng.randint(1, max(1, min(4, 131072 // (nx * ny * nz)))),
                    relu=rng.random() < 0.5)
    if kind == "convback":
        return dict(kind="convback", nx=nx, ny=ny, nz=nz, batch=rng.randint(1, 2))
    if kind == "predict":
        return dict(kind="predict", nx=nx, ny=ny, nz=nz, count=rng.randint(1, 5), max_batch=4)
    return dict(kind="train", nx=nx, ny=ny, nz=nz, batch=rng.randint(1, 4), samples=rng.randint(4, 9), steps=2)


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _system(case, seed):
    P = _pkg()
    geo = P.GEOM_TOP_SOURCES if case["top"] else P.GEOM_OPPOSITE_FACES
    return P.generate(case["nx"], case["ny"], case["nz"], case["rays"], geo, 1 + seed, 0.02, case["lam"])


def _batch_edges(case):
    """Cubic grids from lo to hi voxels, evenly spread."""
    return [int(round(e)) for e in np.linspace(case["lo"], case["hi"], case["problems"])]


def _batch_inputs(case, seed):
    P = _pkg()
    specs = []
    for p, e in enumerate(_batch_edges(case)):
        own = (1 + seed % 1000003) * 64 + p
        specs.append(dict(grid=(e, e, e), n_rays=case["per_col"] * e ** 3, geometry=P.GEOM_OPPOSITE_FACES, seed=own,
                          lam=0.1, rhs=[(own * 16 + k + 1, 0.01 + 0.01 * k) for k in range(case["rhs"])]))
    return P.generate_batch(specs=specs)


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _fields(case, seed, count):
    """Network inputs and targets, (count, V) float64 on the host: a few Gaussian
    blobs each, the input with the noise of a one-step estimate from data."""
    g = _gen(seed)
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    opt = dict(device="cuda", dtype=torch.float64)
    X, Y, Z = torch.arange(nx, **opt), torch.arange(ny, **opt), torch.arange(nz, **opt)
    ins, outs = [], []
    for _ in range(count):
        f = torch.zeros(nz, ny, nx, **opt)
        for _ in range(5):
            c = torch.rand(4, generator=g, **opt)
            bump = (torch.exp(-(Z - c[2] * nz) ** 2 / 18)[:, None, None] * torch.exp(-(Y - c[1] * ny) ** 2 / 18)[:, None]
                    * torch.exp(-(X - c[0] * nx) ** 2 / 18))
            f += (2 * c[3] - 1) * bump
        noise = torch.randn(nz, ny, nx, generator=g, **opt)
        outs.append(f.reshape(-1))
        ins.append((0.6 * f + 0.05 * noise).reshape(-1))
    return torch.stack(ins).cpu().numpy(), torch.stack(outs).cpu().numpy()


def _layer(case, seed):
    g = _gen(seed)
    V = case["nx"] * case["ny"] * case["nz"]
    x = torch.relu(torch.randn(case["batch"], V, CH, generator=g, device="cuda"))  # activations after a ReLU
    w = torch.randn(TAPS, CH, CH, generator=g, device="cuda") * math.sqrt(2.0 / (TAPS * CH))
    extra = torch.randn(CH, generator=g, device="cuda") * 0.1 if case["kind"] == "conv" else \
        torch.randn(case["batch"], V, CH, generator=g, device="cuda") / (case["batch"] * V)
    return x, w, extra


def prepare(case, seed):
    P = _pkg()
    kind = case["kind"]
    st = dict(case=case)
    if kind in ("lsqr", "exact"):
        s = _system(case, seed)
        st["op"] = P.Operator(s, P.OP_EXACT_ORDER if kind == "exact" else P.OP_DEFAULT)
        st["b"] = torch.from_numpy(s.b.copy()).cuda()
        st["x"] = torch.empty(s.n, dtype=torch.float64, device="cuda")
    elif kind == "aprod":
        s = _system(case, seed)
        st["op"] = P.Operator(s)
        t = torch.float32 if case["f32"] else torch.float64
        x0, y0 = _vectors(case, seed, s.n, s.m_k + s.m_d)
        st["x0"], st["y0"] = x0.to(t), y0.to(t)
        st["x"], st["y"] = torch.empty_like(st["x0"]), torch.empty_like(st["y0"])
        st["stream"] = torch.cuda.ExternalStream(st["op"].lib.plsqr_op_get_stream(st["op"].h))
    elif kind == "batch":
        systems, B, _ = _batch_inputs(case, seed)
        st["bt"] = P.Batch(systems, case["rhs"], flags=P.BATCH_NO_TUNE)
        st["b"] = torch.from_numpy(st["bt"].pack_b(B)).cuda()
        st["x"] = torch.empty(sum(s.n for s in systems) * case["rhs"], dtype=torch.float64, device="cuda")
    elif kind == "conv":
        st["in"], st["w"], st["bias"] = _layer(case, seed)
        st["out"] = torch.empty_like(st["in"])
        st["lib"] = P.load()
    elif kind == "convback":
        st["in"], st["w"], st["dout"] = (t.cpu().numpy() for t in _layer(case, seed))
        st["P"] = P
    else:
        grid = (case["nx"], case["ny"], case["nz"])
        st["net"] = P.WarmStartNet(grid, max_batch=case.get("max_batch", case.get("batch")), seed=3)
        if kind == "predict":
            st["net"].set_params(np.load(WEIGHTS))
            st["in"] = _fields(case, seed, case["count"])[0]
        else:
            st["net"].set_data(*_fields(case, seed, case["samples"]))
    return st


def _vectors(case, seed, n, m):
    """x0 (n) and y0 (m) in FP64, the values FP32 holds exactly when the case is FP32."""
    g = _gen(seed)
    x0 = torch.randn(n, generator=g, device="cuda", dtype=torch.float64) / math.sqrt(n)
    y0 = torch.randn(m, generator=g, device="cuda", dtype=torch.float64) / math.sqrt(m)
    return (x0.float().double(), y0.float().double()) if case["f32"] else (x0, y0)


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------
def _ptr(t):
    return ctypes.c_void_p(t.data_ptr())


def run(state):
    P = _pkg()
    case = state["case"]
    kind = case["kind"]
    if kind in ("lsqr", "exact"):
        opts = {}
        if case["mixed"]:
            opts = dict(tol=1e-9, precision=P.PREC_MIXED, precond=P.PRECOND_COLSCALE, precond_power=1.5,
                        refine_adaptive=True)
        state["op"].lsqr_device(state["b"].data_ptr(), state["x"].data_ptr(), case["itn"], **opts)
        return state["x"]
    if kind == "aprod":
        op, x, y = state["op"], state["x"], state["y"]
        call = op.aprod_device_f32 if case["f32"] else op.aprod_device
        with torch.cuda.stream(state["stream"]):
            y.copy_(state["y0"])
            call(1, state["x0"].data_ptr(), y.data_ptr())
            x.copy_(state["x0"])
            call(2, x.data_ptr(), state["y0"].data_ptr())
        return dict(y=y, x=x)
    if kind == "batch":
        state["bt"].solve_device(state["b"].data_ptr(), state["x"].data_ptr(), case["itn"])
        return state["x"]
    if kind == "conv":
        rc = state["lib"].plsqr_cnn_conv_forward_noalloc(
            case["nx"], case["ny"], case["nz"], case["batch"], _ptr(state["in"]), _ptr(state["w"]),
            _ptr(state["bias"]), int(case["relu"]), _ptr(state["out"]),
            ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
        if rc:
            raise RuntimeError(state["lib"].plsqr_cnn_last_error(None))
        return state["out"]
    if kind == "convback":
        din, dw, db = P.conv_backward((case["nx"], case["ny"], case["nz"]), state["in"], state["w"], state["dout"])
        return dict(din=din, dw=dw, db=db)
    if kind == "predict":
        return state["net"].predict(state["in"])
    loss = state["net"].train(case["steps"], case["batch"], lr=2e-3, seed=5)
    return dict(loss=loss, params=state["net"].get_params())


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------
def _sizes(case):
    """Rows, columns and nonzeros of a case's system: mean chords of straight rays."""
    nx, ny, nz, rays = case["nx"], case["ny"], case["nz"], case["rays"]
    n = nx * ny * nz
    nnz = rays * (nx + ny + nz) * (0.467 if case["top"] else 0.556)
    xs, ys, zs = max(nx - 2, 0) * ny * nz, nx * max(ny - 2, 0) * nz, nx * ny * max(nz - 2, 0)
    return n, rays, n + xs + ys + zs, nnz, n + 3.0 * (xs + ys + zs)


def _aprod_work(n, mk, md, nk, nd, value, vector):
    """Bytes of mode 1 and of mode 2 (each stored value, index, pointer and vector
    element once, updated vectors read and written) and the flops of both."""
    b1 = (nk + nd) * (value + 4) + 4 * (mk + md) + vector * n + 2 * vector * (mk + md)
    b2 = (nk + nd) * (value + 4) + 8 * n + vector * (mk + md) + 2 * vector * n
    return b1, b2, 4 * (nk + nd)


def work(case):
    kind = case["kind"]
    if kind in ("lsqr", "exact"):
        n, mk, md, nk, nd = _sizes(case)
        value = 4 if case["mixed"] else 8
        b1, b2, fl = _aprod_work(n, mk, md, nk, nd, value, value)
        its = 180 if case["mixed"] else case["itn"]  # the mixed solve stops on its own test
        return dict(bytes=its * (b1 + b2 + 5 * 8 * n), flops=its * (fl + 6 * n + 4 * (mk + md)))
    if kind == "aprod":
        value = 4 if case["f32"] else 8
        b1, b2, fl = _aprod_work(*_sizes(case), value, value)
        return dict(bytes=b1 + b2, flops=fl)
    if kind == "batch":
        total = dict(bytes=0.0, flops=0.0)
        for e in _batch_edges(case):
            n, mk, md, nk, nd = _sizes(dict(nx=e, ny=e, nz=e, rays=case["per_col"] * e ** 3, top=False))
            K = case["rhs"]  # the matrix once for all right-hand sides
            total["bytes"] += case["itn"] * (2 * 12 * (nk + nd) + K * 8 * (8 * n + 3 * (mk + md)))
            total["flops"] += case["itn"] * K * (4 * (nk + nd) + 6 * n + 4 * (mk + md))
        return total
    V = case["nx"] * case["ny"] * case["nz"]
    layer = 2.0 * V * TAPS * CH * CH  # flops of one full layer and one sample
    net = 2.0 * V * TAPS * (CH + 2 * CH * CH + CH)  # the network's first layer has one input, its last one output
    if kind == "conv":
        return dict(bytes=case["batch"] * V * CH * 8 + 4 * LAYER, flops=case["batch"] * layer)
    if kind == "convback":
        return dict(bytes=case["batch"] * V * CH * 12 + 8 * LAYER, flops=2 * case["batch"] * layer)
    if kind == "predict":
        return dict(bytes=case["count"] * V * 16 + 4 * LAYERS * LAYER, flops=case["count"] * net)
    per = case["batch"] * V  # activations of three layers (bf16) written, read forward and twice backward
    return dict(bytes=case["steps"] * (per * (8 + 3 * CH * 2 * 4 + 3 * CH * 2 * 3) + 4 * 28 * LAYERS * LAYER),
                flops=case["steps"] * 3 * case["batch"] * net)


# ---------------------------------------------------------------------------
# the same results in 64 bits, in plain torch
# ---------------------------------------------------------------------------
class _Matrix:
    """[A_k; D] and its transpose as CSR on the GPU, for vectors or (length, K) arrays."""

    def __init__(self, s):
        def cu(a):
            return torch.from_numpy(np.array(a)).cuda()
        kc = torch.repeat_interleave(torch.arange(s.n, device="cuda"), cu(np.diff(s.k_col_ptr)).long())
        dr = torch.repeat_interleave(torch.arange(s.m_d, device="cuda"), cu(np.diff(s.d_row_ptr)).long()) + s.m_k
        r = torch.cat([cu(s.k_row_idx).long(), dr])
        c = torch.cat([kc, cu(s.d_col_idx).long()])
        v = torch.cat([cu(s.k_val), cu(s.d_val)])
        self.m, self.n = s.m_k + s.m_d, s.n
        self.a = self._csr(r, c, v, self.m, self.n)
        self.at = self._csr(c, r, v, self.n, self.m)

    @staticmethod
    def _csr(r, c, v, m, n):
        order = torch.argsort(r * n + c)
        ptr = torch.zeros(m + 1, dtype=torch.int64, device="cuda")
        ptr[1:] = torch.cumsum(torch.bincount(r, minlength=m), 0)
        return torch.sparse_csr_tensor(ptr, c[order], v[order], size=(m, n))

    def mul(self, x):
        return (self.a @ x.reshape(self.n, -1)).reshape((self.m,) + x.shape[1:])

    def tmul(self, y):
        return (self.at @ y.reshape(self.m, -1)).reshape((self.n,) + y.shape[1:])


def _lsqr(A, b, itn):
    """Paige and Saunders' LSQR from zero, itn iterations, for every column of b (m, K)."""
    beta = b.norm(dim=0)
    u = b / beta
    v = A.tmul(u)
    alpha = v.norm(dim=0)
    v = v / alpha
    w, x = v.clone(), torch.zeros_like(v)
    phibar, rhobar = beta, alpha
    for _ in range(itn):
        u = A.mul(v) - alpha * u
        beta = u.norm(dim=0)
        u = u / beta
        v = A.tmul(u) - beta * v
        alpha = v.norm(dim=0)
        v = v / alpha
        rho = torch.hypot(rhobar, beta)
        c, s = rhobar / rho, beta / rho
        theta, rhobar = s * alpha, -c * alpha
        phi, phibar = c * phibar, s * phibar
        x = x + (phi / rho) * w
        w = v - (theta / rho) * w
    return x


def _solution(s, b, itn, to_convergence):
    """x (n, K) for b (m_k, K): after itn iterations, or at the least-squares solution."""
    A = _Matrix(s)
    b = torch.cat([b, torch.zeros(s.m_d, b.shape[1], dtype=torch.float64, device="cuda")])
    if not to_convergence:
        return _lsqr(A, b, itn)
    x = _lsqr(A, b, 350)
    return x + _lsqr(A, b - A.mul(x), 150)


def _taps(case):
    """(offset slices) of the 27 taps on a zero-padded (B, nz, ny, nx, C) tensor."""
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    for t in range(TAPS):
        dz, dy, dx = t // 9, t // 3 % 3, t % 3
        yield t, (slice(None), slice(dz, dz + nz), slice(dy, dy + ny), slice(dx, dx + nx))


def _conv64(case, x, w, b=None):
    """x (B, V, C) float64, w (27, N, C): the layer's sums, (B, V, N)."""
    B = x.shape[0]
    g = torch.nn.functional.pad(x.reshape(B, case["nz"], case["ny"], case["nx"], -1), (0, 0, 1, 1, 1, 1, 1, 1))
    out = torch.zeros(x.shape[0] * x.shape[1], w.shape[1], dtype=torch.float64, device=x.device)
    for t, at in _taps(case):
        out = out + g[at].reshape(-1, x.shape[2]) @ w[t].T
    return (out if b is None else out + b).reshape(B, x.shape[1], -1)


def _bf(t):
    return t.bfloat16().double()


def _net64(case, params, x):
    """The network without rounding: x (B, V) -> (B, V), in units of the gain."""
    h = x[:, :, None]
    for l in range(LAYERS):
        q = params[l * LAYER:(l + 1) * LAYER]
        w, b = q[:TAPS * CH * CH].reshape(TAPS, CH, CH), q[TAPS * CH * CH:]
        if l == 0:
            w = w[:, :, :1]
        if l == LAYERS - 1:
            w, b = w[:, :1], b[:1]
        h = _conv64(case, h, w, b)
        if l < LAYERS - 1:
            h = torch.relu(h)
    return h[:, :, 0]


def _exact_predict(case, seed):
    x = torch.from_numpy(_fields(case, seed, case["count"])[0]).cuda()
    p = torch.from_numpy(np.load(WEIGHTS)).cuda().double()
    s = x.square().mean(1, keepdim=True).sqrt()
    return torch.cat([s[i:i + 1] * p[-1] * _net64(case, p, x[i:i + 1] / s[i:i + 1]) for i in range(len(x))])


def exact(case, seed):
    kind = case["kind"]
    if kind in ("lsqr", "exact"):
        s = _system(case, seed)
        b = torch.from_numpy(s.b.copy()).cuda()[:, None]
        return _solution(s, b, case["itn"], kind == "lsqr" and case["itn"] > 20)[:, 0]
    if kind == "aprod":
        s = _system(case, seed)
        A = _Matrix(s)
        x0, y0 = _vectors(case, seed, s.n, A.m)
        return dict(y=y0 + A.mul(x0), x=x0 + A.tmul(y0))
    if kind == "batch":
        systems, B, _ = _batch_inputs(case, seed)
        return torch.cat([_solution(s, torch.from_numpy(np.array(b)).cuda().T.contiguous(), 0, True).T.reshape(-1)
                          for s, b in zip(systems, B)])
    if kind == "conv":  # the entry point's operands are bf16, its sums are not
        x, w, b = _layer(case, seed)
        out = _conv64(case, _bf(x), _bf(w), b.double())
        return torch.relu(out) if case["relu"] else out
    if kind == "convback":
        x, w, d = _layer(case, seed)
        x, w, d = _bf(x), _bf(w), _bf(d)
        din = _conv64(case, d, w.flip(0).transpose(1, 2))
        grid = (x.shape[0], case["nz"], case["ny"], case["nx"], CH)
        g = torch.nn.functional.pad(x.reshape(grid), (0, 0, 1, 1, 1, 1, 1, 1))
        dw = torch.stack([d.reshape(-1, CH).T @ g[at].reshape(-1, CH) for _, at in _taps(case)])
        return dict(din=din, dw=dw, db=d.sum((0, 1)))
    if kind == "predict":
        return _exact_predict(case, seed)
    return None  # a training step's bf16 activations have no counterpart in 64 bits
