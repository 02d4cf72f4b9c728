"""The workloads this framework's performance is judged on.

Each case is one thing a program does with the framework through its public entry points: an
escape-time image, a fused elementwise chain, row and column reductions, a training step and
inference of bf16 MLPs, inference of int8 MLPs, per-pixel programs and a vertex transform.
`listed()` names twelve of them; `draw(rng)` gives more of the same kinds with sizes spread over
their whole ranges (ragged ones among them).  A case is a dict whose "kind" selects the functions
below; `prepare` makes the inputs from the seed on the GPU, with the plan a program keeps (compiled
chains and programs, a captured step with its packed weights), and `run` makes one pass, returning
the framework's own device buffers as torch tensors without a copy.
"""
from __future__ import annotations

import math

import torch

from vernondsl_amd import graph as vgraph
from vernondsl_amd import kernels, spec
from vernondsl_amd import mapchain as mc
from vernondsl_amd import pixprog as pp
from vernondsl_amd.rhi import Device, Queue, Tensor

_TYPESTR = {"f32": "<f4", "bf16": "<i2", "i8": "|i1", "i32": "<i4"}
_NAMES = {0: "f32", 1: "bf16", 2: "i8", 3: "i32"}


# ---- the device, and its buffers as torch tensors ------------------------------------------------
class _Context:
    """The device and the queue every case runs on, opened at first use."""
    dev = None
    queue = None


def _open():
    if _Context.dev is None:
        torch.cuda.init()
        _Context.dev = Device(0)
        _Context.queue = Queue(_Context.dev)
    return _Context.dev, _Context.queue


class _Exported:
    """A framework tensor in the form torch takes device memory in; keeps the tensor alive."""

    def __init__(self, t: Tensor):
        self.tensor = t
        self.__cuda_array_interface__ = {"shape": t.shape, "typestr": _TYPESTR[_NAMES[t.dtype]], "version": 2,
                                         "data": (t.buffer.address(), False), "strides": None}


def _torch(t: Tensor) -> torch.Tensor:
    """The same memory as a torch tensor (bf16 is held as 16-bit words by the framework)."""
    x = torch.as_tensor(_Exported(t), device="cuda")
    return x.view(torch.bfloat16) if _NAMES[t.dtype] == "bf16" else x


def _put(values: torch.Tensor, dtype: str) -> Tensor:
    """A framework tensor holding `values`."""
    dev, _ = _open()
    t = Tensor(dev, tuple(values.shape), dtype)
    _torch(t).copy_(values)
    return t


def _empty(shape, dtype: str) -> Tensor:
    return Tensor(_open()[0], shape, dtype)


def _generator(seed: int) -> torch.Generator:
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _normal(g, shape, sigma=1.0):
    return torch.randn(shape, generator=g, device="cuda") * sigma


def _uniform(g, shape, lo, hi):
    return torch.rand(shape, generator=g, device="cuda") * (hi - lo) + lo


# ---- escape-time images --------------------------------------------------------------------------
def _escape_params(c, seed):
    r = torch.Generator().manual_seed(int(seed))
    u, v = (float(x) for x in torch.rand(2, generator=r))
    if c["family"] == "julia":  # fractal.py's frame at some time of its animation
        p = spec.julia_paint_params(6.0 * u, c["nj"])
        p.update(ni=c["ni"], max_iter=c["max_iter"], out_scale=-1.0 / c["max_iter"])
        return p
    p = spec.mandelbrot_params(1024, c["max_iter"])
    p.update(ni=c["ni"], nj=c["nj"], re_den=float(c["ni"]), im_den=float(c["nj"]),
             re_post=-2.0 + 0.1 * (u - 0.5), im_post=-1.5 + 0.1 * (v - 0.5))
    return p


def _prepare_escape(c, seed):
    _, q = _open()
    p = kernels.escape_time_params(**_escape_params(c, seed))
    out = _empty((c["ni"], c["nj"]), "f32" if c["family"] == "julia" else "i32")
    return {"q": q, "p": p, "out": out, "result": _torch(out)}


def _run_escape(s):
    kernels.escape_time(s["q"], s["p"], s["out"])
    return s["result"]


def _work_escape(c):
    # 8 operations per pixel and iteration; the mean count over these windows is about 0.19 of the
    # limit for the Mandelbrot set and about 0.4 of it for the Julia frames.
    n = c["ni"] * c["nj"]
    return {"bytes": 4 * n, "flops": 8 * n * c["max_iter"] * (0.4 if c["family"] == "julia" else 0.19)}


# ---- elementwise chains --------------------------------------------------------------------------
def _chain(name):
    if name == "tanh":  # tanh(a x + b) * exp(-x^2) + bias[col]
        return mc.compile(spec.map_chain_expr())
    return mc.compile(mc.sigmoid(mc.Input(0)) * mc.Input(1, "col") + mc.Input(0) * mc.Input(0))


def _chain_inputs(c, seed):
    g = _generator(seed)
    x = _normal(g, (c["rows"], c["cols"]))
    return x, _uniform(g, (c["cols"] if c["chain"] == "tanh" else c["rows"],), -1.0, 1.0)


def _prepare_map(c, seed):
    _, q = _open()
    x, v = _chain_inputs(c, seed)
    out = _empty((c["rows"], c["cols"]), "f32")
    return {"q": q, "prog": _chain(c["chain"]), "ins": [_put(x, "f32"), _put(v, "f32")], "out": out, "result": _torch(out)}


def _run_map(s):
    kernels.map_chain(s["q"], s["prog"], s["ins"], s["out"])
    return s["result"]


def _work_map(c):
    n, side = c["rows"] * c["cols"], c["cols"] if c["chain"] == "tanh" else c["rows"]
    return {"bytes": 8 * n + 4 * side, "flops": (30 if c["chain"] == "tanh" else 16) * n}


def _exact_map(c, seed):
    x, v = (t.double() for t in _chain_inputs(c, seed))
    if c["chain"] == "tanh":
        return torch.tanh(x * spec.MAP_A + spec.MAP_B) * torch.exp(-x * x) + v
    return torch.sigmoid(x) * v[:, None] + x * x


# ---- reductions ----------------------------------------------------------------------------------
def _reduce_input(c, seed):
    """N(0, sigma 2), with a +20 outlier in 1% of the rows."""
    g = _generator(seed)
    x = _normal(g, (c["rows"], c["cols"]), 2.0)
    n = max(1, c["rows"] // 100)
    rows = torch.randint(c["rows"], (n,), generator=g, device="cuda")
    cols = torch.randint(c["cols"], (n,), generator=g, device="cuda")
    x[rows, cols] += 20.0
    return x.to(torch.bfloat16) if c["dtype"] == "bf16" else x


def _prepare_softmax(c, seed):
    _, q = _open()
    x = _put(_reduce_input(c, seed), c["dtype"])
    out = [_empty((c["rows"],), "f32"), _empty((c["rows"],), "f32"), _empty((c["rows"], c["cols"]), c["dtype"])]
    return {"q": q, "x": x, "out": out, "result": [_torch(t) for t in out]}


def _run_softmax(s):
    row_sum, row_max, softmax = s["out"]
    kernels.row_reduce_softmax(s["q"], s["x"], row_sum, row_max, softmax)
    return s["result"]


def _work_softmax(c):
    n, size = c["rows"] * c["cols"], 2 if c["dtype"] == "bf16" else 4
    return {"bytes": 2 * size * n + 8 * c["rows"], "flops": 8 * n}


def _exact_softmax(c, seed):
    x = _reduce_input(c, seed).double()
    return [x.sum(1), x.amax(1), torch.softmax(x, 1)]


def _prepare_columns(c, seed):
    _, q = _open()
    x = _put(_reduce_input(c, seed), c["dtype"])
    out = [_empty((c["cols"],), "f32"), _empty((c["cols"],), "f32")]
    return {"q": q, "x": x, "out": out, "result": [_torch(t) for t in out]}


def _run_columns(s):
    kernels.col_reduce(s["q"], s["x"], s["out"][0], s["out"][1])
    return s["result"]


def _work_columns(c):
    n, size = c["rows"] * c["cols"], 2 if c["dtype"] == "bf16" else 4
    return {"bytes": size * n + 8 * c["cols"], "flops": 2 * n}


def _exact_columns(c, seed):
    x = _reduce_input(c, seed).double()
    return [x.sum(0), x.amax(0)]


# ---- bf16 MLPs -----------------------------------------------------------------------------------
def _weight(g, n_out, n_in):
    b = math.sqrt(6.0 / (n_in + n_out))
    return _uniform(g, (n_out, n_in), -b, b).to(torch.bfloat16)


def _train_inputs(c, seed):
    g = _generator(seed)
    x = _normal(g, (c["batch"], c["d_in"])).to(torch.bfloat16)
    return (x, _weight(g, c["hidden"], c["d_in"]), _weight(g, c["d_out"], c["hidden"]),
            _normal(g, (c["batch"], c["d_out"])))


def _compiled(graph, values):
    """The graph's executable with its inputs and weights in place, captured as a step."""
    dev, q = _open()
    exe = graph.compile(dev)
    for name, v in values.items():
        _torch(exe.t[name]).copy_(v)
    torch.cuda.synchronize()
    return {"q": q, "exe": exe, "step": exe.capture(q)}


def _run_step(s):
    s["step"].launch(s["q"])
    return s["result"]


def _prepare_train(c, seed):
    graph, grads = vgraph.mlp_train_graph(c["batch"], c["d_in"], c["hidden"], c["d_out"])
    s = _compiled(graph, dict(zip(("X", "W1", "W2", "T"), _train_inputs(c, seed))))
    names = ["loss", "Y", grads["W1"].name, grads["W2"].name]
    s["result"] = [_torch(s["exe"].t[n]) for n in names]
    return s


def _work_train(c):
    b, i, h, o = c["batch"], c["d_in"], c["hidden"], c["d_out"]
    return {"bytes": 2 * b * i + 2 * h * (i + o) + 8 * b * o + 4 * h * (i + o) + 4, "flops": spec.mlp_flops(b, i, h, o)}


def _gelu(x):
    return 0.5 * x * torch.erfc(-x / math.sqrt(2.0))


def _exact_train(c, seed):
    x, w1, w2, t = (v.double() for v in _train_inputs(c, seed))
    pre = x @ w1.t()
    h = _gelu(pre)
    y = h @ w2.t()
    d = y - t
    dy = d * (2.0 / d.numel())
    slope = 0.5 * torch.erfc(-pre / math.sqrt(2.0)) + pre * torch.exp(-0.5 * pre * pre) / math.sqrt(2.0 * math.pi)
    da = (dy @ w2) * slope
    return [(d * d).mean().reshape(1), y, da.t().contiguous() @ x, dy.t().contiguous() @ h]


def _infer_widths(c):
    return [c["d_in"]] + [c["hidden"]] * (c["layers"] - 1) + [c["d_out"]]


def _infer_inputs(c, seed):
    g = _generator(seed)
    x = _normal(g, (c["batch"], c["d_in"])).to(torch.bfloat16)
    w = _infer_widths(c)
    return x, [_weight(g, w[k + 1], w[k]) for k in range(c["layers"])]


def _prepare_infer(c, seed):
    x, ws = _infer_inputs(c, seed)
    graph = vgraph.Graph(pack_weights=True)
    h, values = graph.input("X", tuple(x.shape), "bf16"), {"X": x}
    for k, w in enumerate(ws):
        last = k == len(ws) - 1
        p = graph.param(f"W{k}", tuple(w.shape), "bf16", requires_grad=False)
        h = graph.linear(h, p, act="none" if last else "gelu", out_dtype="f32" if last else None,
                         name="Y" if last else f"H{k}")
        values[f"W{k}"] = w
    s = _compiled(graph, values)
    s["result"] = [_torch(s["exe"].t[f"H{k}"]) for k in range(len(ws) - 1)] + [_torch(s["exe"].t["Y"])]
    return s


def _work_infer(c):
    w = _infer_widths(c)
    mn = sum(w[k] * w[k + 1] for k in range(c["layers"]))
    return {"bytes": 2 * mn + 2 * c["batch"] * w[0] + c["batch"] * (2 * sum(w[1:-1]) + 4 * w[-1]), "flops": 2 * c["batch"] * mn}


def _exact_infer(c, seed):
    x, ws = _infer_inputs(c, seed)
    h, out = x.double(), []
    for k, w in enumerate(ws):
        h = h @ w.double().t()
        h = h if k == len(ws) - 1 else _gelu(h)
        out.append(h)
    return out


# ---- int8 MLPs -----------------------------------------------------------------------------------
def _int8_widths(c):
    return [c["width"]] * c["layers"] + [c["d_out"]]


def _int8_inputs(c, seed):
    g = _generator(seed)
    x = _normal(g, (c["batch"], c["width"])).to(torch.bfloat16)
    w = _int8_widths(c)
    layers = []
    for k in range(c["layers"]):
        q = torch.randint(-127, 128, (w[k + 1], w[k]), generator=g, device="cuda", dtype=torch.int8)
        layers.append((q, _uniform(g, (w[k + 1],), 0.005, 0.02)))
    return x, layers


def _prepare_int8(c, seed):
    x, layers = _int8_inputs(c, seed)
    values = {"X": x}
    for k, (w, scale) in enumerate(layers):
        values[f"W{k}"], values[f"S{k}"] = w, scale
    s = _compiled(vgraph.w8a8_infer_graph(c["batch"], tuple(_int8_widths(c))), values)
    s["result"] = [_torch(s["exe"].t[n]) for n in [f"H{k}" for k in range(c["layers"] - 1)] + ["Y"]]
    return s


def _work_int8(c):
    w = _int8_widths(c)
    mn = sum(w[k] * w[k + 1] for k in range(c["layers"]))
    return {"bytes": mn + 4 * sum(w[1:]) + 2 * c["batch"] * sum(w), "flops": 2 * c["batch"] * mn}


def _exact_int8(c, seed):
    # the quantisation (f32 scale and quotient, halves to even) and the bf16 activations between
    # layers are the operation's definition; the products and the scaling are in 64 bits
    x, layers = _int8_inputs(c, seed)
    h, out = x, []
    for k, (w, scale) in enumerate(layers):
        f = h.float()
        s = f.abs().amax(1, keepdim=True) / 127.0
        q = torch.where(s > 0, torch.clamp(torch.round(f / s), -127, 127), torch.zeros_like(f)).double()
        y = (q @ w.double().t()) * s.double() * scale.double()
        y = y if k == len(layers) - 1 else torch.relu(y)
        out.append(y)
        h = y.float().to(torch.bfloat16)
    return out


# ---- per-pixel programs --------------------------------------------------------------------------
def _heat_program(ni, nj):
    """A step of explicit heat diffusion: a five-point stencil, indices clamped at the border."""
    b = pp.Builder()
    i, j = b.index(0), b.index(1)
    at = b.load_at(0, i, j)
    lap = b.load_at(0, b.op("max", b.op("add", i, -1.0), 0.0), j)
    lap = b.op("add", lap, b.load_at(0, b.op("min", b.op("add", i, 1.0), float(ni - 1)), j))
    lap = b.op("add", lap, b.load_at(0, i, b.op("max", b.op("add", j, -1.0), 0.0)))
    lap = b.op("add", lap, b.load_at(0, i, b.op("min", b.op("add", j, 1.0), float(nj - 1))))
    lap = b.op("sub", lap, b.op("mul", at, 4.0))
    return pp.compile_program(b, out=b.op("add", at, b.op("mul", lap, 0.2)))


def _heat_input(c, seed):
    return _uniform(_generator(seed), (c["ni"], c["nj"]), 0.0, 1.0)


def _prepare_heat(c, seed):
    _, q = _open()
    u, v = _put(_heat_input(c, seed), "f32"), _empty((c["ni"], c["nj"]), "f32")
    return {"q": q, "prog": _heat_program(c["ni"], c["nj"]), "ins": [u], "out": v, "result": _torch(v)}


def _run_heat(s):
    kernels.pixel_program(s["q"], s["prog"], s["ins"], s["out"])
    return s["result"]


def _work_heat(c):
    n = c["ni"] * c["nj"]
    return {"bytes": 8 * n, "flops": 7 * n}


def _exact_heat(c, seed):
    u = _heat_input(c, seed).double()
    up, down = torch.cat([u[:1], u[:-1]]), torch.cat([u[1:], u[-1:]])
    left, right = torch.cat([u[:, :1], u[:, :-1]], 1), torch.cat([u[:, 1:], u[:, -1:]], 1)
    k = float(torch.tensor(0.2, dtype=torch.float32))
    return u + k * (up + down + left + right - 4.0 * u)


def _histogram_program(bins):
    """Adds 1 to the bin of each pixel's value in [0, 1)."""
    b = pp.Builder()
    at = b.op("floor", b.op("mul", b.load(0), float(bins)))
    return pp.compile_program(b, out=None, effects=[b.scatter_add(1, 0.0, at, 1.0)], in_dtypes=[pp.F32, pp.I32],
                              in_extents=[None, (1, bins)])


def _histogram_input(c, seed):
    # a smooth distribution of values, heavier at the low end, all below 1
    x = torch.rand((c["ni"], c["nj"]), generator=_generator(seed), device="cuda")
    return (x * (0.25 + 0.75 * x)).clamp(max=0.999)


def _prepare_histogram(c, seed):
    _, q = _open()
    x, h = _put(_histogram_input(c, seed), "f32"), _empty((1, c["bins"]), "i32")
    return {"q": q, "prog": _histogram_program(c["bins"]), "x": x, "hist": h, "grid": (c["ni"], c["nj"]), "result": _torch(h)}


def _run_histogram(s):
    s["hist"].buffer.fill_u32(s["q"], 0)
    kernels.pixel_program(s["q"], s["prog"], [s["x"], s["hist"]], None, grid=s["grid"])
    return s["result"]


def _work_histogram(c):
    n = c["ni"] * c["nj"]
    return {"bytes": 4 * n + 4 * c["bins"], "flops": 3 * n}


# ---- vertex transform ----------------------------------------------------------------------------
def _vertex_inputs(c, seed):
    g = _generator(seed)
    return _normal(g, (c["n"], 3)), _normal(g, (3, 4, 4))


def _prepare_vertices(c, seed):
    _, q = _open()
    pos, mats = (_put(v, "f32") for v in _vertex_inputs(c, seed))
    out, varying = _empty((c["n"], 4), "f32"), _empty((c["n"], 3), "f32")
    return {"q": q, "pos": pos, "mats": mats, "out": out, "varying": varying, "result": [_torch(out), _torch(varying)]}


def _run_vertices(s):
    kernels.vec_transform(s["q"], s["pos"], s["mats"], s["out"], s["varying"])
    return s["result"]


def _work_vertices(c):
    return {"bytes": 40 * c["n"] + 192, "flops": 96 * c["n"]}


def _exact_vertices(c, seed):
    pos, mats = _vertex_inputs(c, seed)
    v = torch.cat([pos, torch.ones_like(pos[:, :1])], 1).double()
    for m in mats.double():
        v = v @ m.t()
    return [v, pos.double()]


# ---- the kinds -----------------------------------------------------------------------------------
# kind: (prepare, run, work, exact or None, tolerance or None for bit equality).  The tolerances are
# what another summation order, or another correctly working evaluation of exp, tanh and erfc in f32,
# moves the outputs by: f32 results 1e-6; bf16 results, and f32 results of sums over bf16 activations,
# by the activations that then round the other way.
_KINDS = {
    "escape": (_prepare_escape, _run_escape, _work_escape, None, None),
    "map": (_prepare_map, _run_map, _work_map, _exact_map, {"rel": 1e-6, "max": 4e-6}),
    "softmax": (_prepare_softmax, _run_softmax, _work_softmax, _exact_softmax, {"rel": 1e-6, "max": 4e-6}),
    "columns": (_prepare_columns, _run_columns, _work_columns, _exact_columns, {"rel": 1e-6, "max": 4e-6}),
    "train": (_prepare_train, _run_step, _work_train, _exact_train, {"rel": 2e-3, "max": 5e-2}),
    "infer": (_prepare_infer, _run_step, _work_infer, _exact_infer, {"rel": 2e-3, "max": 5e-2}),
    "int8": (_prepare_int8, _run_step, _work_int8, _exact_int8, None),
    "heat": (_prepare_heat, _run_heat, _work_heat, _exact_heat, None),
    "histogram": (_prepare_histogram, _run_histogram, _work_histogram, None, None),
    "vertices": (_prepare_vertices, _run_vertices, _work_vertices, _exact_vertices, None),
}


def listed():
    return [
        # one frame of fractal.py's animation, the program the framework exists to run: the smallest
        # call, where launching counts
        {"name": "frame_640x320", "kind": "escape", "family": "julia", "ni": 640, "nj": 320, "max_iter": 50},
        # the Mandelbrot image of the benchmark
        {"name": "mandelbrot_1024", "kind": "escape", "family": "mandelbrot", "ni": 1024, "nj": 1024, "max_iter": 256},
        # the benchmark's fused elementwise chain at full size
        {"name": "map_8192", "kind": "map", "chain": "tanh", "rows": 8192, "cols": 8192},
        # a softmax over a width that is no power of two (a vocabulary, a class count)
        {"name": "softmax_f32_3000x5003", "kind": "softmax", "rows": 3000, "cols": 5003, "dtype": "f32"},
        # the benchmark's softmax in bf16
        {"name": "softmax_bf16_16384x4096", "kind": "softmax", "rows": 16384, "cols": 4096, "dtype": "bf16"},
        # column statistics of the same tensor in f32 (per-feature sums and maxima, bias gradients)
        {"name": "columns_16384x4096", "kind": "columns", "rows": 16384, "cols": 4096, "dtype": "f32"},
        # the benchmark's training step: forward, loss and backward of a two-layer MLP
        {"name": "train_2048x4096", "kind": "train", "batch": 2048, "d_in": 4096, "hidden": 4096, "d_out": 4096},
        # a small classifier's training step with a batch that is no multiple of a tile
        {"name": "train_300x784", "kind": "train", "batch": 300, "d_in": 784, "hidden": 1000, "d_out": 10},
        # serving a bf16 MLP to a few requests at a time: bound by reading the weights
        {"name": "infer_8x4096", "kind": "infer", "batch": 8, "layers": 4, "d_in": 4096, "hidden": 4096, "d_out": 4096},
        # the benchmark's int8 MLP at its batch
        {"name": "int8_512x8192", "kind": "int8", "batch": 512, "layers": 4, "width": 8192, "d_out": 1024},
        # the same model serving a few requests at a time
        {"name": "int8_8x8192", "kind": "int8", "batch": 8, "layers": 4, "width": 8192, "d_out": 1024},
        # a heat-diffusion step over a large plate by a general per-pixel program
        {"name": "heat_8192", "kind": "heat", "ni": 8192, "nj": 8192},
    ]


def _spread(rng, lo, hi):
    """An integer in [lo, hi], spread evenly over its logarithm."""
    return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def _extent(rng, lo, hi, grains):
    """Such an integer, made a multiple of one of `grains`."""
    g = rng.choice(grains)
    return max(g, _spread(rng, lo, hi) // g * g)


def draw(rng):
    kind = rng.choice(sorted(_KINDS))
    if kind == "escape":
        if rng.random() < 0.5:
            n = _spread(rng, 60, 720)
            return {"kind": kind, "family": "julia", "ni": 2 * n, "nj": n, "max_iter": _spread(rng, 40, 200)}
        return {"kind": kind, "family": "mandelbrot", "ni": _spread(rng, 100, 1536), "nj": _spread(rng, 100, 1536),
                "max_iter": _spread(rng, 50, 512)}
    if kind == "map":
        return {"kind": kind, "chain": rng.choice(["tanh", "sigmoid"]), "rows": _spread(rng, 1, 8192),
                "cols": _extent(rng, 4, 8192, (1, 4, 64))}
    if kind in ("softmax", "columns"):
        cols = _extent(rng, 3, 16384, (1, 1, 8, 256))
        return {"kind": kind, "rows": _spread(rng, 1, min(16384, (1 << 26) // cols)), "cols": cols,
                "dtype": rng.choice(["f32", "bf16"])}
    if kind == "train":
        grains = (1, 8, 64, 256)
        return {"kind": kind, "batch": _extent(rng, 16, 2048, (1, 8, 128)), "d_in": _extent(rng, 64, 4096, grains),
                "hidden": _extent(rng, 64, 4096, grains), "d_out": _extent(rng, 4, 4096, (1, 8, 256))}
    if kind == "infer":
        grains = (8, 64, 256, 256)
        return {"kind": kind, "batch": _spread(rng, 1, 512), "layers": rng.randint(2, 4), "d_in": _extent(rng, 256, 4096, grains),
                "hidden": _extent(rng, 256, 4096, grains), "d_out": _extent(rng, 16, 4096, (1, 32, 256))}
    if kind == "int8":
        return {"kind": kind, "batch": _spread(rng, 1, 512), "layers": rng.randint(1, 4),
                "width": _extent(rng, 512, 8192, (16, 64, 512, 512)), "d_out": _extent(rng, 32, 8192, (1, 32, 256))}
    if kind == "heat":
        return {"kind": kind, "ni": _spread(rng, 64, 8192), "nj": _spread(rng, 64, 8192)}
    if kind == "histogram":
        return {"kind": kind, "ni": _spread(rng, 64, 8192), "nj": _spread(rng, 64, 8192), "bins": _spread(rng, 8, 8192)}
    return {"kind": kind, "n": _spread(rng, 1000, 1 << 24)}


def prepare(case, seed):
    state = dict(_KINDS[case["kind"]][0](case, seed), run=_KINDS[case["kind"]][1])
    torch.cuda.synchronize()  # the inputs are in place before the framework's own queue reads them
    return state


def run(state):
    return state["run"](state)


def work(case):
    return _KINDS[case["kind"]][2](case)


def tolerance(case):
    t = _KINDS[case["kind"]][4]
    if t is None:
        return "exact"
    if case["kind"] == "softmax" and case["dtype"] == "bf16":
        return {"rel": 1e-4, "max": 1e-2}
    return dict(t)


def exact(case, seed):
    f = _KINDS[case["kind"]][3]
    return None if f is None else f(case, seed)
