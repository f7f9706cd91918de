"""Performance cases of the framework: what its users run, with the sizes they run it at.

Two kinds of entry point are driven, both as a program drives them: the engine's C API (include/nc.h through
newch_amd.abi: tensors, autograd, optimizers) for whole steps and blocks, and the kernel layer (include/nc_hip.h
through newch_amd.hip.Kernels on device buffers) for single operations.  Every state's work goes to one stream,
as one program's does.

listed() names the cases; draw() gives more of the same families over their whole ranges.  run() makes one pass
and returns whole outputs (gradients and updated weights included); exact() is the same in 64 bits by plain torch.
"""
import ctypes
import math

import torch
import torch.nn.functional as F

from newch_amd import abi, hip

DEV = "cuda"
EPS = 1e-5            # LayerNorm
LR, MOMENTUM = 0.05, 0.9
ACTS = ("gelu", "silu", "sigmoid", "tanh", "hardswish", "relu6", "relu")


def listed():
    return [
        # the MNIST-CNN bias-ReLU-pool chain of the framework's smallest configuration, with its backward
        {"name": "conv_bias_chain", "family": "chain", "n": 64, "c": 16, "h": 28, "w": 28},
        # one training step of a small image classifier at the usual batch: launches and small products
        {"name": "classifier_step", "family": "classifier", "batch": 64, "features": 784, "hidden": 128, "classes": 10},
        # a transformer's MLP block in training: norm, two linears, GELU, residual, forward and backward
        {"name": "mlp_block", "family": "mlp_block", "tokens": 2048, "d": 768, "hidden": 3072},
        # the 1000-class head of a vision model in training, both gradients and the bias gradient
        {"name": "linear_head", "family": "linear", "m": 4096, "k": 2048, "n": 1000},
        # one linear of a model that serves a few sequences at a time, a token each
        {"name": "linear_decode", "family": "decode", "m": 8, "k": 4096, "n": 4096},
        # attention over 14 x 14 patches and a class token, 8 images of 12 heads, forward and backward
        {"name": "attention", "family": "attention", "heads": 96, "s": 197, "d": 64},
        # a language model's loss over its vocabulary, whose size is odd, and the logits' gradient
        {"name": "vocabulary_loss", "family": "loss", "rows": 2048, "classes": 50257},
        # LayerNorm of a mid-sized transformer in training
        {"name": "layer_norm", "family": "rows", "op": "layer_norm", "rows": 16384, "cols": 768},
        # an activation over a large tensor, forward and backward: the headline configuration's size
        {"name": "activation", "family": "activation", "op": "gelu", "n": 1 << 28},
        # broadcast add over 2^30 outputs with both sum-to-shape gradients: the broadcast configuration's chunk
        {"name": "broadcast", "family": "broadcast", "op": "add", "form": "outer", "p": 64 * 512, "h": 512, "w": 64},
        # an int8 linear that serves a small batch
        {"name": "int8_linear", "family": "int8", "m": 16, "k": 4096, "n": 4096},
        # a wide MLP's weight quantized for inference and expanded back
        {"name": "quantize", "family": "quantize", "rows": 4096, "cols": 11008},
    ]


def _log_int(rng, lo, hi):
    """lo .. hi, spread over the logarithm; as often as not rounded down to a multiple of 16 where it is large."""
    v = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    if v >= 64 and rng.random() < 0.5:
        v -= v % 16
    return max(lo, min(hi, v))


def draw(rng):
    family = rng.choice(("chain", "classifier", "mlp_block", "linear", "decode", "attention", "loss", "rows",
                         "activation", "broadcast", "int8", "quantize"))
    L = _log_int
    while True:
        if family == "chain":
            c = {"n": L(rng, 1, 256), "c": L(rng, 1, 256), "h": L(rng, 5, 64), "w": L(rng, 5, 64)}
            ok = c["n"] * c["c"] * c["h"] * c["w"] <= 1 << 26
        elif family == "classifier":
            c = {"batch": L(rng, 4, 1024), "features": L(rng, 32, 2048), "hidden": L(rng, 32, 2048),
                 "classes": L(rng, 2, 1000)}
            ok = True
        elif family == "mlp_block":
            c = {"tokens": L(rng, 16, 4096), "d": L(rng, 64, 1024), "hidden": L(rng, 128, 4096)}
            ok = 12 * c["tokens"] * c["d"] * c["hidden"] <= 10 ** 11
        elif family == "linear":
            c = {"m": L(rng, 16, 8192), "k": L(rng, 16, 4096), "n": L(rng, 8, 4096)}
            ok = 6 * c["m"] * c["k"] * c["n"] <= 10 ** 11
        elif family == "decode":
            c = {"m": L(rng, 1, 64), "k": L(rng, 256, 8192), "n": L(rng, 256, 8192)}
            ok = True
        elif family == "attention":
            c = {"heads": L(rng, 4, 256), "s": L(rng, 16, 1024), "d": rng.choice((32, 40, 64, 80, 96, 128))}
            ok = c["heads"] * c["s"] ** 2 <= 1 << 26
        elif family == "loss":
            c = {"rows": L(rng, 16, 16384), "classes": L(rng, 10, 65536)}
            ok = c["rows"] * c["classes"] <= 1 << 27
        elif family == "rows":
            c = {"op": rng.choice(("layer_norm", "layer_norm", "softmax", "log_softmax")), "rows": L(rng, 64, 65536),
                 "cols": L(rng, 16, 8192)}
            ok = c["rows"] * c["cols"] <= 1 << 26
        elif family == "activation":
            c = {"op": rng.choice(ACTS), "n": L(rng, 1 << 10, 1 << 28)}
            ok = True
        elif family == "broadcast":
            # outer: a[p, 1, w] op b[h, w]; channel: x[p, h, w] op b[h, 1]; bias: x[p, h * w] op b[h * w]
            c = {"op": rng.choice(("add", "mul", "div")), "form": rng.choice(("outer", "channel", "bias")),
                 "p": L(rng, 1, 65536), "h": L(rng, 3, 1024), "w": L(rng, 4, 4096)}
            ok = 1 << 12 <= c["p"] * c["h"] * c["w"] <= 1 << 28
        elif family == "int8":
            c = {"m": L(rng, 1, 4096), "k": L(rng, 256, 8192), "n": L(rng, 256, 8192)}
            ok = c["m"] * c["k"] * c["n"] <= 1 << 36
        else:
            c = {"rows": L(rng, 64, 32768), "cols": L(rng, 64, 16384)}
            ok = c["rows"] * c["cols"] <= 1 << 28
        if ok:
            return dict(c, family=family)


# ---- inputs: plain torch, from the seed alone ---------------------------------------------------------
def _inputs(case, seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed))

    def normal(*shape, std=1.0, mean=0.0):
        t = torch.randn(shape, generator=g, device=DEV)
        if std != 1.0:
            t.mul_(std)
        return t.add_(mean) if mean else t

    def uniform(lo, hi, *shape):
        return torch.rand(shape, generator=g, device=DEV).mul_(hi - lo).add_(lo)

    def labels(n, c):
        return torch.randint(0, c, (n,), generator=g, device=DEV, dtype=torch.int32)

    f = case["family"]
    if f == "chain":
        return {"x": uniform(-1, 1, case["n"], case["c"], case["h"], case["w"]),
                "b": uniform(-0.1, 0.1, 1, case["c"], 1, 1)}
    if f == "classifier":
        i, h, o = case["features"], case["hidden"], case["classes"]
        return {"x": uniform(0, 1, case["batch"], i), "y": labels(case["batch"], o),
                "w1": normal(h, i, std=i ** -0.5), "b1": normal(h, std=0.01),
                "w2": normal(o, h, std=h ** -0.5), "b2": normal(o, std=0.01)}
    if f == "mlp_block":
        t, d, h = case["tokens"], case["d"], case["hidden"]
        return {"x": normal(t, d), "target": normal(t, d), "gamma": normal(d, std=0.1, mean=1.0),
                "beta": normal(d, std=0.1), "w1": normal(h, d, std=d ** -0.5), "b1": normal(h, std=0.1),
                "w2": normal(d, h, std=h ** -0.5), "b2": normal(d, std=0.1)}
    if f == "linear":
        m, k, n = case["m"], case["k"], case["n"]
        return {"x": normal(m, k), "w": normal(n, k, std=k ** -0.5), "b": normal(n, std=0.1), "g": normal(m, n)}
    if f == "decode" or f == "int8":
        m, k, n = case["m"], case["k"], case["n"]
        return {"x": normal(m, k), "w": normal(n, k, std=0.02), "b": normal(n, std=0.1)}
    if f == "attention":
        shape = (case["heads"], case["s"], case["d"])
        return {"q": normal(*shape), "k": normal(*shape), "v": normal(*shape), "target": normal(*shape)}
    if f == "loss":
        return {"x": normal(case["rows"], case["classes"], std=2.0), "y": labels(case["rows"], case["classes"])}
    if f == "rows":
        r, c = case["rows"], case["cols"]
        ins = {"x": normal(r, c, std=2.0), "g": normal(r, c)}
        if case["op"] == "layer_norm":
            ins.update(gamma=normal(c, std=0.1, mean=1.0), beta=normal(c, std=0.1))
        return ins
    if f == "activation":
        return {"x": normal(case["n"]), "g": normal(case["n"])}
    if f == "broadcast":
        sa, sb, so = _bcast_shapes(case)
        return {"a": normal(*sa), "b": uniform(0.5, 2.0, *sb), "g": normal(*so)}
    w = normal(case["rows"], case["cols"], std=0.02)
    outliers = torch.rand(w.shape, generator=g, device=DEV) < 0.001
    return {"w": torch.where(outliers, w * 50, w)}


def _bcast_shapes(case):
    p, h, w = case["p"], case["h"], case["w"]
    if case["form"] == "outer":
        return (p, 1, w), (1, h, w), (p, h, w)
    if case["form"] == "channel":
        return (p, h, w), (1, h, 1), (p, h, w)
    return (p, h * w), (1, h * w), (p, h * w)


def _bcast_strides(shape, out):
    st, s = [], 1
    for n, o in zip(reversed(shape), reversed(out)):
        st.append(0 if n == 1 and o != 1 else s)
        s *= n
    return tuple(reversed(st))


# ---- the framework's side --------------------------------------------------------------------------------
_shared = {}


def _lib():
    if not _shared:
        lib = abi.load()
        _shared.update(lib=lib, kernels=hip.Kernels(lib), stream=torch.cuda.Stream())
    return _shared["lib"]


def _stream():
    _lib()
    return _shared["stream"].cuda_stream


class _Engine:
    """One context of the engine; freed with the last tensor or view that lives in it."""

    def __init__(self):
        self.lib = _lib()
        self.ctx = self.lib.nc_init(ctypes.byref(abi.Config(0, 1, 0, 0)))
        self.lib.nc_set_stream(self.ctx, _stream())

    def check(self):
        if not self.lib.nc_ok(self.ctx):
            raise RuntimeError(self.lib.nc_error(self.ctx).decode())

    def tensor(self, t, param=False):
        """A persistent tensor (or parameter) with t's values."""
        L, (nd, shape) = self.lib, abi.shape_arg(t.shape)
        dt = abi.I32 if t.dtype == torch.int32 else abi.F32
        if param:
            n = L.nc_parameter(self.ctx, L.nc_from_device(self.ctx, dt, t.data_ptr(), nd, shape), nd, shape)
        else:
            L.nc_persistent_begin(self.ctx)
            n = L.nc_from_device(self.ctx, dt, t.data_ptr(), nd, shape)
            L.nc_persistent_end(self.ctx)
        self.check()
        return n

    def __del__(self):
        if self.ctx:
            self.lib.nc_free_ctx(self.ctx)
            self.ctx = None


class _Memory:
    """An engine tensor's device memory, for torch to look at in place."""

    def __init__(self, engine, ptr, shape):
        self.engine = engine
        self.__cuda_array_interface__ = {"data": (ptr, False), "shape": shape, "typestr": "<f4", "version": 2}


class _State:
    """A program's tensors in an engine context; views of the engine's memory are made once for each place."""

    def __init__(self, ins, params, others=()):
        self.e = _Engine()
        torch.cuda.synchronize()
        self.t = {k: self.e.tensor(ins[k], True) for k in params}
        self.t.update({k: self.e.tensor(ins[k]) for k in others})
        self.params = [self.t[k] for k in params]
        self.seen = {}
        self.e.lib.nc_synchronize(self.e.ctx)
        self.e.lib.nc_step_end(self.e.ctx)
        self.e.check()

    def view(self, t, *shape):
        key = (self.e.lib.nc_device_ptr(t), shape)
        if key not in self.seen:
            self.e.check()
            self.seen[key] = torch.as_tensor(_Memory(self.e, key[0], shape), device=DEV)
        return self.seen[key]

    def grad(self, name, *shape):
        return self.view(self.e.lib.nc_grad(self.t[name]), *shape)

    def begin(self):
        """A new step: the last one's temporaries go back, gradients start from zero."""
        self.e.lib.nc_step_end(self.e.ctx)
        for p in self.params:
            self.e.lib.nc_zero_grad(p)


def prepare(case, seed):
    ins = _inputs(case, seed)
    f = case["family"]
    _lib()
    state = {"case": case}
    if f == "chain":
        state["s"] = _State(ins, ("x", "b"))
    elif f == "classifier":
        s = state["s"] = _State(ins, ("w1", "b1", "w2", "b2"), ("x", "y"))
        opts = abi.OptimOpts(LR, MOMENTUM, 0.0, 0.0, 0.0, 0.0)
        state["opt"] = s.e.lib.nc_sgd(s.e.ctx, abi.ptr_array(s.params), len(s.params), opts)
        s.e.check()
    elif f == "mlp_block":
        state["s"] = _State(ins, ("x", "gamma", "beta", "w1", "b1", "w2", "b2"), ("target",))
    elif f == "decode":
        s = state["s"] = _State(ins, (), ("x", "w", "b"))
        s.e.lib.nc_set_grad_enabled(s.e.ctx, 0)
    elif f == "int8":
        s = state["s"] = _State(ins, (), ("x", "w", "b"))
        L, scale = s.e.lib, ctypes.c_void_p()
        L.nc_set_grad_enabled(s.e.ctx, 0)
        L.nc_persistent_begin(s.e.ctx)
        s.t["wq"] = L.nc_quantize_rows(s.t["w"], ctypes.byref(scale))
        s.t["ws"] = scale.value
        L.nc_persistent_end(s.e.ctx)
        s.e.check()
        L.nc_synchronize(s.e.ctx)
        L.nc_release(s.t.pop("w"))
    elif f == "attention":
        state["s"] = _State(ins, ("q", "k", "v"), ("target",))
    elif f == "loss":
        state["s"] = _State(ins, ("x",), ("y",))
    else:  # the kernel layer on the program's own buffers: outputs and workspaces beside the inputs
        K = _shared["kernels"]
        state["b"] = b = dict(ins)

        def buffer(*shape, dtype=torch.float32):
            return torch.empty(shape, device=DEV, dtype=dtype)

        def workspace(n):
            return buffer(max(int(n), 256), dtype=torch.uint8)

        if f == "linear":
            m, k, n = case["m"], case["k"], case["n"]
            b.update(y=buffer(m, n), gx=buffer(m, k), gw=buffer(n, k), gb=buffer(n),
                     ws=workspace(K.binary_bwd_workspace((m, n), (0, 1))))
        elif f == "rows":
            r, c = case["rows"], case["cols"]
            b.update(y=buffer(r, c), gx=buffer(r, c))
            if case["op"] == "layer_norm":
                b.update(stats=buffer(r, 2), gw=buffer(c), gb=buffer(c), ws=workspace(K.layer_norm_bwd_workspace(r, c)))
        elif f == "activation":
            b.update(y=buffer(case["n"]), gx=buffer(case["n"]))
        elif f == "broadcast":
            sa, sb, so = _bcast_shapes(case)
            ta, tb, to = (_bcast_strides(s, so) for s in (sa, sb, so))
            b.update(o=buffer(*so), ga=buffer(*sa), gb=buffer(*sb))
            state.update(shape=so, ta=ta, tb=tb, to=to)
            if case["form"] == "outer":
                b["ws"] = workspace(K.binary_bwd2_workspace(so, ta, tb))
            else:
                b["ws"] = workspace(max(K.binary_bwd_workspace(so, ta), K.binary_bwd_workspace(so, tb)))
        else:
            r, c = case["rows"], case["cols"]
            b.update(q=buffer(r, c, dtype=torch.int8), scale=buffer(r), out=buffer(r, c))
    torch.cuda.synchronize()
    return state


def run(state):
    return _RUN[state["case"]["family"]](state, state["case"])


def _run_chain(state, case):
    s = state["s"]
    L, t = s.e.lib, s.t
    s.begin()
    h = L.nc_relu(L.nc_add(t["x"], t["b"]))
    p = L.nc_sum(L.nc_sum(h, 3, 1), 2, 1)
    L.nc_backward(L.nc_sum(p, abi.ALL_AXES, 0))
    n, c, hh, ww = case["n"], case["c"], case["h"], case["w"]
    return s.view(p, n, c), s.grad("x", n, c, hh, ww), s.grad("b", c)


def _run_classifier(state, case):
    s = state["s"]
    L, t = s.e.lib, s.t
    L.nc_step_end(s.e.ctx)
    h = L.nc_relu(L.nc_linear_fn(t["x"], t["w1"], t["b1"]))
    logits = L.nc_linear_fn(h, t["w2"], t["b2"])
    loss = L.nc_cross_entropy(logits, t["y"])
    L.nc_optim_zero_grad(state["opt"])
    L.nc_backward(loss)
    L.nc_optim_step(state["opt"])
    n, i, d, o = case["batch"], case["features"], case["hidden"], case["classes"]
    return (s.view(logits, n, o), s.view(loss), s.view(t["w1"], d, i), s.view(t["b1"], d), s.view(t["w2"], o, d),
            s.view(t["b2"], o))


def _run_mlp_block(state, case):
    s = state["s"]
    L, t = s.e.lib, s.t
    s.begin()
    z = L.nc_layer_norm(t["x"], 1, t["gamma"], t["beta"], EPS)
    h = L.nc_gelu(L.nc_linear_fn(z, t["w1"], t["b1"]), 0)
    y = L.nc_add(t["x"], L.nc_linear_fn(h, t["w2"], t["b2"]))
    loss = L.nc_mse_loss(y, t["target"])
    L.nc_backward(loss)
    m, d, hd = case["tokens"], case["d"], case["hidden"]
    return (s.view(y, m, d), s.view(loss), s.grad("x", m, d), s.grad("gamma", d), s.grad("beta", d),
            s.grad("w1", hd, d), s.grad("b1", hd), s.grad("w2", d, hd), s.grad("b2", d))


def _run_linear(state, case):
    K, b, st = _shared["kernels"], state["b"], _stream()
    m, k, n = case["m"], case["k"], case["n"]
    x, w, g, y, gb, ws = (b[i].data_ptr() for i in ("x", "w", "g", "y", "gb", "ws"))
    K.gemm_f32_bias(0, 1, m, n, k, 1.0, x, k, w, k, b["b"].data_ptr(), y, n, stream=st)
    K.gemm_f32(0, 0, m, k, n, 1.0, g, n, w, k, 0.0, b["gx"].data_ptr(), k, stream=st)
    K.gemm_f32(1, 0, n, k, m, 1.0, g, n, x, k, 0.0, b["gw"].data_ptr(), k, stream=st)
    K.binary_bwd("add", 1, (m, n), g, (n, 1), g, (n, 1), gb, (0, 1), gb, (0, 1), ws, b["ws"].numel(),
                 accumulate=False, stream=st)
    return b["y"], b["gx"], b["gw"], b["gb"]


def _run_decode(state, case):
    s = state["s"]
    s.e.lib.nc_step_end(s.e.ctx)
    y = s.e.lib.nc_linear_fn(s.t["x"], s.t["w"], s.t["b"])
    return (s.view(y, case["m"], case["n"]),)


def _run_int8(state, case):
    s = state["s"]
    s.e.lib.nc_step_end(s.e.ctx)
    y = s.e.lib.nc_linear_int8(s.t["x"], s.t["wq"], s.t["ws"], s.t["b"])
    return (s.view(y, case["m"], case["n"]),)


def _run_attention(state, case):
    s = state["s"]
    L, t = s.e.lib, s.t
    s.begin()
    scores = L.nc_scale(L.nc_matmul(t["q"], L.nc_transpose(t["k"], 1, 2)), case["d"] ** -0.5)
    o = L.nc_matmul(L.nc_softmax(scores), t["v"])
    loss = L.nc_mse_loss(o, t["target"])
    L.nc_backward(loss)
    shape = (case["heads"], case["s"], case["d"])
    return s.view(o, *shape), s.view(loss), s.grad("q", *shape), s.grad("k", *shape), s.grad("v", *shape)


def _run_loss(state, case):
    s = state["s"]
    L, t = s.e.lib, s.t
    s.begin()
    loss = L.nc_cross_entropy(t["x"], t["y"])
    L.nc_backward(loss)
    return s.view(loss), s.grad("x", case["rows"], case["classes"])


def _run_rows(state, case):
    K, b, st = _shared["kernels"], state["b"], _stream()
    r, c = case["rows"], case["cols"]
    x, g, y, gx = (b[i].data_ptr() for i in ("x", "g", "y", "gx"))
    if case["op"] == "layer_norm":
        gamma, beta, stats, gw, gb = (b[i].data_ptr() for i in ("gamma", "beta", "stats", "gw", "gb"))
        K.layer_norm_fwd(r, c, x, gamma, beta, EPS, y, stats, stream=st)
        K.fill(gw, 4, 0, c, stream=st)  # the column gradients are added into
        K.fill(gb, 4, 0, c, stream=st)
        K.layer_norm_bwd(r, c, x, gamma, stats, g, gx, gw, gb, b["ws"].data_ptr(), b["ws"].numel(), accumulate=False,
                         stream=st)
        return b["y"], b["gx"], b["gw"], b["gb"]
    log = case["op"] == "log_softmax"
    K.softmax_fwd(log, r, c, x, y, stream=st)
    K.softmax_bwd(log, r, c, y, g, gx, accumulate=False, stream=st)
    return b["y"], b["gx"]


def _run_activation(state, case):
    K, b, st = _shared["kernels"], state["b"], _stream()
    x, g, y, gx = (b[i].data_ptr() for i in ("x", "g", "y", "gx"))
    K.unary_fwd(case["op"], x, y, case["n"], stream=st)
    K.unary_bwd(case["op"], x, y, g, gx, case["n"], accumulate=False, stream=st)
    return b["y"], b["gx"]


def _run_broadcast(state, case):
    K, m, st = _shared["kernels"], state["b"], _stream()
    op, shape, ta, tb, to = case["op"], state["shape"], state["ta"], state["tb"], state["to"]
    a, b, g, o, ga, gb, ws = (m[i].data_ptr() for i in ("a", "b", "g", "o", "ga", "gb", "ws"))
    nws = m["ws"].numel()
    K.binary_fwd(op, shape, a, ta, b, tb, o, to, stream=st)
    if case["form"] == "outer":
        K.binary_bwd2(op, shape, g, to, a, ta, b, tb, ga, ta, gb, tb, ws, nws, accumulate=False, stream=st)
    else:
        K.binary_bwd(op, 0, shape, g, to, a, ta, b, tb, ga, ta, ws, nws, accumulate=False, stream=st)
        K.binary_bwd(op, 1, shape, g, to, a, ta, b, tb, gb, tb, ws, nws, accumulate=False, stream=st)
    return m["o"], m["ga"], m["gb"]


def _run_quantize(state, case):
    K, b, st = _shared["kernels"], state["b"], _stream()
    r, c = case["rows"], case["cols"]
    w, q, scale, out = (b[i].data_ptr() for i in ("w", "q", "scale", "out"))
    K.quantize_rows(r, c, w, q, scale, stream=st)
    K.dequantize_rows(r, c, q, scale, out, stream=st)
    return b["q"], b["scale"], b["out"]


_RUN = {"chain": _run_chain, "classifier": _run_classifier, "mlp_block": _run_mlp_block, "linear": _run_linear,
        "decode": _run_decode, "int8": _run_int8, "attention": _run_attention, "loss": _run_loss, "rows": _run_rows,
        "activation": _run_activation, "broadcast": _run_broadcast, "quantize": _run_quantize}


# ---- what a pass cannot do without --------------------------------------------------------------------------
def work(case):
    """Bytes: each call's inputs read once and its results written once (float32 unless said); flops: the
    products' multiply-adds and a few a value for the rest.  What a later call of the same pass reads again is
    counted once where it is small (weights, block activations), and for each call where it is the tensor itself."""
    f = case["family"]
    if f == "chain":
        n = case["n"] * case["c"] * case["h"] * case["w"]
        return {"bytes": 4 * (2 * n + case["n"] * case["c"] + 2 * case["c"]), "flops": 4 * n}
    if f == "classifier":
        b, i, h, o = case["batch"], case["features"], case["hidden"], case["classes"]
        weights = h * i + h + o * h + o
        return {"bytes": 4 * (b * i + b + b * o + 4 * weights), "flops": 2 * b * (2 * i * h + 3 * h * o)}
    if f == "mlp_block":
        t, d, h = case["tokens"], case["d"], case["hidden"]
        return {"bytes": 4 * (4 * t * d + 2 * (2 * d * h + h + 3 * d)), "flops": 12 * t * d * h}
    if f == "linear":
        m, k, n = case["m"], case["k"], case["n"]
        return {"bytes": 4 * (2 * m * k + 2 * n * k + 2 * m * n + 2 * n), "flops": 6 * m * k * n}
    if f == "decode":
        m, k, n = case["m"], case["k"], case["n"]
        return {"bytes": 4 * (m * k + n * k + n + m * n), "flops": 2 * m * k * n}
    if f == "int8":
        m, k, n = case["m"], case["k"], case["n"]
        return {"bytes": 4 * m * k + n * k + 8 * n + 4 * m * n, "flops": 2 * m * k * n}
    if f == "attention":
        b, s, d = case["heads"], case["s"], case["d"]
        return {"bytes": 4 * 8 * b * s * d, "flops": 12 * b * s * s * d}
    if f == "loss":
        n = case["rows"] * case["classes"]
        return {"bytes": 12 * n + 4 * case["rows"], "flops": 8 * n}
    if f == "rows":
        n = case["rows"] * case["cols"]
        return {"bytes": 20 * n, "flops": 16 * n}
    if f == "activation":
        return {"bytes": 20 * case["n"], "flops": 40 * case["n"]}
    if f == "broadcast":
        sa, sb, so = (math.prod(s) for s in _bcast_shapes(case))
        small = 2 if case["op"] == "add" else 3  # mul and div read their operands again for the gradients
        return {"bytes": 4 * (2 * so + small * (sa + sb)), "flops": 3 * so}
    n = case["rows"] * case["cols"]
    return {"bytes": 10 * n + 8 * case["rows"], "flops": 4 * n}


def tolerance(case):
    """About four times what the float32 path shows against 64 bits over these ranges: 3.2e-7 (largest value 9e-6
    off) where there are products of long rows, 1e-7 (2e-6) elsewhere.  int8 values, their scales and what they expand
    to are defined bit for bit, an int8 product's sums too."""
    f = case["family"]
    if f == "quantize":
        return "exact"
    if f in ("classifier", "mlp_block", "linear", "decode", "attention"):
        return {"rel": 1.5e-6, "max": 4e-5}
    return {"rel": 5e-7, "max": 1e-5}


# ---- the same in 64 bits ----------------------------------------------------------------------------------------
def exact(case, seed):
    ins = _inputs(case, seed)
    f = case["family"]
    d = {k: v.double() for k, v in ins.items() if v.dtype == torch.float32}
    if f == "chain":
        h = torch.relu(d["x"] + d["b"])
        on = (h > 0).double()
        return h.sum((2, 3)), on, on.sum((0, 2, 3))
    if f == "classifier":
        p = {k: d[k].requires_grad_(True) for k in ("w1", "b1", "w2", "b2")}
        logits = F.linear(torch.relu(F.linear(d["x"], p["w1"], p["b1"])), p["w2"], p["b2"])
        loss = F.cross_entropy(logits, ins["y"].long())
        loss.backward()
        return (logits.detach(), loss.detach()) + tuple((v - LR * v.grad).detach() for v in p.values())
    if f == "mlp_block":
        p = {k: d[k].requires_grad_(True) for k in ("x", "gamma", "beta", "w1", "b1", "w2", "b2")}
        z = F.layer_norm(p["x"], (case["d"],), p["gamma"], p["beta"], EPS)
        y = p["x"] + F.linear(F.gelu(F.linear(z, p["w1"], p["b1"])), p["w2"], p["b2"])
        loss = F.mse_loss(y, d["target"])
        loss.backward()
        return (y.detach(), loss.detach()) + tuple(v.grad for v in p.values())
    if f == "linear":
        return (d["x"] @ d["w"].T + d["b"], d["g"] @ d["w"], d["g"].T @ d["x"], d["g"].sum(0))
    if f == "decode":
        return (d["x"] @ d["w"].T + d["b"],)
    if f == "int8":
        xq, xs = _quantized(ins["x"])
        wq, ws = _quantized(ins["w"])
        return ((xq.double() @ wq.double().T) * xs.double()[:, None] * ws.double() + d["b"],)
    if f == "attention":
        q, k, v = (d[i].requires_grad_(True) for i in ("q", "k", "v"))
        scores = torch.matmul(q, k.transpose(1, 2).contiguous()) * case["d"] ** -0.5
        o = torch.matmul(torch.softmax(scores, -1), v)
        loss = F.mse_loss(o, d["target"])
        loss.backward()
        return o.detach(), loss.detach(), q.grad, k.grad, v.grad
    if f == "loss":
        x = d["x"].requires_grad_(True)
        loss = F.cross_entropy(x, ins["y"].long())
        loss.backward()
        return loss.detach(), x.grad
    if f == "rows":
        x = d["x"].requires_grad_(True)
        if case["op"] == "layer_norm":
            w, b = d["gamma"].requires_grad_(True), d["beta"].requires_grad_(True)
            y = F.layer_norm(x, (case["cols"],), w, b, EPS)
            y.backward(d["g"])
            return y.detach(), x.grad, w.grad, b.grad
        y = F.softmax(x, -1) if case["op"] == "softmax" else F.log_softmax(x, -1)
        y.backward(d["g"])
        return y.detach(), x.grad
    if f == "activation":
        fn = {"gelu": F.gelu, "silu": F.silu, "sigmoid": torch.sigmoid, "tanh": torch.tanh, "hardswish": F.hardswish,
              "relu6": F.relu6, "relu": torch.relu}[case["op"]]
        x = d["x"].requires_grad_(True)
        y = fn(x)
        y.backward(d["g"])
        return y.detach(), x.grad
    if f == "broadcast":
        sa, sb, _ = _bcast_shapes(case)
        a, b, g = d["a"], d["b"], d["g"]
        if case["op"] == "add":
            return a + b, _sum_to(g, sa), _sum_to(g, sb)
        if case["op"] == "mul":
            return a * b, _sum_to(g * b, sa), _sum_to(g * a, sb)
        return a / b, _sum_to(g / b, sa), _sum_to(-(g * a) / (b * b), sb)
    q, scale = _quantized(ins["w"])
    return None, scale.double(), q.double() * scale.double()[:, None]


def _quantized(w):
    """Symmetric int8 rows as the format defines them, in float32: absmax / 127, round to nearest even."""
    amax = w.abs().amax(1)
    scale = torch.where(amax > 0, amax / torch.full_like(amax, 127), torch.ones_like(amax))
    return torch.round(w * (1 / scale)[:, None]).clamp_(-127, 127), scale


def _sum_to(t, shape):
    dims = [i for i, n in enumerate(shape) if n == 1 and t.shape[i] != 1]
    return t.sum(dims, keepdim=True) if dims else t
