"""The workloads this framework is measured on.

Each case is one piece of a training step, taken through the Python entry
points of ``tensors_amd.ops`` on memory that the program already holds on the
GPU: a whole small step, Linear layers forward and backward in fp32 and bf16,
a classifier head with its loss, convolutions, LayerNorm, the cross entropy
and the optimiser.  ``listed()`` names the fixed ones, ``draw()`` gives more
of the same ranges.  A forward pass and the backward pass of a layer are one
case; the backward takes the activation that the forward of its micro-batch
saved (an input of the case), so a pre-activation that rounds to the other
side of zero does not change the gradients that are compared.
"""
import numpy as np
import torch
import torch.nn.functional as F

from tensors_amd import _lib, ops
from tensors_amd.device import BF16, Context, DeviceArray

_CTX = None


def _ctx():
    """The program's one context (device 0)."""
    global _CTX
    if _CTX is None:
        _CTX = Context(0)
    return _CTX


class Borrowed(DeviceArray):
    """A DeviceArray over a contiguous torch tensor's memory."""

    _TYPES = {torch.float32: np.float32, torch.int64: np.int64, torch.bfloat16: BF16}

    def __init__(self, t):
        assert t.is_contiguous()
        self.ctx, self.tensor, self.ptr = _ctx(), t, t.data_ptr()
        self.shape, self.dtype = tuple(t.shape), self._TYPES[t.dtype]
        self.size, self.nbytes = t.numel(), t.numel() * t.element_size()

    def free(self):
        self.ptr = self.tensor = None


def listed():
    return [
        # A whole step of a small MLP (784-256-128-10, batch 64): launches and
        # host work count here, not bytes.
        {"name": "mlp_step", "kind": "mlp_step", "batch": 64, "inputs": 784, "hidden1": 256, "hidden2": 128,
         "classes": 10},
        # One fp32 Linear + ReLU layer at 2048 cubed.
        {"name": "linear_f32", "kind": "linear", "dtype": "f32", "batch": 2048, "inputs": 2048, "outputs": 2048},
        # The first layer over flattened 3 x 32 x 32 images with an odd width
        # and the last, incomplete batch of an epoch.
        {"name": "linear_f32_odd", "kind": "linear", "dtype": "f32", "batch": 999, "inputs": 3072, "outputs": 1001},
        # The widest layer of the bf16 MLP 4096-8192-8192-4096-1000, batch 4096.
        {"name": "linear_bf16", "kind": "linear", "dtype": "bf16", "batch": 4096, "inputs": 8192, "outputs": 8192},
        # Its first layer at one of eight data-parallel ranks' share.
        {"name": "linear_bf16_b512", "kind": "linear", "dtype": "bf16", "batch": 512, "inputs": 4096,
         "outputs": 8192},
        # Its classifier with the loss: 1000 outputs, bf16 logits.
        {"name": "head_bf16", "kind": "head", "dtype": "bf16", "batch": 4096, "inputs": 4096, "outputs": 1000},
        # The second convolution of the 32 x 32 image network.
        {"name": "conv_s2", "kind": "conv", "batch": 128, "channels": 32, "size": 32, "filters": 64, "kernel": 3,
         "stride": 2, "pad": 1},
        # A convolution of a larger image network: more channels and pixels
        # than one block's LDS holds.
        {"name": "conv_56", "kind": "conv", "batch": 32, "channels": 64, "size": 56, "filters": 64, "kernel": 3,
         "stride": 1, "pad": 1},
        # LayerNorm at the isolated size, and over activations as wide as the
        # bf16 MLP's.
        {"name": "layernorm", "kind": "layernorm", "rows": 1024, "cols": 1024},
        {"name": "layernorm_wide", "kind": "layernorm", "rows": 4096, "cols": 8192},
        # The loss and its gradient over fp32 logits.
        {"name": "cross_entropy", "kind": "cross_entropy", "rows": 4096, "cols": 1024},
        # The optimiser over all parameters of the bf16 MLP, with the bf16
        # copies of its weights.
        {"name": "sgd", "kind": "sgd", "widths": "4096,8192,8192,4096,1000", "bf16_copy": True},
    ]


def _log(rng, lo, hi, odd=0.35):
    """A size from lo to hi, spread over its logarithm: a multiple of 64 (of 8
    below 512) where that is in range, or with chance `odd` any number."""
    v = int(round(lo * (hi / lo) ** rng.random()))
    if rng.random() >= odd:
        step = 64 if v >= 512 else 8
        v = (v + step // 2) // step * step
    return max(lo, min(hi, v))


def draw(rng):
    kind = rng.choice(["mlp_step", "linear", "linear", "linear", "head", "conv", "conv", "layernorm", "cross_entropy",
                       "sgd"])
    if kind == "mlp_step":
        c = {"kind": kind, "batch": _log(rng, 16, 512), "inputs": _log(rng, 64, 3072),
             "hidden1": _log(rng, 32, 512), "hidden2": _log(rng, 32, 512), "classes": rng.randint(2, 16)}
        # The largest product that the small-layer entry points take.
        while c["batch"] * c["inputs"] * c["hidden1"] > 1 << 27:
            c["batch"] //= 2
        return c
    if kind == "linear":
        if rng.random() < 0.5:
            return {"kind": kind, "dtype": "f32", "batch": _log(rng, 32, 2048), "inputs": _log(rng, 64, 4096),
                    "outputs": _log(rng, 32, 4096)}
        return {"kind": kind, "dtype": "bf16", "batch": _log(rng, 64, 4096), "inputs": _log(rng, 256, 8192, 0.15),
                "outputs": _log(rng, 256, 8192, 0.15)}
    if kind == "head":
        return {"kind": kind, "dtype": rng.choice(["f32", "bf16"]), "batch": _log(rng, 32, 4096),
                "inputs": _log(rng, 64, 4096, 0.2), "outputs": _log(rng, 10, 1024)}
    if kind == "conv":
        size, k, s = rng.choice([(8, 3, 1), (14, 3, 1), (16, 3, 2), (28, 3, 1), (28, 5, 1), (32, 3, 1), (32, 3, 2),
                                 (33, 3, 1), (56, 3, 1), (56, 1, 1), (15, 5, 2)])
        c = {"kind": kind, "batch": _log(rng, 8, 128), "channels": rng.choice([1, 3, 8, 16, 24, 32, 64, 128]),
             "size": size, "filters": rng.choice([8, 16, 32, 48, 64, 128]), "kernel": k, "stride": s, "pad": k // 2}
        while _conv_out(c) ** 2 * c["batch"] * c["channels"] * k * k > 1 << 26:
            c["batch"] = max(1, c["batch"] // 2)
        return c
    if kind == "layernorm":
        c = {"kind": kind, "rows": _log(rng, 64, 8192), "cols": _log(rng, 64, 8192)}
    elif kind == "cross_entropy":
        c = {"kind": kind, "rows": _log(rng, 64, 8192), "cols": _log(rng, 10, 32768)}
    else:
        return {"kind": kind, "widths": ",".join(str(_log(rng, 64, 4096)) for _ in range(rng.randint(2, 6))),
                "bf16_copy": rng.random() < 0.5}
    while c["rows"] * c["cols"] > 1 << 25:
        c["rows"] = max(1, c["rows"] // 2)
    return c


def _conv_out(c):
    return ops.conv_out(c["size"], c["kernel"], c["stride"], c["pad"], 1)


def _widths(c):
    w = [int(v) for v in c["widths"].split(",")]
    return list(zip(w[:-1], w[1:]))


class _Make:
    """Inputs on the GPU from one seed."""

    def __init__(self, seed):
        self.g = torch.Generator(device="cuda")
        self.g.manual_seed(int(seed))

    def normal(self, *shape, std=1.0, dtype=torch.float32):
        return (torch.randn(shape, generator=self.g, device="cuda") * std).to(dtype)

    def hidden(self, *shape, dtype=torch.float32):
        """A ReLU's output."""
        return torch.randn(shape, generator=self.g, device="cuda").relu_().to(dtype)

    def weight(self, out, fan_in, *rest, dtype=torch.float32):
        n = fan_in
        for r in rest:
            n *= r
        w = torch.rand((out, fan_in, *rest), generator=self.g, device="cuda")
        return ((w * 2 - 1) * n ** -0.5).to(dtype)

    def labels(self, n, classes):
        return torch.randint(0, classes, (n,), generator=self.g, device="cuda")


def _inputs(c, seed):
    """The case's input tensors by name."""
    m, kind = _Make(seed), c["kind"]
    if kind == "mlp_step":
        b, d0, d1, d2, n = (c[k] for k in ("batch", "inputs", "hidden1", "hidden2", "classes"))
        # Normalised pixels, 0..255 / 255 by mean 0.1307 and deviation 0.3081.
        x = (torch.randint(0, 256, (b, d0), generator=m.g, device="cuda").float() / 255 - 0.1307) / 0.3081
        return {"x": x, "t": m.labels(b, n), "w1": m.weight(d1, d0), "w2": m.weight(d2, d1), "w3": m.weight(n, d2),
                "b3": m.normal(n, std=0.01), "v1": m.normal(d1, d0, std=0.01), "v2": m.normal(d2, d1, std=0.01),
                "v3": m.normal(n, d2, std=0.01), "vb3": m.normal(n, std=0.01)}
    if kind in ("linear", "head"):
        dt = torch.bfloat16 if c["dtype"] == "bf16" else torch.float32
        b, i, o = c["batch"], c["inputs"], c["outputs"]
        t = {"x": m.hidden(b, i, dtype=dt), "w": m.weight(o, i, dtype=dt), "b": m.normal(o, std=0.05)}
        if kind == "head":
            t["t"] = m.labels(b, o)
        else:
            t["y_saved"] = m.hidden(b, o, dtype=dt)
            t["dy"] = m.normal(b, o, std=1.0 / b, dtype=dt)
        return t
    if kind == "conv":
        n, ci, s, co, k, p = c["batch"], c["channels"], c["size"], c["filters"], c["kernel"], _conv_out(c)
        return {"x": m.hidden(n, ci, s, s), "w": m.weight(co, ci, k, k), "b": m.normal(co, std=0.05),
                "y_saved": m.hidden(n, co, p, p), "dy": m.normal(n, co, p, p, std=1.0 / n)}
    if kind == "layernorm":
        r, k = c["rows"], c["cols"]
        return {"x": m.normal(r, k), "gamma": m.normal(k, std=0.1) + 1, "beta": m.normal(k, std=0.1),
                "dy": m.normal(r, k, std=1.0 / r)}
    if kind == "cross_entropy":
        return {"x": m.normal(c["rows"], c["cols"], std=3.0), "t": m.labels(c["rows"], c["cols"])}
    t = {}
    for n, (i, o) in enumerate(_widths(c)):
        t["p%d" % (2 * n)], t["p%d" % (2 * n + 1)] = m.weight(o, i), m.normal(o, std=0.05)
        for a, std in (("g", 1e-3), ("v", 1e-2)):
            t[a + "%d" % (2 * n)], t[a + "%d" % (2 * n + 1)] = m.normal(o, i, std=std), m.normal(o, std=std)
    return t


def prepare(case, seed):
    c = dict(case)
    s = {k: Borrowed(v) for k, v in _inputs(c, seed).items()}
    s["case"] = c

    def out(name, *shape, dtype=torch.float32):
        s[name] = Borrowed(torch.zeros(shape, dtype=dtype, device="cuda"))

    kind = c["kind"]
    if kind == "mlp_step":
        b, d0, d1, d2, n = (c[k] for k in ("batch", "inputs", "hidden1", "hidden2", "classes"))
        for name, shape in (("h1", (b, d1)), ("h2", (b, d2)), ("z", (b, n)), ("loss", (1,)), ("dz", (b, n)),
                            ("dh2", (b, d2)), ("dh1", (b, d1)), ("dw1", (d1, d0)), ("dw2", (d2, d1)), ("dw3", (n, d2)),
                            ("db3", (n,))):
            out(name, *shape)
    elif kind in ("linear", "head"):
        dt = torch.bfloat16 if c["dtype"] == "bf16" else torch.float32
        b, i, o = c["batch"], c["inputs"], c["outputs"]
        out("y", b, o, dtype=dt)
        out("dz", b, o, dtype=dt)
        out("dx", b, i, dtype=dt)
        out("dw", o, i)
        out("db", o)
        if kind == "head":
            out("loss", 1)
    elif kind == "conv":
        n, ci, h, co, k, p = c["batch"], c["channels"], c["size"], c["filters"], c["kernel"], _conv_out(c)
        out("y", n, co, p, p)
        out("dz", n, co, p, p)
        out("dx", n, ci, h, h)
        out("dw", co, ci, k, k)
        out("db", co)
        # What the column form of the convolution needs, for geometries that
        # the kernels without column buffers do not take.
        out("col", n, ci * k * k, p * p)
    elif kind == "layernorm":
        r, k = c["rows"], c["cols"]
        out("y", r, k)
        out("dx", r, k)
        out("mean", r)
        out("rstd", r)
        out("dgamma", k)
        out("dbeta", k)
    elif kind == "cross_entropy":
        out("loss", 1)
        out("dx", c["rows"], c["cols"])
    elif kind == "sgd" and c["bf16_copy"]:
        for n, (i, o) in enumerate(_widths(c)):
            out("s%d" % (2 * n), o, i, dtype=torch.bfloat16)
    # The context launches on a stream of its own.
    torch.cuda.synchronize()
    return s


def _give(s, *names):
    return {n: s[n].tensor for n in names}


def _mlp_step(s):
    """Forward, loss, backward and update of three Linear layers, the hidden
    two without bias."""
    ops.gemm(s["x"], s["w1"], s["h1"], trans_b=True, relu=True)
    ops.gemm(s["h1"], s["w2"], s["h2"], trans_b=True, relu=True)
    ops.gemm(s["h2"], s["w3"], s["z"], trans_b=True, bias=s["b3"])
    ops.ce_fwd_bwd(s["z"], s["t"], s["loss"], s["dz"])
    if s["case"]["hidden2"] % 4 == 0:
        ops.linear_bwd_narrow(s["dz"], s["h2"], s["w3"], s["dh2"], s["dw3"], s["db3"])
    else:
        ops.gemm(s["dz"], s["w3"], s["dh2"])
        ops.gemm(s["dz"], s["h2"], s["dw3"], trans_a=True)
        ops.colsum(s["dz"], s["db3"])
    ops.linear_bwd_small(s["dh2"], s["h1"], s["w2"], s["dh1"], s["dw2"], mask=s["h2"])
    ops.gemm_relu_masked(s["dh1"], s["h1"], s["x"], s["dw1"], trans_a=True)
    ops.sgd_momentum_multi([s["w1"], s["w2"], s["w3"], s["b3"]], [s["dw1"], s["dw2"], s["dw3"], s["db3"]],
                           [s["v1"], s["v2"], s["v3"], s["vb3"]], 0.01, 0.9)
    return _give(s, "loss", "z", "dw1", "dw2", "dw3", "db3", "w1", "w2", "w3", "b3", "v1")


def _linear(s):
    """relu(x w^T + b), and the gradients of x, w and b behind the ReLU."""
    ops.gemm(s["x"], s["w"], s["y"], trans_b=True, bias=s["b"], relu=True)
    ops.relu_bwd_colsum(s["dy"], s["y_saved"], s["dz"], s["db"])
    ops.gemm(s["dz"], s["w"], s["dx"])
    ops.gemm(s["dz"], s["x"], s["dw"], trans_a=True)
    return _give(s, "y", "dx", "dw", "db")


def _head(s):
    """Logits, mean cross entropy and all gradients; a head of at most 16 fp32
    outputs takes its backward in one call."""
    c = s["case"]
    ops.gemm(s["x"], s["w"], s["y"], trans_b=True, bias=s["b"])
    if c["dtype"] == "bf16":
        ops.ce_fwd_bwd_bf16(s["y"], s["t"], s["loss"], s["dz"])
    else:
        ops.ce_fwd_bwd(s["y"], s["t"], s["loss"], s["dz"])
    if c["dtype"] == "f32" and c["outputs"] <= 16 and c["inputs"] % 4 == 0:
        ops.linear_bwd_narrow(s["dz"], s["x"], s["w"], s["dx"], s["dw"], s["db"])
    else:
        ops.colsum(s["dz"], s["db"])
        ops.gemm(s["dz"], s["w"], s["dx"])
        ops.gemm(s["dz"], s["x"], s["dw"], trans_a=True)
    return _give(s, "y", "loss", "dx", "dw", "db")


def _taken(fn, *args, **kw):
    """Whether the kernel takes the geometry."""
    try:
        fn(*args, **kw)
        return True
    except _lib.TFError as e:
        if e.status != _lib.TF_ERR_UNSUPPORTED:
            raise
        return False


def _conv(s):
    """relu(conv(x, w) + b), and all gradients behind the ReLU; a pass whose
    geometry does not fit takes the column form, as nn::Conv2dModule does."""
    c, x, w, col = s["case"], s["x"], s["w"], s["col"]
    n, ci, co, k = c["batch"], c["channels"], c["filters"], c["kernel"]
    kk, p = col.shape[1:]
    geo = {"stride": (c["stride"],) * 2, "pad": (c["pad"],) * 2}
    have_col = not _taken(ops.conv2d_fwd, x, w, s["y"], bias=s["b"], relu=True, **geo)
    if have_col:
        ops.im2col(x, col, k, k, **geo)
        ops.gemm_ex(w, col, s["y"], co, p, kk, lda=kk, ldb=p, ldc=p, stride_b=kk * p, stride_c=co * p, batch=n,
                    epilogue=_lib.TF_EPI_ROW_BIAS_RELU, bias=s["b"])
    if have_col or not _taken(ops.conv2d_bwd_weight, x, s["dy"], s["dw"], db=s["db"], relu_y=s["y_saved"], dz=s["dz"],
                              **geo):
        ops.relu_bwd(s["dy"], s["y_saved"], s["dz"])
        if not have_col:
            ops.im2col(x, col, k, k, **geo)
        ops.gemm_ex(s["dz"], col, s["dw"], co, kk, p, lda=p, ldb=p, ldc=kk, trans_b=True, stride_a=co * p,
                    stride_b=kk * p, batch=n, reduce_batch=True)
        ops.chansum_nchw(s["dz"], s["db"])
    if not _taken(ops.conv2d_bwd_data, s["dz"], w, s["dx"], **geo):
        # The columns of x are no longer needed: theirs hold the gradient's.
        ops.gemm_ex(w, s["dz"], col, kk, p, co, lda=kk, ldb=p, ldc=p, trans_a=True, stride_b=co * p, stride_c=kk * p,
                    batch=n)
        ops.col2im(col, s["dx"], k, k, **geo)
    return _give(s, "y", "dx", "dw", "db")


def _layernorm(s):
    ops.layernorm_fwd(s["x"], s["gamma"], s["beta"], s["y"], s["mean"], s["rstd"])
    ops.layernorm_bwd(s["dy"], s["x"], s["gamma"], s["mean"], s["rstd"], s["dx"], s["dgamma"], s["dbeta"])
    return _give(s, "y", "mean", "rstd", "dx", "dgamma", "dbeta")


def _cross_entropy(s):
    ops.ce_fwd_bwd(s["x"], s["t"], s["loss"], s["dx"])
    return _give(s, "loss", "dx")


def _sgd(s):
    n = 2 * len(_widths(s["case"]))
    group = lambda a: [s.get("%s%d" % (a, i)) for i in range(n)]  # noqa: E731
    ops.sgd_momentum_multi(group("p"), group("g"), group("v"), 0.01, 0.9,
                           group("s") if s["case"]["bf16_copy"] else None)
    return _give(s, *(k for k in s if k[0] in "pvs" and k[1:].isdigit()))


_RUN = {"mlp_step": _mlp_step, "linear": _linear, "head": _head, "conv": _conv, "layernorm": _layernorm,
        "cross_entropy": _cross_entropy, "sgd": _sgd}


def run(state):
    return _RUN[state["case"]["kind"]](state)


def work(case):
    c, kind = case, case["kind"]
    if kind == "mlp_step":
        b, d0, d1, d2, n = (c[k] for k in ("batch", "inputs", "hidden1", "hidden2", "classes"))
        p = d0 * d1 + d1 * d2 + d2 * n + n
        # The first layer's input needs no gradient.
        return {"bytes": 4 * (b * d0 + 4 * p) + 8 * b, "flops": 2 * b * (2 * d0 * d1 + 3 * d1 * d2 + 3 * d2 * n) + 4 * p}
    if kind in ("linear", "head"):
        b, i, o, e = c["batch"], c["inputs"], c["outputs"], 2 if c["dtype"] == "bf16" else 4
        # x, w, bias in, y out; dy and the saved activation (or the labels)
        # in, dx, dw and db out.
        n = e * (2 * b * i + o * i + b * o) + 4 * (o * i + 2 * o)
        return {"bytes": n + (e * 2 * b * o if kind == "linear" else 8 * b), "flops": 6 * b * i * o}
    if kind == "conv":
        n, ci, h, co, k, p = c["batch"], c["channels"], c["size"], c["filters"], c["kernel"], _conv_out(c) ** 2
        return {"bytes": 4 * (2 * n * ci * h * h + 3 * n * co * p + 2 * co * ci * k * k + 2 * co),
                "flops": 6 * n * co * p * ci * k * k}
    if kind == "layernorm":
        r, k = c["rows"], c["cols"]
        return {"bytes": 4 * (4 * r * k + 2 * r + 4 * k), "flops": 24 * r * k}
    if kind == "cross_entropy":
        r, k = c["rows"], c["cols"]
        return {"bytes": 8 * r * k + 8 * r, "flops": 6 * r * k}
    n, w = sum((i + 1) * o for i, o in _widths(c)), sum(i * o for i, o in _widths(c))
    return {"bytes": 20 * n + (2 * w if c["bf16_copy"] else 0), "flops": 4 * n}


def tolerance(case):
    kind = case["kind"]
    if case.get("dtype") == "bf16":
        # One rounding to bf16 of y and dx (2^-9 at most, 1.7e-3 in the mean).
        return {"rel": 7e-3}
    if kind == "sgd":
        # Two rounded multiply-adds a value; the bf16 copy one rounding more.
        return {"rel": 7e-3 if case["bf16_copy"] else 2e-7}
    # fp32 sums of up to 10^5 terms: 1e-7 to 6e-7 against 64 bits, and other
    # orders of the sums up to twice that apart.
    return {"rel": 4e-6}


def exact(case, seed):
    t = _inputs(dict(case), seed)
    d = {k: v.double() if v.is_floating_point() else v for k, v in t.items()}
    return _EXACT[case["kind"]](case, d)


def _exact_loss(z, t):
    b = z.shape[0]
    logp = F.log_softmax(z, 1)
    loss = -logp.gather(1, t[:, None]).mean().reshape(1)
    dz = (logp.exp() - F.one_hot(t, z.shape[1])) / b
    return loss, dz


def _exact_mlp(c, d):
    h1 = (d["x"] @ d["w1"].T).relu()
    h2 = (h1 @ d["w2"].T).relu()
    z = h2 @ d["w3"].T + d["b3"]
    loss, dz = _exact_loss(z, d["t"])
    g = {"w3": dz.T @ h2, "b3": dz.sum(0)}
    dh2 = dz @ d["w3"] * (h2 > 0)
    g["w2"] = dh2.T @ h1
    dh1 = dh2 @ d["w2"] * (h1 > 0)
    g["w1"] = dh1.T @ d["x"]
    v = {k: 0.9 * d["v" + (k[1:] if k != "b3" else "b3")] + g[k] for k in g}
    out = {"loss": loss, "z": z, "v1": v["w1"]}
    for k in g:
        out["d" + k], out[k] = g[k], d[k] - 0.01 * v[k]
    return out


def _exact_linear(c, d):
    dz = d["dy"] * (d["y_saved"] > 0)
    return {"y": (d["x"] @ d["w"].T + d["b"]).relu(), "dx": dz @ d["w"], "dw": dz.T @ d["x"], "db": dz.sum(0)}


def _exact_head(c, d):
    y = d["x"] @ d["w"].T + d["b"]
    loss, dz = _exact_loss(y, d["t"])
    return {"y": y, "loss": loss, "dx": dz @ d["w"], "dw": dz.T @ d["x"], "db": dz.sum(0)}


def _exact_conv(c, d):
    k, h, n, p = c["kernel"], c["size"], c["batch"], _conv_out(c)
    geo = {"kernel_size": k, "padding": c["pad"], "stride": c["stride"]}
    w = d["w"].flatten(1)
    dz = (d["dy"] * (d["y_saved"] > 0)).flatten(2)
    y, dx, dw = [], [], torch.zeros_like(w)
    for i in range(n):
        col = F.unfold(d["x"][i:i + 1], **geo)[0]
        y.append((w @ col + d["b"][:, None]).relu())
        dw += dz[i] @ col.T
        dx.append(F.fold((w.T @ dz[i])[None], (h, h), **geo)[0])
    return {"y": torch.stack(y).reshape(n, -1, p, p), "dx": torch.stack(dx), "dw": dw.reshape(d["w"].shape),
            "db": dz.sum((0, 2))}


def _exact_layernorm(c, d):
    x, dy = d["x"], d["dy"]
    mean = x.mean(1, keepdim=True)
    rstd = ((x - mean).square().mean(1, keepdim=True) + 1e-5).rsqrt()
    xh = (x - mean) * rstd
    g = dy * d["gamma"]
    dx = rstd * (g - g.mean(1, keepdim=True) - xh * (g * xh).mean(1, keepdim=True))
    return {"y": xh * d["gamma"] + d["beta"], "mean": mean[:, 0], "rstd": rstd[:, 0], "dx": dx,
            "dgamma": (dy * xh).sum(0), "dbeta": dy.sum(0)}


def _exact_cross_entropy(c, d):
    loss, dz = _exact_loss(d["x"], d["t"])
    return {"loss": loss, "dx": dz}


def _exact_sgd(c, d):
    out = {}
    for i in range(2 * len(_widths(c))):
        v = 0.9 * d["v%d" % i] + d["g%d" % i]
        out["v%d" % i], out["p%d" % i] = v, d["p%d" % i] - 0.01 * v
        if c["bf16_copy"] and i % 2 == 0:
            out["s%d" % i] = out["p%d" % i]
    return out


_EXACT = {"mlp_step": _exact_mlp, "linear": _exact_linear, "head": _exact_head, "conv": _exact_conv,
          "layernorm": _exact_layernorm, "cross_entropy": _exact_cross_entropy, "sgd": _exact_sgd}
