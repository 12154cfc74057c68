"""The workloads that the performance of this library is judged on.

Each case is one training pass of a layer (forward and backward through
``thot_amd.ops``), or a whole training step of one of the host models
(``thot_amd._nott_host``), as a training program runs it.  ``listed()`` names
a dozen; ``draw()`` gives further cases of the same kinds over the same
ranges: batches from a few samples up, widths and lengths that are whole tiles
and ones that are not, fp32 and bf16, with the options that layers are built
with (bias, fused ReLU, causal masks, label smoothing, a residual input).
"""
import math

import torch
import torch.nn.functional as F

from thot_amd import ops

_DT = {"f32": torch.float32, "bf16": torch.bfloat16}


def listed():
    return [
        # The small CNN's whole training step (forward, loss, backward, Adam)
        # at its usual batch: about thirty dependent launches of a few
        # microseconds, so launches and latency are what counts.
        {"name": "small_cnn_step_f32", "kind": "small_cnn", "batch": 64},
        # ResNet-18's whole training step in fp32 (the reference's arithmetic).
        {"name": "resnet18_step_f32", "kind": "resnet18", "batch": 64},
        # The classifier head of ResNet-18: the smallest single layer call.
        {"name": "head_f32", "kind": "linear", "dtype": "f32", "m": 64, "kin": 512, "nout": 1000, "relu": False},
        # The packed q/k/v projection of multi-head attention, 8 x 1024 tokens.
        {"name": "projection_bf16", "kind": "linear", "dtype": "bf16", "m": 8192, "kin": 1024, "nout": 3072,
         "relu": False},
        # A feed-forward layer on 8 sequences of 197 tokens: the token count
        # is no multiple of any tile.
        {"name": "ffn_ragged_bf16", "kind": "linear", "dtype": "bf16", "m": 1576, "kin": 768, "nout": 3072,
         "relu": True},
        # The benchmark's convolution layer.
        {"name": "conv3x3_bf16", "kind": "conv", "dtype": "bf16", "n": 128, "c": 64, "h": 56, "w": 56, "k": 128,
         "r": 3, "stride": 1, "bias": False, "relu": False},
        # A down-sampling convolution, the entry of ResNet-18's third stage.
        {"name": "conv3x3_s2_bf16", "kind": "conv", "dtype": "bf16", "n": 64, "c": 128, "h": 28, "w": 28, "k": 256,
         "r": 3, "stride": 2, "bias": False, "relu": False},
        # The benchmark's attention core, q/k/v as the packed projection leaves them.
        {"name": "attention_bf16", "kind": "attention", "dtype": "bf16", "b": 8, "h": 16, "t": 1024, "s": 1024,
         "dh": 64, "causal": True, "token_major": True},
        # Wide heads on sequences that end inside a tile.
        {"name": "attention_wide_bf16", "kind": "attention", "dtype": "bf16", "b": 4, "h": 8, "t": 1000, "s": 1000,
         "dh": 128, "causal": False, "token_major": False},
        # The LayerNorm of a wide transformer.
        {"name": "layernorm_bf16", "kind": "layernorm", "dtype": "bf16", "rows": 4096, "d": 4096},
        # The last BatchNorm of a residual branch: skip addition and ReLU with it.
        {"name": "batchnorm_bf16", "kind": "batchnorm", "dtype": "bf16", "n": 64, "c": 128, "h": 28, "w": 28,
         "residual": True},
        # Softmax cross-entropy over a vocabulary whose rows are not 16-byte aligned.
        {"name": "xent_f32", "kind": "xent", "dtype": "f32", "n": 4096, "c": 50257, "smoothing": 0.0},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _size(rng, lo, hi):
    """Spread over the logarithm; half whole 64s, a quarter whole 8s, a quarter any."""
    v, kind = _log(rng, lo, hi), rng.random()
    step = 64 if kind < 0.5 else 8 if kind < 0.75 else 1
    return max(lo, min(hi, v // step * step if v >= step else v))


def _draw_conv(rng):
    dtype = rng.choice(["bf16", "bf16", "f32"])
    first = rng.random() < 0.12           # a network's first layer
    r, stride = rng.choice([(3, 1), (5, 1), (7, 2)] if first else
                           [(3, 1), (3, 1), (3, 1), (3, 2), (3, 2), (1, 1), (1, 2), (5, 1)])
    c = rng.choice([1, 3]) if first else rng.choice([16, 24, 32, 48, 64, 64, 96, 128, 128, 256, 512])
    k = rng.choice([32, 64]) if first else rng.choice([16, 32, 48, 64, 64, 96, 128, 128, 256, 512])
    h = rng.choice([28, 32, 64, 112, 224]) if first else rng.choice([7, 8, 13, 14, 16, 28, 28, 30, 32, 35, 56, 56, 64])
    w = h if rng.random() < 0.85 else h + rng.choice([1, 4, 8])
    p = stride
    flops = 6 * c * k * r * r * (-(-h // p)) * (-(-w // p))
    most = min(128, max(1, int((2.5e11 if dtype == "bf16" else 6e10) / flops)), max(1, int(6e7 / (max(c, k) * h * w))))
    return {"kind": "conv", "dtype": dtype, "n": _log(rng, min(8, most), most), "c": c, "h": h, "w": w, "k": k, "r": r,
            "stride": stride, "bias": rng.random() < 0.4, "relu": rng.random() < 0.4}


def _draw_linear(rng):
    dtype = rng.choice(["bf16", "bf16", "f32"])
    kin, nout = _size(rng, 64, 4096), rng.choice([10, 100, 1000, 0, 0, 0, 0, 0]) or _size(rng, 64, 4096)
    most = min(16384, max(32, int((2.5e11 if dtype == "bf16" else 5e10) / (6 * kin * nout))))
    return {"kind": "linear", "dtype": dtype, "m": _size(rng, 16, most), "kin": kin, "nout": nout,
            "relu": rng.random() < 0.4}


def _draw_attention(rng):
    dtype = rng.choice(["bf16", "bf16", "bf16", "f32"])
    dh = rng.choice([32, 40, 64, 64, 64, 80, 96, 128] if dtype == "bf16" else [32, 48, 64])
    t = _size(rng, 32, 2048)
    causal, token_major = rng.random() < 0.5, rng.random() < 0.5
    s = t if causal or token_major or rng.random() < 0.7 else _size(rng, 32, 2048)
    most = max(1, int((1.2e11 if dtype == "bf16" else 2e10) / (14 * t * s * dh)))
    h = rng.choice([4, 8, 12, 16])
    b = _log(rng, 1, max(1, min(32, most // h)))
    return {"kind": "attention", "dtype": dtype, "b": b, "h": min(h, most), "t": t, "s": s, "dh": dh, "causal": causal,
            "token_major": token_major}


def _draw_layernorm(rng):
    d = _size(rng, 64, 8192)
    return {"kind": "layernorm", "dtype": rng.choice(["bf16", "f32"]), "rows": _log(rng, 64, min(32768, 60_000_000 // d)),
            "d": d}


def _draw_batchnorm(rng):
    c, h = rng.choice([16, 32, 64, 96, 128, 256, 512]), rng.choice([7, 13, 14, 28, 35, 56, 112])
    return {"kind": "batchnorm", "dtype": rng.choice(["bf16", "f32"]),
            "n": _log(rng, 4, min(128, max(8, 60_000_000 // (c * h * h)))), "c": c, "h": h, "w": h,
            "residual": rng.random() < 0.5}


def _draw_xent(rng):
    c = rng.choice([0, 0, 10, 100, 1000, 32000, 50257, 128256]) or _size(rng, 10, 150000)
    return {"kind": "xent", "dtype": rng.choice(["bf16", "f32"]), "n": _log(rng, 64, min(16384, 200_000_000 // c)), "c": c,
            "smoothing": rng.choice([0.0, 0.0, 0.1])}


def _draw_small_cnn(rng):
    return {"kind": "small_cnn", "batch": _log(rng, 4, 512)}


def draw(rng):
    return rng.choice([_draw_conv, _draw_conv, _draw_conv, _draw_linear, _draw_linear, _draw_attention, _draw_attention,
                       _draw_layernorm, _draw_batchnorm, _draw_xent, _draw_small_cnn])(rng)


# ------------------------------------------------------------------ inputs
class _Maker:
    def __init__(self, seed):
        self.g = torch.Generator(device="cuda").manual_seed(seed)

    def normal(self, *shape, std=1.0, mean=0.0, dtype=torch.float32):
        return torch.randn(shape, generator=self.g, device="cuda").mul_(std).add_(mean).to(dtype)

    def labels(self, n, c):
        return torch.randint(0, c, (n,), generator=self.g, device="cuda")


def _inputs(case, seed):
    """The tensors of a case, made from the seed alone."""
    mk, kind = _Maker(seed), case["kind"]
    if kind == "small_cnn":
        return {"x": mk.normal(case["batch"], 1, 28, 28), "labels": mk.labels(case["batch"], 10)}
    if kind == "resnet18":
        return {"x": mk.normal(case["batch"], 3, 224, 224), "labels": mk.labels(case["batch"], 1000)}
    dt = _DT[case["dtype"]]
    if kind == "linear":
        m, kin, nout = case["m"], case["kin"], case["nout"]
        x = mk.normal(m, kin, dtype=dt)
        return {"x": torch.relu(x) if case["relu"] else x, "w": mk.normal(nout, kin, std=kin ** -0.5, dtype=dt),
                "b": mk.normal(nout, std=0.1), "dy": mk.normal(m, nout, std=1e-2, dtype=dt)}
    if kind == "conv":
        d = _conv(case)
        xs, ys = ops._conv_shapes(d)
        return {"x": mk.normal(*xs, dtype=dt), "w": mk.normal(d.k, d.c, d.r, d.s, std=(d.c * d.r * d.s) ** -0.5, dtype=dt),
                "b": mk.normal(d.k, std=0.1) if case["bias"] else None, "dy": mk.normal(*ys, std=1e-2, dtype=dt)}
    if kind == "attention":
        b, h, t, s, dh = (case[n] for n in ("b", "h", "t", "s", "dh"))
        if case["token_major"]:
            return {"qkv": mk.normal(b, t, 3, h, dh, dtype=dt), "do": mk.normal(b, t, h, dh, std=1e-2, dtype=dt)}
        return {"q": mk.normal(b, h, t, dh, dtype=dt), "k": mk.normal(b, h, s, dh, dtype=dt),
                "v": mk.normal(b, h, s, dh, dtype=dt), "do": mk.normal(b, h, t, dh, std=1e-2, dtype=dt)}
    if kind == "layernorm":
        r, d = case["rows"], case["d"]
        return {"x": mk.normal(r, d, std=1.5, mean=0.3, dtype=dt), "gamma": mk.normal(d, std=0.1, mean=1.0, dtype=dt),
                "beta": mk.normal(d, std=0.1, dtype=dt), "dy": mk.normal(r, d, std=1e-2, dtype=dt)}
    if kind == "batchnorm":
        s = (case["n"], case["c"], case["h"], case["w"])
        return {"x": mk.normal(*s, std=1.5, mean=0.3, dtype=dt), "gamma": mk.normal(s[1], std=0.1, mean=1.0),
                "beta": mk.normal(s[1], std=0.1), "dy": mk.normal(*s, std=1e-2, dtype=dt),
                "res": mk.normal(*s, dtype=dt) if case["residual"] else None}
    n, c = case["n"], case["c"]
    labels = mk.labels(n, c)
    if n >= 64:
        labels[::61] = -100               # padding rows that the loss ignores
    return {"logits": mk.normal(n, c, std=2.0, dtype=dt), "labels": labels}


def _conv(case):
    p = (case["r"] - 1) // 2
    return ops.conv_desc((case["n"], case["c"], case["h"], case["w"]), (case["k"], case["c"], case["r"], case["r"]),
                         stride=(case["stride"],) * 2, padding=(p, p))


def prepare(case, seed):
    state = dict(_inputs(case, seed), case=case)
    kind = case["kind"]
    if kind in ("small_cnn", "resnet18"):
        from thot_amd import _nott_host
        if kind == "small_cnn":
            state["trainer"] = _nott_host.SmallCNNTrainer(device=0, seed=seed % 1000, lr=1e-4)
        else:
            state["trainer"] = _nott_host.ResNet18Trainer(device=0, seed=seed % 1000, bf16=False, lr=1e-4)
        # one pass before the loop, as capture() makes: it leaves the model as it
        # was, and the gradients exist after it (views that the trainer keeps)
        state["trainer"].warmup(state["x"], state["labels"], 1)
        state["grads"] = state["trainer"].grads()
    elif kind == "conv":
        state["desc"] = _conv(case)
    elif kind == "attention":
        b, h, t, s, dh = (case[n] for n in ("b", "h", "t", "s", "dh"))
        if case["token_major"]:
            state["desc"] = ops.attn_desc(b, h, t, s, dh, case["causal"], token_major=True, ld_qkv=3 * h * dh)
        else:
            state["desc"] = ops.attn_desc(b, h, t, s, dh, case["causal"])
    elif kind == "batchnorm":
        state["running_mean"] = torch.zeros(case["c"], device="cuda")
        state["running_var"] = torch.ones(case["c"], device="cuda")
    return state


# -------------------------------------------------------------------- pass
def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind in ("small_cnn", "resnet18"):
        # One turn of the training loop: the optimizer takes the gradients of
        # the turn before (none before the first) and clears them, then
        # forward, loss and backward.
        tr = state["trainer"]
        tr.optimizer_step()
        return {"loss": tr.forward_backward(state["x"], state["labels"]), "grads": state["grads"]}
    if kind == "linear":
        y = ops.linear_fwd(state["x"], state["w"], state["b"], relu=case["relu"])
        dx, dw, db = ops.linear_bwd(state["dy"], state["x"], state["w"], relu_input=case["relu"])
        return {"y": y, "dx": dx, "dw": dw, "db": db}
    if kind == "conv":
        d = state["desc"]
        out = {"y": ops.conv2d_fwd(state["x"], state["w"], state["b"], d, relu=case["relu"])}
        out["dw"], db = ops.conv2d_bwd_weight(state["x"], state["dy"], d, need_db=case["bias"])
        if case["bias"]:
            out["db"] = db
        if case["c"] > 3:                 # a first layer has no input gradient
            out["dx"] = ops.conv2d_bwd_data(state["dy"], state["w"], d)
        return out
    if kind == "attention":
        d = state["desc"]
        if case["token_major"]:
            q, k, v = state["qkv"].unbind(2)
            o, lse = ops.attention_fwd(q, k, v, d)
            dqkv = torch.empty_like(state["qkv"])
            ops.attention_bwd(q, k, v, o, state["do"], lse, d, out=dqkv.unbind(2))
            return {"o": o, "lse": lse, "dqkv": dqkv}
        q, k, v = state["q"], state["k"], state["v"]
        o, lse = ops.attention_fwd(q, k, v, d)
        dq, dk, dv = ops.attention_bwd(q, k, v, o, state["do"], lse, d)
        return {"o": o, "lse": lse, "dq": dq, "dk": dk, "dv": dv}
    if kind == "layernorm":
        y, mean, rstd = ops.layernorm_fwd(state["x"], state["gamma"], state["beta"])
        dx, dg, db = ops.layernorm_bwd(state["x"], state["dy"], mean, rstd, state["gamma"])
        return {"y": y, "mean": mean, "rstd": rstd, "dx": dx, "dgamma": dg, "dbeta": db}
    if kind == "batchnorm":
        x, g, b, rm, rv = (state[n] for n in ("x", "gamma", "beta", "running_mean", "running_var"))
        # the branch's last BatchNorm takes the skip addition and the final ReLU,
        # whose backward the next block's fork has already applied to dy
        y, mean, rstd = ops.batchnorm2d_fwd(x, g, b, 1e-5, 0.1, rm, rv, residual=state["res"], relu=case["residual"])
        dx, dg, db = ops.batchnorm2d_bwd(x, state["dy"], mean, rstd, g)
        return {"y": y, "mean": mean, "rstd": rstd, "running_mean": rm, "running_var": rv, "dx": dx, "dgamma": dg,
                "dbeta": db}
    dl, loss = ops.softmax_xent_bwd(state["logits"], state["labels"], label_smoothing=case["smoothing"])
    return {"dlogits": dl, "loss": loss}


# -------------------------------------------------------------------- work
# Multiply-adds of one forward pass per sample, and parameters, of the two models.
_MODEL = {"small_cnn": (9 * 32 * 784 + 9 * 32 * 64 * 196 + 3136 * 128 + 1280, 421_642),
          "resnet18": (1_814_073_344, 11_689_512)}


def work(case):
    kind = case["kind"]
    if kind in _MODEL:
        macs, params = _MODEL[kind]
        pixels = 784 if kind == "small_cnn" else 3 * 224 * 224
        # forward and both gradients; the parameters' update reads p, g, m, v and writes p, m, v and the new g
        return {"bytes": 32 * params + 4 * case["batch"] * pixels, "flops": 6 * macs * case["batch"]}
    e = 2 if case["dtype"] == "bf16" else 4
    if kind == "linear":
        m, kin, nout = case["m"], case["kin"], case["nout"]
        return {"bytes": e * (2 * m * kin + 2 * m * nout + nout * kin) + 4 * (nout * kin + 2 * nout),
                "flops": 6 * m * kin * nout}
    if kind == "conv":
        d = _conv(case)
        xs, ys = (math.prod(v) for v in ops._conv_shapes(d))
        ws = d.k * d.c * d.r * d.s
        dx = case["c"] > 3
        return {"bytes": e * (xs * (2 if dx else 1) + 2 * ys + ws) + 4 * ws + (8 * d.k if case["bias"] else 0),
                "flops": (6 if dx else 4) * ys * d.c * d.r * d.s}
    if kind == "attention":
        b, h, t, s, dh = (case[n] for n in ("b", "h", "t", "s", "dh"))
        pairs = sum(min(i + 1, s) for i in range(t)) if case["causal"] else t * s
        # forward 2 products; backward 5
        return {"bytes": b * h * (e * dh * (4 * t + 4 * s) + 4 * t), "flops": 14 * b * h * pairs * dh}
    if kind == "layernorm":
        r, d = case["rows"], case["d"]
        return {"bytes": e * (4 * r * d + 2 * d) + 8 * r + 8 * d, "flops": 20 * r * d}
    if kind == "batchnorm":
        n = case["n"] * case["c"] * case["h"] * case["w"]
        return {"bytes": e * n * (5 if case["residual"] else 4) + 48 * case["c"], "flops": 20 * n}
    n, c = case["n"], case["c"]
    return {"bytes": 2 * e * n * c + 8 * n, "flops": 8 * n * c}


# --------------------------------------------------------------- tolerance
def tolerance(case):
    kind = case["kind"]
    # A ReLU input within rounding of zero takes the other branch, and its
    # channel's gradients change with it (as measured against 64 bits: 3e-4 of
    # the small CNN's first layer's at batch 487, more at a smaller one; up to
    # 3e-3 of the ResNet's).
    if kind == "small_cnn":
        return {"rel": 1e-2, "max": 0.3}
    if kind == "resnet18":
        return {"rel": 2e-2, "max": 0.9}
    if case["dtype"] == "f32":
        # sums of up to 2^18 terms measure 1e-7 to 4e-7 off the 64-bit result
        return {"rel": 4e-6, "max": 1e-4}
    # one rounding of each result (1.7e-3 off the 64-bit result as measured,
    # 2.2e-3 where the probabilities of attention are rounded as well)
    return {"rel": 8e-3, "max": 4e-2}


# ------------------------------------------------------------------- exact
def exact(case, seed):
    kind = case["kind"]
    if kind == "small_cnn":
        return _head(case, seed, _model_parameters(kind, seed), "fc_6", _small_cnn_trunk)
    if kind == "resnet18":
        # the first turn's AdamW step decays the weights (there are no gradients yet)
        return _head(case, seed, _model_parameters(kind, seed), "fc_13", _resnet18_trunk, decay=1 - 1e-4 * 1e-2)
    s = {n: v.double() if v is not None and v.is_floating_point() else v for n, v in _inputs(case, seed).items()}
    if kind == "linear":
        x, w, dy = s["x"], s["w"], s["dy"]
        y, dx = x @ w.t() + s["b"], dy @ w
        if case["relu"]:
            y, dx = y.relu(), dx * (x > 0)
        return {"y": y, "dx": dx, "dw": dy.t() @ x, "db": dy.sum(0)}
    if kind == "conv":
        return _exact_conv(case, s)
    if kind == "attention":
        return _exact_attention(case, s)
    if kind == "layernorm":
        x, dy, g = s["x"], s["dy"], s["gamma"]
        mean = x.mean(1, keepdim=True)
        rstd = ((x - mean).square().mean(1, keepdim=True) + 1e-5).rsqrt()
        xh = (x - mean) * rstd
        dg = dy * g
        dx = rstd * (dg - dg.mean(1, keepdim=True) - xh * (dg * xh).mean(1, keepdim=True))
        return {"y": xh * g + s["beta"], "mean": mean[:, 0], "rstd": rstd[:, 0], "dx": dx, "dgamma": (dy * xh).sum(0),
                "dbeta": dy.sum(0)}
    if kind == "batchnorm":
        x, count = s["x"], case["n"] * case["h"] * case["w"]
        per = lambda v: v.view(1, -1, 1, 1)
        mean = x.mean((0, 2, 3))
        var = (x - per(mean)).square().mean((0, 2, 3))
        rstd = (var + 1e-5).rsqrt()
        xh = (x - per(mean)) * per(rstd)
        z, dz = xh * per(s["gamma"]) + per(s["beta"]), s["dy"]
        if case["residual"]:
            z = (z + s["res"]).relu()
        dg, db = (dz * xh).sum((0, 2, 3)), dz.sum((0, 2, 3))
        dx = per(s["gamma"] * rstd) * (dz - per(db / count) - xh * per(dg / count))
        return {"y": z, "mean": mean, "rstd": rstd, "running_mean": 0.1 * mean,
                "running_var": 0.9 + 0.1 * var * count / max(1, count - 1), "dx": dx, "dgamma": dg, "dbeta": db}
    logits, labels, eps = s["logits"], s["labels"], case["smoothing"]
    n, c = logits.shape
    used = (labels >= 0).double()
    count = used.sum()
    rows = labels.clamp(min=0)[:, None]
    lse = logits.logsumexp(1)
    loss = lse - (1 - eps) * logits.gather(1, rows)[:, 0] - eps * logits.mean(1)
    p = (logits - lse[:, None]).exp_().sub_(eps / c)
    p.scatter_add_(1, rows, torch.full_like(rows, -(1 - eps), dtype=p.dtype))
    return {"dlogits": p.mul_((used / count)[:, None]), "loss": (loss * used).sum() / count}


def _exact_conv(case, s):
    d = _conv(case)
    p, k = (case["r"] - 1) // 2, (case["r"], case["r"])
    geometry = dict(kernel_size=k, stride=case["stride"], padding=p)
    w, need_dx = s["w"].flatten(1), case["c"] > 3
    y, dx, dw = [], [], 0
    per = max(1, int(2e8 // (w.shape[1] * s["dy"][0, 0].numel())))      # images at a time
    for i in range(0, case["n"], per):
        dy = s["dy"][i:i + per].flatten(2)
        cols = F.unfold(s["x"][i:i + per], **geometry)
        y.append(torch.matmul(w, cols))
        dw = dw + torch.matmul(dy, cols.transpose(1, 2)).sum(0)
        if need_dx:
            dx.append(F.fold(torch.matmul(w.t(), dy), (case["h"], case["w"]), **geometry))
    y = torch.cat(y).view(s["dy"].shape)
    if case["bias"]:
        y = y + s["b"].view(1, -1, 1, 1)
    out = {"y": y.relu() if case["relu"] else y, "dw": dw.view(d.k, d.c, d.r, d.s)}
    if case["bias"]:
        out["db"] = s["dy"].sum((0, 2, 3))
    if need_dx:
        out["dx"] = torch.cat(dx)
    return out


def _exact_attention(case, s):
    t, m, scale = case["t"], case["s"], case["dh"] ** -0.5
    if case["token_major"]:
        q, k, v = (x.transpose(1, 2) for x in s["qkv"].unbind(2))
        do = s["do"].transpose(1, 2)
    else:
        q, k, v, do = s["q"], s["k"], s["v"], s["do"]
    got = []
    for i in range(case["b"]):
        qi, ki, vi, di = (x[i].contiguous() for x in (q, k, v, do))
        sc = qi @ ki.transpose(1, 2) * scale
        if case["causal"]:
            sc.masked_fill_(torch.ones(t, m, dtype=torch.bool, device=sc.device).triu(1), -math.inf)
        lse = sc.logsumexp(2)
        p = (sc - lse[..., None]).exp_()
        o = p @ vi
        ds = p * (di @ vi.transpose(1, 2) - (di * o).sum(2, keepdim=True))
        got.append((o, lse, ds @ ki * scale, ds.transpose(1, 2) @ qi * scale, p.transpose(1, 2) @ di))
    o, lse, dq, dk, dv = (torch.stack(x) for x in zip(*got))
    if case["token_major"]:
        return {"o": o.transpose(1, 2), "lse": lse, "dqkv": torch.stack([x.transpose(1, 2) for x in (dq, dk, dv)], 2)}
    return {"o": o, "lse": lse, "dq": dq, "dk": dk, "dv": dv}


# The whole models.  Only the loss and the last layer's gradients are given:
# below it, which branch a ReLU or a max-pool takes for inputs within rounding
# of each other decides a gradient, so its distance from 64 bits measures luck.
def _model_parameters(model, seed):
    from thot_amd import _nott_host
    return {n: v.double() for n, v in _nott_host.initial_parameters(model, seed % 1000).items()}


def _head(case, seed, p, head, trunk, decay=1.0):
    s = _inputs(case, seed)
    p = {n: v * decay for n, v in p.items()}
    with torch.no_grad():
        x = trunk(s["x"].double().cpu(), p)
    last = [p[head + n].requires_grad_() for n in (".weight", ".bias")]
    loss = F.cross_entropy(F.linear(x, *last), s["labels"].cpu())
    grads = dict.fromkeys(p)
    grads[head + ".weight"], grads[head + ".bias"] = torch.autograd.grad(loss, last)
    return {"loss": loss.detach(), "grads": grads}


def _small_cnn_trunk(x, p):
    for n in ("conv2d_0", "conv2d_2"):
        x = F.max_pool2d(F.conv2d(x, p[n + ".weight"], p[n + ".bias"], padding=1).relu(), 2)
    return F.linear(x.flatten(1), p["fc_5.weight"], p["fc_5.bias"]).relu()


def _resnet18_trunk(x, p):
    def norm(x, key):
        return F.batch_norm(x, None, None, p[key + ".weight"], p[key + ".bias"], True, 0.1, 1e-5)

    x = F.conv2d(x, p["conv2d_0.weight"], stride=2, padding=3)
    x = F.max_pool2d(norm(x, "batchnorm2d_1").relu(), 3, 2, 1)
    for i in range(8):
        key = "residual_block_%d." % (3 + i)
        down = key + "conv2d_4.weight" in p
        skip = F.conv2d(x, p[key + "conv2d_4.weight"], stride=2) if down else x
        x = norm(F.conv2d(x, p[key + "conv2d_0.weight"], stride=2 if down else 1, padding=1), key + "batchnorm2d_1")
        x = norm(F.conv2d(x.relu(), p[key + "conv2d_2.weight"], padding=1), key + "batchnorm2d_3")
        x = (x + skip).relu()
    return x.mean((2, 3))
