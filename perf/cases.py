"""The calls whose speed this package is measured by, and how their results are checked.

Every case goes through the package's public entry points (gemm, bmm, exact_sum, conv2d and its
two gradients, and the Linear and Conv2d layers with autograd), on float32 GPU tensors. Results
are defined bit for bit (one rounding of an exact sum of fixed-point products), so every case's
tolerance is "exact"; exact() gives the real-number result, which the fixed-point rounding of the
inputs leaves about 1e-6 away at S = 3 slices, 1e-4 at S = 2 and 1e-2 at S = 1.

A case is a dict of plain values; its "kind" says which call it is:
  gemm     C[M, N] = op(A) op(B), S slices, ta / tb as in gemm()
  linear   one Linear layer, forward and backward: y, dx, dw, db ([rows, k] -> [rows, n])
  heads    one attention layer's two batched products, scores = Q K^T and P V per head, with the
           heads read in place from [tokens, heads * size] activations
  conv     one convolution: pass "fwd", "dw", "dx", or "step" (a Conv2d layer, all of them and
           the bias gradient)
  sum      out[b] = exact sum of x[a, b, c] over a and c
"""
import torch

import bit_reproducible_training_amd as rg

KINDS = ("gemm", "linear", "heads", "conv", "sum")


def _conv(name, what, n, c, h, w, f, kh, kw, stride, pad):
    return {"name": name, "kind": "conv", "pass": what, "n": n, "c": c, "h": h, "w": w, "f": f,
            "kh": kh, "kw": kw, "stride": stride, "pad": pad}


def listed():
    return [
        # A small square product: what a script's first calls and small models are made of;
        # launch latency and the host's work per call count.
        {"name": "gemm_256", "kind": "gemm", "m": 256, "n": 256, "k": 256, "ta": False, "tb": False, "s": 3},
        # The benchmark's product: the largest dense square GEMM users quote.
        {"name": "gemm_4096", "kind": "gemm", "m": 4096, "n": 4096, "k": 4096, "ta": False, "tb": False, "s": 3},
        # Odd sizes and two slices (14-bit inputs, the faster option), op(A) transposed: a weight
        # gradient of a layer whose widths are not multiples of anything.
        {"name": "gemm_ragged_s2", "kind": "gemm", "m": 1003, "n": 3001, "k": 2049, "ta": True, "tb": False, "s": 2},
        # GPT-2 small's vocabulary projection over one 1024-token sequence: a wide ragged output.
        {"name": "lm_head_1024", "kind": "gemm", "m": 1024, "n": 50257, "k": 768, "ta": False, "tb": True, "s": 3},
        # A training step of GPT-2 small's QKV layer on one sequence of 1024 tokens.
        {"name": "linear_qkv_1024", "kind": "linear", "rows": 1024, "k": 768, "n": 2304},
        # A training step of its MLP's first layer on a batch of 8192 tokens.
        {"name": "linear_mlp_8192", "kind": "linear", "rows": 8192, "k": 768, "n": 3072},
        # Its attention products, 12 heads of 64 over 1024 tokens.
        {"name": "heads_1024", "kind": "heads", "tokens": 1024, "heads": 12, "size": 64},
        # LeNet-5's second convolution at batch 100, a whole training step of the layer.
        _conv("lenet_conv2_step", "step", 100, 6, 14, 14, 16, 5, 5, 1, 0),
        # A ResNet's first-stage 3x3 convolution at batch 32, each direction for itself.
        _conv("resnet_conv_fwd", "fwd", 32, 64, 56, 56, 64, 3, 3, 1, 1),
        _conv("resnet_conv_dw", "dw", 32, 64, 56, 56, 64, 3, 3, 1, 1),
        _conv("resnet_conv_dx", "dx", 32, 64, 56, 56, 64, 3, 3, 1, 1),
        # The bias gradient of a convolution over 256 images (64 channels of 56x56).
        {"name": "sum_conv_bias", "kind": "sum", "a": 256, "b": 64, "c": 3136},
    ]


def _log(rng, lo, hi):
    """A whole number spread over [lo, hi] by its logarithm."""
    return max(lo, min(hi, int(round(lo * (hi / lo) ** rng.random()))))


def _draw_conv(rng):
    what = rng.choice(["fwd", "dw", "dx", "step"])
    k = rng.choice([1, 3, 3, 3, 5, 7])
    return _conv(None, what, _log(rng, 1, 128), _log(rng, 1, 256), _log(rng, 8, 112), _log(rng, 8, 112),
                 _log(rng, 4, 256), k, k, rng.choice([1, 1, 2]), rng.choice([0, k // 2]))


def _draw_gemm(rng):
    return {"kind": "gemm", "m": _log(rng, 1, 8192), "n": _log(rng, 1, 50257), "k": _log(rng, 16, 16384),
            "ta": rng.random() < 0.5, "tb": rng.random() < 0.5, "s": rng.choice([1, 2, 3, 3, 3])}


def _draw_linear(rng):
    return {"kind": "linear", "rows": _log(rng, 1, 8192), "k": _log(rng, 64, 4096), "n": _log(rng, 10, 4096)}


def _draw_heads(rng):
    return {"kind": "heads", "tokens": _log(rng, 33, 2048), "heads": rng.randint(1, 16),
            "size": rng.choice([32, 64, 64, 80, 128])}


def _draw_sum(rng):
    c = rng.choice([1, _log(rng, 2, 8192)])
    return {"kind": "sum", "a": _log(rng, 1, 8192), "b": _log(rng, 1, 16384), "c": c}


def draw(rng):
    """One more case of the same ranges, at most a third of the largest listed cases' work."""
    makers = (_draw_gemm, _draw_linear, _draw_heads, _draw_conv, _draw_sum)
    while True:
        case = rng.choice(makers)(rng)
        case.pop("name", None)
        w = work(case)
        if case["kind"] == "conv":
            oh, ow = _out_size(case)
            if case["n"] * oh * ow * case["c"] * case["kh"] * case["kw"] > 6e7:
                continue  # more unfolded input than the listed layer has
        if 1e4 < w["bytes"] < 3e8 and w["flops"] < 4e10:
            return case


def _out_size(case):
    return ((case["h"] + 2 * case["pad"] - case["kh"]) // case["stride"] + 1,
            (case["w"] + 2 * case["pad"] - case["kw"]) // case["stride"] + 1)


def work(case):
    """Bytes (each input read once, each output written once) and multiply-adds (two operations
    each) of one pass."""
    kind = case["kind"]
    if kind == "gemm":
        m, n, k = case["m"], case["n"], case["k"]
        return {"bytes": 4.0 * (m * k + k * n + m * n), "flops": 2.0 * m * n * k}
    if kind == "linear":
        m, n, k = case["rows"], case["n"], case["k"]
        return {"bytes": 4.0 * (2 * m * k + 2 * n * k + 2 * m * n + 2 * n), "flops": 6.0 * m * n * k + m * n}
    if kind == "heads":
        t, h, d = case["tokens"], case["heads"], case["size"]
        return {"bytes": 4.0 * (4 * t * h * d + 2 * h * t * t), "flops": 4.0 * h * t * t * d}
    if kind == "conv":
        oh, ow = _out_size(case)
        x = case["n"] * case["c"] * case["h"] * case["w"]
        y = case["n"] * case["f"] * oh * ow
        w = case["f"] * case["c"] * case["kh"] * case["kw"]
        one = 2.0 * y * case["c"] * case["kh"] * case["kw"]
        if case["pass"] == "step":
            return {"bytes": 4.0 * (2 * x + 2 * y + 2 * w), "flops": 3 * one + y}
        return {"bytes": 4.0 * (x + y + w), "flops": one}
    n = case["a"] * case["b"] * case["c"]
    return {"bytes": 4.0 * (n + case["b"]), "flops": 1.0 * n}


def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _inputs(case, seed):
    """The case's tensors by name: activations N(0, 1), weights and gradients of the scales that
    training meets."""
    g = _generator(seed)

    def normal(*shape, scale=1.0):
        return torch.randn(*shape, generator=g, device="cuda") * scale

    kind = case["kind"]
    if kind == "gemm":
        m, n, k = case["m"], case["n"], case["k"]
        return {"A": normal(*((k, m) if case["ta"] else (m, k))),
                "B": normal(*((n, k) if case["tb"] else (k, n)))}
    if kind == "linear":
        m, n, k = case["rows"], case["n"], case["k"]
        return {"x": normal(m, k), "weight": normal(n, k, scale=0.02), "bias": normal(n, scale=0.02),
                "dy": normal(m, n, scale=1e-3)}
    if kind == "heads":
        t, h, d = case["tokens"], case["heads"], case["size"]
        p = torch.softmax(normal(h, t, t), dim=-1)
        return {"q": normal(t, h * d), "k": normal(t, h * d), "v": normal(t, h * d), "p": p}
    if kind == "conv":
        oh, ow = _out_size(case)
        return {"x": normal(case["n"], case["c"], case["h"], case["w"]),
                "weight": normal(case["f"], case["c"], case["kh"], case["kw"], scale=0.1),
                "bias": normal(case["f"], scale=0.1),
                "dy": normal(case["n"], case["f"], oh, ow, scale=1e-3)}
    return {"x": normal(case["a"], case["b"], case["c"])}


def _heads_of(t, case):
    """[tokens, heads * size] as one [tokens, size] view per head: [heads, tokens, size]."""
    return t.view(case["tokens"], case["heads"], case["size"]).transpose(0, 1)


def prepare(case, seed):
    state = dict(_inputs(case, seed), case=case)
    if case["kind"] == "linear":
        layer = rg.Linear(case["k"], case["n"], device="cuda")
    elif case["kind"] == "conv" and case["pass"] == "step":
        layer = rg.Conv2d(case["c"], case["f"], (case["kh"], case["kw"]), stride=case["stride"],
                          padding=case["pad"], device="cuda")
    else:
        return state
    with torch.no_grad():
        layer.weight.copy_(state.pop("weight"))
        layer.bias.copy_(state.pop("bias"))
    state["x"].requires_grad_(True)
    state["layer"] = layer
    return state


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "gemm":
        return rg.gemm(state["A"], state["B"], case["m"], case["n"], case["k"], case["ta"],
                       case["tb"], case["s"])
    if kind == "linear" or (kind == "conv" and case["pass"] == "step"):
        layer = state["layer"]
        y = layer(state["x"])
        dx, dw, db = torch.autograd.grad(y, (state["x"], layer.weight, layer.bias), state["dy"])
        return {"y": y.detach(), "dx": dx, "dw": dw, "db": db}
    if kind == "heads":
        scores = rg.bmm(_heads_of(state["q"], case), _heads_of(state["k"], case), tb=True)
        mixed = rg.bmm(state["p"], _heads_of(state["v"], case))
        return {"scores": scores, "mixed": mixed}
    if kind == "conv":
        s, p = case["stride"], case["pad"]
        if case["pass"] == "fwd":
            return rg.conv2d(state["x"], state["weight"], s, s, p, p)
        if case["pass"] == "dw":
            return rg.conv2d_grad_weight(state["dy"], state["x"], case["kh"], case["kw"], s, s, p, p)
        shape = [case["n"], case["c"], case["h"], case["w"]]
        return rg.conv2d_grad_input(state["dy"], state["weight"], shape, s, s, p, p)
    return rg.exact_sum(state["x"], case["a"], case["b"], case["c"])


def tolerance(case):
    """The result's bits are the definition's, whatever the kernels, tiles and splits."""
    return "exact"


def _exact_conv(case, t, what):
    """The forward pass or a gradient through the unfolded windows, one image at a time."""
    n, f = case["n"], case["f"]
    kernel = (case["kh"], case["kw"])
    how = {"stride": case["stride"], "padding": case["pad"]}
    wmat = t["weight"].view(f, -1)
    dy = t["dy"].view(n, f, -1)
    if what == "dx":
        wt = wmat.t().contiguous()
        return torch.cat([torch.nn.functional.fold((wt @ dy[i]).unsqueeze(0), (case["h"], case["w"]), kernel, **how)
                          for i in range(n)])
    if what == "dw":
        total = torch.zeros_like(wmat)
        for i in range(n):
            cols = torch.nn.functional.unfold(t["x"][i:i + 1], kernel, **how)[0]
            total += dy[i] @ cols.t().contiguous()
        return total.view_as(t["weight"])
    oh, ow = _out_size(case)
    return torch.stack([(wmat @ torch.nn.functional.unfold(t["x"][i:i + 1], kernel, **how)[0]).view(f, oh, ow)
                        for i in range(n)])


def exact(case, seed):
    kind = case["kind"]
    t = {k: v.double() for k, v in _inputs(case, seed).items()}
    if kind == "gemm":
        a = t["A"].t().contiguous() if case["ta"] else t["A"]
        b = t["B"].t().contiguous() if case["tb"] else t["B"]
        return a @ b
    if kind == "linear":
        return {"y": t["x"] @ t["weight"].t().contiguous() + t["bias"], "dx": t["dy"] @ t["weight"],
                "dw": t["dy"].t().contiguous() @ t["x"], "db": t["dy"].sum(0)}
    if kind == "heads":
        q, k, v = (_heads_of(t[name], case).contiguous() for name in "qkv")
        return {"scores": torch.stack([q[h] @ k[h].t().contiguous() for h in range(case["heads"])]),
                "mixed": torch.stack([t["p"][h] @ v[h] for h in range(case["heads"])])}
    if kind == "conv":
        if case["pass"] != "step":
            return _exact_conv(case, t, case["pass"])
        return {"y": _exact_conv(case, t, "fwd") + t["bias"].view(1, -1, 1, 1),
                "dx": _exact_conv(case, t, "dx"), "dw": _exact_conv(case, t, "dw"),
                "db": t["dy"].sum((0, 2, 3))}
    return t["x"].sum((0, 2))
