"""Timed cases of the framework's public entry points.

Each case is one pass through ``tracea_amd.ops`` or a captured ``tracea_amd.plan.Plan`` on tensors that are
already in device memory, with the output tensor kept by the caller, the way an inference program calls them.
``listed()`` are the named cases, ``draw()`` gives others of the same ranges.
"""
import math

import torch

from tracea_amd import capi, graph as G, ops
from tracea_amd.plan import Plan

_TYPES = {"f16": torch.float16, "bf16": torch.bfloat16, "f32": torch.float32}
_BYTES = {"f16": 2, "bf16": 2, "f32": 4}


def listed():
    return [
        # a linear layer on a handful of rows: one step of token generation, or a small batch at a network's end.
        # Bound by reading the weights once.
        {"name": "gemm_rows16", "kind": "gemm", "m": 16, "n": 4096, "k": 4096, "dtype": "bf16", "b": "nk", "epilogue": "bias"},
        # the half-precision product of the benchmark, column-major B: a linear layer on a large batch of rows
        {"name": "gemm_4096", "kind": "gemm", "m": 4096, "n": 4096, "k": 4096, "dtype": "f16", "b": "nk", "epilogue": "none"},
        # sizes nobody chose for a tile: row-major operands whose rows are no whole number of 16-byte pieces
        {"name": "gemm_ragged", "kind": "gemm", "m": 1000, "n": 900, "k": 1030, "dtype": "f16", "b": "kn", "epilogue": "bias+relu"},
        # single precision, the size the CPU path of the reference is quoted on
        {"name": "gemm_f32_1024", "kind": "gemm", "m": 1024, "n": 1024, "k": 1024, "dtype": "f32", "b": "kn", "epilogue": "none"},
        # a batched linear layer, every batch with weights of its own (experts, heads, ensembles)
        {"name": "linear_batched", "kind": "linear", "batch": 16, "m": 128, "n": 512, "k": 512, "dtype": "f16", "epilogue": "bias+relu"},
        # the 3x3 convolution of the benchmark
        {"name": "conv_3x3_n32", "kind": "conv", "n": 32, "h": 56, "w": 56, "c": 64, "k": 64, "r": 3, "stride": 1, "pad": 1, "dtype": "f16", "epilogue": "bias+relu"},
        # a downsampling convolution at a small batch
        {"name": "conv_stride2_n8", "kind": "conv", "n": 8, "h": 56, "w": 56, "c": 64, "k": 128, "r": 3, "stride": 2, "pad": 1, "dtype": "bf16", "epilogue": "bias+relu"},
        # a whole network on one image, fused, planned and replayed as a graph: the latency of some twenty small launches
        {"name": "resnet18_b1", "kind": "resnet18", "batch": 1, "dtype": "f16"},
        # prefill of a short prompt (the reference's attention benchmark)
        {"name": "attention_s1024_causal", "kind": "attention", "b": 1, "h": 12, "s": 1024, "d": 64, "causal": True, "dtype": "f16", "layout": "bhsd"},
        # attention over a long sequence, the benchmark's configuration and the largest case here
        {"name": "attention_s4096", "kind": "attention", "b": 4, "h": 32, "s": 4096, "d": 128, "causal": False, "dtype": "bf16", "layout": "bhsd"},
        # a head dimension between the kernels' two, a ragged length, heads interleaved as a projection leaves them
        {"name": "attention_d96_ragged", "kind": "attention", "b": 2, "h": 16, "s": 1000, "d": 96, "causal": True, "dtype": "bf16", "layout": "bshd"},
        # the upsampling layer of an image decoder
        {"name": "conv_transpose_n8", "kind": "conv_transpose", "n": 8, "h": 32, "w": 32, "c": 512, "k": 256, "r": 4, "stride": 2, "pad": 1, "dtype": "f16", "epilogue": "bias+relu"},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _near(v, step):
    return max(step, int(round(v / step)) * step)


def draw(rng):
    kind = rng.choice(["rows", "gemm", "ragged", "f32", "linear", "conv", "conv", "resnet18", "attention", "attention",
                       "attention_any", "conv_transpose"])
    half = rng.choice(["f16", "bf16"])
    epi = rng.choice(["none", "bias", "bias+relu", "gelu", "residual"])
    if kind == "rows":
        return {"kind": "gemm", "m": _log(rng, 1, 64), "n": _near(_log(rng, 512, 16384), 8), "k": _near(_log(rng, 512, 8192), 8),
                "dtype": half, "b": rng.choice(["nk", "nk", "kn"]), "epilogue": epi}
    if kind == "gemm":
        step = rng.choice([8, 64, 128])
        return {"kind": "gemm", "m": _near(_log(rng, 128, 6144), step), "n": _near(_log(rng, 128, 6144), step),
                "k": _near(_log(rng, 128, 6144), step), "dtype": half, "b": rng.choice(["nk", "kn"]), "epilogue": epi}
    if kind == "ragged":
        return {"kind": "gemm", "m": _log(rng, 3, 2000), "n": _log(rng, 3, 2000), "k": _log(rng, 16, 2000),
                "dtype": rng.choice(["f16", "bf16", "f32"]), "b": "kn", "epilogue": rng.choice(["none", "bias+relu"])}
    if kind == "f32":
        return {"kind": "gemm", "m": _near(_log(rng, 64, 3072), 4), "n": _near(_log(rng, 64, 3072), 4),
                "k": _near(_log(rng, 64, 3072), 4), "dtype": "f32", "b": "kn", "epilogue": rng.choice(["none", "bias"])}
    if kind == "linear":
        return {"kind": "linear", "batch": _log(rng, 2, 48), "m": _log(rng, 1, 512), "n": _near(_log(rng, 64, 1024), 8),
                "k": _near(_log(rng, 64, 1024), 8), "dtype": rng.choice([half, half, "f32"]), "epilogue": rng.choice(["none", "bias", "bias+relu"])}
    if kind == "conv":
        r = rng.choice([1, 3, 3, 3, 5, 7])
        size = rng.choice([7, 14, 28, 56, 112, rng.randint(9, 100)])
        stride = rng.choice([1, 1, 2])
        c = rng.choice([3, 8, 16, 64]) if r >= 5 else rng.choice([16, 32, 64, 96, 128, 256, 512])
        k = rng.choice([32, 64, 96, 128, 256, 512])
        n = _log(rng, 1, 32)
        while n > 1 and n * (size // stride) ** 2 * c * k * r * r > 3e10:
            n //= 2
        return {"kind": "conv", "n": n, "h": size, "w": size, "c": c, "k": k, "r": r, "stride": stride, "pad": r // 2, "dtype": half,
                "epilogue": rng.choice(["none", "bias+relu", "bias+relu", "bias+silu", "residual+relu"])}
    if kind == "resnet18":
        return {"kind": "resnet18", "batch": _log(rng, 1, 32), "dtype": half}
    if kind == "attention_any":
        return {"kind": "attention", "b": rng.randint(1, 4), "h": rng.choice([4, 8, 12, 16]), "s": _log(rng, 64, 2048),
                "d": rng.choice([32, 40, 48, 72, 80, 96, 112]), "causal": rng.random() < 0.5, "dtype": half,
                "layout": rng.choice(["bhsd", "bshd"])}
    if kind == "attention":
        s = _log(rng, 64, 4096)
        return {"kind": "attention", "b": rng.choice([1, 1, 2, 4]), "h": rng.choice([8, 12, 16, 32]), "s": s, "d": rng.choice([64, 128]),
                "causal": rng.random() < 0.5, "dtype": half, "layout": rng.choice(["bhsd", "bshd"])}
    r, stride = rng.choice([(2, 2), (3, 2), (4, 2), (4, 2), (3, 1)])
    return {"kind": "conv_transpose", "n": _log(rng, 1, 8), "h": (hw := rng.randint(8, 48)), "w": hw, "c": rng.choice([64, 128, 256, 512]),
            "k": rng.choice([64, 128, 256]), "r": r, "stride": stride, "pad": (r - 1) // 2 if r > 2 else 0, "dtype": half,
            "epilogue": rng.choice(["none", "bias+relu"])}


def _out_size(size, c):
    return (size + 2 * c["pad"] - c["r"]) // c["stride"] + 1


def _out_size_transposed(size, c):
    return (size - 1) * c["stride"] - 2 * c["pad"] + c["r"]


def prepare(case, seed):
    c = case
    capi.init()
    dev = torch.device("cuda:0")
    g = torch.Generator(device=dev).manual_seed(seed)
    dt = _TYPES[c["dtype"]]

    def normal(*shape, scale=1.0):
        return (torch.randn(*shape, device=dev, generator=g) * scale).to(dt)

    s = {"kind": c["kind"]}
    kw = s["kw"] = {}
    epi = c.get("epilogue", "none")
    if c["kind"] == "gemm":
        m, n, k = c["m"], c["n"], c["k"]
        s["args"] = (normal(m, k), normal(n, k, scale=k ** -0.5).t() if c["b"] == "nk" else normal(k, n, scale=k ** -0.5))
        if "bias" in epi:
            kw["bias"] = torch.randn(n, device=dev, generator=g) * 0.1
        if "residual" in epi:
            kw["residual"] = normal(m, n)
        kw.update(epilogue=epi, out=torch.empty(m, n, device=dev, dtype=dt))
        s["call"] = ops.gemm
    elif c["kind"] == "linear":
        b, m, n, k = c["batch"], c["m"], c["n"], c["k"]
        s["args"] = (normal(b, m, k), normal(b, k, n, scale=k ** -0.5))
        if "bias" in epi:
            kw["bias"] = torch.randn(n, device=dev, generator=g) * 0.1
        kw.update(epilogue=epi, out=torch.empty(b, m, n, device=dev, dtype=dt))
        s["call"] = ops.linear
    elif c["kind"] in ("conv", "conv_transpose"):
        n, h, w, ch, k, r = (c[f] for f in ("n", "h", "w", "c", "k", "r"))
        x = normal(n, h, w, ch)
        if c["kind"] == "conv":
            wt = normal(k, r, r, ch, scale=(2.0 / (r * r * ch)) ** 0.5)
            y = torch.empty(n, _out_size(h, c), _out_size(w, c), k, device=dev, dtype=dt)
            s["call"] = ops.conv2d
        else:
            wt = normal(ch, r, r, k, scale=(c["stride"] ** 2 / (r * r * ch)) ** 0.5)
            y = torch.empty(n, _out_size_transposed(h, c), _out_size_transposed(w, c), k, device=dev, dtype=dt)
            s["call"] = ops.conv_transpose2d
        s["args"] = (x, wt)
        if "bias" in epi:
            kw["bias"] = torch.randn(k, device=dev, generator=g) * 0.1
        if "residual" in epi:
            kw["residual"] = normal(*y.shape)
        kw.update(stride=c["stride"], padding=c["pad"], epilogue=epi, out=y)
    elif c["kind"] == "attention":
        b, h, n, d = c["b"], c["h"], c["s"], c["d"]

        def heads(make):
            return make(b, h, n, d) if c["layout"] == "bhsd" else make(b, n, h, d).transpose(1, 2)
        s["args"] = tuple(heads(normal) for _ in range(3))
        kw.update(causal=c["causal"], out=heads(lambda *sh: torch.empty(*sh, device=dev, dtype=dt)))
        s["call"] = ops.attention
    else:
        batch = c["batch"]
        graph, info = G.resnet18_graph(batch)
        plan = Plan(G.fuse(graph), dtype=dt)
        image = torch.zeros(batch, 224, 224, 8, device=dev, dtype=dt)
        image[..., :3] = torch.randn(batch, 224, 224, 3, device=dev, generator=g).to(dt)
        plan.bind(info["input"], image)
        for oid, (k, r, q, ch) in info["convs"].items():
            plan.bind(oid, normal(k, r, q, ch, scale=(2.0 / (r * q * ch)) ** 0.5), "weight")
        for oid, (params, ch) in info["bn"].items():
            vals = [torch.rand(ch, device=dev, generator=g) * 0.5 + 0.75, torch.randn(ch, device=dev, generator=g) * 0.1,
                    torch.randn(ch, device=dev, generator=g) * 0.1, torch.rand(ch, device=dev, generator=g) * 0.5 + 0.75]
            for pid, v in zip(params, vals):
                plan.bind(pid, v)
        plan.bind(info["fc"], normal(512, 1000, scale=512 ** -0.5), "weight")
        plan.capture()
        s.update(plan=plan, logits=plan.output(info["output"], (batch, 1000)))
    return s


def run(state):
    if state["kind"] == "resnet18":
        state["plan"].replay()
        return state["logits"]
    return state["call"](*state["args"], **state["kw"])


def work(case):
    c = case
    e = _BYTES[c["dtype"]]
    epi = c.get("epilogue", "none")
    res = 2 if "residual" in epi else 1
    if c["kind"] == "gemm":
        m, n, k = c["m"], c["n"], c["k"]
        return {"bytes": e * (m * k + k * n + res * m * n) + (4 * n if "bias" in epi else 0), "flops": 2.0 * m * n * k}
    if c["kind"] == "linear":
        b, m, n, k = c["batch"], c["m"], c["n"], c["k"]
        return {"bytes": e * b * (m * k + k * n + m * n) + (4 * n if "bias" in epi else 0), "flops": 2.0 * b * m * n * k}
    if c["kind"] == "conv":
        n, ch, k, r = c["n"], c["c"], c["k"], c["r"]
        out = n * _out_size(c["h"], c) * _out_size(c["w"], c)
        read = 1.0 if r >= c["stride"] else 1.0 / c["stride"] ** 2  # a 1x1 filter at stride 2 skips three pixels of four
        return {"bytes": e * (n * c["h"] * c["w"] * ch * read + k * r * r * ch + res * out * k), "flops": 2.0 * out * k * r * r * ch}
    if c["kind"] == "conv_transpose":
        n, ch, k, r = c["n"], c["c"], c["k"], c["r"]
        out = n * _out_size_transposed(c["h"], c) * _out_size_transposed(c["w"], c)
        return {"bytes": e * (n * c["h"] * c["w"] * ch + k * r * r * ch + out * k), "flops": 2.0 * n * c["h"] * c["w"] * ch * k * r * r}
    if c["kind"] == "attention":
        b, h, s, d = c["b"], c["h"], c["s"], c["d"]
        pairs = s * (s + 1) / 2.0 if c["causal"] else float(s) * s
        return {"bytes": e * 4.0 * b * h * s * d, "flops": 4.0 * b * h * d * pairs}
    # ResNet-18: the image's three channels, every weight, the logits; activations need not leave the chip
    batch = c["batch"]
    flops, weights = 2.0 * batch * 512 * 1000, 512 * 1000
    for node in G.resnet18_graph(batch)[0]["operators"]:
        (kind, body), = node.items()
        if kind == "Conv2d":
            ho = (body["h"] + 2 * body["padding"] - body["r"]) // body["stride"] + 1
            ch = 3 if body["c"] == 8 else body["c"]
            flops += 2.0 * body["n"] * ho * ho * body["k"] * body["r"] * body["s"] * ch
            weights += body["k"] * body["r"] * body["s"] * ch
    return {"bytes": e * (batch * 224 * 224 * 3 + weights + batch * 1000), "flops": flops}


def tolerance(case):
    """Relative error (2-norm) of another correct implementation: about four times what each path shows against
    the same product in 64 bits (the network and the convolutions against 32-bit sums).  Seen: products and
    convolutions 2.1e-4 f16, 1.7e-3 bf16 (the rounding of the result), 4e-7 f32 at k = 1024; attention 3.6e-4 /
    2.9e-3 (probabilities rounded too); ResNet-18 3.0e-4 / 2.4e-3 over its 21 roundings."""
    t = case["dtype"]
    if case["kind"] in ("resnet18", "attention"):
        return {"rel": 1.4e-3 if t == "f16" else 1.2e-2}
    return {"rel": {"f16": 9e-4, "bf16": 7e-3, "f32": 3e-6}[t]}
