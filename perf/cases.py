"""Workloads of the public operations, for timing: what a model or a sampler built on this package
asks of it, from one small call to whole training steps.

A case is a dict of plain values.  `op` is the entry point (`na`: na1d / na2d / na3d by the number
of dimensions, `layer`: NeighborhoodAttention1D/2D/3D, `attention`: dense attention, `packed`:
variable-length dense attention); extents and per-dimension arguments are written "30x48x80";
`train` means forward and backward; `causal` has one letter per dimension."""

import math

import torch

import natten_amd
from natten_amd.utils.varlen import generate_varlen_parameters

DTYPES = {"fp32": torch.float32, "bf16": torch.bfloat16, "fp16": torch.float16, "e4m3": torch.float8_e4m3fn}
NA = {1: natten_amd.na1d, 2: natten_amd.na2d, 3: natten_amd.na3d}
LAYERS = {1: natten_amd.NeighborhoodAttention1D, 2: natten_amd.NeighborhoodAttention2D, 3: natten_amd.NeighborhoodAttention3D}


def _na(name, dtype, batch, layout, heads, head_dim, kernel, stride=None, dilation=None, causal=None, heads_kv=None,
        context=0, lse=False, train=False, op="na"):
    n = layout.count("x") + 1
    ones = "x".join(["1"] * n)
    return {"name": name, "op": op, "dtype": dtype, "batch": batch, "layout": layout, "heads": heads,
            "heads_kv": heads_kv or heads, "head_dim": head_dim, "kernel": kernel, "stride": stride or ones,
            "dilation": dilation or ones, "causal": causal or "F" * n, "context": context, "lse": lse, "train": train}


def _attention(name, dtype, batch, seqlen, heads, head_dim, heads_kv=None, causal=False, train=False):
    return {"name": name, "op": "attention", "dtype": dtype, "batch": batch, "layout": str(seqlen), "heads": heads,
            "heads_kv": heads_kv or heads, "head_dim": head_dim, "causal": "T" if causal else "F", "lse": False, "train": train}


def _packed(name, dtype, lengths, heads, head_dim, heads_kv=None, causal=True, train=False):
    return {"name": name, "op": "packed", "dtype": dtype, "lengths": ",".join(map(str, lengths)), "heads": heads,
            "heads_kv": heads_kv or heads, "head_dim": head_dim, "causal": "T" if causal else "F", "lse": False, "train": train}


def listed():
    return [
        # The smallest call: one short signal through a float32 1-D window (the configuration the CPU
        # reference is quoted on); all latency.
        _na("na1d_signal_fp32", "fp32", 1, "256", 2, 32, "7"),
        # Float32 inference of an image model's attention at its stated precision.
        _na("na2d_image_fp32", "fp32", 2, "64x64", 8, 64, "13x13"),
        # The same layer in bf16: small windows over a small image, called once per layer.
        _na("na2d_image_bf16", "bf16", 2, "64x64", 8, 64, "13x13"),
        # An image layer of a text-conditioned model: the window plus 128 context tokens that every
        # query sees, shared key / value heads, a head dim between the native ones.
        _na("na2d_context_bf16", "bf16", 2, "64x64", 8, 96, "13x13", heads_kv=2, context=128),
        # One head over a long sequence with a sliding window (32K tokens, 2K window).
        _na("na1d_long_fp16", "fp16", 1, "32768", 1, 128, "2048"),
        # The headline video layer: causal in time, strided windows in space, LSE wanted by the caller.
        _na("na3d_video_bf16", "bf16", 1, "30x48x80", 24, 128, "18x24x24", stride="1x8x8", causal="TFF", lse=True),
        # Quantised video inference: e4m3 operands with per-head scales, dilated blocked windows.
        _na("na3d_video_e4m3", "e4m3", 1, "16x64x64", 16, 128, "8x16x16", stride="4x8x8", dilation="1x2x2"),
        # Global attention of an image model: 64 x 64 tokens and a class token (no tile divides it).
        _attention("attention_image_bf16", "bf16", 2, 4097, 16, 64),
        # A training step on packed sequences of very different lengths, causal, shared key / value heads.
        _packed("attention_packed_train_bf16", "bf16", [2048, 1333, 70, 1, 900, 2000, 33, 411, 1024, 517], 16, 128,
                heads_kv=4, train=True),
        # A training step of a whole small-head image layer: projections around 7 x 7 windows.
        _na("na2d_layer_train_bf16", "bf16", 4, "56x56", 8, 32, "7x7", train=True, op="layer"),
        # A training step of blocked image attention.
        _na("na2d_train_fp16", "fp16", 1, "128x128", 16, 128, "32x32", stride="16x16", train=True),
        # The largest: a training step on video whose extents no tile divides, dilated in time.
        _na("na3d_train_bf16", "bf16", 1, "29x46x78", 24, 128, "9x24x24", stride="1x8x8", dilation="2x1x1", train=True),
    ]


# ---- more cases of the same ranges ----------------------------------------------------------------

def _log(rng, lo, hi):
    """An integer between lo and hi, spread over the logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1)))))))


def _text(values):
    return "x".join(str(v) for v in values)


def _window(rng, layout, k_lo, k_hi, strides=0.4, dilations=0.25):
    """Window, stride and dilation per dimension that fit the layout."""
    kernel, stride, dilation = [], [], []
    for x in layout:
        d = rng.choice((2, 3)) if rng.random() < dilations and x >= 4 * k_lo else 1
        k = _log(rng, min(k_lo, x // d), max(min(k_hi, x // d), 2))
        k = max(2, k)
        s = rng.choice([s for s in (1, 2, 4, 8, 16) if s <= k]) if rng.random() < strides else 1
        kernel.append(k)
        stride.append(s)
        dilation.append(d)
    return _text(kernel), _text(stride), _text(dilation)


def _draw_fp32(rng):
    n = rng.choice((1, 2, 2, 3))
    layout = {1: lambda: (_log(rng, 256, 8192),), 2: lambda: (_log(rng, 16, 96), _log(rng, 16, 96)),
              3: lambda: (_log(rng, 6, 16), _log(rng, 10, 32), _log(rng, 10, 32))}[n]()
    k, s, d = _window(rng, layout, 3, {1: 257, 2: 25, 3: 11}[n])
    heads = rng.choice((2, 4, 6, 8))
    return _na(None, "fp32", rng.choice((1, 2)), _text(layout), heads, rng.choice((32, 32, 64, 64, 40, 128)), k, s, d,
               rng.choice("FFT") + "F" * (n - 1), heads_kv=rng.choice((heads, heads, heads // 2)))


def _draw_image(rng):
    layout = (_log(rng, 24, 192), _log(rng, 24, 192))
    k, s, d = _window(rng, layout, 3, 48)
    heads = rng.choice((4, 6, 8, 12, 16))
    return _na(None, rng.choice(("bf16", "fp16")), rng.choice((1, 2, 4)), _text(layout), heads,
               rng.choice((32, 64, 64, 128, 128, 72, 96)), k, s, d, heads_kv=rng.choice((heads, heads, heads // 2)),
               context=rng.choice((0, 0, 0, 77, 128, 256)), lse=rng.random() < 0.3)


def _draw_long(rng):
    length = _log(rng, 2048, 65536)
    k, s, d = _window(rng, (length,), 64, min(4096, length // 3), strides=0.5)
    heads = rng.choice((1, 2, 4, 8))
    return _na(None, rng.choice(("bf16", "fp16")), 1, str(length), heads, rng.choice((64, 128, 128)), k, s, d,
               rng.choice("FT"), lse=rng.random() < 0.3)


def _draw_video(rng):
    layout = (_log(rng, 8, 32), _log(rng, 16, 64), _log(rng, 16, 80))
    k, s, d = _window(rng, layout, 4, 24, strides=0.6, dilations=0.15)
    heads = rng.choice((4, 8, 12, 16, 24))
    return _na(None, rng.choice(("bf16", "bf16", "fp16", "e4m3")), 1, _text(layout), heads, rng.choice((64, 128, 128)), k, s, d,
               rng.choice("FT") + "FF", lse=rng.random() < 0.5)


def _draw_attention(rng):
    heads = rng.choice((4, 8, 16, 24))
    return _attention(None, rng.choice(("bf16", "fp16")), rng.choice((1, 2, 4)), _log(rng, 200, 9000), heads,
                      rng.choice((32, 64, 64, 128, 128, 96)), heads_kv=rng.choice((heads, heads, heads // 2)),
                      causal=rng.random() < 0.4, train=rng.random() < 0.4)


def _draw_packed(rng):
    lengths = [_log(rng, 1, 2048) for _ in range(rng.randint(3, 16))]
    heads = rng.choice((4, 8, 16))
    return _packed(None, rng.choice(("bf16", "fp16")), lengths, heads, rng.choice((32, 64, 128, 128)),
                   heads_kv=rng.choice((heads, heads // 2, heads // 4)), causal=rng.random() < 0.7, train=rng.random() < 0.6)


def _draw_layer(rng):
    n = rng.choice((1, 2, 2, 3))
    layout = {1: lambda: (_log(rng, 512, 8192),), 2: lambda: (_log(rng, 14, 96), _log(rng, 14, 96)),
              3: lambda: (_log(rng, 8, 16), _log(rng, 10, 32), _log(rng, 10, 32))}[n]()
    k, s, d = _window(rng, layout, 3, {1: 129, 2: 13, 3: 7}[n], strides=0.2)
    return _na(None, rng.choice(("bf16", "fp16")), rng.choice((1, 2, 4)), _text(layout), rng.choice((2, 4, 8)),
               rng.choice((32, 32, 64)), k, s, d, rng.choice("FFT") + "F" * (n - 1), train=True, op="layer")


def _draw_train(rng):
    n = rng.choice((2, 3))
    layout = {2: lambda: (_log(rng, 32, 160), _log(rng, 32, 160)),
              3: lambda: (_log(rng, 8, 30), _log(rng, 16, 48), _log(rng, 16, 80))}[n]()
    k, s, d = _window(rng, layout, 4, {2: 48, 3: 24}[n], strides=0.6, dilations=0.15)
    heads = rng.choice((4, 8, 16))
    return _na(None, rng.choice(("bf16", "fp16")), 1, _text(layout), heads, rng.choice((32, 64, 128, 128, 96)), k, s, d,
               rng.choice("FT") + "F" * (n - 1), heads_kv=rng.choice((heads, heads, heads // 2)), train=True)


def draw(rng):
    """One more case of the ranges above: the kind first, then its sizes."""
    kinds = (_draw_fp32, _draw_image, _draw_long, _draw_video, _draw_attention, _draw_packed, _draw_layer, _draw_train)
    kind = rng.choice(kinds)
    while True:
        case = kind(rng)
        del case["name"]
        w = work(case)
        if w["flops"] <= (1e11 if case["dtype"] == "fp32" else 5e12) and w["bytes"] <= 3e9:
            return case


# ---- inputs and one pass --------------------------------------------------------------------------

def _ints(text):
    return tuple(int(x) for x in text.split("x"))


def _lengths(case):
    return [int(x) for x in case["lengths"].split(",")]


def _quantise(x):
    """Per-head absmax scaling into the e4m3 range."""
    scale = x.abs().amax(dim=tuple(range(x.dim() - 2)) + (x.dim() - 1,)).float() / 448.0
    return (x / scale.view(-1, 1)).to(torch.float8_e4m3fn), scale


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    dtype = DTYPES[case["dtype"]]

    def rand(*shape):
        return torch.randn(shape, generator=gen, device="cuda", dtype=torch.float32 if case["dtype"] == "e4m3" else dtype)

    state = {"case": case}
    heads, heads_kv, d = case["heads"], case["heads_kv"], case["head_dim"]
    if case["op"] == "layer":
        layout = _ints(case["layout"])
        layer = LAYERS[len(layout)](heads * d, heads, _ints(case["kernel"]), _ints(case["stride"]), _ints(case["dilation"]),
                                    tuple(c == "T" for c in case["causal"])).to("cuda", dtype)
        with torch.no_grad():
            for p in layer.parameters():
                p.copy_(rand(*p.shape) * (p.shape[-1] ** -0.5 if p.dim() > 1 else 0.02))
        state["layer"] = layer
        state["x"] = rand(case["batch"], *layout, heads * d).requires_grad_(True)
        state["d_out"] = rand(case["batch"], *layout, heads * d)
        return state
    if case["op"] == "packed":
        lead = (1, sum(_lengths(case)))
    else:
        lead = (case["batch"], *_ints(case["layout"]))
    q, k, v = rand(*lead, heads, d), rand(*lead, heads_kv, d), rand(*lead, heads_kv, d)
    kwargs = {}
    if case["op"] == "na":
        kwargs.update(kernel_size=_ints(case["kernel"]), stride=_ints(case["stride"]), dilation=_ints(case["dilation"]),
                      is_causal=tuple(c == "T" for c in case["causal"]))
        if case["context"]:
            kwargs["additional_keys"] = rand(case["batch"], case["context"], heads_kv, d)
            kwargs["additional_values"] = rand(case["batch"], case["context"], heads_kv, d)
    else:
        kwargs["is_causal"] = case["causal"] == "T"
    if case["op"] == "packed":
        lengths = torch.tensor(_lengths(case), dtype=torch.int32, device="cuda")
        cu_q, cu_kv, max_q, max_kv = generate_varlen_parameters(q, k, v, lengths, lengths)
        kwargs.update(cumulative_seqlen_Q=cu_q, cumulative_seqlen_KV=cu_kv, max_seqlen_Q=max_q, max_seqlen_KV=max_kv)
    if case["dtype"] == "e4m3":
        (q, sq), (k, sk), (v, sv) = _quantise(q), _quantise(k), _quantise(v)
        kwargs.update(q_scale=sq, k_scale=sk, v_scale=sv, out_dtype=torch.bfloat16)
    if case["lse"]:
        kwargs["return_lse"] = True
    if case["train"]:
        q, k, v = (t.requires_grad_(True) for t in (q, k, v))
        state["d_out"] = rand(*lead, heads, d)
    state.update(q=q, k=k, v=v, kwargs=kwargs)
    return state


def run(state):
    case = state["case"]
    if case["op"] == "layer":
        leaves = [state["x"], *state["layer"].parameters()]
        out = state["layer"](state["x"])
        return [out.detach(), *torch.autograd.grad(out, leaves, state["d_out"])]
    op = NA[case["layout"].count("x") + 1] if case["op"] == "na" else natten_amd.attention
    out = op(state["q"], state["k"], state["v"], **state["kwargs"])
    if not case["train"]:
        return out
    return [out.detach(), *torch.autograd.grad(out, (state["q"], state["k"], state["v"]), state["d_out"])]


# ---- what a pass cannot do without ----------------------------------------------------------------

def _pairs(x, k, s, d, causal):
    """(query, key) pairs along one dimension."""
    if not causal:
        return x * k
    total = 0
    for g in range(d):
        length = x // d + (1 if g < x % d else 0)
        for i in range(length):
            leader = min((i // s) * s + s - 1, length - 1)
            total += i + 1 - max(leader - k + 1, 0)
    return total


def work(case):
    heads, heads_kv, d = case["heads"], case["heads_kv"], case["head_dim"]
    item = {"fp32": 4, "e4m3": 1}.get(case["dtype"], 2)
    if case["op"] == "packed":
        tokens = sum(_lengths(case))
        pairs = sum(n * (n + 1) // 2 if case["causal"] == "T" else n * n for n in _lengths(case))
    elif case["op"] == "attention":
        n = int(case["layout"])
        tokens = case["batch"] * n
        pairs = case["batch"] * (n * (n + 1) // 2 if case["causal"] == "T" else n * n)
    else:
        layout = _ints(case["layout"])
        tokens, pairs = case["batch"] * math.prod(layout), case["batch"]
        for x, k, s, dil, c in zip(layout, _ints(case["kernel"]), _ints(case["stride"]), _ints(case["dilation"]), case["causal"]):
            pairs *= _pairs(x, k, s, dil, c == "T")
        pairs += tokens * case["context"]
    # two products forward (q k, p v), five backward (the logits again, dp, dv, dq, dk)
    flops = (14 if case["train"] else 4) * pairs * heads * d
    if case["op"] == "layer":
        c = heads * d
        parameters = 4 * c * c + 4 * c
        # four projections forward, each with two products backward; x, d_out in, out, d_x out
        return {"bytes": 2 * (4 * tokens * c + 2 * parameters), "flops": flops + 3 * 2 * tokens * 4 * c * c}
    q, kv = tokens * heads * d, (tokens + case.get("batch", 1) * case.get("context", 0)) * heads_kv * d
    size = item * (q + 2 * kv) + max(item, 2) * q + (4 * tokens * heads if case["lse"] else 0)
    if case["train"]:
        size += item * (q + q + 2 * kv)  # d_out in; d_q, d_k, d_v out
    return {"bytes": size, "flops": flops}


def tolerance(case):
    """About four times the largest error of the present kernels against float64 on smaller problems of
    every kind (relative / largest over rms: float32 7e-7 / 5e-6, bf16 3.3e-3 / 5e-2, fp16 4.7e-4 /
    1e-2, e4m3 2.6e-2 / 0.2, whose probabilities are rounded to three bits)."""
    return {"fp32": {"rel": 4e-6, "max": 3e-5}, "bf16": {"rel": 1.3e-2, "max": 0.2}, "fp16": {"rel": 2e-3, "max": 4e-2},
            "e4m3": {"rel": 3e-2, "max": 0.6}}[case["dtype"]]
