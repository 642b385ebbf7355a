"""The work that users of the library have it do, as cases that can be timed and compared.

Five kinds of work, each through the entry points that a program calls (`torsh_amd.hipq.Context`):

* ``linear``: a quantized Linear forward from fp32 activations, weights int8 per output channel, fp32 result.
  ``layout`` says whether the weights were prepared once (``packed``) or are kept as rows (``rows``); ``scale`` says
  how the activations are quantized: per ``tensor``, per ``token`` or with a calibrated ``static`` scale.
* ``round_trip``: dynamic per-tensor int8 quantize of an fp32 tensor, then dequantize with the parameters on the device.
* ``channel``: per-channel int8 quantize with ranges found on the device, then the dequantize, along one axis of an
  ``[outer, channels, inner]`` tensor (``outer`` = 1: weights; otherwise activations).
* ``conv``: a quantized Conv2d forward with bias and int8 result; ``source`` is ``f32`` (the layer quantizes its fp32
  input itself, prepared filters) or ``u8`` (the input comes quantized from the layer before, filters as rows).
* ``stack``: the Linears of a transformer (qkv, out, fc1, fc2) with LayerNorm, GELU and skip connections, all layers in
  one call, on prepared weights.
"""
import functools
import math

import torch

from torsh_amd import hipq


def listed():
    return [
        # One token through an MLP up projection while text is generated: the weights are the traffic.
        {"name": "decode_one_token", "kind": "linear", "m": 1, "n": 11008, "k": 4096, "layout": "packed", "scale": "token"},
        # A small batch of such tokens through the down projection.
        {"name": "decode_batch_down", "kind": "linear", "m": 16, "n": 4096, "k": 11008, "layout": "packed", "scale": "token"},
        # The headline layer: 512 rows, dynamic per-tensor activations.
        {"name": "linear_512", "kind": "linear", "m": 512, "n": 4096, "k": 4096, "layout": "packed", "scale": "tensor"},
        # A long prompt, or many short ones, through the up projection.
        {"name": "linear_prefill", "kind": "linear", "m": 4096, "n": 11008, "k": 4096, "layout": "packed", "scale": "token"},
        # A classifier on odd sizes, weights kept as the checkpoint has them.
        {"name": "linear_ragged_rows", "kind": "linear", "m": 300, "n": 1000, "k": 1001, "layout": "rows", "scale": "tensor"},
        # One small activation tensor, odd in size: the smallest call there is.
        {"name": "round_trip_small", "kind": "round_trip", "numel": 33333},
        # A weight matrix, or a batch of activations, of ordinary size.
        {"name": "round_trip_4096", "kind": "round_trip", "numel": 4096 * 4096},
        # Image activations with a scale per channel.
        {"name": "channels_nchw", "kind": "channel", "outer": 64, "channels": 256, "inner": 56 * 56},
        # A 3x3 layer in the middle of an image network.
        {"name": "conv_3x3", "kind": "conv", "source": "f32", "nb": 32, "c": 256, "h": 14, "w": 14, "oc": 256, "kernel": 3,
         "stride": 1, "pad": 1},
        # The first layer of an image network: three channels, large windows, stride 2.
        {"name": "conv_stem", "kind": "conv", "source": "u8", "nb": 32, "c": 3, "h": 224, "w": 224, "oc": 64, "kernel": 7,
         "stride": 2, "pad": 3},
        # A transformer's Linears over a full batch of sequences ...
        {"name": "stack_8192", "kind": "stack", "tokens": 8192, "d": 768, "d_ff": 3072, "layers": 12},
        # ... and over one short prompt.
        {"name": "stack_short", "kind": "stack", "tokens": 77, "d": 768, "d_ff": 3072, "layers": 12},
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def _feature_size(rng, lo, hi):
    """A size over the whole range: two times in three a multiple of 64 as layers mostly are, else whatever comes."""
    v = _log_int(rng, lo, hi)
    return max(64, v // 64 * 64) if rng.random() < 2 / 3 else v


def _draw_linear(rng):
    layout = rng.choice(["packed", "packed", "rows"])
    limit = 4096 * 11008 * 4096 if layout == "packed" else 512 * 4096 * 4096
    while True:
        m, n, k = _log_int(rng, 1, 8192), _feature_size(rng, 64, 32000), _feature_size(rng, 64, 16384)
        if m * n * k <= limit and n * k <= 1 << 27:
            return {"kind": "linear", "m": m, "n": n, "k": k, "layout": layout,
                    "scale": rng.choice(["tensor", "token", "static"])}


def _draw_channel(rng):
    while True:
        outer = rng.choice([1, _log_int(rng, 2, 512)])
        channels, inner = _log_int(rng, 16, 8192), _log_int(rng, 16, 16384)
        if outer * channels * inner <= 64 * 256 * 56 * 56:
            return {"kind": "channel", "outer": outer, "channels": channels, "inner": inner}


def _draw_conv(rng):
    while True:
        source = rng.choice(["f32", "u8"])
        kernel = rng.choice([1, 3, 3, 5, 7])
        side = _log_int(rng, max(7, kernel), 224)
        case = {"kind": "conv", "source": source, "nb": _log_int(rng, 1, 64),
                "c": 32 * _log_int(rng, 1, 16) if source == "f32" else rng.choice([1, 3, _log_int(rng, 4, 512)]),
                "h": side, "w": side + rng.randint(0, 3), "oc": _feature_size(rng, 16, 512), "kernel": kernel,
                "stride": 1 if source == "f32" else rng.choice([1, 2]), "pad": kernel // 2}
        w = work(case)
        if w["flops"] <= 16e9 and w["bytes"] <= 128e6:
            return case


def draw(rng):
    kind = rng.choice(["linear", "linear", "linear", "round_trip", "channel", "conv", "conv", "stack"])
    if kind == "linear":
        return _draw_linear(rng)
    if kind == "round_trip":
        return {"kind": "round_trip", "numel": _log_int(rng, 1000, 1 << 25)}
    if kind == "channel":
        return _draw_channel(rng)
    if kind == "conv":
        return _draw_conv(rng)
    d = 128 * rng.randint(1, 8)
    return {"kind": "stack", "tokens": _log_int(rng, 1, 8192), "d": d, "d_ff": min(3072, d * rng.randint(2, 4)),
            "layers": rng.randint(1, 12)}


@functools.lru_cache(maxsize=None)
def _context():
    """A program keeps one context per device."""
    return hipq.Context(0)


def _quantized_weights(ctx, g, n, k):
    q, scales, _, _ = ctx.quantize_per_row(torch.randn(n, k, generator=g, device="cuda") * 0.02)
    return q, scales, torch.randn(n, generator=g, device="cuda") * 0.01


def _prepare_linear(ctx, g, case):
    m, n, k = case["m"], case["n"], case["k"]
    w, w_scales, bias = _quantized_weights(ctx, g, n, k)
    x = torch.randn(m, k, generator=g, device="cuda")
    return {"x": x, "w": ctx.pack_rows(w) if case["layout"] == "packed" else w, "w_scales": w_scales, "bias": bias,
            # a calibrated scale: what four standard deviations of the activations need
            "a_scale": 4.0 / 127, "out": torch.empty(m, n, device="cuda")}


def _prepare_conv(ctx, g, case):
    nb, c, h, w, oc, kernel = (case[key] for key in ("nb", "c", "h", "w", "oc", "kernel"))
    x = torch.relu(torch.randn(nb, c, h, w, generator=g, device="cuda"))
    wq, w_scales, bias = _quantized_weights(ctx, g, oc, c * kernel * kernel)
    wq = wq.view(oc, c, kernel, kernel)
    # a calibrated output scale: four standard deviations of a window's sum (E[relu(x)^2] = 1/2)
    out_scale = 4.0 * 0.02 * math.sqrt(c * kernel * kernel / 2) / 127
    state = {"w_scales": w_scales, "bias": bias, "out_scale": out_scale}
    if case["source"] == "f32":
        packed, sums = ctx.conv2d_pack_weights(wq)
        return {**state, "x": x, "w": packed, "w_sums": sums}
    s_in = 5.0 / 255
    return {**state, "x": ctx.quantize_per_tensor_u8(x, s_in, 0), "s_in": s_in, "w": wq}


def _prepare_stack(ctx, g, case):
    tokens, d, d_ff = case["tokens"], case["d"], case["d_ff"]
    blocks = []
    for _ in range(case["layers"]):
        block = {}
        for name, (n, k) in {"qkv": (3 * d, d), "out": (d, d), "fc1": (d_ff, d), "fc2": (d, d_ff)}.items():
            block["w_" + name], block["s_" + name], block["b_" + name] = _quantized_weights(ctx, g, n, k)
        for ln in ("ln1", "ln2"):
            block[ln + "_gamma"] = torch.rand(d, generator=g, device="cuda") + 0.5
            block[ln + "_beta"] = torch.randn(d, generator=g, device="cuda") * 0.1
        blocks.append(block)
    return {"blocks": ctx.stack_prepare(blocks), "workspace": ctx.stack_workspace_prepared(tokens, d, d_ff),
            "embedded": torch.randn(tokens, d, generator=g, device="cuda"), "x": torch.empty(tokens, d, device="cuda")}


def prepare(case, seed):
    ctx = _context()
    g = torch.Generator(device="cuda").manual_seed(seed)
    if case["kind"] == "linear":
        state = _prepare_linear(ctx, g, case)
    elif case["kind"] == "round_trip":
        state = {"x": torch.randn(case["numel"], generator=g, device="cuda")}
    elif case["kind"] == "channel":
        state = {"x": torch.randn(case["outer"], case["channels"], case["inner"], generator=g, device="cuda")}
    elif case["kind"] == "conv":
        state = _prepare_conv(ctx, g, case)
    else:
        state = _prepare_stack(ctx, g, case)
    return {**state, "case": case, "ctx": ctx}


def _run_linear(ctx, s, case):
    per_token = case["scale"] == "token"
    if case["layout"] == "packed":
        if case["scale"] == "static":
            return ctx.linear_static_packed(s["x"], s["a_scale"], s["w"], s["w_scales"], s["bias"], out=s["out"])
        return ctx.linear_dynamic_packed(s["x"], s["w"], s["w_scales"], s["bias"], per_token=per_token, out=s["out"])
    if case["scale"] == "static":
        return ctx.linear_static(s["x"], s["a_scale"], s["w"], s["w_scales"], s["bias"], out=s["out"])
    return ctx.linear_dynamic(s["x"], s["w"], s["w_scales"], s["bias"], per_token=per_token, out=s["out"])


def run(state):
    ctx, case = state["ctx"], state["case"]
    if case["kind"] == "linear":
        return _run_linear(ctx, state, case)
    if case["kind"] == "round_trip":
        q, params = ctx.quantize_dynamic_per_tensor(state["x"])
        return q, ctx.dequantize_with_params(q, params)
    if case["kind"] == "channel":
        axis = 1
        q, scales, zero_points, _ = ctx.quantize_per_channel_auto(state["x"], axis)
        return q, scales, zero_points, ctx.dequantize_per_channel(q, scales, zero_points, axis)
    if case["kind"] == "conv":
        pad, stride = (case["pad"],) * 2, (case["stride"],) * 2
        if case["source"] == "f32":
            out, _ = ctx.conv2d_dynamic_packed(state["x"], state["w"], state["w_sums"], (case["kernel"],) * 2,
                                               state["w_scales"], state["bias"], state["out_scale"], 0, padding=pad)
            return out
        return ctx.conv2d_i8(state["x"], 0, state["s_in"], state["w"], state["w_scales"], state["bias"],
                             state["out_scale"], 0, stride=stride, padding=pad)
    state["x"].copy_(state["embedded"])  # the stack works in place
    return ctx.stack_forward(state["blocks"], state["x"], case["d_ff"], state["workspace"], prepared=True)


def work(case):
    if case["kind"] == "linear":
        m, n, k = case["m"], case["n"], case["k"]
        return {"bytes": 4 * m * k + n * k + 8 * n + 4 * m * n, "flops": 2 * m * n * k}
    if case["kind"] == "round_trip":
        return {"bytes": 9 * case["numel"], "flops": 4 * case["numel"]}
    if case["kind"] == "channel":
        numel = case["outer"] * case["channels"] * case["inner"]
        return {"bytes": 9 * numel + 8 * case["channels"], "flops": 4 * numel}
    if case["kind"] == "conv":
        nb, c, h, w, oc, kernel = (case[key] for key in ("nb", "c", "h", "w", "oc", "kernel"))
        ho = (h + 2 * case["pad"] - kernel) // case["stride"] + 1
        wo = (w + 2 * case["pad"] - kernel) // case["stride"] + 1
        return {"bytes": nb * c * h * w * (4 if case["source"] == "f32" else 1) + oc * c * kernel * kernel + 8 * oc +
                nb * oc * ho * wo, "flops": 2 * nb * oc * ho * wo * c * kernel * kernel}
    tokens, d, d_ff, layers = case["tokens"], case["d"], case["d_ff"], case["layers"]
    weights = layers * (4 * d * d + 2 * d * d_ff)
    return {"bytes": weights + layers * 4 * (2 * (4 * d + d_ff + d) + 4 * d) + 8 * tokens * d,
            "flops": 2 * tokens * weights}


def tolerance(case):
    if case["kind"] == "stack":
        # LayerNorm sums folded in another order move a value across a rounding edge here and there, and every such
        # code changes a row of the products after it: 2e-3 between the row-major and the prepared form of the stack
        # over 12 layers (d 768 and 1024, 77 to 8192 tokens).
        return {"rel": 8e-3}
    # Codes, int32 sums and each f32 operation after them are fixed by the reference: the bits are the same in any
    # order of the sums.
    return "exact"
