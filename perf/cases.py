"""What a user of this framework runs, as cases that can be timed one by one.

A case is a dict of plain values.  Its "kind" names the public entry point that is called:

    linear            WALinear.forward: one quantized linear, called eagerly
    layer             the linears of a pre-LayerNorm decoder layer (q/k/v as one, out_proj, fc1 with ReLU, fc2),
                      LayerNorm, bias and residual inside the calls as DecoderLayer.forward makes them
    gated             the linears of a gated decoder layer (q/k/v, o, silu(gate) * up, down)
    step              OPTDecoder.greedy_step replayed from a HIP graph: one token per sequence over a filled cache
    prefill           OPTDecoder.forward on whole prompts into an empty cache
    lut_attention     sparse_attention over a block look-up table (q_len == kv_len)
    decode_attention  sparse_attention of one query row per sequence over the KV cache
    pack              WALinear.from_float: quantise and pack an fp16 linear
    dequant           quant.dequant: packed weight -> fp16

listed() holds the cases themselves, draw() makes more over the same ranges.
"""
import math
import os
import sys

import torch
from torch import nn

_PKG = os.path.join(os.getcwd(), "sparse-quant_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import quant  # noqa: E402
from sqamd import lut_layout  # noqa: E402
from sqamd.block_sparse_attention_lut import sparse_attention  # noqa: E402
from sqamd.opt_decode import E2E_SCALE_MIN, E2E_SCALE_STD, OPTDecoder  # noqa: E402
from sqamd.qlinear import WALinear  # noqa: E402

DEV = "cuda"


def listed():
    return [
        # one projection for one token, called from Python: launch and call overhead against 9 MB of weights
        {"name": "linear_1tok", "kind": "linear", "tokens": 1, "k": 4096, "n": 4096, "group": 64, "bits": 4,
         "layout": "l1", "act": "none", "residual": False},
        # a decoder layer's linears for one token: interactive decoding without a graph
        {"name": "layer_1tok", "kind": "layer", "tokens": 1, "hidden": 4096, "ffn": 16384, "group": 128},
        # batched decoding as served: four layers, lm_head and token choice in a HIP graph, 8 sequences, 640 cache rows
        {"name": "step_8seq", "kind": "step", "batch": 8, "rows": 640, "layers": 4},
        # a larger decode batch on a gated MLP
        {"name": "gated_32tok", "kind": "gated", "tokens": 32, "hidden": 4096, "ffn": 11008, "group": 128, "layout": "l1"},
        # a short ragged prompt on weights stored in the tensor-core layout; 13696 = 107 x 128
        {"name": "gated_l2_100tok", "kind": "gated", "tokens": 100, "hidden": 5120, "ffn": 13696, "group": 128,
         "layout": "l2"},
        # a prompt of ordinary length at the default group size
        {"name": "gated_g64_333tok", "kind": "gated", "tokens": 333, "hidden": 4096, "ffn": 11008, "group": 64,
         "layout": "l1"},
        # a long prompt, matrix-core bound
        {"name": "layer_2048tok", "kind": "layer", "tokens": 2048, "hidden": 4096, "ffn": 16384, "group": 128},
        # a batch of short encoder inputs through the sparse attention
        {"name": "lut_encoder_512", "kind": "lut_attention", "batch": 8, "heads": 16, "seq": 512, "dim": 64,
         "density": 0.25, "causal": False},
        # one long causal prompt through the sparse attention
        {"name": "lut_causal_4096", "kind": "lut_attention", "batch": 1, "heads": 32, "seq": 4096, "dim": 128,
         "density": 0.26, "causal": True},
        # the decode branch of the same entry point over long caches
        {"name": "decode_attn_2048", "kind": "decode_attention", "batch": 8, "heads": 32, "rows": 2048, "dim": 128,
         "mask": False},
        # whole prompts through the model: 8 x 512 tokens, sparse attention, cache writes, lm_head
        {"name": "prefill_8x512", "kind": "prefill", "batch": 8, "prompt": 512, "layers": 2, "density": 0.26},
        # loading a model: one fp16 linear quantised and packed
        {"name": "pack_16384x4096", "kind": "pack", "k": 4096, "n": 16384, "group": 128, "bits": 4, "layout": "l1"},
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _multiple(rng, lo, hi, step):
    return max(1, int(round(_log_int(rng, lo, hi) / step))) * step


def draw(rng):
    kind = rng.choice(["linear", "linear", "layer", "layer", "gated", "gated", "step", "prefill", "lut_attention",
                       "lut_attention", "decode_attention", "pack", "dequant"])
    if kind == "linear":
        layout = rng.choice(["l1", "l1", "l1", "l2"])
        group = 128 if layout == "l2" else rng.choice([128, 128, 64, 64, 32])
        return {"kind": kind, "tokens": _log_int(rng, 1, 2048), "k": _multiple(rng, 768, 16384, 128),
                "n": _multiple(rng, 768, 16384, 32), "group": group,
                "bits": rng.choice([4, 4, 4, 2]) if layout == "l1" else 4, "layout": layout,
                "act": rng.choice(["none", "relu", "silu"]), "residual": rng.random() < 0.5}
    if kind == "layer":
        hidden = _multiple(rng, 1024, 5120, 256)
        return {"kind": kind, "tokens": _log_int(rng, 1, 2048), "hidden": hidden, "ffn": 4 * hidden,
                "group": rng.choice([128, 128, 64])}
    if kind == "gated":
        hidden = _multiple(rng, 1024, 5120, 256)
        layout = rng.choice(["l1", "l1", "l2"])
        return {"kind": kind, "tokens": _log_int(rng, 1, 2048), "hidden": hidden,
                "ffn": int(round(hidden * rng.uniform(2.5, 3.0) / 128)) * 128,
                "group": 128 if layout == "l2" else rng.choice([128, 128, 64]), "layout": layout}
    if kind == "step":
        return {"kind": kind, "batch": rng.randint(1, 8), "rows": _log_int(rng, 100, 2000), "layers": rng.randint(3, 4)}
    if kind == "prefill":
        prompt = _multiple(rng, 64, 1024, 1)
        return {"kind": kind, "batch": max(1, min(8, 4096 // prompt, rng.randint(1, 8))), "prompt": prompt,
                "layers": 2, "density": rng.choice([0.0, 0.26, 0.5])}
    if kind == "lut_attention":
        dim = rng.choice([64, 128])
        seq = _log_int(rng, 128, 4096)
        return {"kind": kind, "batch": rng.randint(1, max(1, min(8, 4096 // seq))), "heads": rng.choice([12, 16, 32]),
                "seq": seq, "dim": dim, "density": round(rng.uniform(0.15, 0.5), 2), "causal": rng.random() < 0.5}
    if kind == "decode_attention":
        return {"kind": kind, "batch": rng.randint(1, 8), "heads": rng.choice([12, 16, 32]), "rows": _log_int(rng, 64, 4096),
                "dim": rng.choice([64, 128]), "mask": rng.random() < 0.3}
    k, n = _multiple(rng, 768, 8192, 128), _multiple(rng, 768, 8192, 32)
    layout = rng.choice(["l1", "l1", "l2"])
    return {"kind": kind, "k": k, "n": n, "group": 128 if layout == "l2" else rng.choice([128, 64, 32]),
            "bits": rng.choice([4, 4, 2]) if kind == "pack" and layout == "l1" else 4, "layout": layout}


def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    return g


def _randn(gen, *shape, scale=1.0):
    return (torch.randn(shape, device=DEV, generator=gen) * scale).half()


def _walinear(gen, k, n, group, layout="l1", bits=4, bias=True):
    """Random codes U{0..2^bits - 1}, zeros of the same range, scales |N(0, 0.004)| + 2e-4: the decoder harness's."""
    if layout == "l2":
        m = nn.Linear(k, n, bias=False, device=DEV, dtype=torch.float16)
        m.weight.data = _randn(gen, n, k, scale=0.02)
        lin = WALinear.from_float(m, {"n_bit": bits, "group_size": group}, layout="l2")
        lin.bias = _randn(gen, 1, n, scale=0.01) if bias else None
        return lin
    lin = WALinear(k, n, w_bit=bits, group_size=group, bias=bias, dev=DEV, layout=layout)
    lin.weight = torch.randint(0, 256, (n, k * bits // 8), dtype=torch.uint8, device=DEV, generator=gen)
    z = torch.randint(0, 1 << bits, (n, k // group), device=DEV, generator=gen).half() + 64
    s = (torch.randn((n, k // group), device=DEV, generator=gen).abs() * E2E_SCALE_STD + E2E_SCALE_MIN).half()
    lin.zeros_scales = torch.stack([z, s], dim=-1).reshape(n, 2 * (k // group)).contiguous()
    if bias:
        lin.bias = _randn(gen, 1, n, scale=0.01)
    return lin


def _layernorm(gen, hidden):
    ln = nn.LayerNorm(hidden, device=DEV, dtype=torch.float16)
    ln.weight.data = (1 + torch.randn(hidden, device=DEV, generator=gen) * 0.1).half()
    ln.bias.data = _randn(gen, hidden, scale=0.1)
    return ln


def _lut(case, seed):
    nb = (case["seq"] + 63) // 64
    layout = lut_layout.synth_layout(case["heads"], nb, case["density"], causal=case["causal"], seed=seed)
    return lut_layout.layout2lut_single_density(layout[None])[0].to(DEV)


@torch.no_grad()
def prepare(case, seed):
    kind = case["kind"]
    gen = _gen(seed)
    s = dict(case)
    if kind == "linear":
        s["lin"] = _walinear(gen, case["k"], case["n"], case["group"], case["layout"], case["bits"])
        s["x"] = _randn(gen, 1, case["tokens"], case["k"])
        s["res"] = _randn(gen, 1, case["tokens"], case["n"]) if case["residual"] else None
    elif kind == "layer":
        h, f, g = case["hidden"], case["ffn"], case["group"]
        s["qkv"], s["out"] = _walinear(gen, h, 3 * h, g), _walinear(gen, h, h, g)
        s["fc1"], s["fc2"] = _walinear(gen, h, f, g), _walinear(gen, f, h, g)
        s["ln1"], s["ln2"] = _layernorm(gen, h), _layernorm(gen, h)
        s["x"], s["attn"] = _randn(gen, 1, case["tokens"], h), _randn(gen, 1, case["tokens"], h)
    elif kind == "gated":
        h, f, g, lay = case["hidden"], case["ffn"], case["group"], case["layout"]
        s["qkv"], s["out"] = _walinear(gen, h, 3 * h, g, lay, bias=False), _walinear(gen, h, h, g, lay, bias=False)
        s["gate"], s["up"] = _walinear(gen, h, f, g, lay, bias=False), _walinear(gen, h, f, g, lay, bias=False)
        s["down"] = _walinear(gen, f, h, g, lay, bias=False)
        s["x"], s["attn"] = _randn(gen, 1, case["tokens"], h), _randn(gen, 1, case["tokens"], h)
    elif kind in ("step", "prefill"):
        model = OPTDecoder(layers=case["layers"], dev=DEV, seed=seed)
        for layer in model.layers:
            layer.fuse_qkv()
        s["model"] = model
        b, vocab = case["batch"], model.embed.shape[0]
        if kind == "prefill":
            if case["density"]:
                model.set_prefill_lut(case["prompt"], case["density"], seed=seed)
            s["cache"] = model.new_cache(b, case["prompt"] + 128)
            s["ids"] = torch.randint(0, vocab, (b, case["prompt"]), device=DEV, generator=gen)
        else:
            rows = case["rows"]
            s["cache"] = model.new_cache(b, rows + 8)
            for kc, vc in s["cache"]:
                kc[:, :, :rows] = _randn(gen, b, model.heads, rows, kc.shape[-1])
                vc[:, :, :rows] = _randn(gen, b, model.heads, rows, kc.shape[-1])
            s["next"] = torch.randint(0, vocab, (b, 1), device=DEV, generator=gen)
            s["tok"], s["pos"] = s["next"].clone(), torch.full((1,), rows, dtype=torch.long, device=DEV)
            side = torch.cuda.Stream()
            side.wait_stream(torch.cuda.current_stream())
            with torch.cuda.stream(side):
                model.greedy_step(s["tok"], s["cache"], s["pos"])
            torch.cuda.current_stream().wait_stream(side)
            torch.cuda.synchronize()
            s["graph"] = torch.cuda.CUDAGraph()
            s["tok"].copy_(s["next"])
            s["pos"].fill_(rows)
            with torch.cuda.graph(s["graph"], stream=side):
                s["logits"] = model.greedy_step(s["tok"], s["cache"], s["pos"])
    elif kind == "lut_attention":
        shape = (case["batch"], case["heads"], case["seq"], case["dim"])
        s["q"], s["k"], s["v"] = _randn(gen, *shape), _randn(gen, *shape), _randn(gen, *shape)
        s["lut"] = _lut(case, seed)
    elif kind == "decode_attention":
        b, h, d = case["batch"], case["heads"], case["dim"]
        s["q"] = _randn(gen, b, h, 1, d)
        s["k"], s["v"] = _randn(gen, b, h, case["rows"], d), _randn(gen, b, h, case["rows"], d)
        s["bias"] = None
        if case["mask"]:  # left padding of up to half the cache, as a batched tokenizer leaves it
            pad = torch.randint(0, case["rows"] // 2, (b, 1, 1, 1), device=DEV, generator=gen)
            rows = torch.arange(case["rows"], device=DEV).view(1, 1, 1, -1)
            s["bias"] = torch.where(rows < pad, float("-inf"), 0.0).half()
    elif kind == "pack":
        m = nn.Linear(case["k"], case["n"], bias=True, device=DEV, dtype=torch.float16)
        m.weight.data, m.bias.data = _randn(gen, case["n"], case["k"], scale=0.02), _randn(gen, case["n"], scale=0.01)
        s["module"] = m
    elif kind == "dequant":
        s["lin"] = _walinear(gen, case["k"], case["n"], case["group"], case["layout"], bias=False)
    else:
        raise ValueError("unknown kind %r" % kind)
    return s


@torch.no_grad()
def run(s):
    kind = s["kind"]
    if kind == "linear":
        return s["lin"](s["x"], residual=s["res"], act=s["act"])
    if kind == "layer":
        qkv = s["qkv"](s["x"], pre_ln=s["ln1"])
        x = s["out"](s["attn"], residual=s["x"])
        h = s["fc1"](x, act="relu", pre_ln=s["ln2"])
        return qkv, x, h, s["fc2"](h, residual=x)
    if kind == "gated":
        qkv = s["qkv"](s["x"])
        x = s["out"](s["attn"], residual=s["x"])
        gate, up = s["gate"], s["up"]
        h = quant.gemm_awq_silu_dot_ut(x, gate.weight, up.weight, gate.zeros_scales, up.zeros_scales, None, None,
                                       s["tokens"], s["ffn"], s["hidden"], s["group"])
        return qkv, x, h, s["down"](h, residual=x)
    if kind == "step":
        s["tok"].copy_(s["next"])
        s["pos"].fill_(s["rows"])
        s["graph"].replay()
        return s["logits"], s["tok"], s["cache"]
    if kind == "prefill":
        return s["model"](s["ids"], s["cache"], 0), s["cache"]
    if kind == "lut_attention":
        return sparse_attention(s["q"], s["k"], s["v"], s["dim"] ** -0.5, s["lut"], LT=s["causal"])
    if kind == "decode_attention":
        return sparse_attention(s["q"], s["k"], s["v"], s["dim"] ** -0.5, None, attention_mask=s["bias"])
    if kind == "pack":
        lin = WALinear.from_float(s["module"], {"n_bit": s["bits"], "group_size": s["group"]}, layout=s["layout"])
        return lin.weight, lin.zeros_scales, lin.bias
    lin = s["lin"]
    return quant.dequant(lin.weight, lin.zeros_scales, s["n"], s["k"], s["group"])


def _linear_work(tokens, n, k, group, bits=4):
    return n * k * bits // 8 + (k // group) * n * 4 + tokens * (k + n) * 2, 2 * tokens * n * k


def _kept_pairs(seq, density, causal):
    """Query-key pairs of one head that the look-up table keeps (block 64)."""
    nb = (seq + 63) // 64
    keep = max(1, int(round(density * nb)))
    pairs = 0
    for i in range(nb):
        rows = min(64, seq - 64 * i)
        if causal:
            pairs += rows * (rows + 1) // 2 + min(keep - 1, i) * 64 * rows
        else:
            pairs += min(keep, nb) * 64 * rows
    return pairs


def work(case):
    kind = case["kind"]
    parts = []
    extra_bytes = extra_flops = 0
    if kind == "linear":
        parts = [_linear_work(case["tokens"], case["n"], case["k"], case["group"], case["bits"])]
        extra_bytes = case["n"] * 2 + (case["tokens"] * case["n"] * 2 if case["residual"] else 0)
    elif kind in ("layer", "gated"):
        t, h, f, g = case["tokens"], case["hidden"], case["ffn"], case["group"]
        up = 2 if kind == "gated" else 1
        parts = [_linear_work(t, 3 * h, h, g), _linear_work(t, h, h, g), _linear_work(t, h, f, g)]
        parts += [_linear_work(t, f, h, g)] * up
        extra_bytes = t * h * 2
    elif kind in ("step", "prefill"):
        h, f, vocab = 4096, 16384, 50272
        b = case["batch"]
        t = b if kind == "step" else b * case["prompt"]
        for _ in range(case["layers"]):
            parts += [_linear_work(t, 3 * h, h, 128), _linear_work(t, h, h, 128), _linear_work(t, f, h, 128),
                      _linear_work(t, h, f, 128)]
            if kind == "step":
                extra_bytes += 2 * t * h * (case["rows"] + 1) * 2
                extra_flops += 4 * t * h * (case["rows"] + 1)
            else:
                pairs = _kept_pairs(case["prompt"], case["density"] or 1.0, True)
                extra_bytes += 2 * t * h * 2
                extra_flops += 4 * b * h * pairs
        extra_bytes += vocab * h * 2 + b * vocab * 2
        extra_flops += 2 * b * vocab * h
    elif kind == "lut_attention":
        z = case["batch"] * case["heads"]
        extra_bytes = 4 * z * case["seq"] * case["dim"] * 2
        extra_flops = 4 * z * case["dim"] * _kept_pairs(case["seq"], case["density"], case["causal"])
    elif kind == "decode_attention":
        z = case["batch"] * case["heads"]
        extra_bytes = 2 * z * (case["rows"] + 1) * case["dim"] * 2
        extra_flops = 4 * z * case["rows"] * case["dim"]
    else:
        nk = case["n"] * case["k"]
        extra_bytes = nk * 2 + nk * case["bits"] // 8 + nk // case["group"] * 4
        extra_flops = nk * 2
    return {"bytes": sum(p[0] for p in parts) + extra_bytes, "flops": sum(p[1] for p in parts) + extra_flops}


def tolerance(case):
    """About four times what each path differs by from itself carried out in float64 from the same fp16 inputs
    (measured: linear 2.1e-4..3.6e-4, attention 2.1e-4..3.6e-4, layer and gated up to 7.7e-4 on their worst output,
    step 1.1e-3, prefill 5e-4)."""
    kind = case["kind"]
    if kind in ("pack", "dequant"):
        return "exact"
    if kind in ("layer", "gated"):
        return {"rel": 3e-3}
    if kind == "step":
        return {"rel": 4e-3, "differ": 0.25}  # of up to 8 chosen tokens, the other one of a near tie
    if kind == "prefill":
        return {"rel": 2e-3}
    return {"rel": 1.4e-3}
