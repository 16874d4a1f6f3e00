"""The workloads this framework's speed is judged by: one pass of each through the public Python API.

Every case is a dict of plain values with a "kind" (which call it makes) and the sizes, storage
formats and options of that call; prepare() builds what a program holds before the call (packed
weights, activations, adapters), run() makes one pass, exact() gives the same outputs in 64 bits
with plain torch.  Shapes are those of the models whose linears the framework serves: FLUX.1 and
Wan transformer blocks, SDXL's fp16 U-Net and text encoders, decoder-only text encoders with
prefill and token-by-token decode, stacked mixture-of-experts projections, and the conversion of
dense weights to packed ones and back.
"""
import math
import os
import sys

import torch

_PKG = os.path.join(os.getcwd(), "mlx-gen_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import mlxq  # noqa: E402

_DTYPES = {"bf16": torch.bfloat16, "f32": torch.float32, "f16": torch.float16}
_ACTS = {"none": mlxq.MLXQ_ACT_NONE, "gelu": mlxq.MLXQ_ACT_GELU, "gelu_tanh": mlxq.MLXQ_ACT_GELU_TANH,
         "gelu_exact": mlxq.MLXQ_ACT_GELU_EXACT}


def _linear(name, M, K, N, x="bf16", bits=4, gs=64, bias="none", act="none", rank=0):
    return {"name": name, "kind": "linear", "M": M, "K": K, "N": N, "x": x, "bits": bits, "gs": gs, "bias": bias,
            "act": act, "rank": rank}


def listed():
    return [
        # One token of a 3B-class decoder's SwiGLU MLP: gate and up fused, then down.  The smallest
        # call: launches and latency.
        {"name": "decode_mlp_1", "kind": "mlp", "M": 1, "K": 3072, "F": 8192, "bits": 4, "gs": 64},
        # The same step for five sequences at once on a 7B-class MLP, whose width (86 x 128) does
        # not divide evenly.
        {"name": "decode_mlp_5", "kind": "mlp", "M": 5, "K": 4096, "F": 11008, "bits": 4, "gs": 64},
        # adaLN modulation of a diffusion transformer block: one conditioning row, wide output, bias.
        _linear("modulation", 1, 3072, 18432, bits=8, gs=64, bias="bf16"),
        # Text-encoder prefill of an odd-length prompt: token rows gathered from the packed table,
        # then one projection of them.
        {"name": "prompt", "kind": "prompt", "M": 333, "K": 3072, "N": 4096, "vocab": 32000, "bits": 4, "gs": 64},
        # fp16 text encoder (77 tokens): first feed-forward linear with its activation.
        _linear("clip_fc1", 77, 1280, 5120, x="f16", bits=8, gs=64, bias="bf16", act="gelu"),
        # fp16 U-Net feed-forward projection at 64 x 64 latents.
        _linear("unet_ff", 4096, 1280, 10240, x="f16", bits=4, gs=64, bias="bf16"),
        # bf16 diffusion transformer MLP (4096 image + 512 text tokens): up with GELU, then down.
        {"name": "dit_mlp", "kind": "dit_mlp", "M": 4608, "K": 3072, "F": 12288, "bits": 4, "gs": 64},
        # Joint QKV projection of the same block with bias and a rank-16 LoRA adapter.
        _linear("qkv_lora", 4608, 3072, 9216, bits=8, gs=128, bias="bf16", rank=16),
        # The feed-forward of the same model on its f32 residual stream, with a rank-32 adapter.
        _linear("ff_f32_lora", 4608, 3072, 12288, x="f32", bits=4, gs=64, bias="bf16", act="gelu", rank=32),
        # Gate/up projection of every expert of a mixture-of-experts encoder layer (K: 45 groups).
        {"name": "experts", "kind": "experts", "E": 32, "M": 512, "K": 2880, "N": 5760, "bits": 4, "gs": 64},
        # Converting one attention block's dense weights to packed ones, and unpacking one of them.
        {"name": "pack", "kind": "pack", "count": 4, "N": 5120, "K": 5120, "bits": 8, "gs": 64, "w": "bf16"},
        # A video transformer's attention projection over 32760 tokens.  The largest call.
        _linear("video_proj", 32760, 5120, 5120, bits=8, gs=64, bias="bf16"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _mult(rng, lo, hi, step):
    """A multiple of step, spread over the logarithm of [lo, hi]."""
    return min(hi // step, max(-(-lo // step), round(_log(rng, lo, hi) / step))) * step


def draw(rng):
    kind = rng.choice(["mlp", "prompt", "decode", "prefill", "image", "image", "dit_mlp", "experts", "pack"])
    bits, gs = rng.choice([4, 4, 8]), rng.choice([32, 64, 64, 128])
    if kind == "mlp":
        return {"kind": "mlp", "M": rng.randint(1, 8), "K": _mult(rng, 1024, 4096, 128),
                "F": _mult(rng, 2048, 14336, 128), "bits": bits, "gs": gs}
    if kind == "prompt":
        return {"kind": "prompt", "M": _log(rng, 9, 512), "K": _mult(rng, 768, 4096, 128),
                "N": _log(rng, 768, 8192), "vocab": _log(rng, 4000, 50000), "bits": bits, "gs": gs}
    if kind == "dit_mlp":
        return {"kind": "dit_mlp", "M": _log(rng, 1024, 4608), "K": _mult(rng, 1152, 3072, 128),
                "F": _mult(rng, 4608, 12288, 128), "bits": bits, "gs": gs}
    if kind == "experts":
        return {"kind": "experts", "E": rng.choice([4, 8, 16, 32]), "M": _log(rng, 1, 512),
                "K": _mult(rng, 1024, 2880, gs), "N": 2 * _log(rng, 720, 2880), "bits": bits, "gs": gs}
    if kind == "pack":
        return {"kind": "pack", "count": rng.randint(1, 4), "N": _log(rng, 640, 5120), "K": _mult(rng, 640, 5120, gs),
                "bits": bits, "gs": gs, "w": rng.choice(["bf16", "bf16", "f32"])}
    # Single linears: one to eight rows, a prompt's rows, an image's rows.
    rows = {"decode": (1, 8), "prefill": (9, 512), "image": (513, 4608)}[kind]
    c = _linear(None, _log(rng, *rows), _mult(rng, 640, 6144, gs), _log(rng, 640, 12288),
                x=rng.choice(["bf16", "bf16", "f16", "f32"]), bits=bits, gs=gs, bias=rng.choice(["none", "bf16"]))
    del c["name"]
    if kind == "image":
        c["rank"] = rng.choice([0, 0, 8, 16, 32])
    if kind != "decode":
        c["act"] = rng.choice(["none", "none", "gelu_exact", "gelu_tanh"] if c["x"] == "bf16" else ["none", "none", "gelu"])
    return c


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _randn(g, shape, std=1.0, dtype=torch.bfloat16):
    return (torch.randn(shape, generator=g, device="cuda", dtype=torch.float32) * std).to(dtype)


def _affine(w, gs, bits):
    """Per-group affine quantization in w's own precision: codes [N, K] (int32), scale and bias
    [N, K/gs].  The range end of larger magnitude is reproduced exactly."""
    N, K = w.shape
    g = w.view(N, K // gs, gs)
    lo, hi = g.amin(-1), g.amax(-1)
    s = ((hi - lo) / (2 ** bits - 1)).clamp_min(1e-7)
    side = lo.abs() > hi.abs()
    s = torch.where(side, s, -s)
    edge = torch.where(side, lo, hi)
    q0 = torch.round(edge / s)
    s = torch.where(q0 != 0, edge / torch.where(q0 != 0, q0, torch.ones_like(q0)), s)
    b = torch.where(q0 != 0, edge, torch.zeros_like(edge))
    q = (g - b[..., None]) / s[..., None]
    codes = (torch.sign(q) * torch.floor(q.abs() + 0.5)).clamp(0, 2 ** bits - 1)
    return codes.to(torch.int32).view(N, K), s, b


def _pack(w, gs, bits):
    """The packed triple of w as a checkpoint holds it: 32/bits codes per word, low bits first."""
    codes, s, b = _affine(w.float(), gs, bits)
    N, K = w.shape
    per = 32 // bits
    c = codes.view(N, K // per, per)
    words = c[..., 0].clone()
    for i in range(1, per):
        words |= c[..., i] << (i * bits)
    # scales and biases in one buffer, as the framework's own quantize lays them out
    n = s.numel()
    buf = torch.empty(2 * n + 256, dtype=torch.bfloat16, device=w.device)
    at = (n + 255) // 128 * 128
    sb = buf[:n].view(s.shape), buf[at:at + n].view(s.shape)
    sb[0].copy_(s)
    sb[1].copy_(b)
    return words, sb[0], sb[1]


def _weight(g, N, K, gs, bits):
    return _pack(_randn(g, (N, K), 0.02), gs, bits)


def prepare(case, seed):
    g = _gen(seed)
    k, gs, bits = case["kind"], case["gs"], case["bits"]
    s = {"case": case}
    if k == "linear":
        M, K, N, r = case["M"], case["K"], case["N"], case["rank"]
        s["w"] = _weight(g, N, K, gs, bits)
        s["x"] = _randn(g, (M, K), 1.0, _DTYPES[case["x"]])
        s["bias"] = None if case["bias"] == "none" else _randn(g, (N,), 0.1, _DTYPES[case["bias"]])
        s["a"] = _randn(g, (K, r), 0.01) if r else None
        s["b"] = _randn(g, (r, N), 0.01) if r else None
    elif k in ("mlp", "dit_mlp"):
        s["x"] = _randn(g, (case["M"], case["K"]))
        if k == "mlp":
            s["gate"] = _weight(g, case["F"], case["K"], gs, bits)
        s["up"] = _weight(g, case["F"], case["K"], gs, bits)
        s["down"] = _weight(g, case["K"], case["F"], gs, bits)
    elif k == "prompt":
        s["ids"] = torch.randint(0, case["vocab"], (case["M"],), generator=g, device="cuda", dtype=torch.int32)
        s["table"] = _weight(g, case["vocab"], case["K"], gs, bits)
        s["w"] = _weight(g, case["N"], case["K"], gs, bits)
    elif k == "experts":
        E, M, K, N = case["E"], case["M"], case["K"], case["N"]
        wq, sc, bi = _weight(g, E * N, K, gs, bits)
        s["w"] = wq.view(E, N, -1), sc.view(E, N, -1), bi.view(E, N, -1)
        s["x"] = _randn(g, (M, K))
        s["bias"] = _randn(g, (E, N), 0.1)
    elif k == "pack":
        s["ws"] = [_randn(g, (case["N"], case["K"]), 0.02, _DTYPES[case["w"]]) for _ in range(case["count"])]
    return s


def run(s):
    c = s["case"]
    k, gs, bits = c["kind"], c["gs"], c["bits"]
    if k == "linear":
        return mlxq.linear(s["x"], *s["w"], gs, bits, bias=s["bias"], lora_a=s["a"], lora_b=s["b"], lora_scale=0.75,
                           activation=_ACTS[c["act"]])
    if k == "mlp":
        h = mlxq.swiglu(s["x"], s["gate"], s["up"], gs, bits)
        return mlxq.quantized_matmul(h, *s["down"], True, gs, bits)
    if k == "dit_mlp":
        h = mlxq.linear(s["x"], *s["up"], gs, bits, activation=mlxq.MLXQ_ACT_GELU_EXACT)
        return h, mlxq.quantized_matmul(h, *s["down"], True, gs, bits)
    if k == "prompt":
        h = mlxq.embedding(s["ids"], *s["table"], gs, bits, out_dtype=torch.bfloat16)
        return h, mlxq.quantized_matmul(h, *s["w"], True, gs, bits)
    if k == "experts":
        return mlxq.qmm_experts(s["x"], *s["w"], gs, bits, bias=s["bias"])
    packs = mlxq.quantize_batched(s["ws"], gs, bits)
    return [t for p in packs for t in p], mlxq.dequantize(*packs[0], gs, bits)


def _packed_bytes(N, K, gs, bits, sb=2):
    return N * K * bits / 8 + 2 * N * (K // gs) * sb


def work(case):
    k, gs, bits = case["kind"], case["gs"], case["bits"]
    K = case["K"]
    if k == "linear":
        M, N, r = case["M"], case["N"], case["rank"]
        xb = 4 if case["x"] == "f32" else 2
        yb = 2 if case["x"] == "bf16" and case["act"] != "gelu" else 4
        n = M * K * xb + _packed_bytes(N, K, gs, bits) + M * N * yb + (2 * N if case["bias"] != "none" else 0)
        return {"bytes": n + 2 * r * (K + N), "flops": 2 * M * K * N + 2 * M * r * (K + N)}
    if k == "mlp":
        M, F = case["M"], case["F"]
        return {"bytes": 2 * _packed_bytes(F, K, gs, bits) + _packed_bytes(K, F, gs, bits) + 4 * M * K,
                "flops": 6 * M * K * F}
    if k == "dit_mlp":
        M, F = case["M"], case["F"]
        return {"bytes": _packed_bytes(F, K, gs, bits) + _packed_bytes(K, F, gs, bits) + 4 * M * K + 2 * M * F,
                "flops": 4 * M * K * F}
    if k == "prompt":
        M, N = case["M"], case["N"]
        return {"bytes": 4 * M + _packed_bytes(M, K, gs, bits) + 2 * M * K + _packed_bytes(N, K, gs, bits) + 2 * M * N,
                "flops": 2 * M * K * N}
    if k == "experts":
        E, M, N = case["E"], case["M"], case["N"]
        return {"bytes": 2 * M * K + _packed_bytes(E * N, K, gs, bits) + 2 * E * N + 2 * E * M * N,
                "flops": 2 * E * M * K * N}
    N, wb = case["N"], 4 if case["w"] == "f32" else 2
    return {"bytes": case["count"] * (N * K * wb + _packed_bytes(N, K, gs, bits, wb)) + _packed_bytes(N, K, gs, bits, wb)
            + N * K * wb, "flops": 0}


def tolerance(case):
    if case["kind"] == "pack":
        return "exact"
    if case["kind"] == "linear" and case["x"] != "bf16":
        # f32 results.  Measured against 64 bits: up to 2.8e-6 from fp16 activations and 9.7e-6 from
        # f32 ones (carried on the matrix cores to 16 significant bits).
        return {"rel": 1e-5 if case["x"] == "f16" else 4e-5}
    # bf16 results: 1.6e-3 to 2.9e-3 measured for one linear, up to 4.2e-3 where the decode MLP and
    # the GELUs round at several points on the way.
    return {"rel": 1e-2}


def _dense64(w, gs, bits, tile_bf16):
    """The dequantized weights in 64 bits; with tile_bf16 rounded to bf16 first, as the product of
    bf16 operands over more than 8 rows is defined (dequantize, then a bf16 matmul)."""
    wq, s, b = w
    per = 32 // bits
    shift = torch.arange(0, 32, bits, device=wq.device, dtype=torch.int32)
    codes = ((wq[..., None] >> shift) & (2 ** bits - 1)).view(wq.shape[0], wq.shape[1] * per)
    d = codes.view(wq.shape[0], -1, gs).double() * s.double()[..., None] + b.double()[..., None]
    d = d.view(codes.shape)
    return d.float().to(torch.bfloat16).double() if tile_bf16 else d


def _act64(y, act):
    if act == "none":
        return y
    if act == "gelu_tanh":
        return 0.5 * y * (1 + torch.tanh(math.sqrt(2 / math.pi) * (y + 0.044715 * y ** 3)))
    return 0.5 * y * (1 + torch.erf(y / math.sqrt(2)))


def exact(case, seed):
    s = prepare(case, seed)
    k, gs, bits = case["kind"], case["gs"], case["bits"]
    if k == "linear":
        x = s["x"].double()
        y = x @ _dense64(s["w"], gs, bits, case["x"] == "bf16" and case["M"] > 8).t().contiguous()
        if s["bias"] is not None:
            y += s["bias"].double()
        if s["a"] is not None:
            y += 0.75 * ((x @ s["a"].double()) @ s["b"].double())
        return _act64(y, case["act"])
    if k == "mlp":
        x = s["x"].double()
        gate = x @ _dense64(s["gate"], gs, bits, False).t().contiguous()
        h = gate * torch.sigmoid(gate) * (x @ _dense64(s["up"], gs, bits, False).t().contiguous())
        return h @ _dense64(s["down"], gs, bits, False).t().contiguous()
    if k == "dit_mlp":
        h = _act64(s["x"].double() @ _dense64(s["up"], gs, bits, True).t().contiguous(), "gelu")
        return h, h @ _dense64(s["down"], gs, bits, True).t().contiguous()
    if k == "prompt":
        rows = tuple(t[s["ids"].long()] for t in s["table"])
        h = _dense64(rows, gs, bits, False)
        return h, h @ _dense64(s["w"], gs, bits, case["M"] > 8).t().contiguous()
    if k == "experts":
        x = s["x"].double()
        return torch.stack([x @ _dense64(tuple(t[e] for t in s["w"]), gs, bits, case["M"] > 8).t().contiguous()
                            + s["bias"][e].double() for e in range(case["E"])])
    out, w0 = [], None
    for w in s["ws"]:
        codes, sc, bi = _affine(w.double(), gs, bits)
        out += [None, sc, bi]
        if w0 is None:
            r = lambda t: t.to(w.dtype).double().repeat_interleave(gs, 1)  # noqa: E731
            w0 = codes.double() * r(sc) + r(bi)
    return out, w0
