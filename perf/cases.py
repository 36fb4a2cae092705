"""The workloads this library's speed is measured on.

Each case is one call of a public entry point of ``nn_amd`` as an inference program makes it:
a quantized linear, the SwiGLU MLP, the LM head or the mixture-of-experts layer, at decode
(one token), batched decode (a few tokens) and prefill (hundreds to thousands of tokens).

``listed`` gives the fixed cases, ``draw`` further ones of the same ranges, ``prepare`` the
weights and inputs, ``run`` one pass, ``work`` the bytes and operations it cannot do without,
``exact`` its result in 64 bits from a decode of the same block bytes in plain torch.
"""
from __future__ import annotations

import math

import torch

import nn_amd

DEV = "cuda:0"
DTYPES = {"f32": torch.float32, "bf16": torch.bfloat16}
FORMATS = {"q8_0": nn_amd.QuantType.Q8_0, "q4_k": nn_amd.QuantType.Q4_K, "q6_k": nn_amd.QuantType.Q6_K}
# nn-gguf's layout is the only Q6_K layout there is
LAYOUTS = {"q8_0": nn_amd.Layout.GGUF, "q4_k": nn_amd.Layout.GGUF, "q6_k": nn_amd.Layout.NN_GGUF}


def linear(fmt, m, n, k, x="bf16", out="f32", bias=False):
    return {"kind": "linear", "fmt": fmt, "m": m, "n": n, "k": k, "x": x, "out": out, "bias": bias}


def mlp(m, hidden, inter, x="bf16", out="f32"):
    return {"kind": "mlp", "m": m, "hidden": hidden, "inter": inter, "x": x, "out": out}


def head(n, k):
    return {"kind": "head", "n": n, "k": k}


def moe(m, experts, top_k, hidden, inter, x="bf16", router=True):
    return {"kind": "moe", "m": m, "experts": experts, "top_k": top_k, "hidden": hidden, "inter": inter, "x": x,
            "router": router}


def listed():
    cases = {
        # one token through a Q8_0 attention projection, f32 as the op's default: the smallest call
        "decode_q8_0": linear("q8_0", 1, 4096, 4096, x="f32"),
        # one token through a Q4_K Qwen3-8B MLP: most of a decode step's weight bytes
        "decode_mlp_q4_k": mlp(1, 4096, 12288),
        # greedy decoding's LM head over the whole vocabulary: logits and their argmax
        "decode_head_q6_k": head(151936, 4096),
        # the LM head of a served batch of eight sequences
        "batch8_head_q6_k": linear("q6_k", 8, 151936, 4096),
        # a served batch of a dozen sequences through a biased Q8_0 projection
        "batch12_q8_0": linear("q8_0", 12, 4096, 4096, out="bf16", bias=True),
        # six speculated tokens through the down projection, f32 activations
        "batch6_q4_k_f32": linear("q4_k", 6, 4096, 12288, x="f32"),
        # a prompt of odd length in the reference's own dtype through the up projection
        "prefill203_q4_k_f32": linear("q4_k", 203, 12288, 4096, x="f32"),
        # a prompt of 512 tokens through the whole MLP
        "prefill512_mlp_q4_k": mlp(512, 4096, 12288, out="bf16"),
        # the same prompt through the Q6_K down projection that mixed Q4_K files hold
        "prefill512_q6_k": linear("q6_k", 512, 4096, 12288, out="bf16"),
        # one token through a GPT-OSS expert layer: router, four experts, combine
        "decode_moe": moe(1, 32, 4, 2880, 2880),
        # a short prompt or a served batch through the same layer: every expert in use
        "prefill256_moe": moe(256, 32, 4, 2880, 2880),
        # a long prompt, routing decided by the caller: many rows per expert
        "prefill2048_moe": moe(2048, 32, 4, 2880, 2880, router=False),
    }
    return [dict(name=name, **case) for name, case in cases.items()]


def _log_uniform(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(("linear", "linear", "linear", "linear", "linear", "mlp", "mlp", "head", "moe", "moe"))
    x = rng.choice(("bf16", "bf16", "f32"))
    out = rng.choice(("bf16", "f32"))
    if kind == "linear":
        fmt = rng.choice(("q8_0", "q4_k", "q6_k"))
        k = 256 * _log_uniform(rng, 4, 48)
        if fmt == "q8_0" and rng.random() < 0.25:
            k += 32 * rng.randint(1, 7)  # Q8_0 rows are whole 32-element blocks only
        n = _log_uniform(rng, 512, 24576)
        if rng.random() < 0.7:
            n = (n + 127) // 128 * 128  # models' widths; the rest any number of rows
        m = min(_log_uniform(rng, 1, 2048), int(1.5e11 / (2 * n * k)))
        return linear(fmt, m, n, k, x, out, rng.random() < 0.3)
    if kind == "mlp":
        hidden = 256 * rng.choice((4, 8, 10, 16, 20))
        inter = 256 * _log_uniform(rng, 12, 48)
        m = min(_log_uniform(rng, 1, 2048), int(1.8e11 / (6 * hidden * inter)))
        return mlp(m, hidden, inter, x, out)
    if kind == "head":
        return head(_log_uniform(rng, 30000, 152064), 256 * _log_uniform(rng, 4, 20))
    experts = rng.choice((8, 16, 32, 64))
    top_k = rng.choice((1, 2, 4, 4, 6, 8))
    hidden, inter = 32 * _log_uniform(rng, 24, 90), 32 * _log_uniform(rng, 16, 90)
    while experts * hidden * inter > 32 * 2880 * 2880:
        experts //= 2
    m = min(_log_uniform(rng, 1, 2048), int(4e11 / (6 * top_k * hidden * inter)))
    return moe(m, experts, top_k, hidden, inter, x, rng.random() < 0.6)


# ---- inputs --------------------------------------------------------------------------------


def _generator(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed))
    return g


def _activations(g, m, k, dtype):
    """N(0, 1) tokens whose channels differ in size, as a model's hidden states do."""
    channel = torch.exp(0.5 * torch.randn(k, generator=g, device=DEV))
    return (torch.randn(m, k, generator=g, device=DEV) * channel).to(dtype)


def _f16_bytes(t):
    return t.to(torch.float16).contiguous().view(torch.uint8)


def _codes(g, count, length, mean, spread, top):
    """Codes of normally distributed values, uint8 [count, length]."""
    v = torch.randn(count, length, generator=g, device=DEV, dtype=torch.float16).mul_(spread).add_(mean)
    return v.round_().clamp_(0, top).to(torch.uint8)


def _ints(g, lo, hi, shape):
    return torch.randint(lo, hi, shape, generator=g, device=DEV, dtype=torch.int32).to(torch.uint8)


def _q8_0(g, nb):
    """Q8_0 blocks of N(0, 0.02) weights: [d f16][32 int8]."""
    d = 0.02 * (0.9 + 0.4 * torch.rand(nb, 1, generator=g, device=DEV)) * 2.1 / 127
    q = (_codes(g, nb, 32, 128, 55, 255).to(torch.int16) - 128).clamp_(-127, 127).to(torch.int8)
    return torch.cat((_f16_bytes(d), q.view(torch.uint8)), 1)


def _q4_k(g, nb):
    """Q4_K super-blocks of N(0, 0.02) weights: [d, dmin f16][12 scale bytes][128 nibble bytes]."""
    spread = 0.02 * (0.9 + 0.2 * torch.rand(nb, 1, generator=g, device=DEV))
    d, dmin = spread * 4.4 / 15 / 63, spread * 2.4 / 63
    sc, mn = _ints(g, 36, 64, (nb, 8)), _ints(g, 36, 64, (nb, 8))
    packed = torch.cat((sc[:, :4] | (sc[:, 4:] >> 4 << 6), mn[:, :4] | (mn[:, 4:] >> 4 << 6),
                        (sc[:, 4:] & 15) | ((mn[:, 4:] & 15) << 4)), 1)
    q = _codes(g, nb, 256, 7.5, 3.4, 15).view(nb, 4, 2, 32)  # pairs of sub-blocks share their bytes
    return torch.cat((_f16_bytes(d), _f16_bytes(dmin), packed, (q[:, :, 0] | (q[:, :, 1] << 4)).reshape(nb, 128)), 1)


def _q6_k(g, nb):
    """Q6_K super-blocks of N(0, 0.02) weights: [128 low nibbles][64 high crumbs][16 int8][d f16]."""
    d = 0.02 * (0.9 + 0.2 * torch.rand(nb, 1, generator=g, device=DEV)) * 2.2 / 31 / 127
    sc = _ints(g, 70, 128, (nb, 16))
    q = _codes(g, nb, 256, 32, 13, 63)
    lo, hi = q & 15, q >> 4
    return torch.cat((lo[:, 0::2] | (lo[:, 1::2] << 4),
                      hi[:, 0::4] | (hi[:, 1::4] << 2) | (hi[:, 2::4] << 4) | (hi[:, 3::4] << 6), sc, _f16_bytes(d)), 1)


def _weight_bytes(g, fmt, n, k):
    """Block bytes of a weight [n, k] on the device, [blocks, block bytes], in slices that fit."""
    make, block = {"q8_0": (_q8_0, 32), "q4_k": (_q4_k, 256), "q6_k": (_q6_k, 256)}[fmt]
    total, step = n * k // block, (1 << 26) // block
    return torch.cat([make(g, min(step, total - i)) for i in range(0, total, step)])


def _moe_weights(g, experts, k, n):
    """MXFP4 experts [experts, k, n] of N(0, 0.02) weights: packed codes, E8M0 scale bytes, bias."""
    edges = torch.tensor([0.25, 0.75, 1.25, 1.75, 2.5, 3.5, 5.0], device=DEV, dtype=torch.float16)

    def matrix():
        v = torch.randn(k, n, generator=g, device=DEV, dtype=torch.float16).mul_(2.4)
        c = torch.bucketize(v.abs(), edges, out_int32=True).to(torch.uint8) | ((v < 0).to(torch.uint8) << 3)
        return (c[:, 0::2] << 4) | c[:, 1::2]

    packed = torch.stack([matrix() for _ in range(experts)])
    return packed, _ints(g, 119, 122, (experts, k, n // 32)), torch.randn(experts, n, generator=g, device=DEV) * 0.02


def _inputs(case, seed):
    """Everything a case's call takes, as tensors on the device, from the seed alone."""
    g = _generator(seed)
    kind = case["kind"]
    if kind == "linear":
        d = {"w": _weight_bytes(g, case["fmt"], case["n"], case["k"]),
             "x": _activations(g, case["m"], case["k"], DTYPES[case["x"]])}
        d["bias"] = torch.randn(case["n"], generator=g, device=DEV) * 0.1 if case["bias"] else None
        return d
    if kind == "head":
        return {"w": _weight_bytes(g, "q6_k", case["n"], case["k"]),
                "x": _activations(g, 1, case["k"], torch.float32)[0]}
    if kind == "mlp":
        h, i = case["hidden"], case["inter"]
        return {"gate": _weight_bytes(g, "q4_k", i, h), "up": _weight_bytes(g, "q4_k", i, h),
                "down": _weight_bytes(g, "q4_k", h, i), "x": _activations(g, case["m"], h, DTYPES[case["x"]])}
    e, h, i = case["experts"], case["hidden"], case["inter"]
    d = {"gu": _moe_weights(g, e, h, 2 * i), "dn": _moe_weights(g, e, i, h),
         "x": torch.randn(case["m"], h, generator=g, device=DEV).to(DTYPES[case["x"]]), "rw": None, "rb": None,
         "logits": None}
    if case["router"]:
        d["rw"] = torch.randn(e, h, generator=g, device=DEV) * 0.02
        d["rb"] = torch.randn(e, generator=g, device=DEV) * 0.1
    else:
        d["logits"] = torch.randn(case["m"], e, generator=g, device=DEV)
    return d


def prepare(case, seed):
    d = _inputs(case, seed)
    kind = case["kind"]
    state = {"case": case, "x": d["x"]}
    if kind in ("linear", "head"):
        fmt = case.get("fmt", "q6_k")
        state["w"] = nn_amd.QuantizedWeight.from_quantized(d["w"], FORMATS[fmt], (case["n"], case["k"]),
                                                           layout=LAYOUTS[fmt])
        state["bias"] = d.get("bias")
    elif kind == "mlp":
        state["mlp"] = nn_amd.QuantizedMLP(d["gate"], d["up"], d["down"], nn_amd.QuantType.Q4_K, case["hidden"],
                                           case["inter"])
    else:
        host = {name: None if d[name] is None else d[name].cpu().numpy() for name in ("rw", "rb")}
        (gp, gs, gb), (dp, ds, db) = d["gu"], d["dn"]
        state["moe"] = nn_amd.QuantizedMoE(case["experts"], case["hidden"], case["inter"], gp, gs, gb.cpu().numpy(),
                                           dp, ds, db.cpu().numpy(), router_weight=host["rw"],
                                           router_bias=host["rb"])
        state["logits"] = d["logits"]
    return state


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "linear":
        return nn_amd.quantized_linear(state["x"], state["w"], state["bias"], out_dtype=DTYPES[case["out"]])
    if kind == "head":
        return nn_amd.linear_argmax(state["x"], state["w"], check=False)
    if kind == "mlp":
        return state["mlp"].forward(state["x"], out_dtype=DTYPES[case["out"]], check=False)
    if case["router"]:
        return state["moe"].block_forward(state["x"], top_k=case["top_k"], check=False)
    return state["moe"].forward(state["x"], state["logits"], top_k=case["top_k"])


# ---- what a pass cannot do without -----------------------------------------------------------


def work(case):
    size = {"f32": 4, "bf16": 2}
    bits = {"q8_0": 34 / 32, "q4_k": 144 / 256, "q6_k": 210 / 256}
    kind = case["kind"]
    if kind in ("linear", "head"):
        m, n, k = case.get("m", 1), case["n"], case["k"]
        nbytes = n * k * bits[case.get("fmt", "q6_k")] + m * k * size[case.get("x", "f32")]
        nbytes += m * n * size[case.get("out", "f32")] + (4 * n if case.get("bias") else 0)
        return {"bytes": int(nbytes), "flops": 2 * m * n * k}
    if kind == "mlp":
        m, h, i = case["m"], case["hidden"], case["inter"]
        return {"bytes": int(3 * h * i * bits["q4_k"]) + m * h * (size[case["x"]] + size[case["out"]]),
                "flops": 6 * m * h * i}
    m, e, k, h, i = case["m"], case["experts"], case["top_k"], case["hidden"], case["inter"]
    used = e * (1 - (1 - k / e) ** m)  # experts with a token
    nbytes = used * (3 * h * i * 17 / 32 + 4 * (2 * i + h)) + m * h * (size[case["x"]] + 4)
    nbytes += 4 * e * (h + 1) if case["router"] else 4 * m * e
    return {"bytes": int(nbytes), "flops": 6 * m * k * h * i + (2 * m * e * h if case["router"] else 0)}


def tolerance(case):
    if case["kind"] != "moe" and case.get("out") == "bf16":
        return {"rel": 7e-3}  # one rounding to bf16
    if case["kind"] == "mlp" or case.get("fmt") == "q4_k":
        return {"rel": 5e-5}  # f32 sums, offset and minimum terms cancelling in them (1.2e-5 seen)
    return {"rel": 1e-5}  # f32 sums; experts: f32 inputs and the SwiGLU output as pairs of bf16 (2.5e-6 seen)


# ---- the result in 64 bits -------------------------------------------------------------------


def _f16_of(b):
    return b.contiguous().view(torch.float16).double()


def _decode(blocks, fmt, k):
    """Block bytes [blocks, bytes] to weights [rows, k] in f64."""
    nb = blocks.shape[0]
    if fmt == "q8_0":
        w = _f16_of(blocks[:, :2]) * blocks[:, 2:].contiguous().view(torch.int8).double()
    elif fmt == "q4_k":
        d, dmin, s = _f16_of(blocks[:, 0:2]), _f16_of(blocks[:, 2:4]), blocks[:, 4:16]
        sc = torch.cat((s[:, 0:4] & 63, (s[:, 8:12] & 15) | (s[:, 0:4] >> 6 << 4)), 1).double()
        mn = torch.cat((s[:, 4:8] & 63, (s[:, 8:12] >> 4) | (s[:, 4:8] >> 6 << 4)), 1).double()
        q = blocks[:, 16:].reshape(nb, 4, 1, 32)
        q = torch.cat((q & 15, q >> 4), 2).reshape(nb, 8, 32).double()
        w = (d * sc)[:, :, None] * q - (dmin * mn)[:, :, None]
    else:
        lo, hi = blocks[:, :128], blocks[:, 128:192]
        lo = torch.stack((lo & 15, lo >> 4), 2).reshape(nb, 256)
        hi = torch.stack([(hi >> s) & 3 for s in (0, 2, 4, 6)], 2).reshape(nb, 256)
        sc = blocks[:, 192:208].contiguous().view(torch.int8).double()
        w = (_f16_of(blocks[:, 208:210]) * sc)[:, :, None] * ((lo | (hi << 4)).double() - 32).reshape(nb, 16, 16)
    return w.reshape(-1, k)


def _matmul(x, blocks, fmt, n, k):
    """x @ W^T in f64, the weight decoded a slice of rows at a time."""
    per_row = blocks.shape[0] // n
    step = max(1, (1 << 27) // k)
    parts = [x.double() @ _decode(blocks[r * per_row:min(n, r + step) * per_row], fmt, k).t()
             for r in range(0, n, step)]
    return torch.cat(parts, 1)


def _expert(packed, scales):
    lut = torch.tensor([0, 0.5, 1, 1.5, 2, 3, 4, 6], device=DEV, dtype=torch.float64)
    lut = torch.cat((lut, -lut))
    w = torch.stack((lut[(packed >> 4).long()], lut[(packed & 15).long()]), 2).reshape(packed.shape[0], -1)
    return w * torch.exp2(scales.double() - 127).repeat_interleave(32, 1)


def _moe_exact(case, d):
    x = d["x"].double()
    logits = d["logits"].double() if d["rw"] is None else x @ d["rw"].double().t() + d["rb"].double()
    p, idx = torch.topk(torch.softmax(logits, 1), case["top_k"], 1)
    p = p / p.sum(1, keepdim=True)
    (gp, gs, gb), (dp, ds, db) = d["gu"], d["dn"]
    y = torch.zeros_like(x)
    for e in range(case["experts"]):
        t, s = torch.nonzero(idx == e, as_tuple=True)
        if t.numel() == 0:
            continue
        gu = x[t] @ _expert(gp[e], gs[e]) + gb[e].double()
        gate, up = gu[:, :case["inter"]], gu[:, case["inter"]:]
        h = (gate * torch.sigmoid(gate)).clamp(-7.0, 7.0) * up
        y[t] += p[t, s][:, None] * (h @ _expert(dp[e], ds[e]) + db[e].double())
    return y


def exact(case, seed):
    d = _inputs(case, seed)
    kind = case["kind"]
    if kind == "linear":
        y = _matmul(d["x"], d["w"], case["fmt"], case["n"], case["k"])
        return y if d["bias"] is None else y + d["bias"].double()
    if kind == "head":
        y = _matmul(d["x"][None], d["w"], "q6_k", case["n"], case["k"])[0]
        return y, torch.argmax(y)
    if kind == "mlp":
        h, i = case["hidden"], case["inter"]
        gate, up = _matmul(d["x"], d["gate"], "q4_k", i, h), _matmul(d["x"], d["up"], "q4_k", i, h)
        return _matmul(gate * torch.sigmoid(gate) * up, d["down"], "q4_k", h, i)
    return _moe_exact(case, d)
