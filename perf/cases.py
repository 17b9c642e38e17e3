"""Performance cases: the calls a program makes through ``kore_amd.rocm``, over the sizes it makes them at.

Each case goes through the public entry points only, with the buffers a program keeps (weights, activations,
workspaces) made in ``prepare``.  Kinds:

``mlp_i8``      a BitLinear MLP block on int8 codes: pre-quant, gate and up projections, SwiGLU, pre-quant, down
                projection (decode, continuous-batching and prefill token counts);
``linear_f32``  ``BitLinear::forward`` on f32 activations with bias;
``embed_norm``  a model's input: token embedding, then the first layer's RMSNorm;
``rope``        Q and K of one attention layer rotated in place;
``attn_train``  attention probabilities: softmax (causal: one call per head, as the causal entry point counts the
                rows of one matrix) and its backward;
``loss``        cross-entropy backward over the vocabulary;
``norm_train``  RMSNorm forward and backward;
``act``         an element-wise activation over a whole FFN activation.
"""
import torch

from kore_amd import rocm
from kore_amd.rocm import HipBuffer

DEV = 0
NORM_EPS = 1e-6


def listed():
    return [
        # One token through one MLP block of the 2560/6912 BitLinear model: what a decode step repeats per layer.
        {"name": "mlp_i8 decode 1", "kind": "mlp_i8", "tokens": 1, "dim": 2560, "ffn": 6912},
        # A continuous-batching decode step; the batch is whatever is running, so not a round number.
        {"name": "mlp_i8 decode 45", "kind": "mlp_i8", "tokens": 45, "dim": 2560, "ffn": 6912},
        # Prompt processing of the same block at the pre-quant configuration's 4096 tokens.
        {"name": "mlp_i8 prefill 4096", "kind": "mlp_i8", "tokens": 4096, "dim": 2560, "ffn": 6912},
        # BitLinear::forward on f32 activations, one token: the reference's own decode step.
        {"name": "linear_f32 decode 1", "kind": "linear_f32", "tokens": 1, "in": 2560, "out": 6912},
        # The same layer on a decode batch.
        {"name": "linear_f32 decode 64", "kind": "linear_f32", "tokens": 64, "in": 2560, "out": 6912},
        # The FFN's down projection on a prompt of ordinary, ragged length.
        {"name": "linear_f32 prefill 777", "kind": "linear_f32", "tokens": 777, "in": 6912, "out": 2560},
        # The input of a prefill: gather from the 128256 x 4096 table, first RMSNorm.
        {"name": "embed_norm 8192x4096", "kind": "embed_norm", "tokens": 8192, "dim": 4096, "vocab": 128256,
         "float_ids": False},
        # Rotary embedding of a training batch (32 query and 8 key heads).
        {"name": "rope 8x2048", "kind": "rope", "batch": 8, "seq": 2048, "q_heads": 32, "k_heads": 8,
         "head_dim": 128, "start": 0, "interleaved": False},
        # Attention probabilities of a ragged sequence, forward per head and backward over all heads.
        {"name": "attn_train 16x1023", "kind": "attn_train", "heads": 16, "q": 1023, "kv": 1023, "causal": True},
        # The loss of a training step over the vocabulary.
        {"name": "loss 2048x128256", "kind": "loss", "tokens": 2048, "classes": 128256},
        # A norm layer's training step at the width of a large model.
        {"name": "norm_train 4096x8192", "kind": "norm_train", "rows": 4096, "cols": 8192},
        # SwiGLU over a whole FFN activation: the largest element-wise stream.
        {"name": "swiglu 16384x14336", "kind": "act", "op": "swiglu", "tokens": 16384, "width": 14336},
    ]


def draw(rng):
    def log(lo, hi):
        return int(round(lo * (hi / lo) ** rng.random()))

    def width(lo, hi):  # half of them multiples of 64 as models have them, the others anything
        v = log(lo, hi)
        return min(hi, max(lo, (v + 32) // 64 * 64)) if rng.random() < 0.5 else v

    kind = rng.choice(["mlp_i8", "linear_f32", "embed_norm", "rope", "attn_train", "loss", "norm_train", "act"])
    if kind == "mlp_i8":
        dim, ffn = width(512, 3072), width(1024, 6912)
        return {"kind": kind, "tokens": log(1, min(4096, 4096 * 2560 * 6912 // (dim * ffn))), "dim": dim, "ffn": ffn}
    if kind == "linear_f32":
        return {"kind": kind, "tokens": log(1, 1024), "in": width(512, 6912), "out": width(512, 6912)}
    if kind == "embed_norm":
        dim = width(512, 8192)
        return {"kind": kind, "tokens": log(1, 8192 * 4096 // max(dim, 4096)), "dim": dim, "vocab": log(16000, 128256 // 2),
                "float_ids": rng.random() < 0.3}
    if kind == "rope":
        kh = rng.choice([1, 2, 4, 8])
        seq = log(1, 2048)
        return {"kind": kind, "batch": log(1, 8), "seq": seq, "q_heads": kh * rng.choice([1, 2, 4]), "k_heads": kh,
                "head_dim": rng.choice([64, 80, 96, 128]), "start": rng.choice([0, rng.randrange(4096)]),
                "interleaved": rng.random() < 0.5}
    if kind == "attn_train":
        q = log(1, 2048)
        kv = q + rng.choice([0, 0, log(1, 2048)])
        return {"kind": kind, "heads": log(1, min(32, max(1, (1 << 25) // (q * kv)))), "q": q, "kv": kv,
                "causal": rng.random() < 0.5}
    if kind == "loss":
        classes = width(256, 128256)
        return {"kind": kind, "tokens": log(16, min(16384, (1 << 28) // classes)), "classes": classes}
    if kind == "norm_train":
        cols = width(512, 8192)
        return {"kind": kind, "rows": log(32, (1 << 25) // cols), "cols": cols}
    w = width(1024, 14336)
    return {"kind": kind, "op": rng.choice(["gelu", "silu", "swiglu"]), "tokens": log(1, 16384), "width": w}


# ------------------------------------------------------------------ inputs
def _gen(seed):
    return torch.Generator(device="cuda:%d" % DEV).manual_seed(seed)


def _normal(g, *shape, std=1.0, mean=0.0):
    return torch.empty(shape, dtype=torch.float32, device=g.device).normal_(mean, std, generator=g)


def _outliers(g, *shape):
    """N(0, 1) with 1% of the entries scaled by 20, as activations before a norm are."""
    x = _normal(g, *shape)
    return torch.where(torch.rand(shape, device=g.device, generator=g) < 0.01, x * 20.0, x)


def _weights(g, m, k):
    """Uniform trits packed base 243 (five per byte, least significant digit first, zeros past k), and row scales."""
    kp = (k + 4) // 5
    t = torch.randint(0, 3, (m, kp * 5), device=g.device, generator=g, dtype=torch.int32)
    t[:, k:] = 1
    w3 = torch.tensor([1, 3, 9, 27, 81], device=g.device, dtype=torch.int32)
    packed = (t.view(m, kp, 5) * w3).sum(-1).to(torch.uint8)
    return packed, torch.rand(m, device=g.device, generator=g) * 0.02 + 0.01


def _trits(packed, k):
    b = packed.to(torch.int32)
    return torch.stack([b // 3 ** i % 3 - 1 for i in range(5)], -1).view(packed.shape[0], -1)[:, :k].double()


def _ids(g, n, vocab):
    ids = torch.randint(0, vocab, (n,), device=g.device, generator=g)
    rep = torch.rand(n, device=g.device, generator=g) < 0.05  # 5% of the tokens repeat the prompt's first one
    return torch.where(rep, ids[0], ids)


def _inputs(case, seed):
    g, kind = _gen(seed), case["kind"]
    if kind == "mlp_i8":
        t, d, f = case["tokens"], case["dim"], case["ffn"]
        i = {"x": _outliers(g, t, d), "wn": _normal(g, d, std=0.02, mean=1.0), "wh": _normal(g, f, std=0.02, mean=1.0)}
        for name, m, k in (("gate", f, d), ("up", f, d), ("down", d, f)):
            i[name], i[name + "_s"] = _weights(g, m, k)
        return i
    if kind == "linear_f32":
        i = {"x": _normal(g, case["tokens"], case["in"]), "bias": _normal(g, case["out"])}
        i["w"], i["s"] = _weights(g, case["out"], case["in"])
        return i
    if kind == "embed_norm":
        ids = _ids(g, case["tokens"], case["vocab"])
        return {"table": _normal(g, case["vocab"], case["dim"], std=0.02), "wn": _normal(g, case["dim"], std=0.02, mean=1.0),
                "ids": ids.to(torch.float32 if case["float_ids"] else torch.int32)}
    if kind == "rope":
        b, s, d = case["batch"], case["seq"], case["head_dim"]
        return {"q": _normal(g, b, s, case["q_heads"], d), "k": _normal(g, b, s, case["k_heads"], d)}
    if kind == "attn_train":
        shape = (case["heads"], case["q"], case["kv"])
        return {"x": _normal(g, *shape, std=2.0), "dy": _normal(g, *shape)}
    if kind == "loss":
        t = torch.randint(0, case["classes"], (case["tokens"],), device=g.device, generator=g)
        return {"x": _normal(g, case["tokens"], case["classes"], std=2.0), "t": t.to(torch.float32)}
    if kind == "norm_train":
        r, c = case["rows"], case["cols"]
        return {"x": _normal(g, r, c), "dy": _normal(g, r, c), "w": _normal(g, c, std=0.02, mean=1.0)}
    n = (case["tokens"], case["width"])
    return {"a": _normal(g, *n), "b": _normal(g, *n)} if case["op"] == "swiglu" else {"a": _normal(g, *n)}


def _buf(t):
    return HipBuffer.from_tensor(t)


def _empty(*shape, dtype=torch.float32):
    return torch.empty(shape, dtype=dtype, device="cuda:%d" % DEV)


def prepare(case, seed):
    i, kind = _inputs(case, seed), case["kind"]
    s = {"case": case, "in": {k: _buf(v) for k, v in i.items()}}
    if kind == "mlp_i8":
        t, d, f = case["tokens"], case["dim"], case["ffn"]
        s["qx"], s["sx"] = _buf(_empty(t, d, dtype=torch.int8)), _buf(_empty(t))
        s["gate"], s["up"] = _buf(_empty(t, f)), _buf(_empty(t, f))
        s["qh"], s["sh"] = _buf(_empty(t, f, dtype=torch.int8)), _buf(_empty(t))
        s["out"] = {"y": _empty(t, d)}
    elif kind == "linear_f32":
        s["out"] = {"y": _empty(case["tokens"], case["out"])}
    elif kind == "embed_norm":
        s["out"] = {"e": _empty(case["tokens"], case["dim"]), "y": _empty(case["tokens"], case["dim"])}
    elif kind == "rope":
        s["inv"] = rocm.rocm_rope_inv_freq_f32(DEV, case["head_dim"], 10000.0)
        s["out"] = {"q": i["q"], "k": i["k"]}
    elif kind == "attn_train":
        y, dx = torch.empty_like(i["x"]), torch.empty_like(i["x"])
        s["out"] = {"y": y, "dx": dx}
        s["heads"] = [(_buf(i["x"][h]), _buf(y[h])) for h in range(case["heads"])]
    elif kind == "loss":
        s["out"] = {"dx": torch.empty_like(i["x"])}
    elif kind == "norm_train":
        s["out"] = {"y": torch.empty_like(i["x"]), "dx": torch.empty_like(i["x"]), "dw": torch.empty_like(i["w"])}
        ws = rocm.rocm_rms_norm_backward_workspace_bytes(case["rows"], case["cols"])
        s["ws"] = HipBuffer.empty(DEV, max(ws, 16))
    else:
        s["out"] = {"y": torch.empty_like(i["a"])}
    s["buf"] = {k: _buf(v) for k, v in s["out"].items()}
    return s


def run(s):
    c, i, o = s["case"], s["in"], s["buf"]
    kind = c["kind"]
    if kind == "mlp_i8":
        t, d, f = c["tokens"], c["dim"], c["ffn"]
        rocm.rocm_rms_norm_quant_i8(DEV, i["x"], i["wn"], t, d, NORM_EPS, s["qx"], s["sx"])
        rocm.rocm_bit_linear_i8(DEV, i["gate"], i["gate_s"], s["qx"], s["sx"], None, f, t, d, s["gate"])
        rocm.rocm_bit_linear_i8(DEV, i["up"], i["up_s"], s["qx"], s["sx"], None, f, t, d, s["up"])
        rocm.rocm_swiglu_f32(DEV, s["gate"], s["up"], t * f, s["gate"])
        rocm.rocm_rms_norm_quant_i8(DEV, s["gate"], i["wh"], t, f, NORM_EPS, s["qh"], s["sh"])
        rocm.rocm_bit_linear_i8(DEV, i["down"], i["down_s"], s["qh"], s["sh"], None, d, t, f, o["y"])
    elif kind == "linear_f32":
        rocm.rocm_bit_linear_f32(DEV, i["w"], i["s"], i["x"], i["bias"], c["out"], c["tokens"], c["in"], o["y"])
    elif kind == "embed_norm":
        embed = rocm.rocm_embedding_forward_f32 if c["float_ids"] else rocm.rocm_embedding_f32
        embed(DEV, i["table"], i["ids"], c["tokens"], c["vocab"], c["dim"], o["e"])
        rocm.rocm_rms_norm_f32(DEV, o["e"], i["wn"], c["tokens"], c["dim"], NORM_EPS, o["y"])
    elif kind == "rope":
        rocm.rocm_rope_qk_f32(DEV, i["q"], i["k"], s["inv"], c["batch"], c["seq"], c["q_heads"], c["k_heads"],
                              c["head_dim"], c["start"], c["interleaved"])
    elif kind == "attn_train":
        rows = c["heads"] * c["q"]
        if c["causal"]:
            for x, y in s["heads"]:
                rocm.rocm_softmax_causal_f32(DEV, x, c["q"], c["kv"], c["kv"] - c["q"], y)
        else:
            rocm.rocm_softmax_f32(DEV, i["x"], rows, c["kv"], o["y"])
        rocm.rocm_softmax_backward_f32(DEV, i["dy"], o["y"], rows, c["kv"], o["dx"])
    elif kind == "loss":
        rocm.rocm_cross_entropy_backward_f32(DEV, i["x"], i["t"], c["tokens"], c["classes"], o["dx"])
    elif kind == "norm_train":
        rocm.rocm_rms_norm_f32(DEV, i["x"], i["w"], c["rows"], c["cols"], NORM_EPS, o["y"])
        rocm.rocm_rms_norm_backward_f32(DEV, i["dy"], i["x"], i["w"], c["rows"], c["cols"], NORM_EPS, s["ws"], o["dx"],
                                        o["dw"])
    elif c["op"] == "swiglu":
        rocm.rocm_swiglu_f32(DEV, i["a"], i["b"], c["tokens"] * c["width"], o["y"])
    else:
        op = rocm.rocm_gelu_f32 if c["op"] == "gelu" else rocm.rocm_silu_f32
        op(DEV, i["a"], c["tokens"] * c["width"], o["y"])
    return s["out"]


# ------------------------------------------------------------ work and bars
def work(case):
    """Every call's inputs read once and its outputs written once; multiply-adds count two, other terms a few."""
    kind = case["kind"]
    if kind == "mlp_i8":
        t, d, f = case["tokens"], case["dim"], case["ffn"]
        weights = 2 * f * ((d + 4) // 5) + d * ((f + 4) // 5) + 4 * (2 * f + d) + 4 * (d + f)
        norms = 5 * t * (d + f) + 8 * t
        linears = 2 * t * d + t * f + 4 * t * (2 * f + d) + 12 * t
        return {"bytes": weights + norms + linears + 12 * t * f, "flops": 6 * t * d * f}
    if kind == "linear_f32":
        t, k, m = case["tokens"], case["in"], case["out"]
        return {"bytes": m * ((k + 4) // 5) + 8 * m + 4 * t * (k + m), "flops": 2 * t * k * m}
    if kind == "embed_norm":
        n = case["tokens"] * case["dim"]
        return {"bytes": 16 * n + 4 * case["tokens"] + 4 * case["dim"], "flops": 4 * n}
    if kind == "rope":
        n = case["batch"] * case["seq"] * (case["q_heads"] + case["k_heads"]) * case["head_dim"]
        return {"bytes": 8 * n, "flops": 3 * n}
    if kind == "attn_train":
        h, q, kv = case["heads"], case["q"], case["kv"]
        seen = q * (kv - q) + q * (q + 1) // 2 if case["causal"] else q * kv  # what a causal mask leaves to read
        return {"bytes": h * (4 * seen + 16 * q * kv), "flops": h * (4 * seen + 4 * q * kv)}
    if kind == "loss":
        n = case["tokens"] * case["classes"]
        return {"bytes": 8 * n + 4 * case["tokens"], "flops": 4 * n}
    if kind == "norm_train":
        n = case["rows"] * case["cols"]
        return {"bytes": 20 * n + 12 * case["cols"], "flops": 14 * n}
    n = case["tokens"] * case["width"]
    return {"bytes": (12 if case["op"] == "swiglu" else 8) * n, "flops": 8 * n}


def tolerance(case):
    kind = case["kind"]
    if kind in ("linear_f32", "embed_norm"):
        return "exact"  # the reference's own order of every sum: bit-identical by contract
    if kind == "mlp_i8":
        # An ulp in SwiGLU moves a code across a rounding boundary now and then: one step of 127 in one term
        # (2.7e-4 from the result in 64 bits at 4096 tokens).
        return {"rel": 1e-3, "max": 0.1}
    if kind == "rope":
        return {"rel": 2e-7, "max": 1e-5}
    return {"rel": 5e-6, "max": 1e-4}


# -------------------------------------------------------------- in 64 bits
def _norm64(x, w, eps=NORM_EPS):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps) * w


def _codes64(x):
    amax = x.abs().amax(-1, keepdim=True)
    amax = torch.where(amax < 1e-8, torch.ones_like(amax), amax)
    t = x * 127.0 / amax
    return torch.clamp(torch.sign(t) * torch.floor(t.abs() + 0.5), -128, 127), amax / 127.0


def exact(case, seed):
    if work(case)["bytes"] > 4e9:
        return None
    kind, i = case["kind"], _inputs(case, seed)
    if kind == "mlp_i8":
        def linear(name, q, qs, k):
            return q @ _trits(i[name], k).t() * i[name + "_s"].double() * qs

        q, qs = _codes64(_norm64(i["x"].double(), i["wn"].double()))
        gate, up = linear("gate", q, qs, case["dim"]), linear("up", q, qs, case["dim"])
        q, qs = _codes64(_norm64(gate * torch.sigmoid(gate) * up, i["wh"].double()))
        return {"y": linear("down", q, qs, case["ffn"])}
    if kind == "linear_f32":
        return {"y": i["x"].double() @ _trits(i["w"], case["in"]).t() * i["s"].double() + i["bias"].double()}
    if kind == "embed_norm":
        e = i["table"][i["ids"].long()].double()
        return {"e": e, "y": _norm64(e, i["wn"].double())}
    if kind == "rope":
        # The angle is the f32 product of the position and the table's entry, as the operator defines it.
        half = case["head_dim"] // 2
        inv = rope_table(case["head_dim"]).to(i["q"].device)
        pos = torch.arange(case["start"], case["start"] + case["seq"], device=inv.device, dtype=torch.float32)
        angle = (pos[:, None] * inv[None, :]).double()[None, :, None, :]
        cos, sin, out = torch.cos(angle), torch.sin(angle), {}
        for name in ("q", "k"):
            x = i[name].double()
            a, b = (x[..., 0::2], x[..., 1::2]) if case["interleaved"] else (x[..., :half], x[..., half:])
            r0, r1 = a * cos - b * sin, a * sin + b * cos
            out[name] = torch.stack([r0, r1], -1).flatten(-2) if case["interleaved"] else torch.cat([r0, r1], -1)
        return out
    if kind == "attn_train":
        x, dy = i["x"].double(), i["dy"].double()
        if case["causal"]:
            keep = torch.ones(case["q"], case["kv"], dtype=torch.bool, device=x.device).tril(case["kv"] - case["q"])
            x = x.masked_fill(~keep, float("-inf"))
        y = torch.softmax(x, -1)
        return {"y": y, "dx": y * (dy - (y * dy).sum(-1, keepdim=True))}
    if kind == "loss":
        g = torch.softmax(i["x"].double(), -1)
        g[torch.arange(case["tokens"], device=g.device), i["t"].long()] -= 1.0
        return {"dx": g / case["tokens"]}
    if kind == "norm_train":
        x, dy, w = i["x"].double(), i["dy"].double(), i["w"].double()
        inv = 1.0 / torch.sqrt((x * x).mean(-1, keepdim=True) + NORM_EPS)
        coeff = (x * dy * w).sum(-1, keepdim=True) * inv ** 3 / case["cols"]
        return {"y": x * inv * w, "dx": w * inv * dy - coeff * x, "dw": (dy * x * inv).sum(0)}
    a = i["a"].double()
    if case["op"] == "gelu":
        return {"y": 0.5 * a * (1.0 + torch.tanh((2.0 / torch.pi) ** 0.5 * (a + 0.044715 * a ** 3)))}
    y = a * torch.sigmoid(a)
    return {"y": y * i["b"].double() if case["op"] == "swiglu" else y}


def rope_table(head_dim):
    """1 / theta^(2i / D) rounded to f32, theta = 10000."""
    i = torch.arange(head_dim // 2, dtype=torch.float32)
    return 1.0 / torch.pow(torch.tensor(10000.0), 2.0 * i / head_dim)
