"""Performance cases of libdeepinfer_hip: what a Qwen3.6-35B-A3B server asks of one MI355X.

Every case is one call of a public entry point of ``deepinfer_hip`` on the current stream,
as a model's forward pass makes it: GEMV and dense projections, the decode and prefill MoE
layer, the vocabulary head, causal attention over the KV cache and the gated delta rule.
Weights are the model's MLX-affine group-64 matrices in 5 and 8 bits.

listed() holds the fixed cases, draw(rng) more of the same ranges. prepare() makes weights
and inputs on the GPU from the seed, run() makes the call, exact() gives the same outputs
in 64 bits from plain torch. MoE calls add to the residual and the delta rule to its state,
as in a decode loop: a second run() on one state starts from what the first one left.
"""
import math
import os
import sys

import torch

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(_ROOT, "infer.net_amd"))
import deepinfer_hip as dh  # noqa: E402

H, I, TOP = 2048, 512, 8            # hidden width, expert width, experts a token takes
EPSILON = 1e-6
# the model's projections (rows, columns): q with its gate, k or v, o, the linear-attention
# input projection
PROJECTIONS = {"q_gate": (8192, 2048), "kv": (512, 2048), "o": (2048, 4096), "in_proj": (12288, 2048)}


def listed():
    return [
        # one decode token through one 8-bit projection: the smallest call a server makes
        dict(name="qmv8", kind="qmv", bits=8, rows=4096, columns=2048, x="bf16", y="bf16"),
        # one decode token through one MoE layer, both checkpoint precisions, f32 residual
        # and the next layer's norm, as the decode loop runs it 40 times a token
        dict(name="moe_decode8", kind="moe_decode", bits=8, experts=256, residual="f32", norm=True),
        dict(name="moe_decode5", kind="moe_decode", bits=5, experts=256, residual="f32", norm=True),
        # the vocabulary head of one decode token, four slices
        dict(name="lm_head8", kind="lm_head", bits=8, vocab=248320, slices=4),
        # a short prompt, or the ragged end of a long one
        dict(name="moe_prefill5_t77", kind="moe_prefill", bits=5, experts=256, tokens=77, routing="zipf",
             residual="f32", norm=True),
        # a medium prompt with popular and rare experts
        dict(name="moe_prefill8_t512", kind="moe_prefill", bits=8, experts=256, tokens=512, routing="zipf",
             residual="bf16", norm=False),
        # a full prefill chunk
        dict(name="moe_prefill5_t2048", kind="moe_prefill", bits=5, experts=256, tokens=2048, routing="uniform",
             residual="f32", norm=True),
        # the attention output projection of a short, odd-sized prompt
        dict(name="dense8_o_t61", kind="dense", bits=8, projection="o", tokens=61, y="f32"),
        # the query projection of a long chunk
        dict(name="dense8_q_t4096", kind="dense", bits=8, projection="q_gate", tokens=4096, y="bf16"),
        # one decode token against a 32K cache
        dict(name="attention_decode_32k", kind="attention", position=32767, tokens=1, dtype="f32"),
        # the last chunk of a 32K prompt
        dict(name="attention_prefill_32k", kind="attention", position=30720, tokens=2048, dtype="f32"),
        # a full prefill chunk of a linear-attention layer
        dict(name="delta_t2048", kind="delta", tokens=2048),
    ]


def _log_int(rng, low, high):
    """An integer of [low, high], its logarithm uniform."""
    return max(low, min(high, int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))))


def draw(rng):
    kind = rng.choice(["qmv", "moe_decode", "lm_head", "moe_prefill", "moe_prefill", "dense", "dense", "attention",
                       "attention", "delta"])
    bits = rng.choice([5, 8])
    if kind == "qmv":
        return dict(kind=kind, bits=bits, rows=_log_int(rng, 512, 12288), columns=rng.choice([512, 2048, 4096]),
                    x=rng.choice(["bf16", "f32"]), y=rng.choice(["bf16", "f32"]))
    if kind == "moe_decode":
        return dict(kind=kind, bits=bits, experts=rng.randint(64, 256), residual=rng.choice(["f32", "bf16"]),
                    norm=rng.choice([True, False]))
    if kind == "lm_head":
        return dict(kind=kind, bits=bits, vocab=_log_int(rng, 32000, 248320), slices=rng.randint(1, 4))
    if kind == "moe_prefill":
        return dict(kind=kind, bits=bits, experts=rng.choice([64, 128, 256]), tokens=_log_int(rng, 8, 2048),
                    routing=rng.choice(["zipf", "uniform"]), residual=rng.choice(["f32", "bf16"]),
                    norm=rng.choice([True, False]))
    if kind == "dense":
        return dict(kind=kind, bits=bits, projection=rng.choice(sorted(PROJECTIONS)), tokens=_log_int(rng, 2, 4096),
                    y=rng.choice(["f32", "bf16"]))
    if kind == "attention":
        tokens = 1 if rng.random() < 0.4 else _log_int(rng, 2, 2048)
        return dict(kind=kind, position=_log_int(rng, 1, 30720), tokens=tokens, dtype=rng.choice(["f32", "bf16"]))
    return dict(kind=kind, tokens=_log_int(rng, 1, 2048))


# ------------------------------------------------------------------------------ inputs

def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _normal(g, *shape, scale=1.0):
    return torch.randn(shape, device="cuda", generator=g) * scale


def _affine(g, experts, rows, columns, bits):
    """One matrix's checkpoint buffers: codes uniform over their range, group scales that
    give the weights a deviation of about 0.02, biases that centre them."""
    codes = torch.randint(-2**31, 2**31, (experts, rows, columns * bits // 32), dtype=torch.int32, device="cuda",
                          generator=g)
    scales = torch.rand((experts, rows, columns // 64), device="cuda", generator=g)
    scales = ((0.5 + scales) * (0.02 * math.sqrt(12) / 2**bits)).to(torch.bfloat16)
    biases = -(2.0 ** (bits - 1)) * scales.float() + _normal(g, *scales.shape, scale=1e-4)
    return codes, scales, biases.to(torch.bfloat16)


def _zipf(g, tokens, experts):
    """Router logits whose top-8 follow a Zipf(1.1) popularity of the experts."""
    popularity = torch.arange(1, experts + 1, dtype=torch.float64, device="cuda") ** -1.1
    popularity = torch.log(popularity / popularity.sum())[torch.randperm(experts, device="cuda", generator=g)]
    u = torch.rand((tokens, experts), dtype=torch.float64, device="cuda", generator=g).clamp_(1e-12, 1 - 1e-12)
    return (popularity[None, :] - torch.log(-torch.log(u))).to(torch.bfloat16)


def _moe_shapes(case, bits):
    e = case["experts"]
    return [("router", 1, e, H, 8), ("gate", e, I, H, bits), ("up", e, I, H, bits), ("down", e, H, I, bits),
            ("shared_gate", 1, I, H, bits), ("shared_up", 1, I, H, bits), ("shared_down", 1, H, I, bits),
            ("shared_route", 1, 1, H, 8)]


def _inputs(case, seed):
    """Generator of a case's weights (name, buffers, bits), then its tensors as a dict: the
    weights are handed out one at a time, so that only one is held twice."""
    g = _generator(seed)
    kind = case["kind"]
    if kind == "qmv":
        yield "w", _affine(g, 1, case["rows"], case["columns"], case["bits"]), case["bits"]
        x = _normal(g, case["columns"])
        yield dict(x=x.to(torch.bfloat16) if case["x"] == "bf16" else x)
    elif kind == "lm_head":
        n, v = case["slices"], case["vocab"]
        for k in range(n):
            yield f"w{k}", _affine(g, 1, v * (k + 1) // n - v * k // n, H, case["bits"]), case["bits"]
        yield dict(x=_normal(g, H).to(torch.bfloat16))
    elif kind in ("moe_decode", "moe_prefill"):
        for name, e, r, c, b in _moe_shapes(case, case["bits"]):
            if name == "router" and kind == "moe_prefill":
                continue
            yield name, _affine(g, e, r, c, b), b
        t = case.get("tokens", 1)
        out = dict(x=_normal(g, t, H).to(torch.bfloat16), residual=_normal(g, t, H),
                   norm_weight=1.0 + _normal(g, H, scale=0.1))
        if case["residual"] == "bf16":
            out["residual"] = out["residual"].to(torch.bfloat16)
        if kind == "moe_prefill":
            out["logits"] = (_zipf(g, t, case["experts"]) if case["routing"] == "zipf"
                             else _normal(g, t, case["experts"]).to(torch.bfloat16))
        yield out
    elif kind == "dense":
        r, c = PROJECTIONS[case["projection"]]
        yield "w", _affine(g, 1, r, c, case["bits"]), case["bits"]
        yield dict(x=_normal(g, case["tokens"], c).to(torch.bfloat16))
    elif kind == "attention":
        # queries and keys are normed, so that scores are about N(0, 1); the cache is longer
        # than what is filled, as a server allocates it
        t, n = case["tokens"], case["position"] + case["tokens"]
        cache = (n + 255) // 256 * 256
        real = torch.float32 if case["dtype"] == "f32" else torch.bfloat16
        keys = torch.zeros((cache, 512), dtype=torch.bfloat16, device="cuda")
        values = torch.zeros((cache, 512), dtype=torch.bfloat16, device="cuda")
        keys[:n] = _normal(g, n, 512).to(torch.bfloat16)
        values[:n] = _normal(g, n, 512, scale=0.5).to(torch.bfloat16)
        yield dict(q=_normal(g, t, 4096).to(real), keys=keys, values=values, gate=_normal(g, t, 8192).to(real))
    else:
        t = case["tokens"]
        conv = _normal(g, t, 8192, scale=0.1)
        unit = conv[:, :4096].view(t, 32, 128)
        unit /= unit.norm(dim=2, keepdim=True)
        conv[:, :2048] /= math.sqrt(128.0)
        yield dict(conv=conv, raw=_normal(g, t, 8192), decay=0.9 + 0.1 * torch.rand((t, 32), device="cuda", generator=g),
                   beta=torch.rand((t, 32), device="cuda", generator=g),
                   state=_normal(g, 32, 128, 128, scale=0.01), history=_normal(g, 3, 8192))


_device = None


def _dev():
    """The process's one library context."""
    global _device
    if _device is None:
        torch.cuda.init()
        _device = dh.QuantizedHip()
    return _device


class State:
    """A case's matrices and tensors; the matrices are freed with it."""

    def __init__(self, case):
        self.case, self.mats = case, {}

    def __del__(self):
        for m in self.mats.values():
            m.dispose()


def prepare(case, seed):
    dev, s = _dev(), State(case)
    for item in _inputs(case, seed):
        if isinstance(item, dict):
            for k, v in item.items():
                setattr(s, k, v)
            continue
        name, (codes, scales, biases), bits = item
        m = dev.allocate(codes.shape[0], codes.shape[1], codes.shape[2] * 32 // bits, bits)
        s.mats[name] = m
        m.upload_from(0, codes)
        m.upload_from(1, scales)
        m.upload_from(2, biases)
    kind = case["kind"]
    real = {"f32": torch.float32, "bf16": torch.bfloat16}
    if kind == "qmv":
        s.y = torch.zeros(case["rows"], dtype=real[case["y"]], device="cuda")
    elif kind == "lm_head":
        s.slices = list(s.mats.values())
        s.logits = torch.zeros(case["vocab"], device="cuda")
        s.next = torch.zeros(1, dtype=torch.int32, device="cuda")
    elif kind in ("moe_decode", "moe_prefill"):
        s.layer = dh.make_layer(*(s.mats.get(n) for n, *_ in _moe_shapes(case, case["bits"])))
        s.normed = torch.zeros_like(s.residual, dtype=real[case["residual"]]) if case["norm"] else None
        f32 = case["residual"] == "f32"
        s.merge = dh.make_merge(f32, s.norm_weight if case["norm"] else None, EPSILON, s.normed, normed_f32=f32)
    elif kind == "dense":
        s.y = torch.zeros((case["tokens"], s.mats["w"].rows), dtype=real[case["y"]], device="cuda")
    elif kind == "attention":
        s.out = torch.zeros_like(s.q)
    else:
        s.out = torch.zeros((case["tokens"], 4096), device="cuda")
    return s


def _type(name):
    return dh.F32 if name == "f32" else dh.BF16


def run(s):
    case, dev = s.case, _device
    kind = case["kind"]
    if kind == "qmv":
        dh.qmv(dev, s.mats["w"], s.x, s.y, x_dtype=_type(case["x"]), y_dtype=_type(case["y"]))
        return s.y
    if kind == "lm_head":
        dh.lm_head(dev, s.slices, s.x, s.logits, s.next)
        return [s.logits, s.next]
    if kind == "moe_decode":
        dh.moe_decode(dev, s.layer, s.x, s.residual, merge=s.merge)
        return [s.residual, s.normed]
    if kind == "moe_prefill":
        dh.moe_prefill(dev, s.layer, case["tokens"], s.x, s.logits, s.residual, merge=s.merge)
        return [s.residual, s.normed]
    if kind == "dense":
        dh.dense(dev, s.mats["w"], case["tokens"], s.x, s.y, y_dtype=_type(case["y"]))
        return s.y
    if kind == "attention":
        t = _type(case["dtype"])
        dh.attention(dev, s.q, s.keys, s.values, s.gate, s.out, case["position"], case["tokens"], q_dtype=t,
                     gate_dtype=t, out_dtype=t)
        return s.out
    dh.delta_rule(dev, s.state, s.history, s.conv, s.decay, s.beta, s.raw, s.out, case["tokens"])
    return [s.out, s.state, s.history]


# ------------------------------------------------------------------------------ the answer

def _dequantize(buffers, bits, expert=0):
    """float(code) * scale + bias of one expert in 64 bits, [rows, columns]."""
    codes, scales, biases = (b[expert] for b in buffers)
    columns = codes.shape[1] * 32 // bits
    at = torch.arange(columns, device="cuda") * bits
    words = codes.long() & 0xFFFFFFFF
    low = words[:, at >> 5]
    high = words[:, ((at >> 5) + 1).clamp_(max=codes.shape[1] - 1)]
    q = ((low | (high << 32)) >> (at & 31)[None, :]) & ((1 << bits) - 1)
    wide = lambda v: v.double().repeat_interleave(64, dim=1)  # noqa: E731
    return q.double() * wide(scales) + wide(biases)


def _moe_exact(case, w, t):
    x = t["x"].double()
    logits = t["logits"].double() if "logits" in t else x @ _dequantize(*w["router"]).T
    top, ids = torch.sort(logits, dim=1, descending=True, stable=True)
    probs, ids = torch.softmax(top[:, :TOP], dim=1), ids[:, :TOP]

    def expert(x, names, e):
        gate, up, down = (_dequantize(*w[n], expert=e) for n in names)
        return (torch.nn.functional.silu(x @ gate.T) * (x @ up.T)) @ down.T

    y = torch.sigmoid(x @ _dequantize(*w["shared_route"]).T) * expert(x, ("shared_gate", "shared_up", "shared_down"), 0)
    for e in ids.unique().tolist():
        token, slot = (ids == e).nonzero(as_tuple=True)
        y[token] += probs[token, slot, None] * expert(x[token], ("gate", "up", "down"), e)
    r = t["residual"].double() + y
    if not case["norm"]:
        return [r, None]
    return [r, r * torch.rsqrt((r * r).mean(dim=1, keepdim=True) + EPSILON) * t["norm_weight"].double()]


def _attention_exact(case, t):
    position, tokens = case["position"], case["tokens"]
    n = position + tokens
    q = t["q"].double().view(tokens, 16, 256)
    k, v = (t[name][:n].double().view(n, 2, 256) for name in ("keys", "values"))
    out = torch.empty((tokens, 16, 256), dtype=torch.float64, device="cuda")
    last = position + torch.arange(tokens, device="cuda")
    hidden = torch.arange(n, device="cuda")[None, :] > last[:, None]
    for h in range(16):
        p = (q[:, h] @ k[:, h // 8].T / 16.0).masked_fill_(hidden, -math.inf)
        out[:, h] = torch.softmax(p, dim=1) @ v[:, h // 8]
    return (out * torch.sigmoid(t["gate"].double().view(tokens, 16, 512)[:, :, 256:])).view(tokens, 4096)


def _delta_exact(case, t):
    s = t["state"].double()
    conv = t["conv"].double()
    tokens = case["tokens"]
    q, k = (conv[:, a:a + 2048].view(tokens, 16, 128).repeat_interleave(2, dim=1) for a in (0, 2048))
    v = conv[:, 4096:].view(tokens, 32, 128)
    decay, beta = t["decay"].double(), t["beta"].double()
    out = torch.empty((tokens, 32, 128), dtype=torch.float64, device="cuda")
    for i in range(tokens):
        s = s * decay[i, :, None, None]
        c = (v[i] - (s @ k[i, :, :, None])[:, :, 0]) * beta[i, :, None]
        s = s + c[:, :, None] * k[i, :, None, :]
        out[i] = (s @ q[i, :, :, None])[:, :, 0]
    history = torch.cat([t["history"], t["raw"]]).double()[-3:]
    return [out.view(tokens, 4096), s, history]


def exact(case, seed):
    w, t = {}, None
    for item in _inputs(case, seed):
        if isinstance(item, dict):
            t = item
        else:
            w[item[0]] = item[1:]
    kind = case["kind"]
    if kind == "qmv":
        return t["x"].double() @ _dequantize(*w["w"]).T
    if kind == "lm_head":
        return [torch.cat([t["x"].double() @ _dequantize(*m).T for m in w.values()]), None]
    if kind in ("moe_decode", "moe_prefill"):
        return _moe_exact(case, w, t)
    if kind == "dense":
        return t["x"].double() @ _dequantize(*w["w"]).T
    if kind == "attention":
        return _attention_exact(case, t)
    return _delta_exact(case, t)


# ------------------------------------------------------------------------------ measures

def _weight_bytes(experts, rows, columns, bits):
    return experts * rows * (columns * bits // 8 + columns // 64 * 4)


def work(case):
    kind = case["kind"]
    size = lambda name: 4 if name == "f32" else 2  # noqa: E731
    if kind == "qmv":
        r, c = case["rows"], case["columns"]
        return {"bytes": _weight_bytes(1, r, c, case["bits"]) + c * size(case["x"]) + r * size(case["y"]),
                "flops": 2.0 * r * c}
    if kind == "lm_head":
        v = case["vocab"]
        return {"bytes": _weight_bytes(1, v, H, case["bits"]) + 2 * H + 4 * v, "flops": 2.0 * v * H}
    if kind in ("moe_decode", "moe_prefill"):
        t, e, bits = case.get("tokens", 1), case["experts"], case["bits"]
        if kind == "moe_decode":
            touched = TOP
        elif case["routing"] == "uniform":
            touched = e * (1.0 - (1.0 - TOP / e) ** t)
        else:
            # Zipf(1.1): an expert of probability p is drawn by about 8 p of the tokens
            p = [k ** -1.1 for k in range(1, e + 1)]
            touched = sum(1.0 - max(0.0, 1.0 - min(1.0, TOP * v / sum(p))) ** t for v in p)
        expert = 2 * _weight_bytes(1, I, H, bits) + _weight_bytes(1, H, I, bits)
        b = (touched + 1) * expert + _weight_bytes(1, 1, H, 8)
        f = 2.0 * t * (TOP + 1) * 3 * I * H
        if kind == "moe_decode":
            b, f = b + _weight_bytes(1, e, H, 8), f + 2.0 * e * H
        else:
            b += t * e * 2
        b += t * H * (2 + 2 * size(case["residual"]))
        if case["norm"]:
            b += t * H * size(case["residual"]) + 4 * H
        return {"bytes": float(b), "flops": f}
    if kind == "dense":
        r, c = PROJECTIONS[case["projection"]]
        t = case["tokens"]
        return {"bytes": _weight_bytes(1, r, c, case["bits"]) + t * (2 * c + size(case["y"]) * r),
                "flops": 2.0 * t * r * c}
    if kind == "attention":
        t, n, b = case["tokens"], case["position"] + case["tokens"], size(case["dtype"])
        visible = t * case["position"] + t * (t + 1) // 2
        return {"bytes": 2 * n * 512 * 2 + t * 4096 * b * 3, "flops": 1024.0 * 16 * visible}
    t = case["tokens"]
    return {"bytes": t * (8192 + 64 + 4096) * 4 + 2 * 32 * 128 * 128 * 4 + 2 * 3 * 8192 * 4,
            "flops": 8.0 * 128 * 128 * 32 * t}


def tolerance(case):
    """About four times the distance from exact() that was measured: f32 sums of unrounded
    weights for one token, bf16 operands with f32 sums for chunks, f32 for the delta rule. A
    MoE layer's part of its residual is small beside the residual itself."""
    kind = case["kind"]
    if kind == "moe_prefill":
        return {"rel": 2.5e-3 if case["residual"] == "f32" else 8e-3}
    if kind == "attention" or (kind == "dense" and case["tokens"] > 4):
        return {"rel": 1e-2}
    bf16 = case.get("y") == "bf16" or case.get("residual") == "bf16"
    return {"rel": 8e-3 if bf16 else 4e-6}
