"""What is measured of this framework's speed: the operators that a GPT-OSS style
engine calls for every token, through the package's own entry points.

Two kinds of layer block and the head, at the sizes of a GPT-OSS-120B layer
(hidden and expert width 2880, 128 experts of which 4 are used, MXFP4 experts;
Q4_0 attention projections 2880 -> 4096 / 512 / 512 and 4096 -> 2880; a Q8_0 head
of 201,088 rows) and at generic smaller and ragged ones:

  moe   the quantized MoE block: router, top-k, gate/up, SwiGLU, down, combine,
        for `tokens` tokens through `layers` layers of distinct weights.
        "device": activations on the GPU (forward_moe_batch); "host": slices in
        host memory, as a caller outside Python passes them
        (forward_moe_batch_host).
  attn  what surrounds attention in a layer: RMSNorm with Q8_0 output, the fused
        Q/K/V projections of it, and the output projection of the attention
        context with its bias.
  head  the Q8_0 LM head: all logits of one token.

`skew` is how unequal the experts' popularity is: the router's bias of the
expert of rank r is -skew * log(r) (0: every expert alike).
"""
import math
import os
import sys

import numpy as np
import torch

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "stream-pt_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import spt  # noqa: E402

DEVICE = "cuda"
EPS = 1e-5
E2M1 = (0.0, 0.5, 1.0, 1.5, 2.0, 3.0, 4.0, 6.0, -0.0, -0.5, -1.0, -1.5, -2.0, -3.0, -4.0, -6.0)


def _moe(name, tokens, layers=1, skew=0.0, io="device", hidden=2880, inner=2880, experts=128, used=4, bias=True):
    return {"name": name, "kind": "moe", "tokens": tokens, "layers": layers, "skew": skew, "io": io, "hidden": hidden,
            "inner": inner, "experts": experts, "used": used, "bias": bias}


def _attn(name, tokens, hidden=2880, q=4096, kv=512, bias=True):
    return {"name": name, "kind": "attn", "tokens": tokens, "hidden": hidden, "q": q, "kv": kv, "bias": bias}


def _head(name, rows, hidden=2880):
    return {"name": name, "kind": "head", "rows": rows, "hidden": hidden}


def listed():
    return [
        # One sequence being generated: one token through the layers in turn.  Six
        # layers' experts are more bytes than any cache holds.
        _moe("moe_decode_1", 1, layers=6),
        # A few sequences generated together (continuous batching).
        _moe("moe_decode_8", 8, layers=2),
        # A busy server's decode step: most experts are touched by a token or two.
        _moe("moe_decode_64", 64),
        # The same from the host's side: an odd number of sequences, activations in
        # host memory, the caller waits for the result.
        _moe("moe_host_13", 13, io="host"),
        # A prompt's chunk near the engine's default size of 32, popular experts.
        _moe("moe_prefill_37", 37, skew=1.1),
        # A long prompt's chunk, popular experts: groups of one to hundreds.
        _moe("moe_prefill_512", 512, skew=1.1),
        # Large prefill chunks of many prompts, every expert in use.
        _moe("moe_prefill_2000", 2000),
        # The projections around attention: one token, a server's decode batch or
        # small chunk (odd), a prompt's chunk, and a large one (odd).
        _attn("attn_1", 1),
        _attn("attn_29", 29),
        _attn("attn_512", 512),
        _attn("attn_1999", 1999),
        # The logits of a generated token, over the whole vocabulary.
        _head("head_vocab", 201088),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["moe", "moe", "moe", "attn", "attn", "head"])
    # Widths: the model's own, and others that are whole blocks of 32.
    hidden = rng.choice([2880, 2880, 32 * rng.randint(16, 90)])
    if kind == "moe":
        inner = rng.choice([hidden, hidden, 32 * rng.randint(16, 90)])
        experts = rng.choice([128, 128, 64, 32, rng.randint(8, 128)])
        used = rng.choice([4, 4, 2, rng.randint(1, 8)])
        c = _moe("", _log_int(rng, 1, 2000), 1, rng.choice([0.0, 0.6, 1.1]), rng.choice(["device", "device", "device", "host"]),
                 hidden, inner, experts, min(used, experts), rng.random() < 0.8)
        if c["tokens"] * c["used"] > 8000:
            c["tokens"] = 8000 // c["used"]
    elif kind == "attn":
        c = _attn("", _log_int(rng, 1, 2000), hidden, 64 * rng.randint(8, 64), 64 * rng.randint(1, 16), rng.random() < 0.8)
    else:
        c = _head("", _log_int(rng, 8000, 201088), hidden)
    del c["name"]
    return c


# ---- inputs: all from torch's generator on the GPU, in this fixed order ---------


def _generator(seed):
    g = torch.Generator(device=DEVICE)
    g.manual_seed(int(seed))
    return g


def _normal(g, shape, std=1.0):
    return torch.randn(shape, generator=g, device=DEVICE) * std


def _unit_rows(x):
    """Rows of root mean square 1, as a norm leaves them."""
    return x / x.double().square().mean(-1, keepdim=True).sqrt().float()


def _mxfp4(g, experts, rows, cols):
    """MXFP4 blocks: every nibble alike, E8M0 118..124 (weights of about 0.02)."""
    n = experts * rows * (cols // 32)
    w = torch.randint(0, 256, (n, 17), generator=g, device=DEVICE, dtype=torch.uint8)
    w[:, 0] = torch.randint(118, 125, (n,), generator=g, device=DEVICE, dtype=torch.uint8)
    return w.view(experts, rows, cols // 32, 17)


def _scaled_blocks(g, rows, cols, size):
    """Q4_0 (size 18) or Q8_0 (size 34) blocks: every code alike, fp16 scales of about 0.01."""
    n = rows * (cols // 32)
    w = torch.randint(0, 256, (n, size), generator=g, device=DEVICE, dtype=torch.uint8)
    w[:, :2] = (_normal(g, (n,), 0.01).abs()).half().view(torch.uint8).view(n, 2)
    return w.view(rows, cols // 32, size)


def _inputs(case, seed):
    """The tensors of a case; prepare() hands them to the framework, exact() reads them."""
    g = _generator(seed)
    H = case["hidden"]
    if case["kind"] == "moe":
        D, E, T = case["inner"], case["experts"], case["tokens"]
        got = []
        for _ in range(case["layers"]):
            t = {"x": _unit_rows(_normal(g, (T, H))), "router": _normal(g, (E, H), 0.02),
                 "gate": _mxfp4(g, E, D, H), "up": _mxfp4(g, E, D, H), "down": _mxfp4(g, E, H, D)}
            rank = torch.randperm(E, generator=g, device=DEVICE) + 1
            if case["bias"]:
                t["router_bias"] = _normal(g, (E,), 0.02) - case["skew"] * rank.float().log()
                t["gate_bias"], t["up_bias"] = _normal(g, (E, D), 0.02), _normal(g, (E, D), 0.02)
                t["down_bias"] = _normal(g, (E, H), 0.02)
            got.append(t)
        return got
    if case["kind"] == "attn":
        T, Q, KV = case["tokens"], case["q"], case["kv"]
        t = {"x": _normal(g, (T, H), 3.0), "norm": 1.0 + _normal(g, (H,), 0.1), "ctx": _normal(g, (T, Q), 0.5)}
        for n, rows, cols in (("wq", Q, H), ("wk", KV, H), ("wv", KV, H), ("wo", H, Q)):
            t[n] = _scaled_blocks(g, rows, cols, 18)
            if case["bias"]:
                t["b" + n[1]] = _normal(g, (rows,), 0.02)
        return t
    return {"x": _unit_rows(_normal(g, (H,))), "w": _scaled_blocks(g, case["rows"], H, 34)}


# ---- the framework's side -------------------------------------------------------


def _tensor(name, typ, t, shape):
    return spt.Tensor.make(name, typ, shape, t.data_ptr(), t.numel() * t.element_size())


def prepare(case, seed):
    data = _inputs(case, seed)
    s = {"case": case, "data": data, "ctx": spt.Context(0, torch.cuda.current_stream().cuda_stream)}
    H = case["hidden"]
    if case["kind"] == "moe":
        D, E, T = case["inner"], case["experts"], case["tokens"]
        host = case["io"] == "host"
        s["layers"] = []
        for t in data:
            lw = spt.MoELayer()
            lw.ffn_gate_inp = _tensor("ffn_gate_inp.weight", spt.TYPE_F32, t["router"], [H, E])
            lw.ffn_gate_exps = _tensor("ffn_gate_exps.weight", spt.TYPE_MXFP4, t["gate"], [H, D, E])
            lw.ffn_up_exps = _tensor("ffn_up_exps.weight", spt.TYPE_MXFP4, t["up"], [H, D, E])
            lw.ffn_down_exps = _tensor("ffn_down_exps.weight", spt.TYPE_MXFP4, t["down"], [D, H, E])
            if case["bias"]:
                lw.ffn_gate_inp_bias = _tensor("ffn_gate_inp.bias", spt.TYPE_F32, t["router_bias"], [E])
                lw.ffn_gate_exps_bias = _tensor("ffn_gate_exps.bias", spt.TYPE_F32, t["gate_bias"], [D, E])
                lw.ffn_up_exps_bias = _tensor("ffn_up_exps.bias", spt.TYPE_F32, t["up_bias"], [D, E])
                lw.ffn_down_exps_bias = _tensor("ffn_down_exps.bias", spt.TYPE_F32, t["down_bias"], [H, E])
            x = t["x"].cpu().numpy() if host else t["x"]
            out = np.empty((T, H), np.float32) if host else torch.empty(T, H, device=DEVICE)
            s["layers"].append((lw, x, out))
        s["cfg"] = spt.MoEConfig(H, D, E, case["used"])
    elif case["kind"] == "attn":
        T, Q, KV = case["tokens"], case["q"], case["kv"]
        s["norm"] = _tensor("attn_norm.weight", spt.TYPE_F32, data["norm"], [H])
        for n, rows, cols in (("q", Q, H), ("k", KV, H), ("v", KV, H), ("o", H, Q)):
            s["w" + n] = _tensor("attn_%s.weight" % n, spt.TYPE_Q4_0, data["w" + n], [cols, rows])
            s["b" + n] = _tensor("attn_%s.bias" % n, spt.TYPE_F32, data["b" + n], [rows]) if case["bias"] else None
            s[n] = torch.empty(T, rows, device=DEVICE)
        s["y"] = torch.empty(T, H, device=DEVICE)
        s["yq"] = torch.empty(T * (H // 32) * 34, dtype=torch.uint8, device=DEVICE)
    else:
        s["w"] = _tensor("output.weight", spt.TYPE_Q8_0, data["w"], [H, case["rows"]])
        s["logits"] = torch.empty(case["rows"], device=DEVICE)
    return s


def run(s):
    case, ctx = s["case"], s["ctx"]
    if case["kind"] == "moe":
        call = ctx.forward_moe_batch_host if case["io"] == "host" else ctx.forward_moe_batch
        for lw, x, out in s["layers"]:
            call(s["cfg"], lw, x, out, case["tokens"])
        return [out for _, _, out in s["layers"]]
    if case["kind"] == "attn":
        T = case["tokens"]
        ctx.rmsnorm_batch_into(s["norm"], s["data"]["x"], s["y"], T, EPS, s["yq"])
        ctx.mul_q40_qkv_batch_into([s["wq"], s["wk"], s["wv"]], [s["bq"], s["bk"], s["bv"]], None, [s["q"], s["k"], s["v"]],
                                   T, xq=s["yq"], x_len=T * case["hidden"])
        ctx.mul_q40_batch_bias_into(s["wo"], s["bo"], s["data"]["ctx"], s["o"], T)
        return {n: s[n] for n in ("y", "yq", "q", "k", "v", "o")}
    ctx.mul_q80_into(s["w"], s["data"]["x"], s["logits"])
    return s["logits"]


# ---- what a pass cannot do without ----------------------------------------------


def work(case):
    H = case["hidden"]
    if case["kind"] == "moe":
        D, E, T, k = case["inner"], case["experts"], case["tokens"], case["used"]
        # Experts touched by T tokens, each drawing k without replacement: the
        # expected count, under the popularity that the router's bias and noise give
        # (its share is near r^-skew / sum for the expert of rank r).
        p = [r ** -case["skew"] if case["bias"] else 1.0 for r in range(1, E + 1)]
        total = sum(p)
        touched = max(min(E, k), sum(1.0 - (1.0 - min(1.0, k * v / total)) ** T for v in p))
        b = 4 if case["bias"] else 0
        per_expert = 3 * D * (H // 32) * 17 + (2 * D + H) * b
        one = E * (4 * H + b) + touched * per_expert + 8 * T * H
        return {"bytes": case["layers"] * one, "flops": case["layers"] * (2.0 * T * E * H + 6.0 * T * k * D * H)}
    if case["kind"] == "attn":
        T, Q, KV = case["tokens"], case["q"], case["kv"]
        rows = Q + 2 * KV
        b = 4 if case["bias"] else 0
        return {"bytes": (rows * (H // 32) + H * (Q // 32)) * 18 + (rows + H) * b + 4 * H
                + T * (4 * H + 4 * H + (H // 32) * 34 + 4 * rows + 4 * Q + 4 * H),
                "flops": 2.0 * T * (rows * H + H * Q)}
    return {"bytes": case["rows"] * (H // 32) * 34 + 4 * H + 4 * case["rows"], "flops": 2.0 * case["rows"] * H}


def tolerance(case):
    if case["kind"] == "moe":
        # A gate or up value that moves in its last bit can move a code of the
        # expert's 8-bit inner activations by one.  Four times what the framework's
        # own forms (grouped GEMV and GEMM) differ by on the listed cases.
        return {"rel": 4e-4, "max": 0.03}
    # Exact integer sums per block, added over the blocks in 32 bits (2e-7 between
    # two orders); the norm's 8-bit codes are bytes and stay the same.
    return {"rel": 1e-6, "max": 1e-5, "differ": 0.0}


# ---- the same in 64 bits --------------------------------------------------------


def _q8_0(x):
    """GGML Q8_0 of rows of 32: (codes, fp16 scales), the format's 32-bit rule."""
    x = x.float().view(*x.shape[:-1], -1, 32)
    d = x.abs().amax(-1) / 127.0
    inv = torch.where(d != 0, 1.0 / d, torch.zeros_like(d))
    v = x * inv.unsqueeze(-1)
    codes = torch.sign(v) * torch.floor(v.abs().double() + 0.5).float()  # halves away from zero
    return codes.clamp(-127, 127), d.half()


def _q8_values(x):
    c, d = _q8_0(x)
    return (c.double() * d.double().unsqueeze(-1)).flatten(-2)


def _mxfp4_values(w):
    """[rows, blocks, 17] bytes -> [rows, cols] in 64 bits."""
    lut = torch.tensor(E2M1, dtype=torch.float64, device=w.device)
    nib = w[..., 1:].long()
    v = torch.cat([lut[nib & 15], lut[nib >> 4]], -1)
    return (v * torch.exp2(w[..., :1].double() - 127.0)).flatten(-2)


def _q40_values(w):
    d = w[..., :2].contiguous().view(torch.float16).double()
    nib = w[..., 2:].long()
    return (torch.cat([nib & 15, nib >> 4], -1).double().sub(8.0) * d).flatten(-2)


def _exact_moe(case, t):
    x, T, k = t["x"], case["tokens"], case["used"]
    logits = x.double() @ t["router"].double().T
    if case["bias"]:
        logits += t["router_bias"].double()
    top, ids = logits.topk(k, -1)
    weight = torch.softmax(top, -1)
    xq = _q8_values(x)
    out = torch.zeros(T, case["hidden"], dtype=torch.float64, device=x.device)
    for e in ids.unique().tolist():
        tok, rank = (ids == e).nonzero(as_tuple=True)
        gate = xq[tok] @ _mxfp4_values(t["gate"][e]).T
        up = xq[tok] @ _mxfp4_values(t["up"][e]).T
        if case["bias"]:
            gate, up = gate + t["gate_bias"][e].double(), up + t["up_bias"][e].double()
        gate, up = gate.clamp(max=7.0), up.clamp(-7.0, 7.0)
        act = gate * torch.sigmoid(1.702 * gate) * (up + 1.0)
        y = _q8_values(act) @ _mxfp4_values(t["down"][e]).T
        if case["bias"]:
            y = y + t["down_bias"][e].double()
        out.index_add_(0, tok, y * weight[tok, rank].unsqueeze(-1))
    return out


def exact(case, seed):
    data = _inputs(case, seed)
    if case["kind"] == "moe":
        got = [_exact_moe(case, t) for t in data]
        return [o.cpu().numpy() for o in got] if case["io"] == "host" else got
    if case["kind"] == "attn":
        x = data["x"].double()
        y = x * data["norm"].double() / (x.square().mean(-1, keepdim=True) + EPS).sqrt()
        yq, ctx = _q8_values(y), _q8_values(data["ctx"])
        out = {"y": y, "yq": None}
        for n, v in (("q", yq), ("k", yq), ("v", yq), ("o", ctx)):
            out[n] = v @ _q40_values(data["w" + n]).T
            if case["bias"]:
                out[n] += data["b" + n].double()
        return out
    w, x = data["w"], data["x"].double()
    parts = []
    for r in range(0, case["rows"], 16384):
        b = w[r:r + 16384]
        d = b[..., :2].contiguous().view(torch.float16).double()
        parts.append((b[..., 2:].contiguous().view(torch.int8).double() * d).flatten(-2) @ x)
    return torch.cat(parts)
