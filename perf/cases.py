"""Performance cases of Co-ALiBi attention: what a program that uses the package has it do.

A case is a dict of plain values.  ``kind`` says which entry point it goes through:

- ``train``: ``co_alibi_attention`` with gradients, forward and backward (dQ, dK, dV);
- ``prefill``: ``co_alibi_attention`` without gradients;
- ``layer``: ``gpt.CausalCoALiBiAttention``, the attention layer of the GPT training step (QKV
  projection, attention, output projection), forward and backward under bf16 autocast;
- ``decode``: ``co_alibi_decode``, one new token against a key / value cache.

``layout`` of a train or prefill case: "bhsd" hands over contiguous (B, H, S, D) tensors, "bshd"
transposed views of (B, S, H, D) ones, the form in which a model's projections leave them.
``full_work`` switches the library's tail skip off around the call.

Inputs are N(0, 1) times ``scale``, as in the package's benchmark workloads (0.3 and 0.5 there;
1.0 stands for trained projections, whose logits spread more).
"""
import math

import torch

from co_alibi_attn import _native, co_alibi_attention, co_alibi_decode
from co_alibi_attn.gpt import CausalCoALiBiAttention, GPTConfig

DTYPES = {"fp16": torch.float16, "bf16": torch.bfloat16, "fp32": torch.float32}


def _train(name, B, Hq, Hkv, Sq, Skv, D, dtype, causal=True, scale=0.5, layout="bhsd", full_work=False, kind="train"):
    c = {"kind": kind, "B": B, "Hq": Hq, "Hkv": Hkv, "Sq": Sq, "Skv": Skv, "D": D, "dtype": dtype, "causal": causal,
         "scale": scale, "layout": layout, "full_work": full_work}
    return dict(c, name=name) if name else c


def _layer(name, B, S, n_head, head_dim, scale=1.0):
    c = {"kind": "layer", "B": B, "S": S, "n_head": n_head, "head_dim": head_dim, "scale": scale}
    return dict(c, name=name) if name else c


def _decode(name, B, Hq, Hkv, L, cap, D, dtype, ragged, scale=0.5):
    c = {"kind": "decode", "B": B, "Hq": Hq, "Hkv": Hkv, "L": L, "cap": cap, "D": D, "dtype": dtype, "ragged": ragged,
         "scale": scale}
    return dict(c, name=name) if name else c


def listed():
    return [
        # The fp32 validation configuration: one short sequence, where latency and launches count.
        _train("train_tiny_fp32", 1, 2, 2, 128, 128, 64, "fp32", scale=1.0),
        # fp32 validation of a model-sized layer with a ragged length.
        _train("train_fp32", 2, 12, 12, 1000, 1000, 64, "fp32"),
        # The attention layer of the 12-layer GPT training step (B 8, S 1024, d_model 768, 12 heads).
        _layer("train_gpt_layer", 8, 1024, 12, 64),
        # The headline operator.
        _train("train_headline", 4, 16, 16, 4096, 4096, 128, "fp16"),
        # The headline heads with every visible key processed, as a comparison with other
        # implementations does it (half the batch, which keeps its pass near the headline's).
        _train("train_full_work", 2, 16, 16, 4096, 4096, 128, "fp16", full_work=True),
        # Grouped-query long context.
        _train("train_gqa", 1, 32, 8, 8192, 8192, 128, "bf16"),
        # Small head dim, very long sequence.
        _train("train_long", 1, 8, 8, 16384, 16384, 64, "fp16", scale=0.3),
        # Non-causal attention of a short ragged query block over a longer ragged context
        # (cross attention, an encoder's memory), with gradients.
        _train("train_cross", 2, 16, 16, 333, 2047, 128, "fp16", causal=False, layout="bshd"),
        # A prompt of ordinary ragged length through the grouped-query model, one request.
        _train("prefill_prompt", 1, 32, 8, 1741, 1741, 128, "bf16", layout="bshd", kind="prefill"),
        # The next token after a long prompt, one sequence in a larger cache.
        _decode("decode_one", 1, 32, 8, 8192, 16384, 128, "bf16", False),
        # The next token of 16 sequences of different lengths (a serving batch).
        _decode("decode_serving", 16, 32, 8, 8192, 8192, 128, "bf16", True),
        # The next token of one very long sequence.
        _decode("decode_long", 1, 32, 8, 131072, 131072, 128, "bf16", False),
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def _cost(c):
    """Products of one pass, weighted by how the data type's matrix rate differs: bounds a draw."""
    if c["kind"] == "layer":
        C = c["n_head"] * c["head_dim"]
        return 3 * 8 * c["B"] * c["S"] * C * C + 14 * c["head_dim"] * c["B"] * c["n_head"] * c["S"] ** 2 / 2
    if c["kind"] == "decode":  # bytes bound it
        return 200 * 4 * c["B"] * c["Hkv"] * c["cap"] * c["D"]
    pairs = c["B"] * c["Hq"] * _visible_pairs(c)
    return pairs * c["D"] * (14 if c["kind"] == "train" else 4) * (16 if c["dtype"] == "fp32" else 1)


def draw(rng):
    most = max(_cost(c) for c in listed())
    while True:
        kind = rng.choices(("train", "prefill", "layer", "decode"), (8, 4, 2, 6))[0]
        if kind == "layer":
            c = _layer(None, _log_int(rng, 1, 16), _log_int(rng, 64, 4096), rng.choice((2, 4, 6, 8, 12, 16)),
                       rng.choice((64, 64, 128)), rng.choice((0.5, 1.0)))
            if _cost(c) <= 0.2 * most:
                return c
            continue
        hkv = rng.choice((1, 2, 4, 6, 8, 12, 16, 32))
        hq = hkv * rng.choice([g for g in (1, 1, 1, 2, 4, 8) if g * hkv <= 32])
        D = rng.choices((32, 64, 128, 256), (1, 4, 5, 1))[0]
        scale = rng.choice((0.3, 0.5, 0.5, 1.0))
        if kind == "decode":
            L = _log_int(rng, 16, 131072)
            cap = L + rng.choice((0, 0, rng.randrange(1, L + 1)))
            c = _decode(None, _log_int(rng, 1, 64), hq, hkv, L, cap, D, rng.choice(("bf16", "bf16", "fp16")),
                        rng.random() < 0.5, scale)
            if 4 * c["B"] * hkv * cap * D <= 2 << 30:
                return c
            continue
        dtype = rng.choices(("fp16", "bf16", "fp32"), (4, 4, 1))[0]
        if dtype == "fp32" and D == 256:
            continue
        causal = rng.random() < 0.75
        sq = _log_int(rng, 32, 16384)
        skv = sq if causal else _log_int(rng, 32, 8192)
        c = _train(None, _log_int(rng, 1, 16), hq, hkv, sq, skv, D, dtype, causal, scale, rng.choice(("bhsd", "bshd")),
                   rng.random() < 0.15, kind)
        elements = c["B"] * D * (hq * sq + hkv * skv)
        if _cost(c) <= most and elements <= 1 << 26:
            return c


# ------------------------------------------------------------------ inputs


def _normal(gen, shape, scale):
    return torch.randn(shape, generator=gen, device="cuda") * scale


def _inputs(c, seed):
    """The case's tensors as the caller holds them, before any is marked as needing a gradient."""
    gen = torch.Generator(device="cuda").manual_seed(seed)
    dt = DTYPES[c.get("dtype", "bf16")]
    if c["kind"] == "layer":
        C = c["n_head"] * c["head_dim"]
        # A LayerNorm's output, and the gradient of the residual stream; weights of std 1/sqrt(C)
        # keep q and k at the inputs' scale.
        x = _normal(gen, (c["B"], c["S"], C), c["scale"])
        wqkv = _normal(gen, (3 * C, C), C ** -0.5)
        wproj = _normal(gen, (C, C), C ** -0.5)
        g = _normal(gen, (c["B"], c["S"], C), 1.0)
        return x, wqkv, wproj, g
    if c["kind"] == "decode":
        B, Hq, Hkv, D = c["B"], c["Hq"], c["Hkv"], c["D"]
        q = _normal(gen, (B, Hq, 1, D), c["scale"]).to(dt)
        k = _normal(gen, (B, Hkv, c["cap"], D), c["scale"]).to(dt)
        v = _normal(gen, (B, Hkv, c["cap"], D), c["scale"]).to(dt)
        lens = None
        if c["ragged"]:
            lens = torch.randint((c["L"] + 7) // 8, c["L"] + 1, (B,), generator=gen, device="cuda", dtype=torch.int32)
        return q, k, v, lens
    B, D = c["B"], c["D"]

    def heads(H, S, scale):
        if c["layout"] == "bshd":
            return _normal(gen, (B, S, H, D), scale).to(dt).transpose(1, 2)
        return _normal(gen, (B, H, S, D), scale).to(dt)

    q = heads(c["Hq"], c["Sq"], c["scale"])
    k = heads(c["Hkv"], c["Skv"], c["scale"])
    v = heads(c["Hkv"], c["Skv"], c["scale"])
    do = heads(c["Hq"], c["Sq"], 1.0) if c["kind"] == "train" else None
    return q, k, v, do


def prepare(case, seed):
    t = _inputs(case, seed)
    if case["kind"] == "layer":
        x, wqkv, wproj, g = t
        cfg = GPTConfig(n_layer=1, n_head=case["n_head"], d_model=case["n_head"] * case["head_dim"])
        layer = CausalCoALiBiAttention(cfg, co_alibi_attention).cuda()
        with torch.no_grad():
            layer.qkv.weight.copy_(wqkv)
            layer.proj.weight.copy_(wproj)
        return {"case": case, "layer": layer, "x": x.requires_grad_(), "g": g.to(torch.bfloat16)}
    if case["kind"] == "train":
        for x in t[:3]:
            x.requires_grad_()
    return {"case": case, "t": t}


# ------------------------------------------------------------------ one pass


def run(state):
    c = state["case"]
    if c["kind"] == "layer":
        layer = state["layer"]
        with torch.autocast(device_type="cuda", dtype=torch.bfloat16):
            y = layer(state["x"])
        dx, dwqkv, dwproj = torch.autograd.grad(y, (state["x"], layer.qkv.weight, layer.proj.weight), state["g"])
        return {"y": y.detach(), "dx": dx, "dwqkv": dwqkv, "dwproj": dwproj}
    if c["kind"] == "decode":
        q, k, v, lens = state["t"]
        return co_alibi_decode(q, k, v, seq_len=c["L"] if lens is None else lens, max_seq_len=c["L"])
    if c["full_work"]:
        with _native.tail_skip(False):
            return _attend(c, *state["t"])
    return _attend(c, *state["t"])


def _attend(c, q, k, v, do):
    if c["kind"] == "prefill":
        with torch.no_grad():
            return co_alibi_attention(q, k, v, causal=c["causal"])
    o = co_alibi_attention(q, k, v, causal=c["causal"])
    dq, dk, dv = torch.autograd.grad(o, (q, k, v), do)
    return {"o": o.detach(), "dq": dq, "dk": dk, "dv": dv}


# ------------------------------------------------------------------ the work a pass cannot do without


def _slopes(n_heads, bias_max=8.0):
    """Penalty slope of every query head: twice the ALiBi slope."""
    n = 1 << (n_heads.bit_length() - 1)
    s = [2.0 ** (-bias_max * (h + 1) / n) for h in range(n)]
    s += [2.0 ** (-(bias_max / 2) * (2 * t + 1) / n) for t in range(n_heads - n)]
    return [2.0 * x for x in s]


def _visible_pairs(c):
    sq, skv = c["Sq"], c["Skv"]
    if not c["causal"]:
        return sq * skv
    m = min(sq, skv)
    return m * (m + 1) // 2 + (sq - m) * skv


def _weighty_pairs(c):
    """Pairs per batch entry, over all query heads, whose softmax weight the result can show.  The
    penalty of a key grows by slope * log2(e) / 2 binary digits per key to its right (a sigmoid is
    about 1/2), so a row cannot show the keys more than 26 (fp16), 32 (bf16) or 64 (fp32) digits
    left of its newest one.  Every visible pair counts where the caller asks for full work."""
    if c["full_work"]:
        return c["Hq"] * _visible_pairs(c)
    digits = {"fp16": 26, "bf16": 32, "fp32": 64}[c["dtype"]]
    total = 0
    for lam in _slopes(c["Hq"]):
        w = max(1, math.ceil(digits / (0.5 * lam * math.log2(math.e))))
        if not c["causal"]:
            total += c["Sq"] * min(w, c["Skv"])
        else:  # row i sees min(i + 1, Skv) keys, of which at most w count
            w = min(w, c["Skv"])
            m = min(w, c["Sq"])
            total += m * (m + 1) // 2 + (c["Sq"] - m) * w
    return total


def work(case):
    c = case
    if c["kind"] == "layer":
        C, T = c["n_head"] * c["head_dim"], c["B"] * c["S"]
        a = _train(None, c["B"], c["n_head"], c["n_head"], c["S"], c["S"], c["head_dim"], "bf16")
        # x in and dx, y out (y and g in bf16, the rest fp32), the two weights and their gradients.
        bytes_ = T * C * (4 + 4 + 2 + 2) + 2 * 4 * (3 * C * C + C * C)
        return {"bytes": bytes_, "flops": 3 * 2 * T * 4 * C * C + 14 * c["head_dim"] * c["B"] * _weighty_pairs(a)}
    size = 4 if c["dtype"] == "fp32" else 2
    if c["kind"] == "decode":
        rows = c["B"] * c["L"] * (0.5625 if c["ragged"] else 1.0)  # lengths uniform in [L/8, L]
        return {"bytes": size * (2 * rows * c["Hkv"] * c["D"] + 2 * c["B"] * c["Hq"] * c["D"]),
                "flops": 4 * c["D"] * c["Hq"] * rows}
    nq, nk = c["B"] * c["Hq"] * c["Sq"] * c["D"], c["B"] * c["Hkv"] * c["Skv"] * c["D"]
    pairs = c["B"] * _weighty_pairs(c)
    if c["kind"] == "prefill":
        return {"bytes": size * (2 * nq + 2 * nk), "flops": 4 * c["D"] * pairs}
    return {"bytes": size * (4 * nq + 4 * nk), "flops": 14 * c["D"] * pairs}


def tolerance(case):
    """About four times the error against float64 measured over the listed and 24 drawn cases: up to
    3.6e-7 in fp32, 3.8e-4 in fp16, 2.5e-3 in bf16 and 6.0e-3 for a layer's gradients (the
    operands and scores of the products are rounded to the data type; fp32 leaves room for
    another order of its sums at longer sequences)."""
    if case["kind"] == "layer":
        return {"rel": 2.5e-2}
    return {"rel": {"fp32": 5e-6, "fp16": 1.5e-3, "bf16": 1e-2}[case["dtype"]]}


# ------------------------------------------------------------------ the results in 64 bits


def _head_exact(q, k, v, do, lam, scale, causal):
    """(o, dq, dk, dv) of one head in float64, in blocks of rows; the gradients are None without do."""
    sq, skv = q.shape[0], k.shape[0]
    rows = max(16, min(sq, (1 << 25) // skv))
    o = torch.zeros_like(q)
    grads = None if do is None else (torch.zeros_like(q), torch.zeros_like(k), torch.zeros_like(v))
    for r0 in range(0, sq, rows):
        r1 = min(sq, r0 + rows)
        n = min(skv, r1) if causal else skv
        kk, vv = k[:n], v[:n]
        t = (q[r0:r1] @ kk.T) * scale
        sig = torch.sigmoid(t)
        ok = None
        if causal:
            ok = torch.arange(n, device=q.device)[None, :] <= torch.arange(r0, r1, device=q.device)[:, None]
            sig = torch.where(ok, sig, 0.0)
        z = sig.flip(1).cumsum(1).flip(1)
        t = t - lam * z
        del z
        if causal:
            t = torch.where(ok, t, -math.inf)
        p = torch.softmax(t, 1)
        del t
        o[r0:r1] = p @ vv
        if do is None:
            continue
        dq, dk, dv = grads
        g = do[r0:r1]
        dv[:n] += p.T @ g
        da = p * (g @ vv.T - (g * o[r0:r1]).sum(1, keepdim=True))
        ds = da - lam * sig * (1.0 - sig) * da.cumsum(1)
        dq[r0:r1] = (ds @ kk) * scale
        dk[:n] += (ds.T @ q[r0:r1]) * scale
    return o, grads


def _attention_exact(q, k, v, do, dtype, causal):
    """float64 (B, H, S, D) attention of inputs of any type, with gradients if do is given."""
    B, Hq, _, D = q.shape
    Hkv = k.shape[1]
    lams = torch.tensor(_slopes(Hq), dtype=torch.float32).to(dtype).double().tolist()
    scale = D ** -0.5
    o = torch.empty(q.shape, dtype=torch.float64, device=q.device)
    dq = dk = dv = None
    if do is not None:
        dq = torch.empty_like(o)
        dk = torch.zeros(k.shape, dtype=torch.float64, device=q.device)
        dv = torch.zeros_like(dk)
    for b in range(B):
        for h in range(Hq):
            g = h // (Hq // Hkv)
            out, grads = _head_exact(q[b, h].double(), k[b, g].double(), v[b, g].double(),
                                     None if do is None else do[b, h].double(), lams[h], scale, causal)
            o[b, h] = out
            if do is not None:
                dq[b, h] = grads[0]
                dk[b, g] += grads[1]
                dv[b, g] += grads[2]
    return o, dq, dk, dv


def exact(case, seed):
    t = _inputs(case, seed)
    if case["kind"] == "layer":
        x, wqkv, wproj, g = t
        x, wqkv, wproj, g = x.double(), wqkv.double(), wproj.double(), g.to(torch.bfloat16).double()
        B, S, C = x.shape
        H, D = case["n_head"], case["head_dim"]
        qkv = (x.view(-1, C) @ wqkv.T).view(B, S, 3, H, D)
        q, k, v = (qkv[:, :, i].transpose(1, 2) for i in range(3))
        da = (g.view(-1, C) @ wproj).view(B, S, H, D).transpose(1, 2)
        o, dq, dk, dv = _attention_exact(q, k, v, da, torch.bfloat16, True)
        o = o.transpose(1, 2).reshape(-1, C)
        dqkv = torch.stack([t.transpose(1, 2) for t in (dq, dk, dv)], 2).reshape(-1, 3 * C)
        return {"y": (o @ wproj.T).view(B, S, C), "dx": (dqkv @ wqkv).view(B, S, C), "dwqkv": dqkv.T @ x.view(-1, C),
                "dwproj": g.view(-1, C).T @ o}
    if case["kind"] == "decode":
        q, k, v, lens = t
        B, Hq, _, D = q.shape
        out = []
        for b in range(B):
            n = case["L"] if lens is None else int(lens[b])
            out.append(_attention_exact(q[b:b + 1], k[b:b + 1, :, :n], v[b:b + 1, :, :n], None, q.dtype, False)[0])
        return torch.cat(out)
    q, k, v, do = t
    o, dq, dk, dv = _attention_exact(q, k, v, do, q.dtype, case["causal"])
    return o if do is None else {"o": o, "dq": dq, "dk": dk, "dv": dv}
