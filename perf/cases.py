"""Timed workloads of the operator library: what a transformer's (and a convolution stack's) forward pass asks of
`ntops_amd.torch`, each through its public function.

`listed()` names the workloads, `draw(rng)` gives another one of the same ranges; `prepare` / `run` / `work` /
`tolerance` / `exact` serve both.  A case is a dict of plain values; "op" selects the family."""

import math

import torch
import torch.nn.functional as F

import ntops_amd

T = ntops_amd.torch

DTYPES = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}


def listed():
    return [
        # One decode step's residual add + norm: a handful of token rows, bound by launch and host latency.
        {"name": "norm_decode", "op": "add_rms_norm", "dtype": "bf16", "rows": 8, "cols": 4096},
        # The norm of a prefill whose width is not a multiple of the 16-byte pack (4100: ragged rows).
        {"name": "norm_ragged", "op": "layer_norm", "dtype": "bf16", "rows": 16384, "cols": 4100},
        # The activation over a prefill's hidden states in full precision.
        {"name": "activation", "op": "silu", "dtype": "f32", "rows": 8192, "cols": 4096},
        # Attention scores of a batch under a causal pattern (-inf above the diagonal), normalised over the keys.
        {"name": "softmax_scores", "op": "softmax", "dtype": "bf16", "batch": 4, "heads": 32, "q_len": 2048, "kv_len": 2048},
        # Rotary embedding of a prefill's q and k (grouped-query: 4 q heads to a k head), half-rotation layout.
        {"name": "rope_prefill", "op": "rope", "dtype": "bf16", "batch": 4, "seq": 4096, "q_heads": 32, "k_heads": 8, "dim": 128},
        # One decode step's projection of a small batch: streams the (out, in) weight once.
        {"name": "linear_decode", "op": "linear", "dtype": "bf16", "m": 8, "k": 4096, "n": 14336, "weight": "out_in", "bias": False},
        # A prefill's projection, weight stored (out, in) as F.linear's: matrix-bound, the largest case.
        {"name": "linear_prefill", "op": "linear", "dtype": "bf16", "m": 8192, "k": 4096, "n": 14336, "weight": "out_in", "bias": False},
        # The vocabulary projection of a GPT-2 sized model: 50257 columns, so output rows start at any 2-byte offset.
        {"name": "lm_head", "op": "linear", "dtype": "f16", "m": 8192, "k": 768, "n": 50257, "weight": "out_in", "bias": False},
        # Causal self-attention of a prefill.
        {"name": "attention_prefill", "op": "attention", "kind": "causal", "dtype": "bf16", "batch": 4, "q_heads": 32, "kv_heads": 32, "q_len": 2048, "kv_len": 2048, "dim": 128},
        # One decode step's attention over a grouped-query KV cache: the step's key and value are written into their
        # slot, then one query row per head reads the whole cache.
        {"name": "attention_decode", "op": "attention", "kind": "cache", "dtype": "bf16", "batch": 16, "q_heads": 32, "kv_heads": 8, "q_len": 1, "kv_len": 4096, "dim": 128},
        # Attention of a right-padded batch: one boolean mask (causal and not padding) per sequence, ragged length.
        {"name": "attention_masked", "op": "attention", "kind": "bool", "dtype": "f16", "batch": 8, "q_heads": 16, "kv_heads": 16, "q_len": 1000, "kv_len": 1000, "dim": 64},
        # A 3 x 3 layer of a convolution stack with its bias.
        {"name": "conv_3x3", "op": "conv2d", "dtype": "bf16", "batch": 32, "c": 256, "hw": 56, "out": 256, "kernel": 3, "stride": 1},
    ]


def _log(rng, lo, hi):
    """A whole number spread over the logarithm of [lo, hi]."""
    return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def _ragged(rng, v, unit):
    """`v` as it is (odd and ragged sizes) or, as often, a multiple of `unit`."""
    return max(unit, v // unit * unit) if rng.random() < 0.5 else v


def draw(rng):
    op = rng.choice(["add_rms_norm", "layer_norm", "silu", "softmax", "rope", "linear", "linear", "linear", "causal", "cache", "mask", "conv2d"])
    half = rng.choice(["bf16", "bf16", "f16"])
    dtype = rng.choice(["bf16", "f16", "f32"])
    if op in ("add_rms_norm", "layer_norm"):
        # decode to prefill rows; widths from 512 to 8192, ragged ones among them
        cols = _ragged(rng, _log(rng, 512, 8192), 64)
        most = (16384 * 4100 if dtype != "f32" else 8192 * 4100) // cols
        return {"op": op, "dtype": dtype, "rows": _log(rng, 1, min(most, 16384)), "cols": cols}
    if op == "silu":
        cols = _ragged(rng, _log(rng, 512, 14336), 64)
        return {"op": op, "dtype": dtype, "rows": _log(rng, 1, 8192 * 4096 // cols), "cols": cols}
    if op == "softmax":
        kv = _ragged(rng, _log(rng, 64, 4096), 64)
        heads = rng.choice([8, 12, 16, 32])
        batch = rng.choice([1, 2, 4])
        q = 1 if rng.random() < 0.25 else min(kv, 4 * 32 * 2048 * 2048 // (2 * kv * heads * batch))
        return {"op": op, "dtype": dtype, "batch": batch, "heads": heads, "q_len": q, "kv_len": kv}
    if op == "rope":
        seq = 1 if rng.random() < 0.25 else _ragged(rng, _log(rng, 16, 4096), 16)
        heads = rng.choice([8, 16, 32])
        return {"op": op, "dtype": half, "batch": rng.choice([1, 2, 4]), "seq": seq, "q_heads": heads, "k_heads": heads // rng.choice([1, 4, 8]), "dim": rng.choice([64, 128])}
    if op == "linear":
        # decode (a few rows) to prefill (thousands) over the projections of small to large layers, and the
        # vocabulary projection; weights stored (out, in) or (in, out), with or without a bias
        m = _log(rng, 1, 8192)
        k, n = rng.choice([(768, 2304), (768, 3072), (1024, 1024), (1600, 6400), (4096, 4096), (4096, 6144), (4096, 14336), (14336, 4096), (768, 50257), (1024, 32000)])
        weight = rng.choice(["out_in", "out_in", "in_out"])
        if dtype == "f32":
            m = min(m, 2048 if k * n <= 4096 * 4096 else 512)
        elif rng.random() < 0.5:
            dtype = half
        return {"op": op, "dtype": dtype, "m": m, "k": k, "n": n, "weight": weight, "bias": rng.random() < 0.5}
    if op == "conv2d":
        kernel, stride = rng.choice([(1, 1), (3, 1), (3, 1), (3, 2)])
        c, out = rng.choice([(64, 64), (64, 128), (128, 128), (128, 256), (256, 256), (512, 512)])
        hw = _log(rng, 7, 7168 // c)
        return {"op": op, "dtype": half, "batch": _log(rng, 1, 32), "c": c, "hw": hw, "out": out, "kernel": kernel, "stride": stride}
    dim = rng.choice([64, 128, 128])
    q_heads = rng.choice([8, 16, 32])
    group = rng.choice([1, 1, 4, 8])
    if op == "cache":
        batch = _log(rng, 1, 32)
        kv = _log(rng, 64, 16384)
        kv = max(64, min(kv, 16 * 8 * 4096 * 128 // (batch * (q_heads // group) * dim)))
        return {"op": "attention", "kind": "cache", "dtype": half, "batch": batch, "q_heads": q_heads, "kv_heads": q_heads // group, "q_len": 1, "kv_len": kv, "dim": dim}
    s = _ragged(rng, _log(rng, 64, 2048), 64)
    kind = "causal" if op == "causal" else rng.choice(["bool", "float"])
    batch = rng.choice([1, 2, 4]) if kind == "causal" else rng.choice([1, 2, 4, 8])
    if kind != "causal":
        dim = rng.choice([64, 64, 80, 128])
    return {"op": "attention", "kind": kind, "dtype": half, "batch": batch, "q_heads": q_heads, "kv_heads": q_heads // group, "q_len": s, "kv_len": s, "dim": dim}


def _lengths(case):
    """Attended keys of each sequence of a right-padded batch: from half the length to all of it."""
    b, s = case["batch"], case["kv_len"]
    return [s - (s // 2) * i // max(1, b) for i in range(b)]


def _mask(case, device):
    """True where query i of a sequence may attend key j: j <= i and j is not padding.  (batch, 1, q, kv)."""
    s = case["kv_len"]
    keep = torch.ones(case["q_len"], s, dtype=torch.bool, device=device).tril()
    real = torch.arange(s, device=device)[None, :] < torch.tensor(_lengths(case), device=device)[:, None]
    return keep[None, None] & real[:, None, None]


def prepare(case, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    dt = DTYPES[case["dtype"]]

    def normal(*shape, std=1.0, mean=0.0):
        t = torch.randn(*shape, generator=g, device="cuda")
        return (t.mul_(std) if std != 1.0 else t).add_(mean).to(dt) if mean else (t.mul_(std) if std != 1.0 else t).to(dt)

    op = case["op"]
    st = {"case": case}
    if op in ("add_rms_norm", "layer_norm"):
        rows, cols = case["rows"], case["cols"]
        st["x"] = normal(rows, cols)
        st["w"] = normal(cols, std=0.02, mean=1.0)
        if op == "add_rms_norm":
            st["res"] = normal(rows, cols)
        else:
            st["b"] = normal(cols, std=0.02)
    elif op == "silu":
        st["x"] = normal(case["rows"], case["cols"])
    elif op == "softmax":
        q, kv = case["q_len"], case["kv_len"]
        x = normal(case["batch"], case["heads"], q, kv, std=1 / math.sqrt(128))
        st["x"] = x.masked_fill_(torch.ones(q, kv, dtype=torch.bool, device="cuda").triu(kv - q + 1), float("-inf"))
    elif op == "rope":
        b, s, d = case["batch"], case["seq"], case["dim"]
        st["q"] = normal(b, s, case["q_heads"], d)
        st["k"] = normal(b, s, case["k_heads"], d)
        angle = torch.arange(s, device="cuda", dtype=torch.float64)[:, None] * (10000.0 ** (-torch.arange(0, d, 2, device="cuda", dtype=torch.float64) / d))
        angle = torch.cat([angle, angle], dim=1)
        st["sin"], st["cos"] = angle.sin().to(dt), angle.cos().to(dt)
    elif op == "linear":
        m, k, n = case["m"], case["k"], case["n"]
        st["x"] = normal(m, k)
        st["w"] = normal(n, k, std=0.02).t() if case["weight"] == "out_in" else normal(k, n, std=0.02)
        if case["bias"]:
            st["bias"] = normal(n, std=0.02)
    elif op == "attention":
        b, hq, hk, sq, skv, d = (case[x] for x in ("batch", "q_heads", "kv_heads", "q_len", "kv_len", "dim"))
        st["q"] = normal(b, hq, sq, d)
        if case["kind"] == "cache":  # the cache was allocated for more tokens than it holds
            room = -(-skv // 256) * 256 + 256
            st["k"], st["v"] = (normal(b, hk, room, d)[:, :, :skv] for _ in range(2))
            st["k_new"], st["v_new"] = (normal(b, hk, 1, d) for _ in range(2))
        else:
            st["k"], st["v"] = (normal(b, hk, skv, d) for _ in range(2))
        if case["kind"] == "bool":
            st["mask"] = _mask(case, "cuda")
        elif case["kind"] == "float":
            st["mask"] = torch.zeros(b, 1, sq, skv, dtype=dt, device="cuda").masked_fill_(~_mask(case, "cuda"), float("-inf"))
    else:
        n, c, hw, out, ks = (case[x] for x in ("batch", "c", "hw", "out", "kernel"))
        st["x"] = normal(n, c, hw, hw)
        st["w"] = normal(out, c, ks, ks, std=1 / math.sqrt(c * ks * ks))
        st["bias"] = normal(out, std=0.02)
    return st


def run(st):
    case = st["case"]
    op = case["op"]
    if op == "add_rms_norm":
        return T.add_rms_norm(st["x"], st["res"], (case["cols"],), st["w"], 1e-6)
    if op == "layer_norm":
        return T.layer_norm(st["x"], (case["cols"],), st["w"], st["b"], 1e-5)
    if op == "silu":
        return T.silu(st["x"])
    if op == "softmax":
        return T.softmax(st["x"], -1)
    if op == "rope":
        return T.rotary_position_embedding_qk(st["q"], st["k"], st["sin"], st["cos"], interleaved=False)
    if op == "linear":
        if case["bias"]:
            return T.addmm(st["bias"], st["x"], st["w"])
        return T.mm(st["x"], st["w"])
    if op == "attention":
        gqa = case["q_heads"] != case["kv_heads"]
        if case["kind"] == "causal":
            return T.scaled_dot_product_attention(st["q"], st["k"], st["v"], is_causal=True, enable_gqa=gqa)
        if case["kind"] == "cache":
            last = case["kv_len"] - 1
            k_slot, v_slot = st["k"][:, :, last:], st["v"][:, :, last:]
            out = T.scaled_dot_product_attention(
                st["q"], st["k"], st["v"], enable_gqa=gqa, present_key=st["k_new"], present_value=st["v_new"],
                present_key_slot=k_slot, present_value_slot=v_slot)
            return out, k_slot, v_slot
        return T.scaled_dot_product_attention(st["q"], st["k"], st["v"], attn_mask=st["mask"], enable_gqa=gqa)
    return T.conv2d(st["x"], st["w"], st["bias"], stride=case["stride"], padding=case["kernel"] // 2)


def _size(case):
    return 4 if case["dtype"] == "f32" else 2


def work(case):
    e, op = _size(case), case["op"]
    if op == "add_rms_norm":
        n = case["rows"] * case["cols"]
        return {"bytes": e * (4 * n + case["cols"]), "flops": 5 * n}
    if op == "layer_norm":
        n = case["rows"] * case["cols"]
        return {"bytes": e * (2 * n + 2 * case["cols"]), "flops": 8 * n}
    if op == "silu":
        n = case["rows"] * case["cols"]
        return {"bytes": e * 2 * n, "flops": 4 * n}
    if op == "softmax":
        n = case["batch"] * case["heads"] * case["q_len"] * case["kv_len"]
        return {"bytes": e * 2 * n, "flops": 4 * n}
    if op == "rope":
        n = case["batch"] * case["seq"] * (case["q_heads"] + case["k_heads"]) * case["dim"]
        return {"bytes": e * (2 * n + 2 * case["seq"] * case["dim"]), "flops": 3 * n}
    if op == "linear":
        m, k, n = case["m"], case["k"], case["n"]
        return {"bytes": e * (m * k + k * n + m * n + (n if case["bias"] else 0)), "flops": 2 * m * n * k}
    if op == "attention":
        b, hq, hk, sq, skv, d = (case[x] for x in ("batch", "q_heads", "kv_heads", "q_len", "kv_len", "dim"))
        nbytes = e * d * (2 * b * hq * sq + 2 * b * hk * skv)
        if case["kind"] == "causal":
            pairs = b * sq * (sq + 1) // 2
        elif case["kind"] == "cache":
            pairs = b * sq * skv
            nbytes += e * d * 4 * b * hk
        else:
            pairs = sum(length * (length + 1) // 2 + (sq - length) * length for length in _lengths(case))
            nbytes += b * sq * skv * (1 if case["kind"] == "bool" else e)
        return {"bytes": nbytes, "flops": 4 * d * hq * pairs}
    n, c, hw, out, ks = (case[x] for x in ("batch", "c", "hw", "out", "kernel"))
    p = (hw + 2 * (ks // 2) - ks) // case["stride"] + 1
    return {"bytes": e * (n * c * hw * hw + out * c * ks * ks + out + n * out * p * p), "flops": 2 * n * out * c * ks * ks * p * p}


def tolerance(case):
    # About four times the error against 64 bits as measured: one rounding to the output's type is 1.7e-3 (bf16) and
    # 2.1e-4 (f16) of the result's 2-norm; rope rounds its products too (2.4e-3), and attention the probabilities
    # before the second product (2.3e-3 and 2.5e-4).  32-bit sums are 1e-6 off and less, in any order.
    if case["dtype"] == "f32":
        return {"rel": 1e-5}
    if case["op"] == "attention":
        return {"rel": 1.2e-2} if case["dtype"] == "bf16" else {"rel": 1.5e-3}
    if case["op"] == "rope":
        return {"rel": 1e-2} if case["dtype"] == "bf16" else {"rel": 1.2e-3}
    return {"rel": 6.6e-3} if case["dtype"] == "bf16" else {"rel": 8.5e-4}


def exact(case, seed):
    st = prepare(case, seed)
    op = case["op"]
    d = {name: t.double() for name, t in st.items() if torch.is_tensor(t) and t.is_floating_point()}
    if op == "add_rms_norm":
        res = (st["x"] + st["res"]).double()  # the new residual is a rounded sum; the norm reads it
        return res * torch.rsqrt(res.square().mean(-1, keepdim=True) + 1e-6) * d["w"], d["x"] + d["res"]
    if op == "layer_norm":
        x = d["x"] - d["x"].mean(-1, keepdim=True)
        return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + 1e-5) * d["w"] + d["b"]
    if op == "silu":
        return d["x"] * torch.sigmoid(d["x"])
    if op == "softmax":
        return torch.softmax(d["x"], -1)
    if op == "rope":
        def rotate(x):
            a, b = x.chunk(2, -1)
            return x * d["cos"][None, :, None] + torch.cat([-b, a], -1) * d["sin"][None, :, None]
        return rotate(d["q"]), rotate(d["k"])
    if op == "linear":
        out = d["x"] @ d["w"]
        return out + d["bias"] if case["bias"] else out
    if op == "attention":
        group = case["q_heads"] // case["kv_heads"]
        if case["kind"] == "cache":
            d["k"][:, :, -1:], d["v"][:, :, -1:] = d["k_new"], d["v_new"]
        out = torch.empty_like(d["q"])
        for i in range(case["batch"]):
            for h in range(case["kv_heads"]):
                heads = slice(h * group, (h + 1) * group)
                s = torch.matmul(d["q"][i, heads], d["k"][i, h].t().contiguous()) / math.sqrt(case["dim"])
                if case["kind"] == "causal":
                    s = s.masked_fill_(torch.ones(s.shape[-2:], dtype=torch.bool, device="cuda").triu(1), float("-inf"))
                elif "mask" in st:
                    s = s.masked_fill_(~_mask(case, "cuda")[i], float("-inf"))
                out[i, heads] = torch.matmul(torch.softmax(s, -1), d["v"][i, h])
        return (out, d["k_new"], d["v_new"]) if case["kind"] == "cache" else out
    ks = case["kernel"]
    w = d["w"].flatten(1)
    out = []
    for x in d["x"]:
        cols = F.unfold(x[None], ks, padding=ks // 2, stride=case["stride"])[0]
        out.append(w @ cols + d["bias"][:, None])
    out = torch.stack(out)
    p = math.isqrt(out.shape[-1])
    return out.view(*out.shape[:2], p, p)
