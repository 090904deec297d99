"""Measured cases: what a program asks of this package through its public calls.

Each case is one call a user makes again and again: an attention forward (inference) or a forward with its
backward (training), with the sizes, types and options the package is used with, and one encoder stack as a
whole.  ``run`` returns every output whole; ``exact`` gives the same outputs in 64 bits from plain torch.
"""
import math

import torch
import torch.nn.functional as F

import elsa_amd

DTYPES = {"fp16": torch.float16, "bf16": torch.bfloat16, "fp32": torch.float32}
DEV = "cuda"


def _attn(name, mode, dtype, b, h, n, d, causal=False, bias="none"):
    return {"name": name, "kind": "attention", "mode": mode, "dtype": dtype, "b": b, "h": h, "n": n, "d": d,
            "causal": causal, "bias": bias}


def listed():
    return [
        # one image through a small vision transformer's attention layer (196 patches and a class token):
        # the smallest call, where launches and the host side count
        _attn("fwd_short_fp16", "fwd", "fp16", 1, 3, 197, 64),
        # a training step's attention layer at 224 px, batch 8
        _attn("train_short_fp16", "train", "fp16", 8, 3, 197, 64),
        # the whole inference call of a 12-layer encoder on the same tokens
        {"name": "encoder_fp16", "kind": "encoder", "dtype": "fp16", "b": 8, "n": 197, "dim": 192, "heads": 3,
         "depth": 12},
        # a training step's attention layer at 512 px (1024 patches and a class token), bf16
        _attn("train_mid_bf16", "train", "bf16", 8, 3, 1025, 64),
        # the long-sequence training step the package is quoted on
        _attn("train_long_fp16", "train", "fp16", 1, 8, 16384, 64),
        # decoder training, one token past a power of two
        _attn("train_causal_bf16", "train", "bf16", 2, 8, 4097, 64, causal=True),
        # prefill of a long prompt at head dim 128
        _attn("fwd_causal_d128_bf16", "fwd", "bf16", 1, 16, 8192, 128, causal=True),
        # training at head dim 128
        _attn("train_d128_fp16", "train", "fp16", 2, 8, 2048, 128),
        # full-precision inference over a long sequence
        _attn("fwd_fp32", "fwd", "fp32", 1, 8, 8192, 64),
        # full-precision training
        _attn("train_fp32", "train", "fp32", 1, 8, 4096, 64),
        # 7 x 7 shifted windows (inference): relative-position bias plus mask for every window
        _attn("windows_fwd_fp16", "fwd", "fp16", 512, 3, 49, 32, bias="full"),
        # 7 x 7 windows (training): the relative-position bias of each head, with its gradient
        _attn("windows_train_fp16", "train", "fp16", 512, 3, 49, 32, bias="heads"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    mode = rng.choice(["fwd", "train"])
    dtype = rng.choice(["fp16", "bf16", "fp32"])
    if rng.random() < 0.25:  # windows and other short biased calls
        side = rng.randint(6, 16)
        n, h = side * side, rng.choice([3, 4, 6, 8, 12])
        b = _log_int(rng, 1, max(1, 60_000_000 // (h * n * n)))
        return {k: v for k, v in _attn("", mode, dtype, min(b, 1024), h, n, 32,
                                       bias=rng.choice(["heads", "full"])).items() if k != "name"}
    d = rng.choice([32, 64, 64, 64, 80, 128])
    n = _log_int(rng, 49, 16384)
    # heads so that the work stays below the long training step's (fp32: a 16th of it, as its units are slower)
    cap = 1.9e12 / (16 if dtype == "fp32" else 1) / (3.5 if mode == "train" else 1)
    bh = max(1, min(256, int(cap / (4.0 * n * n * d))))
    bh = _log_int(rng, 1, bh)
    h = rng.choice([x for x in (1, 2, 3, 4, 6, 8, 12, 16) if x <= bh])
    return {k: v for k, v in _attn("", mode, dtype, max(1, bh // h), h, n, d, causal=rng.random() < 0.4).items()
            if k != "name"}


# ------------------------------------------------------------------ inputs
def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _attention_inputs(case, seed):
    g, dt = _gen(seed), DTYPES[case["dtype"]]
    shape = (case["b"], case["h"], case["n"], case["d"])
    q, k, v, do = (torch.randn(shape, generator=g, device=DEV, dtype=torch.float32).to(dt) for _ in range(4))
    bias = None
    if case["bias"] != "none":
        n = case["n"]
        bias = 0.5 * torch.randn((1, case["h"], n, n), generator=g, device=DEV, dtype=torch.float32)
        if case["bias"] == "full":  # a third of the windows masks a band of its keys, as shifted windows do
            win = torch.arange(case["b"], device=DEV).view(-1, 1, 1, 1)
            tok = torch.arange(n, device=DEV)
            other = (tok.view(-1, 1) < n // 2) != (tok.view(1, -1) < n // 2)
            bias = bias + torch.where((win % 3 == 0) & other, -100.0, 0.0)
        bias = bias.to(dt)
    return q, k, v, do, bias


def _encoder_weights(case, seed):
    g, c = _gen(seed + 1), case["dim"]
    dt = DTYPES[case["dtype"]]

    def normal(*shape, std):
        return (std * torch.randn(shape, generator=g, device=DEV, dtype=torch.float32)).to(dt)

    w = {}
    for i in range(case["depth"]):
        for name, out, inp in (("qkv", 3 * c, c), ("proj", c, c), ("fc1", 4 * c, c), ("fc2", c, 4 * c)):
            w[f"layers.{i}.{name}.weight"] = normal(out, inp, std=inp ** -0.5)
            w[f"layers.{i}.{name}.bias"] = normal(out, std=0.02)
        for name in ("norm1", "norm2"):
            w[f"layers.{i}.{name}.weight"] = 1 + normal(c, std=0.1)
            w[f"layers.{i}.{name}.bias"] = normal(c, std=0.02)
    w["norm.weight"] = 1 + normal(c, std=0.1)
    w["norm.bias"] = normal(c, std=0.02)
    return w


def _encoder_tokens(case, seed):
    return torch.randn((case["b"], case["n"], case["dim"]), generator=_gen(seed), device=DEV,
                       dtype=torch.float32).to(DTYPES[case["dtype"]])


def prepare(case, seed):
    if case["kind"] == "encoder":
        model = elsa_amd.TransformerEncoder(dim=case["dim"], depth=case["depth"], heads=case["heads"], backend="elsa")
        model = model.to(device=DEV, dtype=DTYPES[case["dtype"]])
        model.load_state_dict(_encoder_weights(case, seed))
        return {"case": case, "model": model.eval(), "x": _encoder_tokens(case, seed)}
    q, k, v, do, bias = _attention_inputs(case, seed)
    if case["mode"] == "train":
        for t in (q, k, v) + ((bias,) if bias is not None else ()):
            t.requires_grad_(True)
    return {"case": case, "q": q, "k": k, "v": v, "do": do, "bias": bias}


def run(state):
    case = state["case"]
    if case["kind"] == "encoder":
        with torch.no_grad():
            return state["model"](state["x"])
    q, k, v, bias = state["q"], state["k"], state["v"], state["bias"]
    if case["mode"] == "fwd":
        return elsa_amd.twopass_attention(q, k, v, bias=bias, is_causal=case["causal"])
    out = elsa_amd.twopass_attention_train(q, k, v, bias=bias, is_causal=case["causal"])
    wrt = (q, k, v) if bias is None else (q, k, v, bias)
    return (out.detach(), *torch.autograd.grad(out, wrt, state["do"]))


# ------------------------------------------------------------------ work
def work(case):
    size = 4 if case["dtype"] == "fp32" else 2
    if case["kind"] == "encoder":
        tokens, c = case["b"] * case["n"], case["dim"]
        linear = 2.0 * tokens * 12 * c * c
        attention = 4.0 * case["b"] * case["n"] ** 2 * c
        weights = case["depth"] * (12 * c * c + 13 * c) + 2 * c
        return {"bytes": size * (weights + 2 * tokens * c), "flops": case["depth"] * (linear + attention)}
    b, h, n, d = case["b"], case["h"], case["n"], case["d"]
    pairs = n * (n + 1) / 2 if case["causal"] else float(n) * n
    forward = 4.0 * b * h * pairs * d
    tensor = size * b * h * n * d
    bias = {"none": 0, "heads": size * h * n * n, "full": size * b * h * n * n}[case["bias"]]
    if case["mode"] == "fwd":
        return {"bytes": 4 * tensor + bias, "flops": forward}
    # q, k, v, dO in; out, dq, dk, dv and the bias gradient out; five products in the backward
    return {"bytes": 8 * tensor + 2 * bias, "flops": 3.5 * forward}


# About four times the largest relative error against 64 bits that these calls showed: 4.2e-4 (fp16), 2.9e-3
# (bf16), 2.0e-6 (fp32, 11726 keys), 1.0e-3 (the encoder's twelve fp16 layers).
def tolerance(case):
    if case["kind"] == "encoder":
        return {"rel": 4e-3}
    return {"rel": {"fp16": 1.6e-3, "bf16": 1.2e-2, "fp32": 8e-6}[case["dtype"]]}


# ------------------------------------------------------------------ 64-bit results
def _exact_head(q, k, v, do, bias, causal, train):
    """One (batch, head) in chunks of rows: out and, in training, dq, dk, dv and the bias gradient."""
    n, d = q.shape
    scale = 1.0 / math.sqrt(d)
    out, dq = torch.empty_like(q), torch.empty_like(q)
    dk, dv = torch.zeros_like(k), torch.zeros_like(v)
    db = torch.zeros((n, n), dtype=torch.float64, device=q.device) if train and bias is not None else None
    key = torch.arange(n, device=q.device)
    for r0 in range(0, n, 4096):
        r = slice(r0, min(n, r0 + 4096))
        s = (q[r] @ k.t()) * scale
        if bias is not None:
            s = s + bias[r]
        if causal:
            s.masked_fill_(key.view(1, -1) > key[r].view(-1, 1), float("-inf"))
        p = torch.softmax(s, dim=-1)
        out[r] = p @ v
        if train:
            dp = do[r] @ v.t()
            ds = p * (dp - (do[r] * out[r]).sum(-1, keepdim=True))
            dq[r] = (ds @ k) * scale
            dk += (ds.t() @ q[r]) * scale
            dv += p.t() @ do[r]
            if db is not None:
                db[r] = ds
    return out, dq, dk, dv, db


def _exact_batched(q, k, v, do, bias, causal, train):
    """All heads at once, for short sequences."""
    scale = 1.0 / math.sqrt(q.shape[-1])
    s = torch.matmul(q, k.transpose(-1, -2).contiguous()) * scale
    if bias is not None:
        s = s + bias
    if causal:
        n = q.shape[-2]
        s.masked_fill_(torch.ones((n, n), dtype=torch.bool, device=q.device).triu(1), float("-inf"))
    p = torch.softmax(s, dim=-1)
    out = torch.matmul(p, v)
    if not train:
        return out
    dp = torch.matmul(do, v.transpose(-1, -2).contiguous())
    ds = p * (dp - (do * out).sum(-1, keepdim=True))
    dq = torch.matmul(ds, k) * scale
    dk = torch.matmul(ds.transpose(-1, -2).contiguous(), q) * scale
    dv = torch.matmul(p.transpose(-1, -2).contiguous(), do)
    if bias is None:
        return out, dq, dk, dv
    return out, dq, dk, dv, (ds.sum(0, keepdim=True) if bias.shape[0] != ds.shape[0] else ds)


def _exact_encoder(case, seed):
    w = {k: t.double() for k, t in _encoder_weights(case, seed).items()}
    x = _encoder_tokens(case, seed).double()
    b, n, c = x.shape
    h = case["heads"]

    def norm(y, name):
        return F.layer_norm(y, (c,), w[name + ".weight"], w[name + ".bias"], 1e-5)

    def linear(y, name):
        return y @ w[name + ".weight"].t() + w[name + ".bias"]

    for i in range(case["depth"]):
        p = f"layers.{i}."
        qkv = linear(norm(x, p + "norm1"), p + "qkv").view(b, n, 3, h, c // h).permute(2, 0, 3, 1, 4)
        y = _exact_batched(qkv[0].contiguous(), qkv[1], qkv[2].contiguous(), None, None, False, False)
        x = x + linear(y.transpose(1, 2).reshape(b, n, c), p + "proj")
        y = linear(norm(x, p + "norm2"), p + "fc1")
        x = x + linear(0.5 * y * (1 + torch.erf(y / math.sqrt(2.0))), p + "fc2")
    return norm(x, "norm")


def exact(case, seed):
    if case["kind"] == "encoder":
        return _exact_encoder(case, seed)
    q, k, v, do, bias = _attention_inputs(case, seed)
    train, causal = case["mode"] == "train", case["causal"]
    q, k, v, do = (t.double() for t in (q, k, v, do))
    bias = None if bias is None else bias.double()
    b, h, n, _ = q.shape
    if n <= 512:
        return _exact_batched(q, k, v, do, bias, causal, train)
    outs = [torch.empty_like(q) for _ in range(4 if train else 1)]
    for i in range(b):
        for j in range(h):
            got = _exact_head(q[i, j], k[i, j], v[i, j], do[i, j], None, causal, train)
            for dst, src in zip(outs, got):
                dst[i, j] = src
    return tuple(outs) if train else outs[0]
