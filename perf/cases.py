"""The work that a user of this framework has it do, as cases that can be timed.

Every case goes through the torch-facing entry points of ``inferno_amd`` (attention forward and
backward, decode against a KV cache, the standalone softmax, and the layers of the GPT training
step around the attention), on inputs that are in device memory before the call.

``listed()`` holds the named cases, ``draw(rng)`` gives further ones of the same ranges.
``prepare(case, seed)`` makes the inputs, ``run(state)`` is one pass, ``exact(case, seed)`` the same
outputs in 64 bits from plain torch, ``work(case)`` the bytes and operations that a pass cannot do
without (causal scores counted by half), ``tolerance(case)`` the largest relative error (2-norm) that
another correct implementation at the same precision would show.
"""
from __future__ import annotations

import math

import numpy as np
import torch

import inferno_amd as ia

# AdamW's hyper-parameters, as the optimizer holds them (32 bits).
LR, BETA1, BETA2, EPS, DECAY = (float(np.float32(x)) for x in (3e-4, 0.9, 0.95, 1e-8, 0.1))


def listed():
    return [
        # One layer's attention in a training step, the headline shape: GPT-2-small heads, 8 sequences.
        dict(name="attn_step_f32", kind="attn", B=8, H=12, T=1024, D=64, dtype="f32", sigma=1.0, packed=False),
        # The same layer on bf16 activations as the attention module calls it: q, k and v are columns of
        # one [B, T, 3C] projection, and the sequences end at a ragged length.
        dict(name="attn_step_bf16", kind="attn", B=8, H=12, T=1000, D=64, dtype="bf16", sigma=1.0, packed=True),
        # Long-context training with wide heads and sharp scores (standard deviation 3), in both types.
        dict(name="attn_long_f32", kind="attn", B=1, H=16, T=8192, D=128, dtype="f32", sigma=3.0, packed=False),
        dict(name="attn_long_bf16", kind="attn", B=1, H=16, T=8192, D=128, dtype="bf16", sigma=3.0, packed=False),
        # One user's prompt of odd length on its way into the KV cache: forward only, a small grid.
        dict(name="prefill_f32", kind="prefill", B=1, H=12, T=333, Tk=333, D=64, dtype="f32", causal=True, packed=True),
        # A served batch in steady state: one new token per sequence against 2048 cached keys.
        dict(name="decode_f32", kind="decode", B=32, H=12, Tk=2048, D=64, dtype="f32"),
        # One user's next token, bf16 cache: all launch and latency.
        dict(name="decode_one_bf16", kind="decode", B=1, H=12, Tk=777, D=64, dtype="bf16"),
        # The unfused chain's Softmax over [B, H, T, T] scores, forward and backward.
        dict(name="softmax_f32", kind="softmax", rows=98304, cols=1024, dtype="f32"),
        # The feed-forward block of a training step (Linear, GELU, Linear; gradients of all of it).
        dict(name="mlp_f32", kind="mlp", rows=8192, C=768, dtype="f32"),
        # Into the first block and back: token embedding, positions, LayerNorm, and their gradients.
        dict(name="stem_f32", kind="stem", B=8, T=1024, C=768, V=8192, dtype="f32"),
        # The loss of a training step over the vocabulary, and the gradient of the logits.
        dict(name="loss_f32", kind="loss", rows=8192, V=8192, dtype="f32"),
        # The optimizer over a 12-layer model's parameters, in one call.
        dict(name="adamw_f32", kind="adamw", L=12, C=768, V=8192, dtype="f32"),
    ]


def _log(rng, lo, hi):
    """An integer between lo and hi, spread over its logarithm."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["attn"] * 4 + ["prefill"] * 2 + ["decode"] * 2 + ["softmax", "mlp", "mlp", "stem", "loss", "adamw"])
    if kind in ("attn", "prefill"):
        D = rng.choice([32, 64, 64, 128])
        H = rng.randint(1, 16)
        T = _log(rng, 17, 8192 if D == 128 else 4096)
        # up to the longest listed one's scores times head dim, and 8192 tokens a batch or so
        B = max(1, min(rng.randint(1, 16), 16384 // T, int(16 * 8192**2 * 128 / (H * T * T * D))))
        c = dict(kind=kind, B=B, H=H, T=T, D=D, dtype=rng.choice(["f32", "bf16"]), packed=rng.random() < 0.5)
        if kind == "attn":
            c["sigma"] = rng.choice([1.0, 1.0, 3.0])
        else:
            # the rest of a prompt behind keys that are cached already, or (seldom) no mask
            c["Tk"] = T + (_log(rng, 1, 1024) if rng.random() < 0.4 and not c["packed"] else 0)
            c["causal"] = rng.random() < 0.85
        return c
    if kind == "decode":
        Tk = _log(rng, 64, 8192)
        B, H, D = _log(rng, 1, 64), rng.randint(1, 16), rng.choice([32, 64, 64, 128])
        return dict(kind=kind, B=max(1, min(B, 2**23 // (H * Tk))), H=H, Tk=Tk, D=D, dtype=rng.choice(["f32", "bf16"]))
    if kind == "softmax":
        cols = _log(rng, 32, 12288)
        return dict(kind=kind, rows=_log(rng, 64, max(65, min(200000, 98304 * 1024 // cols))), cols=cols,
                    dtype=rng.choice(["f32", "f32", "bf16"]))
    if kind == "mlp":
        return dict(kind=kind, rows=_log(rng, 32, 8192), C=4 * rng.randint(32, 224), dtype="f32")
    if kind == "stem":
        return dict(kind=kind, B=rng.randint(1, 8), T=_log(rng, 32, 1024), C=4 * rng.randint(16, 256),
                    V=_log(rng, 64, 22197), dtype="f32")
    if kind == "loss":
        return dict(kind=kind, rows=_log(rng, 64, 8192), V=_log(rng, 64, 22197), dtype="f32")
    return dict(kind="adamw", L=rng.randint(1, 12), C=4 * rng.randint(16, 192), V=_log(rng, 64, 22197), dtype="f32")


def _dtype(case):
    return torch.bfloat16 if case["dtype"] == "bf16" else torch.float32


def _normal(gen, shape, dtype=torch.float32, std=1.0):
    x = torch.randn(shape, generator=gen, device="cuda", dtype=torch.float32)
    return (x * std if std != 1.0 else x).to(dtype)


def _heads(gen, case, T, n):
    """n [B, H, T, D] tensors; packed: views of one [B, T, n C] projection, as the module makes them."""
    B, H, D, dt, std = case["B"], case["H"], case["D"], _dtype(case), case.get("sigma", 1.0)
    if case.get("packed"):
        x = _normal(gen, (B, T, n * H * D), dt, std)
        return [x[:, :, i * H * D:(i + 1) * H * D].view(B, T, H, D).transpose(1, 2) for i in range(n)]
    return [_normal(gen, (B, H, T, D), dt, std) for _ in range(n)]


def _adamw_shapes(case):
    L, C, V = case["L"], case["C"], case["V"]
    block = [(C, 3 * C), (3 * C,), (C, C), (C,), (C, 4 * C), (4 * C,), (4 * C, C), (C,), (C,), (C,), (C,), (C,)]
    return [(V, C)] + block * L + [(C,), (C,)]


def prepare(case, seed):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(int(seed) * 7919 + 11)
    kind, dt, s = case["kind"], _dtype(case), {"case": case}
    if kind == "attn":
        s["q"], s["k"], s["v"] = _heads(gen, case, case["T"], 3)
        # the gradient that comes back through the output projection: [B, T, C], its heads as views
        do = _normal(gen, (case["B"], case["T"], case["H"], case["D"]), dt, 0.05)
        s["do"] = do.transpose(1, 2) if case["packed"] else do.transpose(1, 2).contiguous()
    elif kind == "prefill":
        if case["packed"]:
            s["q"], s["k"], s["v"] = _heads(gen, case, case["T"], 3)
        else:
            s["q"] = _heads(gen, case, case["T"], 1)[0]
            s["k"], s["v"] = _heads(gen, case, case["Tk"], 2)
    elif kind == "decode":
        s["q"] = _normal(gen, (case["B"], case["H"], 1, case["D"]), dt)
        s["k"] = _normal(gen, (case["B"], case["H"], case["Tk"], case["D"]), dt)
        s["v"] = _normal(gen, (case["B"], case["H"], case["Tk"], case["D"]), dt)
    elif kind == "softmax":
        s["x"] = _normal(gen, (case["rows"], case["cols"]), dt, 2.0)
        s["dy"] = _normal(gen, (case["rows"], case["cols"]), dt, 0.05)
    elif kind == "mlp":
        C = case["C"]
        s["x"] = _normal(gen, (case["rows"], C))
        s["w1"], s["b1"] = _normal(gen, (C, 4 * C), std=C**-0.5), _normal(gen, (4 * C,), std=0.1)
        s["w2"], s["b2"] = _normal(gen, (4 * C, C), std=(4 * C)**-0.5), _normal(gen, (C,), std=0.1)
        s["dy"] = _normal(gen, (case["rows"], C), std=0.05)
    elif kind == "stem":
        n, C, V = case["B"] * case["T"], case["C"], case["V"]
        s["ids"] = torch.randint(0, V, (n,), generator=gen, device="cuda", dtype=torch.int32)
        s["table"], s["pos"] = _normal(gen, (V, C), std=0.5), _normal(gen, (case["T"], C), std=0.5)
        s["gamma"], s["beta"] = 1.0 + _normal(gen, (C,), std=0.1), _normal(gen, (C,), std=0.1)
        s["dy"] = _normal(gen, (n, C), std=0.05)
    elif kind == "loss":
        s["logits"] = _normal(gen, (case["rows"], case["V"]), std=2.0)
        s["targets"] = torch.randint(0, case["V"], (case["rows"],), generator=gen, device="cuda", dtype=torch.int32)
        s["one"] = torch.ones(1, device="cuda")
    else:
        # the parameters, gradients and moments of a model lie in four flat buffers, one slice per tensor
        shapes = _adamw_shapes(case)
        sizes = [math.prod(sh) for sh in shapes]
        s["flat"] = [_normal(gen, (sum(sizes),), std=std) for std in (0.05, 0.01, 0.01, 0.01)]
        s["flat"][3].square_()
        s["params"] = [tuple(t.view(sh) for t in ts) for sh, ts in zip(shapes, zip(*(f.split(sizes) for f in s["flat"])))]
    return s


def run(state):
    s, kind = state, state["case"]["kind"]
    if kind == "attn":
        o, lse = ia.attn_fwd(s["q"], s["k"], s["v"])
        dq, dk, dv = ia.attn_bwd(s["q"], s["k"], s["v"], o, s["do"], lse)
        return {"o": o, "lse": lse, "dq": dq, "dk": dk, "dv": dv}
    if kind == "prefill":
        o, lse = ia.attn_fwd(s["q"], s["k"], s["v"], causal=s["case"]["causal"])
        return {"o": o, "lse": lse}
    if kind == "decode":
        return ia.attn_decode(s["q"], s["k"], s["v"])
    if kind == "softmax":
        y = ia.softmax_fwd(s["x"])
        return {"y": y, "dx": ia.softmax_bwd(y, s["dy"])}
    if kind == "mlp":
        h = ia.gemm(s["x"], s["w1"], bias=s["b1"])
        a = ia.gelu_fwd(h)
        y = ia.gemm(a, s["w2"], bias=s["b2"])
        dw2 = ia.gemm(a, s["dy"], trans_a=True)
        db2 = ia.col_sum(s["dy"])
        dh = ia.gelu_bwd(h, ia.gemm(s["dy"], s["w2"], trans_b=True))
        dw1 = ia.gemm(s["x"], dh, trans_a=True)
        db1 = ia.col_sum(dh)
        return {"y": y, "dx": ia.gemm(dh, s["w1"], trans_b=True), "dw1": dw1, "db1": db1, "dw2": dw2, "db2": db2}
    if kind == "stem":
        x = ia.binary_bcast(0, ia.embedding_fwd(s["ids"], s["table"]), s["pos"])
        y, mean, invstd = ia.layernorm_fwd(x, s["gamma"], s["beta"])
        dx, dgamma, dbeta = ia.layernorm_bwd(x, s["dy"], s["gamma"], mean, invstd)
        return {"y": y, "dgamma": dgamma, "dbeta": dbeta, "dx": dx,
                "dtable": ia.embedding_bwd(s["ids"], dx, s["table"].shape[0])}
    if kind == "loss":
        loss, lse = ia.cross_entropy_fwd(s["logits"], s["targets"])
        return {"loss": loss, "dlogits": ia.cross_entropy_bwd(s["logits"], s["targets"], lse, s["one"])}
    ia.adamw_step_multi(s["params"], 10, lr=LR, beta1=BETA1, beta2=BETA2, eps=EPS, weight_decay=DECAY)
    return {"p": s["flat"][0], "m": s["flat"][2], "v": s["flat"][3]}


def _scores(case):
    """Visible (query, key) pairs of one head, causal ones counted as half the square."""
    T, Tk = case["T"], case.get("Tk", case["T"])
    return T * Tk - T * T / 2 if case.get("causal", True) else T * Tk


def work(case):
    kind, e = case["kind"], 2 if case["dtype"] == "bf16" else 4
    if kind in ("attn", "prefill"):
        BH, T, Tk, D = case["B"] * case["H"], case["T"], case.get("Tk", case["T"]), case["D"]
        fwd = 4 * BH * _scores(case) * D
        if kind == "prefill":
            return {"bytes": BH * ((2 * T + 2 * Tk) * D * e + 4 * T), "flops": fwd}
        # forward and backward are two calls: the backward reads q, k, v, o, dO and lse again
        return {"bytes": BH * (12 * T * D * e + 8 * T), "flops": 3.5 * fwd}
    if kind == "decode":
        BH, Tk, D = case["B"] * case["H"], case["Tk"], case["D"]
        return {"bytes": BH * (2 * Tk + 2) * D * e, "flops": 4 * BH * Tk * D}
    if kind == "softmax":
        n = case["rows"] * case["cols"]
        return {"bytes": 5 * n * e, "flops": 8 * n}
    if kind == "mlp":
        r, C = case["rows"], case["C"]
        # six products of 2 r C 4C operations each; every call's operands and results once
        act, w = r * C * e, 4 * C * C * e
        return {"bytes": 6 * (5 * act + w) + 5 * 4 * act + 5 * act, "flops": 48 * r * C * C}
    if kind == "stem":
        n, C, V = case["B"] * case["T"], case["C"], case["V"]
        return {"bytes": e * C * (10 * n + case["T"] + V), "flops": 30 * n * C}
    if kind == "loss":
        n = case["rows"] * case["V"]
        return {"bytes": 3 * n * e, "flops": 8 * n}
    n = sum(math.prod(sh) for sh in _adamw_shapes(case))
    return {"bytes": 7 * n * e, "flops": 15 * n}


def tolerance(case):
    # About four times the distance to exact() that was measured.  bf16: results are rounded to 8 bits, and P
    # and dS inside the products too (0.2-0.5%).  32 bits: the order of the sums; with sharp scores
    # (standard deviation 3) the rounding of a score moves its probability by up to 4e-6.
    if case["dtype"] == "bf16":
        return {"rel": 2e-2 if case.get("sigma", 1.0) > 1.0 else 1e-2}
    if case["kind"] == "attn":
        return {"rel": 1.6e-5 if case["sigma"] > 1.0 else 4e-6}
    return {"rel": {"mlp": 7e-6, "adamw": 1e-6, "prefill": 2e-6}.get(case["kind"], 1e-6)}


def exact(case, seed):
    return _EXACT[case["kind"]](case, prepare(case, seed))


def _scale(D):
    """1 / sqrt(D) as the library takes it by default (32 bits)."""
    return float(np.float32(1.0) / np.sqrt(np.float32(D)))


def _exact_attn(case, s):
    # head by head, as plain 2-D products
    B, H, T, D = s["q"].shape
    Tk, c = s["k"].shape[2], _scale(D)
    out = {"o": torch.empty((B, H, T, D), dtype=torch.float64, device="cuda"),
           "lse": torch.empty((B, H, T), dtype=torch.float64, device="cuda")}
    if "do" in s:
        out.update({n: torch.empty((B, H, t, D), dtype=torch.float64, device="cuda")
                    for n, t in (("dq", T), ("dk", Tk), ("dv", Tk))})
    hidden = torch.ones((T, Tk), dtype=torch.bool, device="cuda").triu_(1 + Tk - T) if case.get("causal", True) else None
    for b in range(B):
        for h in range(H):
            q, k, v = (s[n][b, h].double().contiguous() for n in ("q", "k", "v"))
            x = (q @ k.t().contiguous()).mul_(c)
            if hidden is not None:
                x.masked_fill_(hidden, -math.inf)
            lse = torch.logsumexp(x, dim=1)
            p = x.sub_(lse[:, None]).exp_()
            o = p @ v
            out["o"][b, h], out["lse"][b, h] = o, lse
            if "do" in s:
                do = s["do"][b, h].double().contiguous()
                out["dv"][b, h] = p.t().contiguous() @ do
                ds = (do @ v.t().contiguous()).sub_((do * o).sum(1, keepdim=True)).mul_(p).mul_(c)
                out["dq"][b, h] = ds @ k
                out["dk"][b, h] = ds.t().contiguous() @ q
    return out


def _exact_decode(case, s):
    q, k, v = (s[n].double() for n in ("q", "k", "v"))
    p = torch.softmax((q * k).sum(-1) * _scale(q.shape[3]), dim=-1)
    return (p[..., None] * v).sum(2, keepdim=True)


def _exact_softmax(case, s):
    x, dy = s["x"].double(), s["dy"].double()
    y = torch.softmax(x, dim=1)
    # the backward starts from the y that the forward handed on, in its own type
    yr = y.to(s["x"].dtype).double() if s["x"].dtype == torch.bfloat16 else y
    return {"y": y, "dx": yr * (dy - (dy * yr).sum(1, keepdim=True))}


_GELU_A, _GELU_B = 0.7978845608028654, 0.044715


def _exact_mlp(case, s):
    x, w1, b1, w2, b2, dy = (s[n].double() for n in ("x", "w1", "b1", "w2", "b2", "dy"))
    h = x @ w1 + b1
    t = torch.tanh(_GELU_A * (h + _GELU_B * h**3))
    a = 0.5 * h * (1 + t)
    da = dy @ w2.t().contiguous()
    dh = da * (0.5 * (1 + t) + 0.5 * h * (1 - t * t) * _GELU_A * (1 + 3 * _GELU_B * h * h))
    return {"y": a @ w2 + b2, "dx": dh @ w1.t().contiguous(), "dw1": x.t().contiguous() @ dh, "db1": dh.sum(0),
            "dw2": a.t().contiguous() @ dy, "db2": dy.sum(0)}


def _exact_stem(case, s):
    ids, n, C = s["ids"].long(), s["ids"].numel(), case["C"]
    gamma, beta, dy = (s[k].double() for k in ("gamma", "beta", "dy"))
    x = s["table"].double()[ids] + s["pos"].double().repeat(case["B"], 1)
    mean = x.mean(1, keepdim=True)
    invstd = (((x - mean)**2).mean(1, keepdim=True) + 1e-5).rsqrt()
    xh, dxh = (x - mean) * invstd, dy * gamma
    dx = invstd * (dxh - dxh.mean(1, keepdim=True) - xh * (dxh * xh).mean(1, keepdim=True))
    dtable = torch.zeros((case["V"], C), dtype=torch.float64, device="cuda").index_add_(0, ids, dx)
    return {"y": xh * gamma + beta, "dgamma": (dy * xh).sum(0), "dbeta": dy.sum(0), "dx": dx, "dtable": dtable}


def _exact_loss(case, s):
    x, t = s["logits"].double(), s["targets"].long()
    lse = torch.logsumexp(x, dim=1)
    loss = (lse - x.gather(1, t[:, None])[:, 0]).mean().reshape(1)
    g = x.sub_(lse[:, None]).exp_()
    g.scatter_add_(1, t[:, None], torch.full((g.shape[0], 1), -1.0, dtype=torch.float64, device="cuda"))
    return {"loss": loss, "dlogits": g.div_(g.shape[0])}


def _exact_adamw(case, s):
    bc1, bc2 = (float(np.float32(1.0) - np.power(np.float32(b), np.float32(10))) for b in (BETA1, BETA2))
    p, g, m, v = (t.double() for t in s["flat"])
    m = BETA1 * m + (1.0 - BETA1) * g
    v = BETA2 * v + (1.0 - BETA2) * g * g
    return {"p": p - LR * ((m / bc1) / ((v / bc2).sqrt() + EPS) + DECAY * p), "m": m, "v": v}


_EXACT = {"attn": _exact_attn, "prefill": _exact_attn, "decode": _exact_decode, "softmax": _exact_softmax,
          "mlp": _exact_mlp, "stem": _exact_stem, "loss": _exact_loss,
          "adamw": _exact_adamw}
