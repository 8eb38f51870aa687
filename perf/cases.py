"""The work a user of this package has it do, as timed cases.

Each case is one pass through the package's public entry points: attention in
the forward alone (inference) and as a training step, the norms, the softmax
along the ragged axis and the packed <-> padded conversions.  ``listed()``
gives the fixed cases, ``draw(rng)`` one more of the ranges they stand for.

A case is a dict of plain values; ``prepare(case, seed)`` makes the inputs on
the GPU, ``run(state)`` makes one pass and returns its outputs whole,
``exact(case, seed)`` gives the same outputs in 64 bits from plain torch,
``work(case)`` the bytes and operations a pass cannot do without and
``tolerance(case)`` the error another correct implementation of the same
precision shows.
"""

from __future__ import annotations

import math

import numpy as np
import torch

import scree_amd
from scree_amd import kernels
from scree_amd.kernels import hip

DTYPES = {"fp32": torch.float32, "fp16": torch.float16, "bf16": torch.bfloat16}
DEVICE = "cuda"


# ------------------------------------------------------------------- cases
def _attn(name, *, dtype, heads, kv_heads, head_dim, seqs, mean_len, sigma, len_seed, causal, train,
          total=0):
    return {"name": name, "kind": "attn", "dtype": dtype, "heads": heads, "kv_heads": kv_heads,
            "head_dim": head_dim, "seqs": seqs, "mean_len": mean_len, "sigma": sigma,
            "len_seed": len_seed, "total": total, "causal": causal, "train": train}


def _norm(name, *, norm, dtype, rows, heads, dim, train):
    # heads > 1: rows x heads x dim, normalised over the last axis (per-head norm)
    return {"name": name, "kind": "norm", "norm": norm, "dtype": dtype, "rows": rows, "heads": heads,
            "dim": dim, "train": train}


def _ragged(name, kind, *, dtype, features, seqs, mean_len, sigma, len_seed, train=False, total=0):
    return {"name": name, "kind": kind, "dtype": dtype, "features": features, "seqs": seqs,
            "mean_len": mean_len, "sigma": sigma, "len_seed": len_seed, "total": total,
            "train": train}


def listed():
    return [
        # A short request batch: 16 short sequences of a small model, forward
        # only.  A few microseconds of GPU work, so the call itself counts.
        _attn("attn_fwd_small_fp16", dtype="fp16", heads=4, kv_heads=4, head_dim=32, seqs=16,
              mean_len=128, sigma=0.6, len_seed=0, causal=True, train=False),
        # Prefill of a mixed batch of prompts on a decoder with grouped-query
        # attention (32 query heads on 8 K/V heads of 128).
        _attn("attn_prefill_gqa_bf16", dtype="bf16", heads=32, kv_heads=8, head_dim=128, seqs=8,
              mean_len=1024, sigma=0.6, len_seed=0, causal=True, train=False),
        # The benchmark's training step: 16 sequences, 12,160 tokens, 16 heads
        # of 64, forward and backward.
        _attn("attn_train_fp16_16x64", dtype="fp16", heads=16, kv_heads=16, head_dim=64, seqs=16,
              mean_len=760, sigma=0.6, len_seed=0, causal=True, train=True, total=12160),
        # Long-context pretraining of a large decoder: 32 sequences up to
        # 16k tokens, 32 heads of 128 (the largest case).
        _attn("attn_train_bf16_32x128", dtype="bf16", heads=32, kv_heads=32, head_dim=128, seqs=32,
              mean_len=2048, sigma=1.2, len_seed=0, causal=True, train=True),
        # An encoder's training step: no mask, many short sequences, 12 heads
        # of 64.
        _attn("attn_train_encoder_bf16", dtype="bf16", heads=12, kv_heads=12, head_dim=64, seqs=48,
              mean_len=256, sigma=0.6, len_seed=1, causal=False, train=True),
        # Training in fp32 (the dtype an Array of fp32 values is computed in):
        # 16 sequences of mean 256, 8 heads of 64.
        _attn("attn_train_fp32_8x64", dtype="fp32", heads=8, kv_heads=8, head_dim=64, seqs=16,
              mean_len=256, sigma=0.6, len_seed=0, causal=True, train=True),
        # The hidden-state RMSNorm of a decoder block in training: 19,758
        # packed tokens of 4,096.
        _norm("rmsnorm_train_bf16_4096", norm="rms", dtype="bf16", rows=19758, heads=1, dim=4096,
              train=True),
        # LayerNorm of a base-size encoder in training (hidden 768 = 12 x 64).
        _norm("layernorm_train_fp16_768", norm="layer", dtype="fp16", rows=12160, heads=1, dim=768,
              train=True),
        # Per-head RMSNorm of the queries (tokens, heads, head_dim) in
        # training, as decoders that normalise q and k apply it.
        _norm("headnorm_train_bf16_16x128", norm="rms", dtype="bf16", rows=12160, heads=16, dim=128,
              train=True),
        # The residual add + RMSNorm of one decode step: 64 tokens of 4,096,
        # forward only.  Latency.
        _norm("add_rmsnorm_decode_bf16", norm="add_rms", dtype="bf16", rows=64, heads=1, dim=4096,
              train=False),
        # Softmax along the ragged axis in training, at the size the
        # benchmark times it: 64 sequences, 19,758 rows of 4,096 columns.
        _ragged("softmax_train_bf16_4096", "softmax", dtype="bf16", features=4096, seqs=64,
                mean_len=256, sigma=0.6, len_seed=0, train=True),
        # Hidden states to a padded batch and back (a padded model inside a
        # packed pipeline): 16 sequences, 12,160 tokens of 1,024.
        _ragged("pad_unpad_bf16_1024", "pad", dtype="bf16", features=1024, seqs=16, mean_len=760,
                sigma=0.6, len_seed=0, total=12160),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["attn", "attn", "attn", "attn32", "norm", "norm", "norm", "softmax", "pad"])
    sigma = round(rng.uniform(0.2, 1.2), 2)
    len_seed = rng.randrange(1 << 20)
    if kind in ("attn", "attn32"):
        f32 = kind == "attn32"
        head_dim = rng.choice([32, 64, 64, 128, 128, 256] if not f32 else [32, 64, 64, 128])
        kv_heads = rng.choice([2, 3, 4, 6, 8, 12, 16])
        group = rng.choice([1, 1, 1, 2, 4])
        heads = kv_heads * group
        seqs = _log_int(rng, 1, 96)
        tokens = _log_int(rng, 256, 32768 if not f32 else 8192)
        # as much attention as the largest listed case (fp32: a fiftieth of it) at most
        cap = 3.0e12 if not f32 else 6.0e10
        while 4.0 * heads * head_dim * tokens * tokens / seqs * math.exp(sigma * sigma) > cap:
            tokens = tokens * 2 // 3
        return _attn(None, dtype="fp32" if f32 else rng.choice(["fp16", "bf16"]), heads=heads,
                     kv_heads=kv_heads, head_dim=head_dim, seqs=seqs,
                     mean_len=max(1, tokens // seqs), sigma=sigma, len_seed=len_seed,
                     causal=rng.random() < 0.75, train=rng.random() < 0.6)
    if kind == "norm":
        heads = rng.choice([1, 1, 1, 8, 16, 32])
        if heads > 1:
            dim, rows = rng.choice([32, 64, 96, 128, 256]), _log_int(rng, 16, 16384)
        else:
            dim, rows = _log_int(rng, 64, 8192), _log_int(rng, 16, 20000)
            if rng.random() < 0.75:  # most models' widths are multiples of 64, some are not
                dim = max(64, dim // 64 * 64)
        return _norm(None, norm=rng.choice(["rms", "layer", "add_rms"]),
                     dtype=rng.choice(["fp32", "fp16", "bf16", "bf16"]), rows=rows, heads=heads,
                     dim=dim, train=rng.random() < 0.7)
    seqs = _log_int(rng, 4, 96)
    mean_len = _log_int(rng, 32, 1024)
    features = _log_int(rng, 1 if kind == "softmax" else 16, 4096)
    if features > 16 and rng.random() < 0.75:
        features = features // 16 * 16
    while seqs * mean_len * features > 64 << 20:
        mean_len = max(1, mean_len * 2 // 3)
    return _ragged(None, kind, dtype=rng.choice(["fp32", "fp16", "bf16"]), features=features,
                   seqs=seqs, mean_len=mean_len, sigma=sigma, len_seed=len_seed,
                   train=kind == "softmax" and rng.random() < 0.6)


# ------------------------------------------------------------------ inputs
def _lengths(case):
    """Log-normal sequence lengths, as the benchmark's sampler draws them;
    rescaled to ``total`` tokens when that is set."""
    rng = np.random.default_rng(case["len_seed"])
    x = rng.lognormal(mean=np.log(case["mean_len"]), sigma=case["sigma"], size=case["seqs"])
    if case["total"]:
        x = x * (case["total"] / x.sum())
    n = [min(16384, max(1, int(v))) for v in x]
    if case["total"]:
        n[int(np.argmax(n))] += case["total"] - sum(n)
    return n


def _rows(case):
    return case["rows"] if case["kind"] == "norm" else sum(_lengths(case))


def _offsets(lengths):
    off = np.zeros(len(lengths) + 1, dtype=np.int32)
    off[1:] = np.cumsum(lengths)
    return torch.from_numpy(off).to(DEVICE)


def _randn(gen, shape, dtype, scale=1.0, mean=0.0):
    x = torch.randn(shape, generator=gen, device=DEVICE, dtype=torch.float32)
    return (x * scale + mean).to(dtype) if (scale != 1.0 or mean != 0.0) else x.to(dtype)


def _inputs(case, seed):
    """The case's input tensors by name, from the seed alone."""
    gen = torch.Generator(device=DEVICE).manual_seed(seed)
    dt = DTYPES[case["dtype"]]
    n = _rows(case)
    if case["kind"] == "attn":
        h, hk, d = case["heads"], case["kv_heads"], case["head_dim"]
        t = {"q": _randn(gen, (n, h, d), dt), "k": _randn(gen, (n, hk, d), dt),
             "v": _randn(gen, (n, hk, d), dt)}
        if case["train"]:
            t["dout"] = _randn(gen, (n, h, d), dt)
        return t
    if case["kind"] == "norm":
        d = case["dim"]
        shape = (n, case["heads"], d) if case["heads"] > 1 else (n, d)
        t = {"x": _randn(gen, shape, dt), "w": _randn(gen, (d,), dt, 0.02, 1.0)}
        if case["norm"] == "layer":
            t["b"] = _randn(gen, (d,), dt, 0.02)
        if case["norm"] == "add_rms":
            t["r"] = _randn(gen, shape, dt)
        if case["train"]:
            t["dy"] = _randn(gen, shape, dt)
            if case["norm"] == "add_rms":
                t["dh"] = _randn(gen, shape, dt)
        return t
    f = case["features"]
    t = {"x": _randn(gen, (n, f), dt, 2.0 if case["kind"] == "softmax" else 1.0)}
    if case["train"]:
        t["dy"] = _randn(gen, (n, f), dt)
    return t


GRAD_NAMES = ("q", "k", "v", "x", "r", "w", "b")


def prepare(case, seed):
    t = _inputs(case, seed)
    state = {"case": case, "t": t}
    if case["kind"] != "norm":
        state["cu"] = _offsets(_lengths(case))
    if case["train"]:
        state["leaves"] = [t[k].requires_grad_(True) for k in GRAD_NAMES if k in t]
    if case["kind"] in ("softmax", "pad"):
        state["arr"] = scree_amd.Array(values=t["x"], offsets=state["cu"])
    if case["kind"] == "attn" and case["dtype"] == "fp32":
        # fp32 attention is an Array-level call
        state["qkv"] = [scree_amd.Array(values=t[x], offsets=state["cu"]) for x in ("q", "k", "v")]
    return state


# --------------------------------------------------------------------- run
def _grads(state):
    return tuple(p.grad for p in state["leaves"])


def run(state):
    case, t = state["case"], state["t"]
    if case["train"]:
        for p in state["leaves"]:
            p.grad = None
    if case["kind"] == "attn":
        cu = state["cu"]
        if case["dtype"] == "fp32":
            out = kernels.varlen_attention(*state["qkv"], causal=case["causal"]).values
        elif case["train"]:
            out = hip.varlen_attention_hip_autograd(t["q"], t["k"], t["v"], cu, causal=case["causal"])
        else:
            return hip.varlen_attention_hip(t["q"], t["k"], t["v"], cu, causal=case["causal"])
        if not case["train"]:
            return out
        out.backward(t["dout"])
        return (out.detach(),) + _grads(state)
    if case["kind"] == "norm":
        if case["norm"] == "add_rms":
            h, y = hip.varlen_add_rmsnorm_hip(t["x"], t["r"], t["w"])
            if not case["train"]:
                return h, y
            torch.autograd.backward((h, y), (t["dh"], t["dy"]))
            return (h.detach(), y.detach()) + _grads(state)
        if case["norm"] == "layer":
            y = hip.varlen_layernorm_hip(t["x"], t["w"], t["b"])
        else:
            y = hip.varlen_rmsnorm_hip(t["x"], t["w"])
        if not case["train"]:
            return y
        y.backward(t["dy"])
        return (y.detach(),) + _grads(state)
    if case["kind"] == "softmax":
        y = kernels.varlen_softmax(state["arr"]).values
        if not case["train"]:
            return y
        y.backward(t["dy"])
        return (y.detach(),) + _grads(state)
    padded, mask = scree_amd.to_padded(state["arr"])
    back = scree_amd.from_padded(padded, mask)
    return padded, mask, back.values, back.offsets


# ---------------------------------------------------------- work, tolerance
def _pairs(case):
    n = _lengths(case)
    return sum(x * (x + 1) // 2 for x in n) if case["causal"] else sum(x * x for x in n)


def work(case):
    s = DTYPES[case["dtype"]].itemsize
    if case["kind"] == "attn":
        n, d = _rows(case), case["head_dim"]
        q, kv = s * n * case["heads"] * d, s * n * case["kv_heads"] * d
        flops = 4.0 * case["heads"] * d * _pairs(case)
        if not case["train"]:
            return {"bytes": 2 * q + 2 * kv, "flops": flops}
        # read q, k, v, dout; write out, dq, dk, dv; two products forward, five backward
        return {"bytes": 4 * q + 4 * kv, "flops": 3.5 * flops}
    if case["kind"] == "norm":
        e = s * case["rows"] * case["heads"] * case["dim"]
        if case["norm"] == "add_rms":
            return {"bytes": (4 + (3 if case["train"] else 0)) * e, "flops": 0}
        # forward x, y; backward dy, dx (x is the same input)
        return {"bytes": (4 if case["train"] else 2) * e, "flops": 0}
    e = s * _rows(case) * case["features"]
    if case["kind"] == "softmax":
        return {"bytes": (4 if case["train"] else 2) * e, "flops": 0}
    padded = case["seqs"] * max(_lengths(case)) * (s * case["features"] + 1)
    return {"bytes": 2 * e + padded, "flops": 0}


def tolerance(case):
    # About four times the largest error against 64 bits seen over the listed
    # and some drawn cases: 2.5e-3 in bf16 and 3.1e-4 in fp16 (the rounding of
    # the stored outputs and, in attention, of the weights as operands), 4.5e-7
    # in fp32 (sums of up to thousands of terms).
    if case["kind"] == "pad":
        return "exact"
    return {"rel": {"fp32": 1.8e-6, "fp16": 1.3e-3, "bf16": 1e-2}[case["dtype"]]}


# ------------------------------------------------------------------- exact
def _exact_attn(case, t):
    lengths = _lengths(case)
    h, hk, d = case["heads"], case["kv_heads"], case["head_dim"]
    group, scale = h // hk, 1.0 / math.sqrt(d)
    x = {k: v.detach().double().transpose(0, 1).contiguous() for k, v in t.items()}  # (heads, n, d)
    names = ["out"] + (["q", "k", "v"] if case["train"] else [])
    res = {k: torch.zeros_like(x["q" if k == "out" else k]) for k in names}
    a = 0
    for n in lengths:
        rows = slice(a, a + n)
        a += n
        keep = torch.ones(n, n, dtype=torch.bool, device=DEVICE).tril() if case["causal"] else None
        step = max(1, (1 << 28) // (n * n) // group)  # K/V heads at a time
        for k0 in range(0, hk, step):
            k1 = min(hk, k0 + step)
            qs = slice(k0 * group, k1 * group)
            q = x["q"][qs, rows].contiguous()
            k = x["k"][k0:k1, rows].repeat_interleave(group, dim=0)
            v = x["v"][k0:k1, rows].repeat_interleave(group, dim=0)
            p = torch.matmul(q, k.transpose(1, 2).contiguous()) * scale
            if keep is not None:
                p.masked_fill_(~keep, -math.inf)
            p = torch.softmax(p, dim=-1)
            out = torch.matmul(p, v)
            res["out"][qs, rows] = out
            if not case["train"]:
                continue
            do = x["dout"][qs, rows].contiguous()
            dv = torch.matmul(p.transpose(1, 2).contiguous(), do)
            ds = torch.matmul(do, v.transpose(1, 2).contiguous())
            ds.sub_((out * do).sum(-1, keepdim=True)).mul_(p).mul_(scale)
            res["q"][qs, rows] = torch.matmul(ds, k)
            dk = torch.matmul(ds.transpose(1, 2).contiguous(), q)
            res["k"][k0:k1, rows] = dk.view(k1 - k0, group, n, d).sum(1)
            res["v"][k0:k1, rows] = dv.view(k1 - k0, group, n, d).sum(1)
    outs = tuple(res[k].transpose(0, 1).contiguous() for k in names)
    return outs if case["train"] else outs[0]


def _exact_norm(case, t):
    eps = 1e-5 if case["norm"] == "layer" else 1e-6
    leaves = {k: t[k].detach().double().requires_grad_(case["train"]) for k in GRAD_NAMES if k in t}
    x = leaves["x"]
    h = None
    if case["norm"] == "add_rms":
        # the stored sum is rounded to the activations' dtype, and that is normalised
        s = x + leaves["r"]
        x = s + (s.detach().float().to(t["x"].dtype).double() - s.detach())
        h = x
    if case["norm"] == "layer":
        c = x - x.mean(-1, keepdim=True)
        y = c * torch.rsqrt((c * c).mean(-1, keepdim=True) + eps) * leaves["w"] + leaves["b"]
    else:
        y = x * torch.rsqrt((x * x).mean(-1, keepdim=True) + eps) * leaves["w"]
    outs = (y,) if h is None else (h, y)
    if not case["train"]:
        return outs if h is not None else y
    gs = (t["dy"].double(),) if h is None else (t["dh"].double(), t["dy"].double())
    torch.autograd.backward(outs, gs)
    return tuple(o.detach() for o in outs) + tuple(p.grad for p in leaves.values())


def _exact_softmax(case, t):
    x = t["x"].detach().double()
    y, dx = torch.empty_like(x), torch.empty_like(x)
    a = 0
    for n in _lengths(case):
        rows = slice(a, a + n)
        a += n
        y[rows] = torch.softmax(x[rows], dim=0)
        if case["train"]:
            g = t["dy"][rows].double()
            dx[rows] = y[rows] * (g - (y[rows] * g).sum(0, keepdim=True))
    return (y, dx) if case["train"] else y


def exact(case, seed):
    if case["kind"] == "pad":
        return None
    t = _inputs(case, seed)
    if case["kind"] == "attn":
        return _exact_attn(case, t)
    return _exact_norm(case, t) if case["kind"] == "norm" else _exact_softmax(case, t)
