"""What the speed of this framework is measured on: the calls a program makes
through the public attention API, from a single small layer to long training
sequences and large KV caches.

``listed()`` holds the fixed cases, ``draw(rng)`` gives another one of the same
ranges.  ``prepare`` makes what the caller has in hand (inputs on the GPU),
``run`` is one pass through the public entry points, ``work`` the bytes and
operations a pass cannot do without, ``exact`` the same outputs from plain
torch in float64 and ``tolerance`` how far another correct implementation at
the same precision may be from this one.

Case kinds
  attention       ``mha`` / ``dot_product_attention`` over whole sequences:
                  forward, or forward and gradients with ``backward``
  decode          ``mha`` with one or a few query rows over a KV cache
  latent_decode   absorbed ``mla`` over a latent cache
  latent_project  ``mla`` with its K/V projections
"""

from __future__ import annotations

import math

import torch

from probjax_amd import masks
from probjax_amd.attention import dot_product_attention, mha, mla

DTYPES = {"f32": torch.float32, "bf16": torch.bfloat16, "f16": torch.float16}
SIZE = {"f32": 4, "bf16": 2, "f16": 2}


def _attention(name, dtype, batch, heads, kv_heads, length, head_dim, mask, backward, *,
               window=0, documents=0, bias="none"):
    c = dict(kind="attention", dtype=dtype, batch=batch, heads=heads, kv_heads=kv_heads, length=length,
             head_dim=head_dim, mask=mask, backward=backward, window=window, documents=documents, bias=bias)
    return dict(c, name=name) if name else c


def _decode(name, dtype, batch, heads, kv_heads, q_len, capacity, head_dim, shortest):
    c = dict(kind="decode", dtype=dtype, batch=batch, heads=heads, kv_heads=kv_heads, q_len=q_len,
             capacity=capacity, head_dim=head_dim, shortest=shortest)
    return dict(c, name=name) if name else c


def _latent_decode(name, dtype, batch, heads, q_len, capacity, rank, v_dim, shortest):
    c = dict(kind="latent_decode", dtype=dtype, batch=batch, heads=heads, q_len=q_len, capacity=capacity,
             rank=rank, v_dim=v_dim, shortest=shortest)
    return dict(c, name=name) if name else c


def _latent_project(name, dtype, batch, heads, length, rank, head_dim, backward):
    c = dict(kind="latent_project", dtype=dtype, batch=batch, heads=heads, length=length, rank=rank,
             head_dim=head_dim, backward=backward)
    return dict(c, name=name) if name else c


def listed():
    return [
        # One layer of a small float32 model (the library's default dtype): launch and latency bound.
        _attention("f32_small_causal", "f32", 1, 4, 4, 512, 64, "causal", False),
        # A float32 training step of an ordinary transformer layer.
        _attention("f32_train_causal", "f32", 4, 8, 8, 1024, 64, "causal", True),
        # Prompt processing of a bf16 language model, the headline shape.
        _attention("bf16_prefill_causal", "bf16", 4, 16, 16, 4096, 128, "causal", False),
        # Training step of a grouped-query bf16 model: the largest case.
        _attention("bf16_train_gqa", "bf16", 2, 16, 4, 4096, 128, "causal", True),
        # Training on documents packed into one row, which must not see each other.
        _attention("bf16_train_packed", "bf16", 2, 16, 16, 2048, 128, "packed", True, documents=6),
        # Training with position information from distance slopes.
        _attention("bf16_train_alibi", "bf16", 2, 12, 12, 1024, 64, "causal", True, bias="alibi"),
        # A sliding-window layer with a head width and a length that are no powers of two, fp16.
        _attention("f16_window_width96", "f16", 2, 12, 12, 1531, 96, "window", True, window=256),
        # Training with a learned additive bias, which gets its gradient, and padded keys.
        _attention("bf16_train_bias", "bf16", 2, 8, 8, 2048, 64, "lengths", True, bias="dense"),
        # Training a latent-attention layer with its K/V projections.
        _latent_project("bf16_train_latent", "bf16", 4, 8, 2048, 128, 64, True),
        # One token for every sequence of a serving batch, caches of different fill.
        _decode("bf16_decode_ragged", "bf16", 32, 32, 8, 1, 8192, 128, 512),
        # One token of one chat against a cache of middle size.
        _decode("bf16_decode_single", "bf16", 1, 32, 8, 1, 4096, 128, 4096),
        # One token for every sequence over compressed latent caches.
        _latent_decode("bf16_latent_decode", "bf16", 16, 16, 1, 4096, 576, 512, 4096),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _cost(case):
    w = work(case)
    # float32 products run at about a sixteenth of the 16-bit rate
    return max(w["bytes"], w["flops"] * (16 if case["dtype"] == "f32" else 1) / 300)


def draw(rng):
    most = max(_cost(c) for c in listed())
    while True:
        case = _draw(rng)
        if _cost(case) <= most:
            return case


def _draw(rng):
    kind = rng.choice(("train", "train", "forward", "forward", "bias", "decode", "decode", "latent_decode",
                       "latent_project"))
    dtype = rng.choice(("bf16", "bf16", "f16", "f32"))
    if kind in ("train", "forward"):
        kv_heads = rng.choice((1, 2, 4, 8))
        heads = kv_heads * rng.choice((1, 1, 2, 4))
        length = _log_int(rng, 64, 2048 if dtype == "f32" else 4096)
        mask = rng.choice(("causal", "causal", "window", "packed", "lengths", "none"))
        bias = rng.choice(("none", "none", "alibi")) if mask == "causal" else "none"
        return _attention(None, dtype, rng.randint(1, 4), heads, kv_heads, length,
                          rng.choice((32, 64, 64, 80, 96, 128, 128)), mask, kind == "train",
                          window=max(16, length // 6) if mask == "window" else 0,
                          documents=rng.randint(2, 8) if mask == "packed" else 0, bias=bias)
    if kind == "bias":
        heads = rng.choice((4, 8, 12))
        return _attention(None, dtype, rng.randint(1, 4), heads, heads,
                          _log_int(rng, 64, 1024 if dtype == "f32" else 2048), rng.choice((32, 64, 64, 128)),
                          rng.choice(("none", "lengths")), rng.random() < 0.5, bias="dense")
    if kind == "decode":
        kv_heads = rng.choice((1, 2, 4, 8))
        capacity = _log_int(rng, 128, 32768)
        batch = max(1, min(32, _log_int(rng, 1, 48), (1 << 18) // capacity))
        return _decode(None, dtype, batch, kv_heads * rng.choice((1, 4, 8)), kv_heads,
                       rng.choice((1, 1, 1, 2, 4)), capacity, rng.choice((64, 80, 128, 128)),
                       max(1, int(capacity * rng.choice((0.0625, 0.5, 1.0)))))
    half = rng.choice(("bf16", "bf16", "f16"))
    if kind == "latent_decode":
        capacity = _log_int(rng, 256, 16384)
        rank, v_dim = rng.choice(((576, 512), (576, 512), (512, 512), (256, 256)))
        return _latent_decode(None, half, max(1, min(32, _log_int(rng, 1, 48), (1 << 17) // capacity)),
                              rng.choice((8, 16, 32)), rng.choice((1, 1, 2)), capacity, rank, v_dim,
                              max(1, int(capacity * rng.choice((0.125, 0.5, 1.0)))))
    return _latent_project(None, half, rng.randint(1, 4), rng.choice((4, 8, 16)), _log_int(rng, 128, 4096),
                           rng.choice((128, 256, 512)), rng.choice((64, 128)), rng.random() < 0.5)


# ---------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------

def _lengths(gen, batch, shortest, longest):
    return torch.randint(shortest, longest + 1, (batch,), generator=gen, device="cuda", dtype=torch.int32)


def _segments(gen, batch, length, documents):
    """Document number of every position: ``documents - 1`` random cuts per row."""
    cuts = torch.rand((batch, documents - 1), generator=gen, device="cuda") * length
    pos = torch.arange(length, device="cuda", dtype=torch.float32)
    return (pos[None, :, None] >= cuts[:, None, :]).sum(-1).to(torch.int32)


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    dtype = DTYPES[case["dtype"]]

    def normal(*shape, scale=1.0, dtype=dtype):
        x = torch.randn(shape, generator=gen, device="cuda", dtype=torch.float32)
        return (x * scale if scale != 1.0 else x).to(dtype)

    s = {"case": case}
    kind, batch = case["kind"], case["batch"]
    if kind == "attention":
        L, H, Hkv, D = case["length"], case["heads"], case["kv_heads"], case["head_dim"]
        s["q"], s["k"], s["v"] = normal(batch, L, H, D), normal(batch, L, Hkv, D), normal(batch, L, Hkv, D)
        s["scale"] = 1.0 / math.sqrt(D)
        mask = case["mask"]
        if mask == "causal":
            s["mask"] = masks.CausalMask()
        elif mask == "window":
            s["mask"] = masks.CausalLocalWindowMask(case["window"])
        elif mask == "packed":
            s["segments"] = _segments(gen, batch, L, case["documents"])
            s["mask"] = masks.BlockDiagonalCausalMask(s["segments"])
        elif mask == "lengths":
            # key padding of about a tenth of every sequence
            s["lengths"] = _lengths(gen, batch, max(1, L - L // 5), L)
            s["mask"] = masks.KVLenMask(s["lengths"])
        else:
            s["mask"] = None
        s["bias"] = None
        if case["bias"] == "dense":
            s["bias_values"] = normal(1, H, L, L, scale=0.5, dtype=torch.float32)
            s["bias"] = masks.DenseBias(s["bias_values"])
        elif case["bias"] == "alibi":
            s["bias"] = masks.CausalAlibiBias()
        if case["backward"]:
            s["do"] = normal(batch, L, H, D)
            for n in ("q", "k", "v", "bias_values"):
                if n in s:
                    s[n].requires_grad_()
    elif kind == "decode":
        S, Hkv, D = case["capacity"], case["kv_heads"], case["head_dim"]
        s["q"] = normal(batch, case["q_len"], case["heads"], D)
        s["k"], s["v"] = normal(batch, S, Hkv, D), normal(batch, S, Hkv, D)
        s["scale"] = 1.0 / math.sqrt(D)
        s["lengths"] = _lengths(gen, batch, case["shortest"], S)
        s["mask"] = masks.KVLenMask(s["lengths"])
    elif kind == "latent_decode":
        s["q"] = normal(batch, case["q_len"], case["heads"], case["rank"])
        s["cache"] = normal(batch, case["capacity"], case["rank"])
        s["scale"] = 1.0 / math.sqrt(192.0)
        s["lengths"] = _lengths(gen, batch, case["shortest"], case["capacity"])
        s["mask"] = masks.KVLenMask(s["lengths"])
    else:
        L, H, D, R = case["length"], case["heads"], case["head_dim"], case["rank"]
        s["q"], s["cache"] = normal(batch, L, H, D), normal(batch, L, R)
        s["wk"], s["wv"] = (normal(H, D, R, scale=1.0 / math.sqrt(R)) for _ in range(2))
        s["scale"] = 1.0 / math.sqrt(D)
        if case["backward"]:
            s["do"] = normal(batch, L, H, D)
            for n in ("q", "cache", "wk", "wv"):
                s[n].requires_grad_()
    return s


# ---------------------------------------------------------------------------
# One pass
# ---------------------------------------------------------------------------

def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "decode":
        return mha(s["q"], s["k"], s["v"], mask=s["mask"], sm_scale=s["scale"])
    if kind == "latent_decode":
        return mla(s["q"], s["cache"], mask=s["mask"], sm_scale=s["scale"], v_dim=case["v_dim"])
    if kind == "latent_project":
        out = mla(s["q"], s["cache"], s["wk"], s["wv"], mask=masks.CausalMask(), sm_scale=s["scale"])
        inputs = {n: s[n] for n in ("q", "cache", "wk", "wv")}
    elif case["bias"] == "dense":
        out = dot_product_attention(s["q"], s["k"], s["v"], mask=s["mask"], bias=s["bias"], sm_scale=s["scale"])
        inputs = {n: s[n] for n in ("q", "k", "v", "bias_values")}
    else:
        out = mha(s["q"], s["k"], s["v"], mask=s["mask"], bias=s["bias"], sm_scale=s["scale"])
        inputs = {n: s[n] for n in ("q", "k", "v")}
    if not case["backward"]:
        return out
    grads = torch.autograd.grad(out, list(inputs.values()), s["do"])
    return {"out": out.detach(), **{"d" + n: g for n, g in zip(inputs, grads)}}


# ---------------------------------------------------------------------------
# Work
# ---------------------------------------------------------------------------

def _pairs(case):
    """Scores of one head of one batch item that the mask keeps (expected)."""
    L = case["length"]
    mask = case["mask"]
    if mask == "causal":
        return L * (L + 1) / 2
    if mask == "window":
        w = min(case["window"], L - 1)
        return (w + 1) * (L - w) + w * (w + 1) / 2
    if mask == "packed":
        return L * L / (case["documents"] + 1)
    if mask == "lengths":
        return L * (L - L // 5 / 2)
    return L * L


def work(case):
    size, kind, batch = SIZE[case["dtype"]], case["kind"], case["batch"]
    if kind == "attention":
        L, H, Hkv, D = case["length"], case["heads"], case["kv_heads"], case["head_dim"]
        q, kv = batch * L * H * D, batch * L * Hkv * D
        values, flops = 2 * q + 2 * kv, 4 * batch * H * D * _pairs(case)
        if case["backward"]:
            values, flops = values + 2 * q + 2 * kv, 3.5 * flops  # dO read; dQ, dK, dV written
        nbytes = values * size
        if case["bias"] == "dense":
            nbytes += 4 * H * L * L * (2 if case["backward"] else 1)
        return {"bytes": nbytes, "flops": flops}
    if kind in ("decode", "latent_decode"):
        keys = batch * (case["shortest"] + case["capacity"]) / 2
        rows = batch * case["q_len"] * case["heads"]
        if kind == "decode":
            D = case["head_dim"]
            return {"bytes": size * (2 * keys * case["kv_heads"] * D + 2 * rows * D),
                    "flops": 4 * case["q_len"] * case["heads"] * keys * D}
        R, dv = case["rank"], case["v_dim"]
        return {"bytes": size * (keys * R + rows * (R + dv)),
                "flops": 2 * case["q_len"] * case["heads"] * keys * (R + dv)}
    L, H, D, R = case["length"], case["heads"], case["head_dim"], case["rank"]
    q, cache, w = batch * L * H * D, batch * L * R, 2 * H * D * R
    project, attend = 4 * batch * L * H * D * R, 2 * batch * H * D * L * (L + 1)
    if not case["backward"]:
        return {"bytes": size * (2 * q + cache + w), "flops": project + attend}
    return {"bytes": size * (4 * q + 2 * cache + 2 * w), "flops": 3 * project + 3.5 * attend}


# ---------------------------------------------------------------------------
# 64-bit results and tolerance
# ---------------------------------------------------------------------------

def _keep(s, b, n_q, n_k):
    """Boolean [Lq, Lk] of the scores batch item ``b`` keeps, or None."""
    case = s["case"]
    i = torch.arange(n_q, device="cuda")[:, None]
    j = torch.arange(n_k, device="cuda")[None, :]
    mask = case.get("mask", "lengths" if "lengths" in s else "causal")
    if mask == "lengths":
        return (j < s["lengths"][b]).expand(n_q, n_k)
    if mask == "none":
        return None
    keep = j <= i
    if mask == "window":
        keep = keep & (j >= i - case["window"])
    elif mask == "packed":
        keep = keep & (s["segments"][b][:, None] == s["segments"][b][None, :])
    return keep


def _attend64(q, k, v, scale, keep, bias, do):
    """float64 attention of one KV head of one batch item: ``q [G, Lq, D]``,
    ``k, v [Lk, D*]`` -> out and, with ``do``, its gradients."""
    p = torch.matmul(q, k.t().contiguous()) * scale
    if bias is not None:
        p = p + bias
    if keep is not None:
        p = p.masked_fill(~keep, float("-inf"))
    p = torch.softmax(p, dim=-1)
    o = torch.matmul(p, v)
    if do is None:
        return o, None
    dv = torch.matmul(p.transpose(1, 2).contiguous(), do).sum(0)
    ds = p * (torch.matmul(do, v.t().contiguous()) - (o * do).sum(-1, keepdim=True))
    dq = torch.matmul(ds, k) * scale
    dk = torch.matmul(ds.transpose(1, 2).contiguous(), q).sum(0) * scale
    return o, (dq, dk, dv, ds)


def _sequence64(s, q, k, v, do, bias=None, slopes=None):
    """float64 ``[B, L, H, D]`` attention over every batch item and KV head."""
    B, n_q, H, _ = q.shape
    n_k, Hkv = k.shape[1], k.shape[2]
    G = H // Hkv
    o = torch.empty((B, n_q, H, v.shape[-1]), dtype=torch.float64, device="cuda")
    grads = None
    if do is not None:
        grads = [torch.empty_like(x) for x in (q, k, v)] + [None if bias is None else torch.zeros_like(bias)]
    far = None
    if slopes is not None:
        pos = torch.arange(n_k, device="cuda", dtype=torch.float64)
        far = pos[None, :] - pos[:n_q, None]
    for b in range(B):
        keep = _keep(s, b, n_q, n_k)
        for h in range(Hkv):
            g = slice(h * G, (h + 1) * G)
            extra = None if bias is None else bias[0, g]
            if far is not None:
                extra = slopes[g, None, None] * far
            out, d = _attend64(q[b, :, g].transpose(0, 1).contiguous(), k[b, :, h].contiguous(),
                               v[b, :, h].contiguous(), s["scale"], keep, extra,
                               None if do is None else do[b, :, g].transpose(0, 1).contiguous())
            o[b, :, g] = out.transpose(0, 1)
            if d is not None:
                grads[0][b, :, g] = d[0].transpose(0, 1)
                grads[1][b, :, h], grads[2][b, :, h] = d[1], d[2]
                if bias is not None:
                    grads[3][0, g] += d[3]
    return o, grads


def exact(case, seed):
    s = prepare(case, seed)
    x = {n: t.detach().double() for n, t in s.items()
         if isinstance(t, torch.Tensor) and n not in ("lengths", "segments")}
    kind = case["kind"]
    do = x.get("do")
    if kind == "decode":
        return _sequence64(s, x["q"], x["k"], x["v"], None)[0]
    if kind == "latent_decode":
        c = x["cache"][:, :, None, :]
        return _sequence64(s, x["q"], c, c[..., :case["v_dim"]], None)[0]
    if kind == "attention":
        slopes = None
        if case["bias"] == "alibi":
            slopes = 2.0 ** -(torch.arange(case["heads"], device="cuda", dtype=torch.float64) + 1)
        o, d = _sequence64(s, x["q"], x["k"], x["v"], do, x.get("bias_values"), slopes)
        if d is None:
            return o
        out = {"out": o, "dq": d[0], "dk": d[1], "dv": d[2]}
        return out if d[3] is None else {**out, "dbias_values": d[3]}
    B, L, R = x["cache"].shape
    H, D = case["heads"], case["head_dim"]
    c2, wk, wv = x["cache"].reshape(B * L, R), x["wk"].reshape(H * D, R), x["wv"].reshape(H * D, R)
    k = torch.matmul(c2, wk.t().contiguous()).reshape(B, L, H, D)
    v = torch.matmul(c2, wv.t().contiguous()).reshape(B, L, H, D)
    o, d = _sequence64(s, x["q"], k, v, do)
    if d is None:
        return o
    dk, dv = d[1].reshape(B * L, H * D), d[2].reshape(B * L, H * D)
    return {"out": o, "dq": d[0], "dcache": (torch.matmul(dk, wk) + torch.matmul(dv, wv)).reshape(B, L, R),
            "dwk": torch.matmul(dk.t().contiguous(), c2).reshape(H, D, R),
            "dwv": torch.matmul(dv.t().contiguous(), c2).reshape(H, D, R)}


# About four times the relative error against float64 that was measured: 5e-7
# in float32 (allowing for longer sums than the listed ones), 3e-4 in fp16 and
# 2.7e-3 in bf16; 3.9e-3 for the latent cache's gradient, which is rounded
# once more on its way through K and V.
_TOLERANCE = {"f32": 5e-6, "f16": 1.2e-3, "bf16": 1.1e-2}


def tolerance(case):
    rel = _TOLERANCE[case["dtype"]]
    return {"rel": 1.5 * rel if case["kind"] == "latent_project" else rel}
