"""float32 attention on bf16 planes (forward and gradients, head dims 64 and
128): every workgroup shape at tile edges against float64, and infinities and
values beyond bf16's range against the same rule in float64.

Bound: a product of planes drops terms below 2^-25 of it and every sum is
float32; over at most a few hundred terms the relative error of an output (in
2-norm) stays below 32 units of 2^-24 = 2e-6 (measured: 2e-7 to 7e-7).
"""

import math

import pytest

from tests._helpers import rng_normal, to_dev

pytestmark = pytest.mark.gpu
REL = 32 * 2.0 ** -24

# D, B, Lq, Lk, Hq, Hkv, causal, forward, dq and dkdv workgroup shapes
CASES = [
    (64, 1, 1, 1, 1, 1, False, "64, 1, 4", "64, 1, 4", "64, 1, 4"),
    (64, 2, 33, 129, 2, 1, False, "64, 1, 4", "64, 1, 4", "64, 1, 4"),
    (64, 1, 257, 255, 4, 4, True, "64, 1, 4", "64, 1, 4", "64, 1, 4"),
    (64, 3, 127, 300, 70, 14, True, "64, 2, 4", "64, 2, 4", "64, 2, 4"),
    (64, 2, 65, 64, 140, 140, False, "64, 4, 2", "64, 4, 2", "64, 4, 2"),
    (64, 1, 129, 191, 260, 260, True, "64, 4, 2", "64, 4, 2", "64, 4, 2"),
    (128, 1, 31, 97, 2, 2, False, "split", "128, 2, 2", "128, 2, 2"),
    (128, 2, 130, 95, 40, 20, True, "128, 2, 2", "128, 2, 2", "128, 2, 2"),
    (128, 1, 161, 129, 260, 260, False, "128, 4, 1", "128, 4, 1", "128, 4, 1"),
]


def _attend64(q, k, v, scale, causal):
    """float64 attention and the q, k, v it used (heads repeated for GQA)."""
    import torch

    q, k, v = (x.double().transpose(1, 2) for x in (q, k, v))
    rep = q.shape[1] // k.shape[1]
    s = torch.matmul(q, k.repeat_interleave(rep, 1).transpose(-1, -2).contiguous()) * scale
    if causal:
        keep = torch.ones(s.shape[-2:], dtype=torch.bool, device=s.device).tril()
        s = s.masked_fill(~keep, float("-inf"))
    return torch.matmul(torch.softmax(s, -1), v.repeat_interleave(rep, 1)).transpose(1, 2)


def _rel(a, b):
    return float((a.double() - b).norm() / b.norm().clamp_min(1e-300))


@pytest.mark.parametrize("case", CASES)
def test_shapes_against_float64(device, case):
    import torch
    from probjax_amd import native
    from probjax_amd.hip_attention import flash_attention_bwd, flash_attention_fwd

    D, B, Lq, Lk, Hq, Hkv, causal, fwd, dq, dkdv = case
    print(f"f32 planes {case}", flush=True)
    q, k, v, do = (to_dev(x, device, torch.float32) for x in rng_normal(
        91, (B, Lq, Hq, D), (B, Lk, Hkv, D), (B, Lk, Hkv, D), (B, Lq, Hq, D)))
    kw = dict(sm_scale=1 / math.sqrt(D), causal=causal)
    o, lse = flash_attention_fwd(q, k, v, return_lse=True, **kw)
    names = native.last_launches()
    grads = flash_attention_bwd(q, k, v, o, do, lse, **kw)
    names += native.last_launches()
    prefix = ("flash_fwd_f32_split_kernel<" if fwd == "split" else f"flash_fwd_f32_planes_kernel<{fwd}",
              f"flash_bwd_dq_f32_planes_kernel<{dq}", f"flash_bwd_dkdv_f32_planes_kernel<{dkdv}")
    assert len(names) == 3 and all(n.startswith(p) for n, p in zip(names, prefix)), names
    x = [t.double().requires_grad_() for t in (q, k, v)]
    want = _attend64(*x, kw["sm_scale"], causal)
    wg = torch.autograd.grad(want, x, do.double())
    errs = [_rel(o, want.detach())] + [_rel(g, w) for g, w in zip(grads, wg)]
    print(f"  rel {errs}", flush=True)
    # one key: the softmax is constant and dq, dk are exactly 0 up to the rounding of dp - delta
    if Lk == 1:
        errs = [errs[0], errs[3]]
    assert max(errs) <= REL, errs


@pytest.mark.parametrize("D,H", [(64, 2), (64, 300), (128, 80)])
def test_values_beyond_bf16_range(device, D, H):
    """Infinite and float32's largest values in K and V take the float32
    MFMAs: -inf scores drop their key, +inf scores make the row NaN, an
    infinite V column is infinite, and finite values stay as accurate."""
    import torch
    from probjax_amd.hip_attention import flash_attention_bwd, flash_attention_fwd

    B, L = 1, 100
    q, k, v, do = (to_dev(x, device, torch.float32) for x in rng_normal(
        92, (B, L, H, D), (B, L, H, D), (B, L, H, D), (B, L, H, D)))
    kw = dict(sm_scale=1 / math.sqrt(D))
    big = torch.finfo(torch.float32).max
    # the largest finite value in V, reached with weight zero (its key's score is -inf)
    k1, v1 = k.clone(), v.clone()
    k1[0, 40] = 0
    k1[0, 40, :, 3] = float("inf")
    v1[0, 40] = big
    o = flash_attention_fwd(q, k1, v1, **kw)
    want = _attend64(q, k1, v1, kw["sm_scale"], False)
    up = (q[0, :, :, 3] > 0)[None]
    assert torch.isnan(o[up]).all()
    assert _rel(o[~up], want[~up]) <= REL
    # infinities in V: rows see them with positive weight
    v2 = v.clone()
    v2[0, 70, :, 5] = float("inf")
    v2[0, 71, :, 6] = float("-inf")
    o = flash_attention_fwd(q, k, v2, **kw)
    assert torch.isposinf(o[..., 5]).all() and torch.isneginf(o[..., 6]).all()
    rest = [i for i in range(D) if i not in (5, 6)]
    want = _attend64(q, k, v, kw["sm_scale"], False)
    assert _rel(o[..., rest], want[..., rest]) <= REL
    # large finite values: K scaled up to float32's end, Q and sm_scale down, so
    # that the scores are those of the unscaled call and dQ is 2^60 times its dQ
    k3 = k * (3.9 / k.abs().max())
    big_k, small_q, scale = k3 * 2.0 ** 126, q * 2.0 ** -60, kw["sm_scale"] * 2.0 ** -66
    assert float(big_k.abs().max()) > 3.3e38
    o3, lse3 = flash_attention_fwd(small_q, big_k, v, sm_scale=scale, return_lse=True)
    x = [t.double().requires_grad_() for t in (q, k3, v)]
    want = _attend64(*x, kw["sm_scale"], False)
    wg = torch.autograd.grad(want, x, do.double())
    dq, _, dv = flash_attention_bwd(small_q, big_k, v, o3, do, lse3, sm_scale=scale)
    assert _rel(o3, want.detach()) <= REL
    assert _rel(dq.double() * 2.0 ** -60, wg[0]) <= REL
    assert _rel(dv, wg[2]) <= REL


@pytest.mark.parametrize("D,H", [(64, 2), (64, 300), (128, 80)])
def test_products_beyond_float32(device, D, H):
    """Finite q and k whose product lies below float32's range drop that key,
    forward and backward, as a score of -inf does."""
    import torch
    from probjax_amd.hip_attention import flash_attention_bwd, flash_attention_fwd

    B, L = 1, 100
    q, k, v, do = (to_dev(x, device, torch.float32) for x in rng_normal(93, *[(B, L, H, D)] * 4))
    q[..., 3] = 1e22 * (1 + q[..., 3].abs())
    k[..., 3] = 0
    k[0, 40, :, 3] = -1e22 * (1 + k[0, 40, :, 4].abs())
    kw = dict(sm_scale=1 / math.sqrt(D))
    o, lse = flash_attention_fwd(q, k, v, return_lse=True, **kw)
    grads = flash_attention_bwd(q, k, v, o, do, lse, **kw)
    rest = [i for i in range(L) if i != 40]
    x = [t.double().requires_grad_() for t in (q, k[:, rest], v[:, rest])]
    want = _attend64(*x, kw["sm_scale"], False)
    wg = torch.autograd.grad(want, x, do.double())
    assert torch.isfinite(lse).all()
    assert not grads[1][:, 40].any() and not grads[2][:, 40].any()
    errs = [_rel(o, want.detach()), _rel(grads[0], wg[0])] + [_rel(g[:, rest], w) for g, w in zip(grads[1:], wg[1:])]
    print(f"  rel {errs}", flush=True)
    assert max(errs) <= REL, errs


@pytest.mark.parametrize("D,H", [(64, 2), (64, 300), (128, 80)])
@pytest.mark.parametrize("which", ["v", "do", "k", "row"])
def test_small_values(device, D, H, which):
    """Operands so small that a bf16 plane would lose bits (V, dO, K against a
    larger scale, some rows of K and V among ordinary ones): as accurate as any."""
    import torch
    from probjax_amd.hip_attention import flash_attention_bwd, flash_attention_fwd

    B, L, scale = 1, 100, 1 / math.sqrt(D)
    for e in (-101, -112, -118):
        q, k, v, do = (to_dev(x, device, torch.float32) for x in rng_normal(94, *[(B, L, H, D)] * 4))
        sm_scale = scale
        if which == "v":
            v *= 2.0 ** e
        elif which == "do":
            do *= 2.0 ** e
        elif which == "k":
            k *= 2.0 ** e
            q *= 2.0 ** 50
            sm_scale *= 2.0 ** (-e - 50)
        else:
            # these rows alone make the last feature block of the output
            v[:, 40:44, :, 32:] *= 2.0 ** e
            v[:, :40, :, 32:] = v[:, 44:, :, 32:] = 0
            k[:, 40:44] *= 2.0 ** e
        kw = dict(sm_scale=sm_scale)
        o, lse = flash_attention_fwd(q, k, v, return_lse=True, **kw)
        grads = flash_attention_bwd(q, k, v, o, do, lse, **kw)
        x = [t.double().requires_grad_() for t in (q, k, v)]
        want = _attend64(*x, sm_scale, False)
        wg = torch.autograd.grad(want, x, do.double())
        errs = [_rel(o, want.detach())] + [_rel(g, w) for g, w in zip(grads, wg)]
        if which == "row":
            errs.append(_rel(o[..., 32:], want.detach()[..., 32:]))
        print(f"  2^{e} rel {errs}", flush=True)
        # dS of a small V or dO is small itself: its products have a test of their own
        checked = {"v": (0, 3), "do": (0, 3)}.get(which, range(len(errs)))
        assert max(errs[i] for i in checked) <= REL, errs


@pytest.mark.parametrize("D,H", [(64, 2), (64, 70), (64, 300), (128, 2), (128, 300)])
@pytest.mark.parametrize("which", ["v", "do", "both"])
def test_small_score_gradients(device, D, H, which):
    """dS is as accurate where V, dO or their product alone make it small."""
    import torch
    from probjax_amd.hip_attention import flash_attention_bwd, flash_attention_fwd

    B, L, kw = 1, 100, dict(sm_scale=1 / math.sqrt(D))
    for e in (-95, -101, -112, -118):
        q, k, v, do = (to_dev(x, device, torch.float32) for x in rng_normal(95, *[(B, L, H, D)] * 4))
        a, b = {"v": (e, 0), "do": (0, e), "both": (e // 2, e - e // 2)}[which]
        v *= 2.0 ** a
        do *= 2.0 ** b
        o, lse = flash_attention_fwd(q, k, v, return_lse=True, **kw)
        grads = flash_attention_bwd(q, k, v, o, do, lse, **kw)
        x = [t.double().requires_grad_() for t in (q, k, v)]
        wg = torch.autograd.grad(_attend64(*x, kw["sm_scale"], False), x, do.double())
        errs = [_rel(g, w) for g, w in zip(grads, wg)]
        print(f"  2^{e} rel {errs}", flush=True)
        assert max(errs) <= REL, errs


@pytest.mark.parametrize("D,H", [(64, 2), (64, 70), (64, 300), (128, 2), (128, 300)])
@pytest.mark.parametrize("bias", [False, True])
def test_large_score_gradients(device, D, H, bias):
    """A dS of ordinary operands' product that is itself huge: infinite where a
    gradient lies beyond float32 (one term alone makes it), accurate elsewhere."""
    import torch
    from probjax_amd.hip_attention import flash_attention_bwd, flash_attention_fwd

    B, L, kw = 1, 100, dict(sm_scale=1 / math.sqrt(D))
    q, k, v, do = (to_dev(x, device, torch.float32) for x in rng_normal(96, *[(B, L, H, D)] * 4))
    # features 3 and 5 are no part of any score
    for t, i in ((q, 5), (k, 3)):
        t[..., i] = 0
        t[0, 41, :, i] = 2.0 ** 34
    q[..., 3] = 0
    k[..., 5] = 0
    v *= 2.0 ** 56
    do *= 2.0 ** 56
    if bias:
        kw["bias"] = torch.zeros(1, 1, L, L, device=device)
    o, lse = flash_attention_fwd(q, k, v, return_lse=True, **kw)
    grads = flash_attention_bwd(q, k, v, o, do, lse, bias_grad=bias, **kw)[:3]
    x = [t.double().requires_grad_() for t in (q, k, v)]
    wg = torch.autograd.grad(_attend64(*x, kw["sm_scale"], False), x, do.double())
    big = torch.finfo(torch.float32).max
    inf = 0
    for g, w in zip(grads, wg):
        assert not torch.isnan(g).any()
        over, under = w.abs() > 1.001 * big, w.abs() < 0.999 * big
        assert torch.equal(g[over], w[over].sign().float() * float("inf"))
        assert torch.isfinite(g[under]).all()
        ordinary = w.abs() < 2.0 ** 120
        assert float((g.double() - w)[ordinary].norm() / w[ordinary].norm()) <= REL
        inf += int(over.sum())
    assert inf > 100


@pytest.mark.parametrize("D,H", [(64, 2), (64, 70), (64, 300), (128, 2), (128, 300)])
def test_one_p_in_both_kernels(device, D, H):
    """The dK/dV kernel's P is the dQ kernel's, bit for bit, also where scores of
    a hundred leave a P fewer digits: with dP = 1, no delta and dO in one
    row, the bias gradient is the one and dV the other."""
    import torch
    from probjax_amd.hip_attention import flash_attention_bwd, flash_attention_fwd

    L, row = 129, 77
    q, k = (to_dev(x, device, torch.float32) for x in rng_normal(98, *[(1, L, H, D)] * 2))
    q *= 20
    v, do = torch.zeros_like(k), torch.zeros_like(q)
    v[..., 0] = 1
    do[0, row, :, 0] = 1
    kw = dict(sm_scale=1 / math.sqrt(D), bias=torch.zeros(1, 1, L, L, device=device))
    _, lse = flash_attention_fwd(q, k, v, return_lse=True, **kw)
    grads = flash_attention_bwd(q, k, v, torch.zeros_like(q), do, lse, bias_grad=True, **kw)
    p = grads[2][0, :, :, 0].t()
    kw["bias"] = kw["bias"].expand(1, H, L, L).contiguous()  # a gradient for every head
    db = flash_attention_bwd(q, k, v, torch.zeros_like(q), do, lse, bias_grad=True, **kw)[3][0, :, row]
    seen = db > 2.0 ** -100  # below, a P is no sum of three planes
    assert seen.sum() > 40 * H and torch.equal(p[seen], db[seen])
