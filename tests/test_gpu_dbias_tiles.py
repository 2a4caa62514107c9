"""dL/d(bias) folded over the broadcast (``pjx_flash_dbias``) against the
per-(batch, head) gradient of the dQ kernel summed afterwards, and rows without
a valid key (``pjx_empty_rows``) against the rule in torch operations.

Both gradients recompute the same float32 P (dP - delta) per score from the
same 16-bit operands (the sums inside a product may be ordered differently,
2^-22 of the terms) and add B * Hq of them in float32: 1e-5 of the largest.
"""

import math

import numpy as np
import pytest

from tests._helpers import rng_normal, to_dev, to_np

pytestmark = pytest.mark.gpu

CASES = [
    # dtype, D, B, Lq, Lk, Hq, Hkv, bias batch, bias heads, causal, kv lengths, window / segments / slopes
    ("bf16", 64, 3, 100, 130, 4, 2, 1, 4, False, [130, 64, 0], None),
    ("f16", 128, 2, 65, 129, 2, 1, 1, 1, True, None, None),
    ("bf16", 128, 2, 64, 128, 4, 4, 2, 4, False, None, None),
    ("bf16", 64, 1, 1, 1, 1, 1, 1, 1, False, None, None),
    ("bf16", 64, 2, 200, 190, 2, 2, 2, 1, True, [190, 77], None),
    ("f16", 64, 2, 150, 150, 4, 2, 1, 4, True, None, "window"),
    ("bf16", 128, 2, 97, 97, 2, 2, 1, 2, True, None, "segments"),
    ("bf16", 64, 2, 97, 161, 2, 2, 1, 2, False, None, "slopes"),
]


@pytest.mark.parametrize("case", CASES)
def test_folded_equals_summed(device, case):
    import torch
    from probjax_amd import hip_attention as hip
    from probjax_amd import native

    dtype, D, B, Lq, Lk, Hq, Hkv, bb, bh, causal, lengths, ext = case
    print(f"dbias {case}", flush=True)
    tdt = torch.bfloat16 if dtype == "bf16" else torch.float16
    q, k, v, do = (to_dev(x, device, tdt) for x in rng_normal(51, (B, Lq, Hq, D), (B, Lk, Hkv, D), (B, Lk, Hkv, D),
                                                              (B, Lq, Hq, D)))
    bias = to_dev(rng_normal(52, (bb, bh, Lq, Lk), scale=0.5)[0], device, torch.float32)
    bias[0, 0, 0, : Lk // 2] = float("-inf")
    mods = None
    if ext == "window":
        mods = hip.ScoreModsArgs(window_left=40)
    elif ext == "segments":
        ids = torch.from_numpy(np.sort(np.random.default_rng(53).integers(0, 4, (B, Lq))).astype(np.int32)).to(device)
        mods = hip.ScoreModsArgs(segment_q=ids, segment_k=ids)
    elif ext == "slopes":
        mods = hip.ScoreModsArgs(alibi_slopes=torch.full((Hq,), 0.25, device=device), alibi_symmetric=True, softcap=9.0)
    L = None if lengths is None else torch.tensor(lengths, dtype=torch.int32, device=device)
    kw = dict(sm_scale=1 / math.sqrt(D), causal=causal, kv_lengths=L, bias=bias, mods=mods)
    o, lse = hip.flash_attention_fwd(q, k, v, return_lse=True, **kw)
    want = hip.flash_attention_bwd(q, k, v, o, do, lse, bias_grad=True, **kw)
    got = hip.flash_attention_bwd(q, k, v, o, do, lse, bias_grad=True, fold_bias_grad=True, **kw)
    E = "Bf16Fmt" if dtype == "bf16" else "F16Fmt"
    assert native.last_launches() == [f"flash_dbias_kernel<{E}, {D}, {D // 32}, {'true' if ext else 'false'}>"]
    torch.cuda.synchronize()
    for a, b in zip(got[:3], want[:3]):
        np.testing.assert_allclose(to_np(a), to_np(b), rtol=2.0 ** -7, atol=2.0 ** -7 * float(b.float().abs().max()))
    a, b = to_np(got[3]), to_np(want[3])
    assert a.shape == b.shape == (bb, bh, Lq, Lk)
    assert np.isfinite(a).all()
    assert np.abs(a - b).max() <= 1e-5 * max(1.0, np.abs(b).max())


@pytest.mark.parametrize("dtype,D,causal,lengths", [
    ("bf16", 64, False, [130, 70]), ("f16", 128, False, [65, 129]), ("bf16", 64, True, [1, 200]), ("bf16", 128, True, [97, 31])])
def test_nonfinite_padding(device, dtype, D, causal, lengths):
    """K and V past a sequence's end may hold anything (a buffer from
    ``torch.empty``): the folded gradient, which also adds the other sequences',
    is bitwise that of finite padding."""
    import torch
    from probjax_amd import hip_attention as hip

    tdt = torch.bfloat16 if dtype == "bf16" else torch.float16
    B, L, H = len(lengths), 200, 2
    q, k, v, do = (to_dev(x, device, tdt) for x in rng_normal(57, *[(B, L, H, D)] * 4))
    bias = to_dev(rng_normal(58, (1, H, L, L), scale=0.5)[0], device, torch.float32)
    kw = dict(sm_scale=1 / math.sqrt(D), causal=causal, bias=bias,
              kv_lengths=torch.tensor(lengths, dtype=torch.int32, device=device))
    o, lse = hip.flash_attention_fwd(q, k, v, return_lse=True, **kw)
    want = hip.flash_attention_bwd(q, k, v, o, do, lse, bias_grad=True, fold_bias_grad=True, **kw)
    for b, n in enumerate(lengths):
        k[b, n:], v[b, n:] = float("nan"), float("inf")
        v[b, n::2] = float("nan")
    got = hip.flash_attention_bwd(q, k, v, o, do, lse, bias_grad=True, fold_bias_grad=True, **kw)
    assert torch.isfinite(want[3]).all() and torch.equal(got[3], want[3])
    assert torch.equal(got[0], want[0])
    for b, n in enumerate(lengths):
        assert torch.equal(got[1][b, :n], want[1][b, :n]) and torch.equal(got[2][b, :n], want[2][b, :n])


@pytest.mark.parametrize("mask", ["causal", "window", "segments", "slopes"])
@pytest.mark.parametrize("D", [64, 128])
def test_nonfinite_at_masked_scores(device, D, mask):
    """What the mask drops has gradient 0 and changes no other, bitwise: an
    infinite or NaN bias there, and V of keys that the rows of a tile do not see."""
    import torch
    from probjax_amd import hip_attention as hip

    B, L, H = 2, 150, 2
    q, k, v, do = (to_dev(x, device, torch.bfloat16) for x in rng_normal(59, *[(B, L, H, D)] * 4))
    bias = to_dev(rng_normal(60, (1, H, L, L), scale=0.5)[0], device, torch.float32)
    i, j = torch.arange(L, device=device)[:, None], torch.arange(L, device=device)[None, :]
    keep, mods = j <= i, None
    if mask == "window":
        keep, mods = keep & (j >= i - 20), hip.ScoreModsArgs(window_left=20)
    elif mask == "segments":
        ids = (j[0] >= 77).to(torch.int32)
        keep, mods = keep & (ids[:, None] == ids[None, :]), hip.ScoreModsArgs(
            segment_q=ids.repeat(B, 1), segment_k=ids.repeat(B, 1))
    elif mask == "slopes":
        mods = hip.ScoreModsArgs(alibi_slopes=torch.full((H,), 0.25, device=device))
    kw = dict(sm_scale=1 / math.sqrt(D), causal=True, mods=mods, bias_grad=True, fold_bias_grad=True)

    def grads(bias):
        o, lse = hip.flash_attention_fwd(q, k, v, return_lse=True, sm_scale=kw["sm_scale"], causal=True, mods=mods,
                                         bias=bias)
        return o, lse, hip.flash_attention_bwd(q, k, v, o, do, lse, bias=bias, **kw)

    o, lse, want = grads(bias)
    assert torch.isfinite(want[3]).all() and not want[3][:, :, ~keep].any()
    for x in ("inf", "nan"):
        got = grads(bias.masked_fill(~keep, float(x)))[2]
        for a, b in zip(got, want):
            assert torch.equal(a, b)
    # the last key's V, seen by the last row alone
    v[:, L - 1] = float("nan")
    got = hip.flash_attention_bwd(q, k, v, o, do, lse, bias=bias, **kw)
    assert torch.equal(got[3][:, :, :-1], want[3][:, :, :-1])


def test_more_heads_than_the_tiles_address(device):
    """Heads whose rows exceed the folded kernel's offsets take the dQ kernel's
    gradient, as ``pjx_flash_bwd`` does for them."""
    import torch
    from probjax_amd import hip_attention as hip

    H, D, L = (1 << 22) // 128 + 1, 128, 2
    q, k, v, do = (to_dev(x, device, torch.bfloat16) for x in rng_normal(61, *[(1, L, H, D)] * 4))
    bias = to_dev(rng_normal(62, (1, 1, L, L))[0], device, torch.float32)
    kw = dict(sm_scale=1 / math.sqrt(D), bias=bias)
    o, lse = hip.flash_attention_fwd(q, k, v, return_lse=True, **kw)
    want = hip.flash_attention_bwd(q, k, v, o, do, lse, bias_grad=True, **kw)
    got = hip.flash_attention_bwd(q, k, v, o, do, lse, bias_grad=True, fold_bias_grad=True, **kw)
    for a, b in zip(got, want):
        assert torch.equal(a, b)


@pytest.mark.parametrize("B,H,L,D,bh,folds", [
    (16, 4, 64, 64, 1, False), (5, 1, 130, 128, 1, False), (4, 3, 100, 64, 3, True), (2, 8, 384, 64, 8, True),
    (6, 4, 384, 128, 1, False), (5, 8, 500, 128, 8, True), (7, 3, 257, 64, 3, False)])
def test_route_by_grid(device, B, H, L, D, bh, folds):
    """Few tiles with many (batch, head) pairs each take the summed copies,
    with the same gradient (the bound of the tests above)."""
    import torch
    from probjax_amd import hip_attention as hip
    from probjax_amd import native

    q, k, v, do = (to_dev(x, device, torch.bfloat16) for x in rng_normal(63, *[(B, L, H, D)] * 4))
    bias = to_dev(rng_normal(64, (1, bh, L, L), scale=0.5)[0], device, torch.float32)
    kw = dict(sm_scale=1 / math.sqrt(D), bias=bias, bias_grad=True)
    o, lse = hip.flash_attention_fwd(q, k, v, return_lse=True, sm_scale=kw["sm_scale"], bias=bias)
    want = hip.flash_attention_bwd(q, k, v, o, do, lse, **kw)
    got = hip.flash_attention_bwd(q, k, v, o, do, lse, fold_bias_grad=True, **kw)
    assert any(n.startswith("flash_dbias_kernel") for n in native.last_launches()) == folds
    a, b = to_np(got[3]), to_np(want[3])
    assert a.shape == b.shape and np.abs(a - b).max() <= 1e-5 * max(1.0, np.abs(b).max())


@pytest.mark.parametrize("dtype,B,Lq,Lk,Hq,Hkv,D", [
    ("bf16", 2, 70, 33, 4, 2, 64), ("f32", 1, 1, 257, 3, 3, 96), ("f16", 2, 300, 5, 8, 1, 256), ("f32", 2, 9, 1, 2, 1, 3)])
def test_empty_rows(device, dtype, B, Lq, Lk, Hq, Hkv, D):
    import torch
    from probjax_amd import attention as A
    from probjax_amd import hip_attention as hip

    tdt = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}[dtype]
    o, v, do = (to_dev(x, device, tdt) for x in rng_normal(54, (B, Lq, Hq, D), (B, Lk, Hkv, D), (B, Lq, Hq, D)))
    lse = torch.zeros((B, Hq, Lq), device=device)
    for share in (0.0, 0.4, 1.0):
        lse[torch.rand(lse.shape, device=device) < share] = float("inf")
        x = v.clone().requires_grad_()
        want = A._flax_empty_rows(o, lse, x)
        (dv,) = torch.autograd.grad(want, x, do)
        got, dgot = o.clone(), torch.zeros_like(v)
        hip.empty_rows(lse, v, got, grad=False)
        hip.empty_rows(lse, do, dgot, grad=True)
        if share == 0.0:
            assert torch.equal(got, o) and not dgot.any()
        # float32 sums in another order that may round to neighbours: one spacing of the format, at most
        # 2^-7 / 2^-10 of the value (torch rounds dV's mean and the sum over heads more often: 4 spacings)
        eps = {"bf16": 2.0 ** -7, "f16": 2.0 ** -10, "f32": 2.0 ** -20}[dtype]
        want, dv = want.detach().float(), dv.float()
        assert float((got.float() - want).abs().max()) <= eps * float(want.abs().max())
        assert float((dgot.float() - dv).abs().max()) <= 4 * eps * max(float(dv.abs().max()), 1e-6)


@pytest.mark.parametrize("dtype,B,Lq,Lk,Hq,Hkv,D,shift", [
    ("bf16", 1, 520, 700, 6, 2, 128, 0), ("f16", 3, 65, 64, 2, 2, 72, 0), ("f32", 1, 257, 66, 1, 1, 20, 0),
    ("bf16", 1, 1, 513, 8, 1, 256, 0), ("bf16", 2, 130, 70, 2, 1, 64, 1), ("f32", 1, 33, 129, 2, 2, 200, 1),
    ("f16", 1, 1030, 5, 40, 1, 8, 0)])
def test_empty_rows_split(device, dtype, B, Lq, Lk, Hq, Hkv, D, shift):
    """The edges of the row chunks, column groups and blocks of 256 rows, and
    tensors that start off 16 bytes (``shift``): sums against float64, to the
    spacing of the format, rows with valid keys untouched."""
    import torch
    from probjax_amd import hip_attention as hip

    tdt = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}[dtype]
    o, v, do, dv = (to_dev(x, device, tdt)[shift:shift + n].view(s) for x, n, s in (
        (rng_normal(65 + i, (math.prod(s) + 8,))[0], math.prod(s), s)
        for i, s in enumerate(((B, Lq, Hq, D), (B, Lk, Hkv, D), (B, Lq, Hq, D), (B, Lk, Hkv, D)))))
    lse = torch.zeros((B, Hq, Lq), device=device)
    for rows in ((Lq - 1,), range(0, Lq, 3), range(Lq)):
        lse[:, :, list(rows)] = float("inf")
        if Hq > 1:
            lse[:, 0] = 0.0  # a head without such rows
        empty = torch.isinf(lse).transpose(1, 2)[..., None]
        mean = v.double().mean(1, keepdim=True).repeat_interleave(Hq // Hkv, 2)
        got, dgot = o.clone(), dv.clone()
        if shift:
            got, dgot = (torch.cat((x.new_zeros(shift), x.flatten()))[shift:].view(x.shape) for x in (got, dgot))
        hip.empty_rows(lse, v, got, grad=False)
        hip.empty_rows(lse, do, dgot, grad=True)
        assert torch.equal(torch.where(empty, 0, got), torch.where(empty, 0, o))
        add = torch.where(empty, do, 0).double().sum(1).view(B, Hkv, Hq // Hkv, D).sum(2)[:, None] / Lk
        # one rounding to the format, and float32 sums of up to 41200 terms of size sqrt of that
        eps = {"bf16": 2.0 ** -8, "f16": 2.0 ** -11, "f32": 0.0}[dtype]
        for x, want in ((got, torch.where(empty, mean, o.double())), (dgot, dv.double() + add)):
            assert float((x.double() - want).abs().max()) <= (eps + 2.0 ** -20) * max(1.0, float(want.abs().max()))


@pytest.mark.parametrize("dtype,D,bias", [("bf16", 64, True), ("f16", 96, False), ("f32", 64, True), ("bf16", 256, False)])
def test_empty_rows_keep_nonfinite_gradients(device, dtype, D, bias):
    """An infinite or NaN dO in a row without a valid key reaches dV alone (the
    row's output is the mean of V): dq, dk and dbias are bitwise those of a
    finite dO there."""
    import torch
    from probjax_amd import attention as A

    tdt = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}[dtype]
    B, L, H = 2, 130, 2
    q, k, v, do = (to_dev(x, device, tdt) for x in rng_normal(55, *[(B, L, H, D)] * 4))
    keep = torch.ones((B, 1, L, L), dtype=torch.bool, device=device)
    keep[0, 0, 5] = False
    keep[1, 0, 64:70] = False
    tb = torch.zeros((H, L, L), device=device).requires_grad_() if bias else None
    leaves = [x.requires_grad_() for x in (q, k, v)] + ([tb] if bias else [])
    bad = do.clone()
    bad[0, 5, 0] = float("inf")
    bad[1, 66, 1] = float("nan")
    out = A.dot_product_attention(q, k, v, mask=keep, bias=tb, implementation="hip")
    want = torch.autograd.grad(out, leaves, do, retain_graph=True)
    got = torch.autograd.grad(out, leaves, bad)
    for i in (i for i in range(len(leaves)) if i != 2):
        assert torch.isfinite(want[i]).all() and torch.equal(got[i], want[i])
    assert not torch.isfinite(got[2][0, :, 0]).any() and not torch.isfinite(got[2][1, :, 1]).any()
    assert torch.equal(got[2][0, :, 1], want[2][0, :, 1])


@pytest.mark.parametrize("dtype,B,L,H,D,shift", [
    ("bf16", 2, 70, 3, 64, 0), ("f16", 1, 33, 1, 8, 0), ("f32", 2, 1, 5, 100, 0), ("f32", 3, 257, 2, 12, 0),
    ("bf16", 1, 40, 2, 256, 1)])
def test_zero_empty_rows(device, dtype, B, L, H, D, shift):
    """A copy with zeros in the rows of +inf lse, bitwise; ``shift`` starts the
    sources off 16 bytes."""
    import torch
    from probjax_amd import hip_attention as hip

    tdt = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}[dtype]
    n = B * L * H * D
    o, do = (to_dev(x, device, tdt)[shift:shift + n].view(B, L, H, D) for x in rng_normal(56, (n + 8,), (n + 8,)))
    lse = torch.zeros((B, H, L), device=device)
    for share in (0.0, 0.4, 1.0):
        lse[torch.rand(lse.shape, device=device) < share] = float("inf")
        empty = torch.isinf(lse).transpose(1, 2)[..., None]
        o_rows, do_rows = hip.zero_empty_rows(lse, o, do)
        assert torch.equal(o_rows, torch.where(empty, 0, o)) and torch.equal(do_rows, torch.where(empty, 0, do))
