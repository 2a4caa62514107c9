"""More (batch, head) pairs than one launch of 512-thread workgroups counts in 32
bits of work-items (2^23): attention over a great many small sets.

The first and last pairs are compared with float64: float32 results to 32 units
of 2^-24 in 2-norm, as elsewhere; 16-bit gradients of the bias, sums of a few
products of values rounded to 2^-9, to 2^-7.
"""

import pytest

pytestmark = pytest.mark.gpu
PAIRS = (1 << 23) + 9
ENDS = [slice(0, 500), slice((1 << 23) - 500, PAIRS)]


def _randn(device, dtype, *shapes):
    import torch

    gen = torch.Generator(device=device).manual_seed(97)
    return [torch.randn(s, generator=gen, device=device, dtype=dtype) for s in shapes]


def _grads64(q, k, v, do, scale, bias=None):
    """float64 output and gradients of one-head sets [B, L, 1, D]."""
    import torch

    x = [t.double().requires_grad_() for t in (q, k, v)] + ([] if bias is None else [bias.double().requires_grad_()])
    s = torch.einsum("bqhd,bkhd->bhqk", x[0], x[1]) * scale
    if bias is not None:
        s = s + x[3]
    o = torch.einsum("bhqk,bkhd->bqhd", torch.softmax(s, -1), x[2])
    return [o.detach(), *torch.autograd.grad(o, x, do.double())]


def _rel(a, b):
    return float((a.double() - b).norm() / b.norm())


def test_float32(device):
    import torch
    from probjax_amd.hip_attention import flash_attention_bwd, flash_attention_fwd

    D = 64
    q, k, v, do = _randn(device, torch.float32, (PAIRS, 1, 1, D), (PAIRS, 2, 1, D), (PAIRS, 2, 1, D), (PAIRS, 1, 1, D))
    kw = dict(sm_scale=D ** -0.5)
    print("float32, 2^23 + 9 pairs", flush=True)
    o, lse = flash_attention_fwd(q, k, v, return_lse=True, **kw)
    got = [o, *flash_attention_bwd(q, k, v, o, do, lse, **kw)]
    for e in ENDS:
        want = _grads64(q[e], k[e], v[e], do[e], D ** -0.5)
        errs = [_rel(g[e], w) for g, w in zip(got, want)]
        print(f"  rel {errs}", flush=True)
        assert max(errs) <= 32 * 2.0 ** -24, errs


def test_bias_gradient(device):
    import torch
    from probjax_amd.hip_attention import flash_attention_bwd, flash_attention_fwd

    D = 128
    q, k, v, do = _randn(device, torch.bfloat16, (PAIRS, 1, 1, D), (PAIRS, 2, 1, D), (PAIRS, 2, 1, D), (PAIRS, 1, 1, D))
    bias, = _randn(device, torch.float32, (PAIRS, 1, 1, 2))
    kw = dict(sm_scale=D ** -0.5, bias=bias)
    print("bias gradient, 2^23 + 9 pairs", flush=True)
    o, lse = flash_attention_fwd(q, k, v, return_lse=True, **kw)
    db = flash_attention_bwd(q, k, v, o, do, lse, bias_grad=True, fold_bias_grad=True, **kw)[3]
    for e in ENDS:
        want = _grads64(q[e], k[e], v[e], do[e], D ** -0.5, bias[e])[4]
        assert _rel(db[e], want) <= 2.0 ** -7


def test_rows_without_a_key(device):
    import torch
    from probjax_amd import hip_attention as hip

    D = 64
    v, out = _randn(device, torch.bfloat16, (PAIRS, 2, 1, D), (PAIRS, 1, 1, D))
    lse = torch.zeros(PAIRS, 1, 1, device=device)
    lse[::3] = float("inf")
    empty = torch.isinf(lse[:, 0, 0])
    print("rows without a key, 2^23 + 9 pairs", flush=True)
    dst = out.clone()
    hip.empty_rows(lse, v, dst, grad=False)
    mean = v.float().mean(1, keepdim=True).bfloat16()
    assert torch.equal(dst[empty], mean[empty]) and torch.equal(dst[~empty], out[~empty])
    dv = v.clone()
    hip.empty_rows(lse, out, dv, grad=True)
    want = (v.float() + out.float() / 2).bfloat16()
    assert torch.equal(dv[empty], want[empty]) and torch.equal(dv[~empty], v[~empty])


def test_float32_row_of_many_heads(device):
    """Rows of all heads so long that 8 of them are more than 32-bit offsets hold."""
    import torch
    from probjax_amd.hip_attention import flash_attention_fwd

    D, L, H = 64, 10, (1 << 21) + (1 << 19)
    q, k, v = _randn(device, torch.float32, (1, 1, H, D), (1, L, H, D), (1, L, H, D))
    kw = dict(sm_scale=D ** -0.5)
    print("float32, 2.6 million heads", flush=True)
    lengths = torch.tensor([L - 1], dtype=torch.int32, device=device)
    o = flash_attention_fwd(q, k, v, kv_lengths=lengths, **kw)
    for e in (slice(0, 500), slice(H // 2, H // 2 + 500), slice(H - 500, H)):
        x = [t[0, :L - 1, e].transpose(0, 1).double() for t in (q, k, v)]
        s = torch.matmul(x[1], x[0].transpose(1, 2)) * D ** -0.5
        assert _rel(o[0, 0, e], (torch.softmax(s, 1) * x[2]).sum(1)) <= 32 * 2.0 ** -24
