"""Split-KV decode on rows narrower than the kernel's width
(``pjx_splitkv_decode_rows``): bitwise what the kernel of that width gives on
explicitly zero-padded inputs, whose parity with the oracle is tested on its
own.  One and several row blocks, one and several chunks, empty and one-key
sequences, a start off 16 bytes."""

from __future__ import annotations

import pytest
import torch

from probjax_amd import native

pytestmark = pytest.mark.gpu

CASES = [  # B, Lq, S, Hq, Hkv, D, lengths, chunk
    (1, 1, 1, 1, 1, 8, None, 0),
    (2, 1, 1500, 8, 2, 80, [1500, 333], 0),
    (3, 2, 700, 24, 2, 96, [700, 0, 1], 128),
    (2, 5, 300, 20, 2, 120, [299, 31], 128),
    (2, 1, 4097, 4, 4, 40, None, 2048),
    (1, 9, 257, 16, 2, 56, None, 0),
    (1, 3, 129, 4, 1, 72, [129], 128),
]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("B,Lq,S,Hq,Hkv,D,lengths,chunk", CASES)
def test_rows_equal_explicit_padding(device, dtype, B, Lq, S, Hq, Hkv, D, lengths, chunk):
    from probjax_amd import hip_attention as hip

    g = torch.Generator().manual_seed(S + D)

    def draw(*shape, offset=0):
        x = torch.randn(*shape, generator=g).to(dtype).to(device)
        if not offset:
            return x
        buf = torch.empty(x.numel() + offset, dtype=dtype, device=device)
        buf[offset:] = x.flatten()
        return buf[offset:].view(shape)

    q, k, v = draw(B, Lq, Hq, D), draw(B, S, Hkv, D, offset=1), draw(B, S, Hkv, D)
    L = None if lengths is None else torch.tensor(lengths, dtype=torch.int32, device=device)
    W = hip.rows_width(D, Hq)
    o, lse = hip.splitkv_decode(q, k, v, sm_scale=0.3, kv_lengths=L, chunk=chunk, return_lse=True, width=W)
    nrb = {1: 1, 2: 2}.get(-(-Lq * (Hq // Hkv) // 16), 4)
    fmt = "Bf16Fmt" if dtype == torch.bfloat16 else "F16Fmt"
    assert native.last_launches()[0] == f"gqa_decode_rows_kernel<{fmt}, {W}, {nrb}>"
    pad = lambda x: torch.nn.functional.pad(x, (0, W - D))
    want, wlse = hip.splitkv_decode(pad(q), pad(k), pad(v), sm_scale=0.3, kv_lengths=L, chunk=chunk, return_lse=True)
    assert o.shape == (B, Lq, Hq, D)
    assert torch.equal(o, want[..., :D].contiguous()) and torch.equal(lse, wlse)


def test_decode_route_takes_rows(device):
    from probjax_amd import attention as A
    from probjax_amd.masks import KVLenMask

    n = torch.tensor([1200, 77], dtype=torch.int32, device=device)
    q, k, v = (torch.randn(2, t, h, 80, device=device, dtype=torch.bfloat16) for t, h in ((1, 8), (1200, 2), (1200, 2)))
    o = A.mha(q, k, v, mask=KVLenMask(n), sm_scale=0.1)
    assert native.last_launches()[0].startswith("gqa_decode_rows_kernel")
    assert torch.equal(A.splitkv_forward(q, k, v, sm_scale=0.1, kv_lengths=n), o)
    q.requires_grad_()  # with a gradient: padded, as before
    assert torch.equal(A.mha(q, k, v, mask=KVLenMask(n), sm_scale=0.1).detach(), o)
    with pytest.raises(ValueError):  # float32 rows keep the padding
        from probjax_amd import hip_attention as hip
        hip.splitkv_decode(q.detach().float(), k.float(), v.float(), sm_scale=0.1, width=128)
