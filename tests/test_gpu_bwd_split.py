"""dK / dV with a key block's steps spread over several workgroups
(``pjx_flash_bwd_split_workspace_size``): against the one-workgroup result of
the same inputs and the oracle's rule for which sizes split.

Both sum the same float32 terms, in another order, and round once to 16 bits:
they differ by at most one rounding step of the value (2^-8 in bf16, 2^-11 in
fp16), or of the largest value where terms cancel.
"""

import math

import numpy as np
import pytest

from tests._helpers import rng_normal, to_dev, to_np

CASES = [
    # dtype, D, B, Lq, Lk, Hq, Hkv, causal, kv lengths, bias, splits
    ("bf16", 128, 1, 1024, 1024, 8, 2, True, None, False, 4),
    ("f16", 64, 2, 1000, 777, 8, 1, False, [777, 130], False, 8),  # ragged, an empty key block
    ("bf16", 64, 1, 4033, 4033, 8, 8, True, None, False, 2),
    ("bf16", 128, 1, 513, 129, 32, 4, False, None, True, 4),
    ("bf16", 64, 1, 2048, 1, 2, 1, False, None, False, 4),  # one key
]


def _size(lib, case):
    dtype, D, B, Lq, Lk, Hq, Hkv, causal = case[:8]
    return lib.pjx_flash_bwd_split_workspace_size(2 if dtype == "f16" else 1, B, Hq, Hkv, Lq, Lk, D, int(causal))


@pytest.mark.parametrize("case", CASES)
def test_split_workspace_size(case):
    from probjax_amd import native

    lib = native.load()
    dtype, D, B, Lq, Lk, Hq, Hkv, causal, _, _, ns = case
    lead = -(-lib.pjx_flash_bwd_workspace_size(B, Hq, Lq) // 256) * 256
    assert _size(lib, case) == lead + ns * 8 * B * Lk * Hkv * D
    # not in float32, at head dim 256, for blocks that already fill the device or with few steps
    assert lib.pjx_flash_bwd_split_workspace_size(0, B, Hq, Hkv, Lq, Lk, D, 1) == 0
    assert lib.pjx_flash_bwd_split_workspace_size(1, B, Hq, Hkv, Lq, Lk, 256, 1) == 0
    assert lib.pjx_flash_bwd_split_workspace_size(1, 4, 16, 16, 4096, 4096, 128, 1) == 0
    assert lib.pjx_flash_bwd_split_workspace_size(1, 1, 2, 2, 300, 300, 128, 1) == 0


@pytest.mark.gpu
@pytest.mark.parametrize("case", CASES)
def test_split_equals_one_workgroup(device, case):
    import torch
    from probjax_amd import native
    from probjax_amd.hip_attention import flash_attention_bwd, flash_attention_fwd

    dtype, D, B, Lq, Lk, Hq, Hkv, causal, lengths, with_bias, ns = case
    print(f"split {case}", flush=True)
    tdt = torch.bfloat16 if dtype == "bf16" else torch.float16
    q, k, v, do = (to_dev(x, device, tdt) for x in rng_normal(71, (B, Lq, Hq, D), (B, Lk, Hkv, D), (B, Lk, Hkv, D),
                                                              (B, Lq, Hq, D)))
    kw = dict(sm_scale=1 / math.sqrt(D), causal=causal)
    if lengths is not None:
        kw["kv_lengths"] = torch.tensor(lengths, dtype=torch.int32, device=device)
    if with_bias:
        kw["bias"] = to_dev(rng_normal(72, (1, Hq, Lq, Lk), scale=0.5)[0], device, torch.float32)
    o, lse = flash_attention_fwd(q, k, v, return_lse=True, **kw)
    got = flash_attention_bwd(q, k, v, o, do, lse, **kw)
    names = native.last_launches()
    plain = torch.empty(native.load().pjx_flash_bwd_workspace_size(B, Hq, Lq), dtype=torch.uint8, device=device)
    want = flash_attention_bwd(q, k, v, o, do, lse, workspace=plain, **kw)
    assert len(names) == 3 and names[2].startswith("bwd_split_reduce_kernel"), names
    assert len(native.last_launches()) == 2
    again = flash_attention_bwd(q, k, v, o, do, lse, **kw)
    torch.cuda.synchronize()
    step = 2.0 ** (-8 if dtype == "bf16" else -11)
    assert torch.equal(got[0], want[0])
    for name, a, b, c in zip(("dk", "dv"), got[1:], want[1:], again[1:]):
        assert torch.equal(a, c), name
        a, b = to_np(a), to_np(b)
        assert (np.abs(a - b) <= step * (np.abs(b) + np.abs(b).max())).all(), f"{name}: {np.abs(a - b).max()}"
        if lengths is not None:
            for i, n in enumerate(lengths):
                assert not a[i, n:].any()
