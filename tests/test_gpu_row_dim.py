"""Head dims between the kernels' widths, taken as they lie in memory
(``pjx_flash_fwd_rows`` / ``pjx_flash_bwd_rows``), against the same call on
inputs padded with zero features: the same kernels on the same values, so every
output is bitwise equal (float32 at head dim 128 may take another kernel for
small grids; there 2e-6 of the largest value, 32 units of 2^-24)."""

import math

import numpy as np
import pytest

from tests._helpers import rng_normal, to_dev

pytestmark = pytest.mark.gpu

CASES = [
    # dtype, D, B, Lq, Lk, Hq, Hkv, causal, kv lengths, bias, extended masks
    ("bf16", 96, 2, 300, 300, 4, 2, True, None, None, None),
    ("f16", 72, 1, 129, 257, 2, 2, False, [200], None, None),
    ("bf16", 40, 2, 128, 128, 3, 1, True, None, None, "window"),
    ("f16", 8, 1, 65, 64, 2, 2, False, None, None, "segments"),
    ("bf16", 120, 1, 100, 190, 2, 1, False, None, None, "softcap"),
    ("bf16", 80, 2, 96, 132, 2, 2, False, [132, 40], "bias", None),  # the bias ring
    ("f16", 32, 1, 97, 131, 2, 2, True, None, "dbias", None),  # bias in registers
    ("bf16", 96, 1, 64, 128, 4, 4, False, None, "fold", None),
    ("bf16", 24, 1, 1024, 1024, 8, 1, True, None, None, None),  # split key blocks
    ("bf16", 96, 2, 256, 256, 300, 300, True, None, None, None),  # 32-key tiles, large grids
    ("f32", 32, 2, 100, 130, 2, 1, True, None, None, None),
    ("f32", 96, 1, 257, 100, 3, 3, False, [77], "dbias", None),
    ("f32", 56, 1, 200, 200, 2, 2, True, None, None, "segments"),
    ("f32", 80, 2, 130, 95, 140, 140, True, None, None, None),
]


def _mods(kind, B, Lq, Lk, device):
    import torch
    from probjax_amd import hip_attention as hip

    if kind == "window":
        return hip.ScoreModsArgs(window_left=37, window_right=11)
    if kind == "segments":
        ids = np.sort(np.random.default_rng(3).integers(0, 4, (B, max(Lq, Lk))), axis=1).astype(np.int32)
        q, k = (torch.from_numpy(np.ascontiguousarray(ids[:, :n])).to(device) for n in (Lq, Lk))
        return hip.ScoreModsArgs(segment_q=q, segment_k=k)
    return hip.ScoreModsArgs(softcap=7.0) if kind == "softcap" else None


@pytest.mark.parametrize("case", CASES)
def test_rows_equal_padding(device, case):
    import torch
    from probjax_amd import hip_attention as hip
    from probjax_amd import native

    dtype, D, B, Lq, Lk, Hq, Hkv, causal, lengths, bias_kind, ext = case
    print(f"rows {case}", flush=True)
    tdt = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}[dtype]
    width = hip.rows_width(D, Hq)
    assert width == (64 if D <= 64 else 128)
    narrow = [to_dev(x, device, tdt) for x in rng_normal(61, (B, Lq, Hq, D), (B, Lk, Hkv, D), (B, Lk, Hkv, D),
                                                         (B, Lq, Hq, D))]
    # a misaligned start is copied
    buf = torch.empty(narrow[0].numel() + 1, dtype=tdt, device=device)
    narrow[0] = buf[1:].view(narrow[0].shape).copy_(narrow[0])
    wide = [torch.nn.functional.pad(x, (0, width - D)) for x in narrow]
    kw = dict(sm_scale=1 / math.sqrt(D), causal=causal, mods=_mods(ext, B, Lq, Lk, device))
    if lengths is not None:
        kw["kv_lengths"] = torch.tensor(lengths, dtype=torch.int32, device=device)
    if bias_kind is not None:
        kw["bias"] = to_dev(rng_normal(62, (1, Hq, Lq, Lk), scale=0.5)[0], device, torch.float32)
    bkw = dict(bias_grad=bias_kind in ("dbias", "fold"), fold_bias_grad=bias_kind == "fold")
    got, want, names = [], [], []
    for (q, k, v, do), out, w in ((wide, want, None), (narrow, got, width)):
        o, lse = hip.flash_attention_fwd(q, k, v, return_lse=True, width=w, **kw)
        names.append(native.last_launches())
        g = hip.flash_attention_bwd(q, k, v, o, do, lse, width=w, **kw, **bkw)
        names[-1] += native.last_launches()
        out += [o, lse, *g]
    torch.cuda.synchronize()
    exact = names[0] == names[1]
    assert exact or dtype == "f32" and width == 128, names
    for name, a, b in zip(("o", "lse", "dq", "dk", "dv", "dbias"), got, want):
        if name not in ("lse", "dbias"):
            assert a.shape[-1] == D and a.is_contiguous()
            assert not b[..., D:].any()
            b = b[..., :D]
        assert torch.isfinite(a).all() or name == "lse"
        if exact:
            assert torch.equal(a, b), f"{name}: {(a - b).abs().max()}"
        else:
            assert float((a - b).abs().max()) <= 2e-6 * max(1.0, float(b.abs().max())), name


def test_api_takes_rows_without_padding(device):
    """mha over D = 96 with gradients launches the kernels on the inputs
    themselves; head dims that are no multiple of 8 are padded as before."""
    import torch
    from probjax_amd import attention as A
    from probjax_amd import hip_attention as hip
    from probjax_amd.masks import CausalMask

    assert [hip.rows_width(d, 8) for d in (8, 20, 64, 72, 128, 136)] == [64, None, 64, 128, 128, None]
    assert hip.rows_width(64, 1 << 20) is None
    for D in (96, 20):
        q, k, v, do = (to_dev(x, device, torch.bfloat16) for x in rng_normal(63, *[(1, 130, 2, D)] * 4))
        x = [t.clone().requires_grad_() for t in (q, k, v)]
        g = torch.autograd.grad(A.mha(*x, mask=CausalMask(), sm_scale=0.1), x, do)
        width = A._kernel_width(D)
        y = [torch.nn.functional.pad(t, (0, width - D)).requires_grad_() for t in (q, k, v)]
        gw = torch.autograd.grad(A.mha(*y, mask=CausalMask(), sm_scale=0.1), y,
                                 torch.nn.functional.pad(do, (0, width - D)))
        for a, b in zip(g, gw):
            assert a.shape[-1] == D and torch.equal(a, b[..., :D])
