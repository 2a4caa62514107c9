"""Segment ids and distance slopes: the kernels that skip and trim by segment
(extended level 2) against the general extended kernels (level 3, reached by
a ``constant`` far below a score's last bit) on the same inputs, forward and
gradients.

Both compute the same scores up to float32 rounding (the slope term is one
fused multiply-add more), so a 16-bit result may differ by one rounding step:
2^-8 (bf16) or 2^-11 (fp16) of the value, and of the largest value where terms
of a sum cancel.
"""

import math

import numpy as np
import pytest

from tests._helpers import rng_normal, to_dev, to_np

pytestmark = pytest.mark.gpu


def _ids(kind, B, n, rng):
    if kind == "sorted":  # packed documents of random lengths
        cuts = np.sort(rng.integers(0, n + 1, size=(B, 4)), axis=1)
        return (np.arange(n)[None, :, None] >= cuts[:, None, :]).sum(-1)
    if kind == "shuffled":  # ids in no order, some negative
        return rng.integers(-3, 3, size=(B, n))
    if kind == "repeated":  # a document that comes back later
        return (np.arange(n)[None] // 37) % 3 + np.zeros((B, 1), np.int64)
    return np.zeros((B, n), np.int64)  # one document


CASES = [
    # dtype, D, B, Lq, Lk, Hq, Hkv, query ids, key ids, slopes, causal, kv lengths
    ("bf16", 128, 2, 300, 300, 4, 2, "sorted", "same", None, True, None),
    ("bf16", 64, 2, 257, 257, 2, 2, "sorted", "same", None, False, [257, 100]),
    ("f16", 128, 1, 128, 320, 2, 1, "shuffled", "shuffled", None, False, None),
    ("bf16", 128, 2, 191, 129, 2, 2, "repeated", "repeated", None, True, None),
    ("bf16", 64, 1, 65, 449, 2, 1, "sorted", "disjoint", None, False, None),
    ("f16", 64, 2, 1, 130, 2, 2, "sorted", "shuffled", None, False, [130, 0]),
    ("bf16", 128, 1, 200, 200, 3, 3, "sorted", "same", "causal", True, None),
    ("bf16", 64, 2, 320, 257, 4, 2, None, None, "symmetric", False, [257, 64]),
    ("f16", 128, 1, 129, 400, 2, 2, None, None, "causal", False, None),
    ("bf16", 64, 1, 64, 64, 1, 1, "one", "same", "symmetric", False, None),
]


@pytest.mark.parametrize("dtype,D,B,Lq,Lk,Hq,Hkv,qids,kids,slopes,causal,lengths", CASES)
def test_level2_equals_general_path(device, dtype, D, B, Lq, Lk, Hq, Hkv, qids, kids, slopes, causal, lengths):
    import torch
    from probjax_amd import hip_attention as hip
    from probjax_amd import native

    rng = np.random.default_rng(81)
    tdt = torch.bfloat16 if dtype == "bf16" else torch.float16
    q, k, v, do = (to_dev(x, device, tdt) for x in rng_normal(82, (B, Lq, Hq, D), (B, Lk, Hkv, D), (B, Lk, Hkv, D),
                                                              (B, Lq, Hq, D)))
    sq = sk = None
    if qids is not None:
        sq = _ids(qids, B, Lq, rng)
        sk = sq if kids == "same" else sq.max() + 1 + _ids("sorted", B, Lk, rng) if kids == "disjoint" else \
            _ids(kids, B, Lk, rng)
        sq, sk = (torch.from_numpy(np.ascontiguousarray(x, np.int32)).to(device) for x in (sq, sk))
    sl = None if slopes is None else torch.tensor([0.5 ** (h + 1) for h in range(Hq)], device=device)
    L = None if lengths is None else torch.tensor(lengths, dtype=torch.int32, device=device)
    got = {}
    for level, constant in ((2, 0.0), (3, 1e-30)):
        m = hip.ScoreModsArgs(segment_q=sq, segment_k=sk, alibi_slopes=sl, alibi_symmetric=slopes == "symmetric",
                              constant=constant)
        print(f"level {level}: D={D} Lq={Lq} Lk={Lk} ids={qids}/{kids} slopes={slopes}", flush=True)
        kw = dict(sm_scale=1 / math.sqrt(D), causal=causal, kv_lengths=L, mods=m)
        o, lse = hip.flash_attention_fwd(q, k, v, return_lse=True, **kw)
        names = native.last_launches()
        grads = hip.flash_attention_bwd(q, k, v, o, do, lse, **kw)
        names += native.last_launches()
        E = "Bf16Fmt" if dtype == "bf16" else "F16Fmt"
        assert names == [f"flash_fwd_bf16_kernel<{E}, {D}, false, {level}>",
                         f"flash_bwd_dq_kernel<{E}, {D}, 0, {level}, 1>",
                         f"flash_bwd_dkdv_kernel<{E}, {D}, false, {level}, 1>"], names
        torch.cuda.synchronize()
        got[level] = [to_np(x) for x in (o, lse, *grads)]
    step = 2.0 ** (-8 if dtype == "bf16" else -11)
    for name, a, b in zip(("o", "lse", "dq", "dk", "dv"), got[2], got[3]):
        if name == "lse":
            np.testing.assert_array_equal(np.isposinf(a), np.isposinf(b))
            fin = np.isfinite(b)
            np.testing.assert_allclose(a[fin], b[fin], rtol=1e-5, atol=1e-5)
            continue
        assert np.isfinite(a).all()
        bound = step * (np.abs(b) + np.abs(b).max(initial=0.0))
        assert (np.abs(a - b) <= bound).all(), f"{name}: {np.abs(a - b).max()}"


@pytest.mark.parametrize("dtype,D", [("f32", 64), ("f32", 128), ("bf16", 64), ("bf16", 128)])
@pytest.mark.parametrize("cut", [1, 2, 3, 130, 133])
def test_documents_start_anywhere(device, dtype, D, cut):
    """A document whose first position is no multiple of 4, at a length that is:
    the query range of a key block starts there, and the ids are read from it."""
    import torch
    from probjax_amd import hip_attention as hip

    B, L, H = 1, 256, 2
    tdt = torch.float32 if dtype == "f32" else torch.bfloat16
    q, k, v, do = (to_dev(x, device, tdt) for x in rng_normal(83, *[(B, L, H, D)] * 4))
    ids = (torch.arange(L, device=device) >= cut).to(torch.int32)[None]
    # document by document, without ids, is the same computation
    got, kw = {}, dict(sm_scale=1 / math.sqrt(D), causal=True)
    for name, spans in (("ids", [(0, L)]), ("alone", [(0, cut), (cut, L)])):
        parts = []
        for a, b in spans:
            x = [t[:, a:b].contiguous() for t in (q, k, v)]
            m = hip.ScoreModsArgs(segment_q=ids, segment_k=ids) if name == "ids" else None
            o, lse = hip.flash_attention_fwd(*x, return_lse=True, mods=m, **kw)
            parts.append([o, *hip.flash_attention_bwd(*x, o, do[:, a:b].contiguous(), lse, mods=m, **kw)])
        got[name] = [torch.cat(t, 1).double() for t in zip(*parts)]
    # float32 sums in another order; one rounding step of bf16
    tol = 32 * 2.0 ** -24 if dtype == "f32" else 2.0 ** -8
    for a, b in zip(got["ids"], got["alone"]):
        assert float((a - b).norm() / b.norm()) <= tol
