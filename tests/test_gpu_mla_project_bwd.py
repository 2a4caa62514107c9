"""Gradients of the latent's up-projection (``pjx_mla_project_bwd``) against the
same products in float64.  Sizes at the edges of its tiles: 64 rows x 64 rank
entries (dcache, whole or in channel splits), 128 channels x 128 rank entries and one or several row splits
(dW); head dims below the width."""

from __future__ import annotations

import pytest
import torch

from probjax_amd import native

pytestmark = pytest.mark.gpu

CASES = [  # B, S, H, R, qk_dim, v_dim, width
    (1, 1, 1, 8, 8, 8, 64),
    (1, 63, 1, 56, 64, 40, 64),
    (2, 65, 3, 64, 64, 64, 64),
    (1, 129, 2, 136, 72, 128, 128),
    (3, 333, 2, 512, 192, 128, 256),
    (2, 2049, 8, 128, 64, 64, 64),
    (1, 100, 17, 72, 64, 64, 64),
    (1, 200, 12, 128, 128, 96, 128),
]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("B,S,H,R,dk,dv,width", CASES)
def test_projection_gradients_match_float64(device, dtype, B, S, H, R, dk, dv, width):
    from probjax_amd import hip_attention as hip

    g = torch.Generator().manual_seed(B * 1000 + S + R)
    draw = lambda *shape: torch.randn(*shape, generator=g, dtype=torch.float32).to(dtype).to(device)
    cache, wk, wv = draw(B, S, R), draw(H, dk, R), draw(H, dv, R)
    dK, dV = draw(B, S, H, width), draw(B, S, H, width)
    # channels past the head dims carry no part of the result
    dK[..., dk:] = float("nan")
    dV[..., dv:] = float("inf")
    assert hip.mla_project_bwd_supported(cache, wk, wv, width)
    got = hip.mla_project_bwd(cache, wk, wv, dK, dV)
    names = [n.split("<")[0] for n in native.last_launches()]
    tiles = ((B * S + 63) // 64) * ((R + 63) // 64)
    split = tiles < 256 and min(512 // tiles, H * width // 32 // 16) > 1
    assert names == (["mla_project_dcache_kernel"] + ["mla_project_dcache_sum_kernel"] * split
                     + ["mla_project_dw_kernel", "mla_project_dw_sum_kernel"])
    again = hip.mla_project_bwd(cache, wk, wv, dK, dV)

    c, a, b = (t.double().cpu() for t in (cache, dK[..., :dk], dV[..., :dv]))
    k, v = wk.double().cpu(), wv.double().cpu()
    rows = lambda t: t.reshape(B * S, -1)
    parts = [
        (rows(a) @ k.reshape(H * dk, R) + rows(b) @ v.reshape(H * dv, R),
         rows(a).abs() @ k.reshape(H * dk, R).abs() + rows(b).abs() @ v.reshape(H * dv, R).abs(), H * (dk + dv)),
        (rows(a).T @ rows(c), rows(a).abs().T @ rows(c).abs(), B * S),
        (rows(b).T @ rows(c), rows(b).abs().T @ rows(c).abs(), B * S),
    ]
    # One rounding to the format (half its spacing) plus a float32 sum of n
    # exact products: at most n units of 2^-23 of the sum of magnitudes.
    half = 2.0 ** -9 if dtype == torch.bfloat16 else 2.0 ** -12
    for x, y, (want, mag, n) in zip(got, again, parts):
        assert torch.equal(x, y)  # the splits are added in a fixed order
        err = (x.double().cpu().reshape(want.shape) - want).abs()
        assert bool((err <= 2 * half * want.abs() + n * 2.0 ** -23 * mag + 2.0 ** -24).all()), err.max()


def test_unaligned_ranks_and_dims_keep_the_general_products(device):
    from probjax_amd import hip_attention as hip

    t = lambda *shape: torch.zeros(*shape, dtype=torch.bfloat16, device=device)
    assert not hip.mla_project_bwd_supported(t(1, 4, 12), t(2, 64, 12), t(2, 64, 12), 64)
    assert not hip.mla_project_bwd_supported(t(1, 4, 16), t(2, 60, 16), t(2, 64, 16), 64)
    assert not hip.mla_project_bwd_supported(t(1, 4, 16).float(), t(2, 64, 16), t(2, 64, 16), 64)
