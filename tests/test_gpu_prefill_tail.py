"""A layer's prompt chunk with more query blocks than CUs: whole rounds of
blocks run unsplit and the blocks of the last, partly filled round are split
over rows, with partials of those alone.

Against ``rope_split4`` and the two multi-row calls (whose query blocks fit
one round and are split all alike, or not at all), bar 2e-3 (fp16) / 2e-2
(bf16) as between any two of these routes.  The tail is part of the noise
pass, all of it with a last origin block, and a lone partial block; the plan
is checked to have one through its workspace size."""

from __future__ import annotations

import numpy as np
import pytest

from conftest import torch_dtype

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tag", ["f16", "bf16"])
@pytest.mark.parametrize("B,Hkv,gr,S,offset", [
    (3, 16, 1, 160, 2048),   # 3 + 3 blocks of 64 heads x 48: the last noise block
    (5, 8, 4, 100, 2049),    # 7 + 2 x 40: an origin block and the noise pass
    (5, 8, 4, 70, 2300),     # 5 + 2 x 40: a noise block of 6 rows
])
def test_split_tail_matches_separate_calls(gpu, B, Hkv, gr, S, offset, tag):
    import torch

    from mlx_motif import _native
    from mlx_motif.kernels import (gda_prefill_attention_from_proj, rope_split4,
                                   sdpa_dual_v_rows)

    print(f"tail B={B} Hkv={Hkv} gr={gr} S={S} offset={offset} {tag}", flush=True)
    D, dt, kv_len = 128, torch_dtype(tag), offset + S
    rows = _native.lib().motif_gda_prefill_workspace_bytes(B, S, Hkv, gr, Hkv, D, kv_len)
    assert 0 < rows < B * Hkv * (gr + 1) * S * 2 * 2 * D * 4  # fewer than every row twice
    gen = torch.Generator(device=gpu).manual_seed(5)
    new = lambda *s: torch.randn(s, generator=gen, device=gpu).to(dt)  # noqa: E731
    q, k, v = new(B, S, Hkv * (gr + 1) * D), new(B, S, 2 * Hkv * D), new(B, S, 2 * Hkv * D)
    slots = [new(B, Hkv, kv_len + 5, D) for _ in range(4)]
    other = [t.clone() for t in slots]
    scale = 1 / np.sqrt(D)
    o, n = gda_prefill_attention_from_proj(q, k, v, slots, offset, Hkv, gr, Hkv, scale)
    q1, q2, k1, k2, v1, v2 = rope_split4(q, k, v, Hkv, gr, Hkv, 1, offset, caches=other)
    tol = 2e-3 if tag == "f16" else 2e-2
    for got, want in ((o, sdpa_dual_v_rows(q1, k1, v1, v2, scale, kv_len=kv_len)),
                      (n, sdpa_dual_v_rows(q2, k2, v1, v2, scale, kv_len=kv_len))):
        assert bool(torch.isfinite(got).all())
        assert float((got.float() - want.float()).abs().max()) <= tol
    for a, b in zip(slots, other):
        assert torch.equal(a, b)
