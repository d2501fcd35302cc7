"""The fused decode step's short contexts: one split per KV head, whose
workgroup applies the GDA epilogue, against the same step in forced 64-row
splits with the merge launch.  Both round o and n to the type before the
epilogue, so they differ by roundings of equal sums only: 2e-3 (fp16) and 2e-2
(bf16), the bars between any two routes of the step.  One row, tile and
workgroup edges, the last length with one split and the first without, head
layouts with idle columns and several origin heads per wave."""

from __future__ import annotations

import numpy as np
import pytest

from conftest import torch_dtype

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tag", ["f16", "bf16"])
@pytest.mark.parametrize("bits", [0, 4, 8])
@pytest.mark.parametrize("gr", [1, 4, 7])
@pytest.mark.parametrize("kv_len", [1, 16, 64, 65, 128, 129])
def test_one_split_matches_merged_splits(gpu, kv_len, gr, bits, tag):
    import torch

    from mlx_motif import _native
    from mlx_motif.kernels import (gda_decode_attention_from_proj,
                                   gda_decode_attention_q4_from_proj, quantize)

    B, H, D, cap, dt = 2, 4, 128, 260, torch_dtype(tag)
    print(f"one split kv_len={kv_len} gr={gr} bits={bits} {tag}", flush=True)
    gen = torch.Generator(device=gpu).manual_seed(kv_len)
    new = lambda *s: torch.randn(s, generator=gen, device=gpu).to(dt)  # noqa: E731
    q, k, v = new(B, 1, H * (gr + 1) * D), new(B, 1, 2 * H * D), new(B, 1, 2 * H * D)
    slots = [new(B, H, cap, D) for _ in range(4)]
    w, lam = new(2 * D), torch.tensor([0.4], device=gpu)
    if bits:
        slots = [quantize(s, 64, bits) for s in slots]

    def step():
        if bits:
            return gda_decode_attention_q4_from_proj(q, k, v, *slots, 1 / np.sqrt(D), w, lam, 0.2,
                                                     gr, kv_len - 1, 64, bits)
        return gda_decode_attention_from_proj(q, k, v, *slots, 1 / np.sqrt(D), w, lam, 0.2, gr,
                                              kv_len - 1)

    y = step()
    _native.set_tuning("rows_per_split", 64)
    try:
        ref = step()
    finally:
        _native.set_tuning("rows_per_split", 0)
    assert bool(torch.isfinite(y).all())
    err = (y.float() - ref.float()).abs().max() / ref.float().abs().max()
    assert float(err) <= (2e-3 if tag == "f16" else 2e-2)
