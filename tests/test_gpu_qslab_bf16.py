"""bf16 verify slabs over the packed cache on producer / consumer waves, the
values and q rows scaled into fp16 by powers of two: against the oracle with
exact dequantisation, relative to the result's largest magnitude, at the bf16
bar of the slab and chunk tests (2e-2).  17, 20, 33 and 64 virtual heads, every
group size, split and unsplit rows, rows past the last step, no mask, values
past fp16's range, poisoned padding rows."""

from __future__ import annotations

import pytest

from test_gpu_qprefill import _run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("B,Hq,Hkv,S,cap,kv_len,causal,gs,sigma", [
    (1, 32, 8, 5, 1024, 1001, True, 64, (1.0, 1.0, 1.0)),
    (1, 4, 4, 17, 320, 33, True, 32, (1.0, 1.0, 1.0)),
    (2, 12, 4, 11, 2048, 2048, True, 128, (1.0, 1.0, 1.0)),
    (1, 64, 8, 8, 512, 500, False, 64, (1.0, 1.0, 1.0)),
    (40, 32, 8, 5, 96, 64, True, 64, (1.0, 1.0, 1.0)),  # one split: writes y
    (1, 32, 8, 5, 1024, 999, True, 64, (1e6, 1e9, 1e12)),
    (1, 32, 8, 8, 1024, 999, True, 64, (1e-9, 1e-5, 1e-5)),
])
def test_bf16_slab_matches_oracle(gpu, rng, B, Hq, Hkv, S, cap, kv_len, causal, gs, sigma, bits):
    _run(gpu, rng, B, Hq, Hkv, S, cap, kv_len, causal, bits, gs, "bf16", sigma)
