"""Prompt chunks over the packed cache (more than 64 virtual heads per KV
head): 32-row tiles dequantised to fp16 in LDS by the workgroup that attends
them, values scaled by a power of two per workgroup and tensor.

Against the oracle with exact dequantisation, relative to the result's largest
magnitude: 2e-3 for fp16 and 2e-2 for bf16, as the slab tests' bars (outputs
rounded to 2^-11 / 2^-8 and the softmax weights and values to 2^-11).  Shapes:
the smallest chunk (65 virtual heads), 4- and 8-wave blocks, one and two column
blocks per wave, splits and none, row counts around the 32-row tile, every
group size, batch 2, no mask, rows that see no key; padding rows with infinite
scales; values and q of magnitudes past fp16's range.
"""

from __future__ import annotations

import numpy as np
import pytest

from conftest import np_to_torch, randn, torch_dtype, torch_to_np
from oracle import oracle as O

pytestmark = pytest.mark.gpu

TOL = {"f16": 2e-3, "bf16": 2e-2}


def _run(gpu, rng, B, Hq, Hkv, S, cap, kv_len, causal, bits, gs, tag, sigma=(1.0, 1.0, 1.0)):
    from mlx_motif.kernels import sdpa_dual_v_q4_rows

    print(f"chunk B={B} Hq={Hq} Hkv={Hkv} S={S} cap={cap} kv_len={kv_len} causal={causal} "
          f"bits={bits} gs={gs} {tag} sigma={sigma}", flush=True)
    dt = torch_dtype(tag)
    q = randn(rng, (B, Hq, S, 128), tag, sigma[0])
    trips = []
    for s in (sigma[1], sigma[2], sigma[2]):
        trips.append(O.quantize(randn(rng, (B, Hkv, cap, 128), tag, s), gs, bits, out_dtype=tag))
    gt = []
    for d, sc, bi in trips:
        t = [np_to_torch(d, None, gpu), np_to_torch(sc, dt, gpu), np_to_torch(bi, dt, gpu)]
        t[1][:, :, kv_len:] = float("inf")  # padding rows: never used
        t[2][:, :, kv_len:] = float("nan")
        gt.append(tuple(t))
    scale = 1 / np.sqrt(128) / (sigma[0] * sigma[1])
    y = torch_to_np(sdpa_dual_v_q4_rows(np_to_torch(q, dt, gpu), *gt, scale, group_size=gs,
                                        bits=bits, kv_len=kv_len, causal=causal))
    ref = O.sdpa_dual_v_q(q, *trips, scale, gs, bits, kv_len, causal=causal)
    assert np.isfinite(y).all()
    err = float(np.max(np.abs(y - ref))) / float(np.max(np.abs(ref)))
    assert err <= TOL[tag], err
    return y


@pytest.mark.parametrize("tag", ["f16", "bf16"])
@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("B,Hq,Hkv,S,cap,kv_len,causal,gs", [
    (1, 2, 2, 65, 96, 65, True, 64),       # 65 heads, one partial 16-column block
    (1, 8, 2, 33, 256, 31, True, 32),      # fewer keys than rows: rows without a key
    (2, 8, 2, 33, 512, 33, True, 128),
    (1, 16, 4, 129, 1028, 1000, True, 64),  # 8 waves, splits
    (1, 8, 2, 200, 300, 257, False, 32),
    (1, 4, 1, 517, 2120, 2113, True, 64),  # two column blocks per wave
])
def test_chunk_matches_oracle(gpu, rng, B, Hq, Hkv, S, cap, kv_len, causal, gs, bits, tag):
    _run(gpu, rng, B, Hq, Hkv, S, cap, kv_len, causal, bits, gs, tag)


@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("tag,sigma", [
    ("bf16", (1e6, 1e9, 1e12)), ("bf16", (1e-9, 1e-5, 1e-5)), ("f16", (1.0, 1.3e4, 1.3e4))])
def test_chunk_value_range(gpu, rng, tag, sigma, bits):
    """Magnitudes past fp16's range (bf16), and an fp16 cache near its end."""
    _run(gpu, rng, 1, 8, 2, 130, 1024, 1001, True, bits, 64, tag, sigma)


@pytest.mark.parametrize("tag", ["f16", "bf16"])
def test_chunk_split_count_forced(gpu, rng, tag):
    from mlx_motif import _native

    ys = []
    for rps in (32, 96, 4096):
        _native.set_tuning("rows_per_split", rps)
        try:
            ys.append(_run(gpu, np.random.default_rng(3), 1, 8, 2, 130, 1024, 1001, True, 8, 64,
                           tag))
        finally:
            _native.set_tuning("rows_per_split", 0)
    for y in ys[1:]:
        assert float(np.max(np.abs(y - ys[0]))) <= TOL[tag]
