"""The dequant bridge of the packed cache: the four slots' live rows in one
dispatch, read where they lie, equal to the oracle's dequantisation bit for
bit (one fp32 multiply, one add, one rounding), for row counts below the
capacity, every group size and type; and a cache restored from views."""

from __future__ import annotations

import numpy as np
import pytest

from conftest import np_to_torch, randn, torch_dtype, torch_to_np
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tag", ["f16", "bf16", "f32"])
@pytest.mark.parametrize("bits,gs,D", [(4, 64, 128), (8, 32, 96), (8, 128, 128), (4, 32, 64)])
@pytest.mark.parametrize("B,H,rows", [(1, 1, 1), (2, 3, 257)])
def test_bridge_equals_oracle(gpu, rng, B, H, rows, bits, gs, D, tag):
    from mlx_motif.cache import MotifGroupedQuantizedKVCache

    print(f"bridge B={B} H={H} rows={rows} bits={bits} gs={gs} D={D} {tag}", flush=True)
    raw = [randn(rng, (B, H, rows, D), tag, 3.0) for _ in range(4)]
    dt = torch_dtype(tag)
    cache = MotifGroupedQuantizedKVCache(group_size=gs, bits=bits)
    outs = cache.update_and_fetch_4(*(np_to_torch(r, dt, gpu) for r in raw))
    slots = (cache.k1, cache.k2, cache.v1, cache.v2)
    for out, slot in zip(outs, slots):
        cut = [torch_to_np(x[:, :, :rows].contiguous()) for x in slot]
        ref = O.dequantize(*cut, group_size=gs, bits=bits, out_dtype=tag)
        assert out.shape == (B, H, rows, D) and out.is_contiguous()
        np.testing.assert_array_equal(torch_to_np(out), np.asarray(ref, np.float64))


def test_restored_views_take_the_per_slot_calls(gpu, rng):
    import torch

    from mlx_motif.cache import MotifGroupedQuantizedKVCache

    raw = [np_to_torch(randn(rng, (2, 2, 300, 128), "f16"), torch.float16, gpu) for _ in range(4)]
    cache = MotifGroupedQuantizedKVCache(group_size=64, bits=4)
    want = cache.update_and_fetch_4(*raw)
    views = MotifGroupedQuantizedKVCache(group_size=64, bits=4)
    views.state, views.meta_state = cache.state, cache.meta_state
    assert not views._uniform((views.k1, views.k2, views.v1, views.v2), 128)
    got = views.update_and_fetch_4(*(r[:, :, :256] for r in raw))  # grows: whole buffers again
    for g, w in zip(got, want):
        assert torch.equal(g[:, :, :300], w)
