# SPDX-License-Identifier: Apache-2.0
"""The dense attention's tile plan (host only): every tile of 128 rows once,
long tiles first, cumulative lengths beside it."""

from __future__ import annotations

import numpy as np
import pytest

from vllm_ascend_quantized_kv_cache.ops import _native

pytestmark = pytest.mark.skipif(not _native.library_path().exists(),
                                reason="libkvq_hip.so not built")


@pytest.mark.parametrize("hq,kvh,d", [(40, 8, 128), (8, 1, 256), (7, 7, 64)])
@pytest.mark.parametrize("q_lens,kv_lens", [
    ([1, 37, 130, 64], [1, 37, 300, 64]),          # one group: longest tile first
    ([2048, 5, 0, 700], [30000, 5, 9, 90000]),     # histories past an L2: requests apart
    ([5, 3], [0, 2]),                              # no keys; fewer keys than queries
    ([0], [4]),
])
@pytest.mark.parametrize("causal", [True, False])
def test_plan_covers_every_tile_once(hq, kvh, d, q_lens, kv_lens, causal):
    from vllm_ascend_quantized_kv_cache.ops.attention import TILE_ROWS, _plan

    rep = hq // kvh
    plan, n = _plan(q_lens, kv_lens, hq, kvh, d, causal)
    b = len(q_lens)
    assert plan[: b + 1].tolist() == [0, *np.cumsum(q_lens)]
    assert plan[b + 1: 2 * (b + 1)].tolist() == [0, *np.cumsum(kv_lens)]
    units = [(u & 0xFFFF, u >> 16) for u in plan[2 * (b + 1):].tolist()]
    want = [(i, t) for i, m in enumerate(q_lens) for t in range(-(-m * rep // TILE_ROWS))]
    assert n == len(units) and sorted(units) == want

    def blocks(i, t):
        last = (min((t + 1) * TILE_ROWS, q_lens[i] * rep) - 1) // rep
        end = min(kv_lens[i], kv_lens[i] - q_lens[i] + last + 1) if causal else kv_lens[i]
        return -(-max(end, 0) // 64)

    apart = sum(kv_lens) * d * 4 * max(1, kvh // 8) > 8 << 20
    cost = [blocks(*u) for u in units]
    if apart:  # a request's tiles together, the long ones first
        seen = [u[0] for u in units]
        assert seen == sorted(seen, key=lambda i: -q_lens[i] * kv_lens[i])
        for i in set(seen):
            mine = [c for c, u in zip(cost, units) if u[0] == i]
            assert mine == sorted(mine, reverse=True)
    else:
        assert cost == sorted(cost, reverse=True)


def test_plan_refuses_negative_lengths():
    from vllm_ascend_quantized_kv_cache.ops.attention import _plan

    with pytest.raises(RuntimeError, match="rejected"):
        _plan([1], [-1], 8, 8, 128, True)


def test_plan_past_the_packed_range_keeps_the_lengths():
    from vllm_ascend_quantized_kv_cache.ops.attention import _plan

    many = [1] * 70000  # requests past 16 bits: the grid without a unit list
    plan, n = _plan(many, many, 1, 1, 128, True)
    assert n == -1
    assert plan[:70001].tolist() == list(range(70001)) == plan[70001:].tolist()


def _lens_call(name, q_lens, kv_lens, *args):
    import ctypes

    arr = ctypes.c_int64 * len(q_lens)
    return getattr(_native.lib(), name)(arr(*q_lens), arr(*kv_lens), len(q_lens), *args)


# the segments follow from the tiles, their key blocks and their rows: what fits the
# chip's slots (two workgroups a CU, one at 256 dims), of at least 4 blocks of 64
# keys, at most 32, where the blocks saved outweigh the partials' way through memory
SEGMENTS = [
    ([16], [8192], 8, 1, 128, 256, 26),           # one tile of 128 blocks: 5 blocks each
    ([16], [8192], 8, 1, 128, 8, 16),             # ... 16 slots
    ([16], [8192], 8, 1, 256, 8, 8),              # ... 8
    ([16] * 3, [8192] * 3, 8, 1, 128, 8, 5),      # three tiles share 16 slots
    ([16], [2000], 8, 1, 128, 256, 8),            # 32 blocks: 8 segments of 4
    ([16], [500], 8, 1, 128, 256, 1),             # 8 blocks: two segments save 4
    ([16], [1024], 8, 1, 128, 256, 4),            # 16 blocks: four segments save 12
    ([1024] * 6, [10240] * 6, 8, 1, 128, 256, 1),   # 384 tiles on 512 slots: one each
    ([1024] * 4, [10240] * 4, 8, 1, 128, 256, 2),   # 256 tiles: two each
    ([1024] * 4, [10240] * 4, 8, 1, 256, 256, 1),   # 256 tiles on 256 slots
    ([700] * 4, [10240] * 4, 40, 8, 128, 256, 1),   # 112 tiles of 8 kv heads: more than slots
    ([0, 0], [5, 5], 8, 1, 128, 256, 1),
    ([60] * 8, [1024] * 8, 64, 8, 128, 256, 1),   # 16 MB of partials a segment for 8 blocks
    ([60] * 8, [6000] * 8, 64, 8, 128, 256, 2),   # ... for 47
    ([60] * 3, [1024] * 3, 64, 8, 128, 256, 1),   # 6 MB a segment, 16 blocks
    ([60] * 3, [2048] * 3, 64, 8, 128, 256, 3),   # ... 32
    ([60] * 3, [1024] * 3, 8, 8, 128, 256, 4),    # 0.7 MB
    ([60] * 8, [768] * 8, 8, 8, 256, 256, 3),     # 4 MB, 12 blocks of 256 dims
]


@pytest.mark.parametrize("q_lens,kv_lens,hq,kvh,d,cus,segs", SEGMENTS)
def test_segments_follow_the_rule(q_lens, kv_lens, hq, kvh, d, cus, segs):
    got = _lens_call("kvq_prefill_attn_segments", q_lens, kv_lens, hq, kvh, d, 1, cus)
    assert got == segs
    # without a device, or one of unknown size, the keys stay whole
    assert _lens_call("kvq_prefill_attn_segments", q_lens, kv_lens, hq, kvh, d, 1, 0) == 1


def test_segments_of_a_plan_past_the_argument():
    """8 x 2048 queries of 5 heads a kv head: 640 tiles, and the argument holds 482."""
    for name, extra in (("kvq_prefill_attn_segments", (256,)),
                        ("kvq_prefill_attn_lens_workspace_bytes", ())):
        got = _lens_call(name, [2048] * 8, [10240] * 8, 40, 8, 128, 1, *extra)
        assert got == _native.KVQ_ERR_CAPACITY


@pytest.mark.gpu
@pytest.mark.parametrize("q_lens,kv_lens,hq,kvh,d,cus,segs", SEGMENTS)
def test_workspace_follows_the_cut(gpu_device, q_lens, kv_lens, hq, kvh, d, cus, segs):
    """Rows of whole tiles, D + 2 floats each, per segment; none for whole keys."""
    import torch

    cus = torch.cuda.get_device_properties(0).multi_processor_count
    segs = _lens_call("kvq_prefill_attn_segments", q_lens, kv_lens, hq, kvh, d, 1, cus)
    tiles = sum(-(-m * (hq // kvh) // 128) for m in q_lens)
    got = _lens_call("kvq_prefill_attn_lens_workspace_bytes", q_lens, kv_lens, hq, kvh, d, 1)
    assert got == (tiles * kvh * segs * 128 * (d + 2) * 4 if segs > 1 else 0)
