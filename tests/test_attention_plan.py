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
    units = [tuple(u) for u in plan[2 * (b + 1):].reshape(-1, 2).tolist()]
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


def test_plan_refuses_unmatched_lengths():
    from vllm_ascend_quantized_kv_cache.ops.attention import _plan

    with pytest.raises(ValueError, match="query lengths"):
        _plan([1, 2], [1], 8, 8, 128, True)
    with pytest.raises(RuntimeError, match="rejected"):
        _plan([1], [-1], 8, 8, 128, True)
