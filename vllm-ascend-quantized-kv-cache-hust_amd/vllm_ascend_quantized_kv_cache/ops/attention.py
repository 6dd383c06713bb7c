# SPDX-License-Identifier: Apache-2.0
"""Dense TND attention on MFMA (HIP kernel ``kvq_prefill_attn``).

Stands in for the NPU fused-attention calls with ``input_layout="TND"`` of the
reference (prefill, chunked prompt rows and the dense fallback of
``pkg/methods/kivi_int4/attention_backend.py:1232-1392``; the INT8 prefill
paths of ``pkg/methods/int8_dynamic/attention_backend.py:207-368``).
"""

from __future__ import annotations

import numpy as np
import torch

from . import _native


#: rows (queries x query heads of a GQA group) of one tile of the kernel
TILE_ROWS = 128


def _plan(q_lens, kv_lens, hq: int, kvh: int, d: int, causal: bool) -> tuple[np.ndarray, int]:
    """``(int32 [cu_q | cu_k | (request, tile) ...], number of tiles)``: the
    cumulative lengths and the tiles in dispatch order, planned natively."""
    if len(q_lens) != len(kv_lens):
        raise ValueError(
            f"prefill_attention: {len(q_lens)} query lengths, {len(kv_lens)} kv lengths")
    lens = np.array([[int(n) for n in q_lens], [int(n) for n in kv_lens]], dtype=np.int64)
    batch = lens.shape[1]
    rep = hq // kvh if kvh else 0
    cap = int(lens[0].sum()) * rep // TILE_ROWS + batch
    plan = np.empty(2 * (batch + 1) + 2 * cap, dtype=np.int32)
    units = int(_native.lib().kvq_plan_prefill_attn(
        lens[0].ctypes.data, lens[1].ctypes.data, batch, hq, kvh, d, 1 if causal else 0,
        plan.ctypes.data, cap))
    _native.check(units if units < 0 else 0, "kvq_plan_prefill_attn")
    return plan[: 2 * (batch + 1 + units)], units


def prefill_attention(
    query: torch.Tensor,
    key: torch.Tensor,
    value: torch.Tensor,
    q_lens: list[int],
    kv_lens: list[int],
    scale: float,
    causal: bool,
    out: torch.Tensor | None = None,
) -> torch.Tensor:
    """Per-request attention over TND tensors.

    ``query [sum q_lens, Hq, D]``, ``key/value [sum kv_lens, KVH, D]``; query
    row ``i`` of a request is kv position ``kv_len - q_len + i``.
    """
    tq, hq, d = query.shape
    kvh = key.shape[1]
    if out is None:
        out = torch.empty_like(query)
    if tq == 0 or not q_lens:
        return out
    _native.require_gpu_tensors("prefill_attention", query, key, value, out)
    q = query.contiguous()
    k = key.contiguous()
    v = value.to(key.dtype).contiguous()
    if q.dtype != k.dtype:
        k = k.to(q.dtype)
        v = v.to(q.dtype)
    target = out if out.is_contiguous() and out.dtype == q.dtype else torch.empty_like(q)
    plan, units = _plan(q_lens, kv_lens, hq, kvh, d, causal)
    batch = len(q_lens)
    plan = torch.from_numpy(plan).to(query.device, non_blocking=True)
    if d in (64, 128, 256) and q.dtype != torch.float32:
        rc = _native.lib().kvq_prefill_attn_planned(
            _native.ptr(q), _native.ptr(k), _native.ptr(v), _native.dtype_code(q.dtype),
            _native.ptr(plan), batch, units, hq, kvh, d, float(scale), 1 if causal else 0,
            _native.ptr(target), _native.stream_of(q),
        )
    else:
        rc = _native.lib().kvq_prefill_attn(
            _native.ptr(q), _native.ptr(k), _native.ptr(v), _native.dtype_code(q.dtype),
            _native.ptr(plan), _native.ptr(plan) + 4 * (batch + 1), batch,
            max(int(x) for x in q_lens), hq, kvh, d, float(scale), 1 if causal else 0,
            _native.ptr(target), _native.stream_of(q),
        )
    _native.check(rc, "kvq_prefill_attn")
    if target is not out:
        out.copy_(target)
    return out


__all__ = ["prefill_attention"]
