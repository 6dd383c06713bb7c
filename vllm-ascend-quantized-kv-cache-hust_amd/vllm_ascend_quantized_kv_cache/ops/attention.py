# SPDX-License-Identifier: Apache-2.0
"""Dense TND attention on MFMA (HIP kernel ``kvq_prefill_attn``).

Stands in for the NPU fused-attention calls with ``input_layout="TND"`` of the
reference (prefill, chunked prompt rows and the dense fallback of
``pkg/methods/kivi_int4/attention_backend.py:1232-1392``; the INT8 prefill
paths of ``pkg/methods/int8_dynamic/attention_backend.py:207-368``).
"""

from __future__ import annotations

import ctypes

import numpy as np
import torch

from . import _native


#: rows (queries x query heads of a GQA group) of one tile of the kernel
TILE_ROWS = 128


def _plan(q_lens: list[int], kv_lens: list[int], hq: int, kvh: int, d: int,
          causal: bool) -> tuple[np.ndarray, int]:
    """``(int32 [cu_q | cu_k | request | tile << 16 ...], number of tiles)``: the
    cumulative lengths and the tiles in dispatch order, planned natively.  The
    lengths alone, and -1, for a batch past what a tile's packing can name."""
    batch = len(q_lens)
    lens = np.array([q_lens, kv_lens], dtype=np.int64)
    cap = int(lens[0].sum()) * (hq // kvh if kvh else 0) // TILE_ROWS + batch
    plan = np.zeros(2 * (batch + 1) + cap, dtype=np.int32)
    units = int(_native.lib().kvq_plan_prefill_attn(
        lens[0].ctypes.data, lens[1].ctypes.data, batch, hq, kvh, d, 1 if causal else 0,
        plan.ctypes.data, cap))
    if units == _native.KVQ_ERR_CAPACITY:
        plan = np.zeros(2 * (batch + 1), dtype=np.int32)
        plan[1:batch + 1] = np.cumsum(lens[0])
        plan[batch + 2:] = np.cumsum(lens[1])
        return plan, -1
    _native.check(units if units < 0 else 0, "kvq_plan_prefill_attn")
    return plan[: 2 * (batch + 1) + units], units


def _launch(q, k, v, q_lens: list[int], kv_lens: list[int], scale: float, causal: int,
            out: torch.Tensor) -> None:
    lib = _native.lib()
    hq, d = q.shape[1:]
    kvh = k.shape[1]
    batch = len(q_lens)
    dtype = _native.dtype_code(q.dtype)
    # keys and values on the 16-byte bounds of the kernel's DMA lanes
    tiled = (d in (64, 128, 256) and q.dtype != torch.float32
             and (k.data_ptr() | v.data_ptr()) % 16 == 0)
    if tiled and batch <= 128:
        # small batches: the lengths and tiles travel with the launch
        lens_t = ctypes.c_int64 * batch
        ql, kl = lens_t(*q_lens), lens_t(*kv_lens)
        nbytes = lib.kvq_prefill_attn_lens_workspace_bytes(ql, kl, batch, hq, kvh, d, causal)
        if nbytes != _native.KVQ_ERR_CAPACITY:
            _native.check(nbytes if nbytes < 0 else 0, "kvq_prefill_attn")
            ws = torch.empty(nbytes, dtype=torch.uint8, device=q.device) if nbytes else None
            rc = lib.kvq_prefill_attn_lens(
                q.data_ptr(), k.data_ptr(), v.data_ptr(), dtype, ql, kl, batch, hq, kvh, d, scale,
                causal, _native.ptr(ws), nbytes, out.data_ptr(), _native.stream_of(q))
            return _native.check(rc, "kvq_prefill_attn")
    plan, units = _plan(q_lens, kv_lens, hq, kvh, d, bool(causal))
    plan = torch.from_numpy(plan).to(q.device, non_blocking=True)
    if tiled and units >= 0:
        rc = lib.kvq_prefill_attn_planned(
            q.data_ptr(), k.data_ptr(), v.data_ptr(), dtype, plan.data_ptr(), batch, units, hq, kvh,
            d, scale, causal, out.data_ptr(), _native.stream_of(q))
    else:
        rc = lib.kvq_prefill_attn(
            q.data_ptr(), k.data_ptr(), v.data_ptr(), dtype, plan.data_ptr(),
            plan.data_ptr() + 4 * (batch + 1), batch, max(q_lens), hq, kvh, d, scale, causal,
            out.data_ptr(), _native.stream_of(q))
    return _native.check(rc, "kvq_prefill_attn")


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
    tq = query.shape[0]
    if out is None:
        out = torch.empty_like(query)
    if tq == 0 or not q_lens:
        return out
    _native.require_gpu_tensors("prefill_attention", query, key, value, out)
    if len(q_lens) != len(kv_lens):
        raise ValueError(
            f"prefill_attention: {len(q_lens)} query lengths, {len(kv_lens)} kv lengths")
    q = query.contiguous()
    k = key.contiguous()
    v = value.to(key.dtype).contiguous()
    if q.dtype != k.dtype:
        k = k.to(q.dtype)
        v = v.to(q.dtype)
    target = out if out.is_contiguous() and out.dtype == q.dtype else torch.empty_like(q)
    _launch(q, k, v, [int(n) for n in q_lens], [int(n) for n in kv_lens], float(scale),
            1 if causal else 0, target)
    if target is not out:
        out.copy_(target)
    return out


__all__ = ["prefill_attention"]
