# SPDX-License-Identifier: Apache-2.0
"""GPU parity of the MFMA dense (prefill / chunked) attention kernel.

Checked against the oracle's fp32 softmax attention within atol/rtol 1e-2 on
ragged batches, GQA ratios, causal and full masks, and query chunks that sit
at the end of a longer key range (chunked prefill with history).
"""

from __future__ import annotations

import pytest
import torch

from oracle import kvq_oracle as ref

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("d", [64, 128, 256])
@pytest.mark.parametrize("hq,kvh", [(8, 8), (40, 8), (8, 1)])
@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_prefill_attention_matches_oracle(gpu_device, d, hq, kvh, causal, dtype):
    from vllm_ascend_quantized_kv_cache.ops.attention import prefill_attention

    g = torch.Generator().manual_seed(d + hq)
    q_lens = [1, 37, 130, 64]
    kv_lens = [1, 37, 300, 64] if causal else [5, 37, 300, 64]  # request 2: chunk with history
    q = torch.randn(sum(q_lens), hq, d, generator=g).to(dtype)
    k = (torch.randn(sum(kv_lens), kvh, d, generator=g) * 2).to(dtype)
    v = torch.randn(sum(kv_lens), kvh, d, generator=g).to(dtype)
    scale = d ** -0.5
    want = ref.attention(q, k, v, q_lens, kv_lens, scale, causal)
    got = prefill_attention(
        q.to(gpu_device), k.to(gpu_device), v.to(gpu_device), q_lens, kv_lens, scale, causal
    )
    torch.testing.assert_close(got.float().cpu(), want, atol=1e-2, rtol=1e-2)


def test_prefill_attention_chunk_after_int4_history(gpu_device):
    """Config-4 shape in miniature: a new chunk attending to a longer prefix."""
    from vllm_ascend_quantized_kv_cache.ops.attention import prefill_attention

    g = torch.Generator().manual_seed(3)
    hq, kvh, d = 40, 8, 128
    q_lens = [256, 128]
    kv_lens = [1280, 640]
    q = torch.randn(sum(q_lens), hq, d, generator=g).to(torch.bfloat16)
    k = (torch.randn(sum(kv_lens), kvh, d, generator=g) * torch.exp(torch.randn(kvh, d, generator=g)))
    k = k.to(torch.bfloat16)
    v = torch.randn(sum(kv_lens), kvh, d, generator=g).to(torch.bfloat16)
    want = ref.attention(q, k, v, q_lens, kv_lens, d ** -0.5, True)
    got = prefill_attention(
        q.to(gpu_device), k.to(gpu_device), v.to(gpu_device), q_lens, kv_lens, d ** -0.5, True
    )
    torch.testing.assert_close(got.float().cpu(), want, atol=1e-2, rtol=1e-2)


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_prefill_attention_growing_and_shrinking_row_maxima(gpu_device, d, dtype):
    """Scores that climb by more than the lazy-offset threshold (8 in log2
    units) every 64-key block for half the heads, and fall for the others:
    the rescale branch runs on almost every block of the first half, never
    after the first block of the second, and both match the oracle."""
    from vllm_ascend_quantized_kv_cache.ops.attention import prefill_attention

    g = torch.Generator().manual_seed(11 + d)
    hq, kvh = 8, 2
    q_lens = [96, 200]
    kv_lens = [300, 200]
    n = sum(kv_lens)
    u = torch.randn(kvh, d, generator=g)
    u = u / u.norm(dim=1, keepdim=True)  # unit direction per kv head
    pos = torch.cat([torch.arange(L, dtype=torch.float32) for L in kv_lens])
    # raw score of key j against a query along u: 8 * (+-0.5 j + noise); with
    # scale d^-0.5 that moves the log2 exponent by about 23 / sqrt(d / 64) per block
    sign = torch.tensor([1.0, -1.0])
    k = (u[None] * (sign[None, :, None] * 0.5 * pos[:, None, None])
         + 0.05 * torch.randn(n, kvh, d, generator=g))
    q = 8.0 * u.repeat_interleave(hq // kvh, dim=0)[None] + 0.05 * torch.randn(
        sum(q_lens), hq, d, generator=g)
    v = torch.randn(n, kvh, d, generator=g)
    q, k, v = q.to(dtype), k.to(dtype), v.to(dtype)
    scale = d ** -0.5
    want = ref.attention(q, k, v, q_lens, kv_lens, scale, True)
    got = prefill_attention(
        q.to(gpu_device), k.to(gpu_device), v.to(gpu_device), q_lens, kv_lens, scale, True
    )
    torch.testing.assert_close(got.float().cpu(), want, atol=1e-2, rtol=1e-2)


@pytest.mark.parametrize("d", [64, 128, 256])
@pytest.mark.parametrize("hq,kvh", [(10, 2), (7, 1), (3, 3)])
def test_prefill_attention_head_rows_across_tiles(gpu_device, d, hq, kvh):
    """Rows of a GQA group's heads share a tile: groups that do not divide the
    128-row tile, requests that end inside a wave, next to an empty one, one
    without keys and one with fewer keys than queries (rows before the first
    key are zero), through the plan and through the grid without one."""
    from vllm_ascend_quantized_kv_cache.ops import _native
    from vllm_ascend_quantized_kv_cache.ops.attention import prefill_attention

    g = torch.Generator().manual_seed(d + hq)
    q_lens = [129, 0, 33, 4, 9]
    kv_lens = [193, 7, 33, 0, 5]
    dtype = torch.bfloat16
    q = torch.randn(sum(q_lens), hq, d, generator=g).to(dtype)
    k = torch.randn(sum(kv_lens), kvh, d, generator=g).to(dtype)
    v = torch.randn(sum(kv_lens), kvh, d, generator=g).to(dtype)
    live = sum(q_lens[:3])
    want = torch.zeros(q.shape)
    want[:live] = ref.attention(q[:live], k[: sum(kv_lens[:3])], v[: sum(kv_lens[:3])],
                                q_lens[:3], kv_lens[:3], d ** -0.5, True)
    want[-5:] = ref.attention(q[-5:], k[-5:], v[-5:], [5], [5], d ** -0.5, True)
    qg, kg, vg = (x.to(gpu_device) for x in (q, k, v))
    got = prefill_attention(qg, kg, vg, q_lens, kv_lens, d ** -0.5, True)
    torch.testing.assert_close(got.float().cpu(), want, atol=1e-2, rtol=1e-2)
    cu = torch.tensor([[0, 129, 129, 162, 166, 175], [0, 193, 200, 233, 233, 238]],
                      dtype=torch.int32, device=gpu_device)
    out = torch.full_like(qg, 7.0)
    rc = _native.lib().kvq_prefill_attn(
        qg.data_ptr(), kg.data_ptr(), vg.data_ptr(), _native.dtype_code(dtype),
        cu[0].data_ptr(), cu[1].data_ptr(), 5, 129, hq, kvh, d, d ** -0.5, 1, out.data_ptr(),
        _native.stream_of(qg))
    assert rc == 0
    torch.testing.assert_close(out, got, atol=0, rtol=0)


@pytest.mark.parametrize("d,hq,kvh,dtype", [(64, 4, 2, torch.float16), (128, 8, 1, torch.bfloat16),
                                            (128, 5, 5, torch.float16), (256, 8, 1, torch.bfloat16)])
@pytest.mark.parametrize("causal", [True, False])
def test_prefill_attention_keys_in_segments(gpu_device, d, hq, kvh, dtype, causal):
    """Few tiles over long keys: every tile's keys in segments, merged.  Requests
    much shorter than the longest one get segments without keys; scores grow
    along the keys, so the segments' maxima differ by powers of two."""
    from vllm_ascend_quantized_kv_cache.ops.attention import prefill_attention

    g = torch.Generator().manual_seed(d + hq)
    q_lens, kv_lens = [17, 1, 2, 3], [3000, 70, 2, 0]
    u = torch.nn.functional.normalize(torch.randn(kvh, d, generator=g), dim=-1)
    grow = torch.cat([torch.arange(n).float() * (20.0 / max(n, 1)) for n in kv_lens])
    k = (grow[:, None, None] * u + 0.2 * torch.randn(sum(kv_lens), kvh, d, generator=g)).to(dtype)
    v = torch.randn(sum(kv_lens), kvh, d, generator=g).to(dtype)
    q = (u.repeat_interleave(hq // kvh, 0)[None] * d ** 0.5
         + torch.randn(sum(q_lens), hq, d, generator=g)).to(dtype)
    got = prefill_attention(q.to(gpu_device), k.to(gpu_device), v.to(gpu_device), q_lens, kv_lens,
                            d ** -0.5, causal).float().cpu()
    want = ref.attention(q[:20], k, v, q_lens[:3], kv_lens[:3], d ** -0.5, causal)
    torch.testing.assert_close(got[:20], want, atol=1e-2, rtol=1e-2)
    assert not got[20:].any()  # no keys


@pytest.mark.parametrize("d", [128, 256])
@pytest.mark.parametrize("where", ["query", "key", "value"])
def test_prefill_attention_of_nans_in_segments(gpu_device, d, where):
    """A NaN among the keys of a segment whose scores are hundreds of powers of two
    under another's reaches the rows that see it, as it does without segments."""
    from vllm_ascend_quantized_kv_cache.ops.attention import prefill_attention

    q_lens, kv_lens, hq = [4], [4000], 8
    g = torch.Generator().manual_seed(d)
    q = torch.ones(4, hq, d, dtype=torch.bfloat16)
    k = torch.zeros(4000, 1, d, dtype=torch.bfloat16)
    k[2000:] = 100.0
    v = torch.randn(4000, 1, d, generator=g).to(torch.bfloat16)
    if where == "query":
        q[1, 5, 3] = float("nan")
    else:
        (k if where == "key" else v)[100, 0, 3] = float("nan")
    got = prefill_attention(q.to(gpu_device), k.to(gpu_device), v.to(gpu_device), q_lens, kv_lens,
                            d ** -0.5, True).isnan().cpu()
    if where == "query":
        assert got[1, 5].all() and int(got.sum()) == d
    elif where == "key":
        assert got.all()
    else:
        assert got[:, :, 3].all() and int(got.sum()) == 4 * hq


@pytest.mark.parametrize("d", [64, 128, 256])
def test_prefill_attention_query_and_output_at_odd_addresses(gpu_device, d):
    """Queries and outputs that start 2 bytes past a 16-byte bound (ordinary vector
    accesses take any address) give what aligned ones give, whole and in segments."""
    from vllm_ascend_quantized_kv_cache.ops.attention import prefill_attention

    def odd(shape):
        n = 1
        for x in shape:
            n *= x
        t = torch.zeros(n + 1, dtype=torch.bfloat16, device=gpu_device)[1:].view(shape)
        assert t.data_ptr() % 16 == 2
        return t

    g = torch.Generator().manual_seed(d)
    for q_lens, kv_lens in (([70, 3], [70, 40]), ([5], [3000])):
        q = torch.randn(sum(q_lens), 4, d, generator=g).to(torch.bfloat16).to(gpu_device)
        k, v = (torch.randn(sum(kv_lens), 2, d, generator=g).to(torch.bfloat16).to(gpu_device)
                for _ in range(2))
        want = prefill_attention(q, k, v, q_lens, kv_lens, d ** -0.5, True)
        got = prefill_attention(odd(q.shape).copy_(q), k, v, q_lens, kv_lens, d ** -0.5, True,
                                out=odd(q.shape))
        assert torch.equal(got, want)


def test_prefill_attention_batch_past_the_launch_argument(gpu_device):
    """More requests, and more tiles, than the plan argument carries."""
    from vllm_ascend_quantized_kv_cache.ops.attention import prefill_attention

    g = torch.Generator().manual_seed(9)
    for q_lens in ([3] * 200, [3, 70000, 4]):
        kv_lens = [n + 2 if n < 100 else 200 for n in q_lens]
        causal = max(q_lens) < 100
        q = torch.randn(sum(q_lens), 1, 64, generator=g).to(torch.bfloat16)
        k = torch.randn(sum(kv_lens), 1, 64, generator=g).to(torch.bfloat16)
        v = torch.randn(sum(kv_lens), 1, 64, generator=g).to(torch.bfloat16)
        want = ref.attention(q, k, v, q_lens, kv_lens, 0.125, causal)
        got = prefill_attention(q.to(gpu_device), k.to(gpu_device), v.to(gpu_device), q_lens,
                                kv_lens, 0.125, causal)
        torch.testing.assert_close(got.float().cpu(), want, atol=1e-2, rtol=1e-2)
