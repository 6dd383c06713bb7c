# SPDX-License-Identifier: Apache-2.0
"""fp8_per_token_head HIP kernels against the oracle (GPU).

* gfx950's E4M3 conversion inside the store kernel, at every rounding
  boundary of the format (rows whose scale is exactly 1, so the kernel's
  quotient is the test value itself), matches the independent encoder;
* rows built so that ``x / scale`` and ``x * (1/scale)`` round to different
  codes follow the division, as the reference semantics does;
* the paged store is bit-exact against the oracle (codes and scales, the
  whole page image, padding slots untouched) for bf16 / fp16 / fp32 inputs,
  int32 / int64 slots and head sizes that exercise every lane width (16, 8
  and 4 codes a lane) and group shape, including partly idle groups;
* the gather is bit-exact against the oracle's dequantize-then-cast, with
  unallocated tail ids;
* attention over the paged codes is within 1e-2 of fp32 attention over the
  oracle's dequantized K/V;
* at a full-size shape (32 requests x 4096 positions, 8 KV heads) a round trip
  of grid values with power-of-two scales is the identity.
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle import kvq_oracle as ref
from tests.test_fp8_per_token_head import E4M3, boundary_points, division_rows, encode_rne
from vllm_ascend_quantized_kv_cache.methods.fp8_per_token_head.byte_cache import (
    Fp8PerTokenHeadLayout,
    fp8_caches_from_byte_tensors,
)
from vllm_ascend_quantized_kv_cache.methods.fp8_per_token_head.semantics import (
    Fp8PerTokenHeadSemantics,
)
from vllm_ascend_quantized_kv_cache.ops import fp8_ops

pytestmark = pytest.mark.gpu

TOL = dict(atol=1e-2, rtol=1e-2)


def _views(device, nb, bs, kvh, d, fill=0):
    """(key buffer, value buffer, (k_data, k_scale, v_data, v_scale)) on device."""
    layout = Fp8PerTokenHeadLayout(nb, bs, kvh, d)
    kb = torch.full((nb, bs, kvh, layout.bytes_per_token_head), fill, dtype=torch.uint8,
                    device=device)
    vb = kb.clone()
    return kb, vb, fp8_caches_from_byte_tensors(kb, vb, layout)


def _store_rows(device, rows: np.ndarray) -> np.ndarray:
    """Codes the store kernel gives for fp32 rows ``[T, 1, D]`` (slot t = row t)."""
    t, kvh, d = rows.shape
    _, _, views = _views(device, 1, t, kvh, d)
    x = torch.from_numpy(rows).to(device)
    fp8_ops.fp8_per_token_head_store(x, x, torch.arange(t, device=device), *views)
    torch.cuda.synchronize()
    return views[0][0].cpu().numpy()


def test_hardware_e4m3_conversion_at_every_rounding_boundary(gpu_device):
    pts = boundary_points()
    per_row = 127
    n = -(-pts.size // per_row)
    rows = np.zeros((n, 1, 128), dtype=np.float32)
    rows[:, 0, 0] = 448.0  # amax 448 -> scale exactly 1
    flat = rows[:, 0, 1:].reshape(-1)
    flat[: pts.size] = pts
    rows[:, 0, 1:] = flat.reshape(n, per_row)
    codes = _store_rows(gpu_device, rows)
    np.testing.assert_array_equal(codes[:, 0, :], encode_rne(rows[:, 0, :]))
    # negative zero keeps its sign bit, as the oracle's cast does
    rows = np.zeros((1, 1, 8), dtype=np.float32)
    rows[0, 0, :3] = (448.0, -0.0, 0.0)
    assert list(_store_rows(gpu_device, rows)[0, 0, :3]) == [0x7E, 0x80, 0x00]


def test_quotient_is_a_division_on_the_gpu(gpu_device):
    rows, want = division_rows(256, seed=11)
    codes = _store_rows(gpu_device, rows)
    np.testing.assert_array_equal(codes[:, 0, 1], want)
    oc, _ = ref.fp8_pth_quantize(torch.from_numpy(rows))
    np.testing.assert_array_equal(codes, oc.numpy())


def _inputs(t, kvh, d, dtype, seed):
    gen = torch.Generator().manual_seed(seed)
    scales = torch.exp(torch.randn((1, kvh, 1), generator=gen) * 2)
    x = torch.randn((t, kvh, d), generator=gen) * scales
    x[0, 0] = 0.0  # an all-zero row: the floor scale
    if t > 2:
        x[2, -1, d // 3] = 3.0e4  # an outlier in one (token, head)
        x[1, 0, : d // 2] = 0.0
    return x.to(dtype)


@pytest.mark.parametrize(
    "dtype,d,kvh,index",
    [
        (torch.bfloat16, 128, 8, torch.int64),
        (torch.bfloat16, 64, 4, torch.int32),
        (torch.float16, 128, 8, torch.int32),
        (torch.float32, 128, 2, torch.int64),
        (torch.bfloat16, 96, 3, torch.int64),   # 12 lanes of a 16-lane group
        (torch.bfloat16, 100, 2, torch.int64),  # D % 8 == 4: 4 codes a lane
        (torch.float32, 36, 5, torch.int32),
        (torch.bfloat16, 256, 2, torch.int64),
        (torch.bfloat16, 512, 1, torch.int32),  # one wave per row
        (torch.float16, 8, 8, torch.int64),     # one lane per row
        (torch.bfloat16, 40, 3, torch.int64),   # 8 codes a lane, 5 lanes of 8
        (torch.float32, 24, 2, torch.int32),    # 8 codes a lane, 3 lanes of 4
    ],
)
def test_store_matches_oracle_bit_exact(gpu_device, dtype, d, kvh, index):
    nb, bs = 9, 16
    t = 100
    x_k = _inputs(t, kvh, d, dtype, seed=d + kvh)
    x_v = _inputs(t, kvh, d, dtype, seed=d * 7 + kvh)
    gen = torch.Generator().manual_seed(d)
    slots = torch.randperm(nb * bs, generator=gen)[:t]
    slots[5] = -1
    slots[40] = -7
    kb, vb, views = _views(gpu_device, nb, bs, kvh, d, fill=0xA5)
    fp8_ops.fp8_per_token_head_store(x_k.to(gpu_device), x_v.to(gpu_device),
                                     slots.to(index).to(gpu_device), *views)
    torch.cuda.synchronize()
    # the oracle writes into the same page images (padding slots keep 0xA5)
    okb = torch.full(kb.shape, 0xA5, dtype=torch.uint8)
    ovb = okb.clone()
    layout = Fp8PerTokenHeadLayout(nb, bs, kvh, d)
    ref.fp8_pth_store(x_k, x_v, slots, *fp8_caches_from_byte_tensors(okb, ovb, layout))
    assert torch.equal(kb.cpu(), okb), "key page image differs"
    assert torch.equal(vb.cpu(), ovb), "value page image differs"


@pytest.mark.parametrize("out_dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("d,kvh", [(128, 8), (100, 2), (64, 4), (40, 3)])
def test_gather_matches_oracle_bit_exact(gpu_device, out_dtype, d, kvh):
    nb, bs = 12, 16
    lens = [37, 16, 0, 70]
    table = torch.tensor([[3, 7, 11, -1, -1], [0, -1, -1, -1, -1], [-1] * 5,
                          [1, 2, 4, 5, 6]])
    gen = torch.Generator().manual_seed(d)
    x_k = _inputs(nb * bs, kvh, d, torch.bfloat16, seed=1)
    x_v = _inputs(nb * bs, kvh, d, torch.bfloat16, seed=2)
    slots = torch.randperm(nb * bs, generator=gen)
    kb, vb, views = _views(gpu_device, nb, bs, kvh, d)
    fp8_ops.fp8_per_token_head_store(x_k.to(gpu_device), x_v.to(gpu_device),
                                     slots.to(gpu_device), *views)
    for index in (torch.int32, torch.int64):
        dk, dv = fp8_ops.fp8_per_token_head_dequant_gather(
            *views, table.to(index).to(gpu_device), lens, out_dtype)
        torch.cuda.synchronize()
        cpu_views = [v.cpu() for v in views]
        wk, wv = ref.fp8_pth_gather(*cpu_views, table, lens, out_dtype)
        assert dk.dtype == out_dtype and dk.shape == (sum(lens), kvh, d)
        assert torch.equal(dk.cpu(), wk) and torch.equal(dv.cpu(), wv)


@pytest.mark.parametrize("index", [torch.int32, torch.int64])
def test_gather_with_lengths_on_the_device_is_the_same(gpu_device, index):
    """The entry point that reads the first rows from device memory, over ragged
    lengths and an empty request."""
    from vllm_ascend_quantized_kv_cache.ops import _native

    nb, bs, kvh, d, lens = 12, 16, 2, 128, [37, 16, 0, 70]
    table = torch.tensor([[3, 7, 11, -1, -1], [0, -1, -1, -1, -1], [-1] * 5, [1, 2, 4, 5, 6]],
                         dtype=index, device=gpu_device)
    _, _, views = _views(gpu_device, nb, bs, kvh, d)
    rows = [_inputs(nb * bs, kvh, d, torch.bfloat16, seed=s).to(gpu_device) for s in (1, 2)]
    fp8_ops.fp8_per_token_head_store(*rows, torch.arange(nb * bs, device=gpu_device), *views)
    want = fp8_ops.fp8_per_token_head_dequant_gather(*views, table, lens, torch.bfloat16)
    cu = torch.tensor([0, 37, 53, 53, 123], dtype=torch.int64, device=gpu_device)
    got = [torch.zeros_like(x) for x in want]
    rc = _native.lib().kvq_fp8_pth_gather(
        *(v.data_ptr() for v in views), nb, bs, kvh, d, table.data_ptr(),
        _native.index_code(index), 5, cu.data_ptr(), 4, got[0].data_ptr(), got[1].data_ptr(),
        _native.dtype_code(torch.bfloat16), _native.stream_of(cu))
    assert rc == 0
    for a, b in zip(got, want):
        assert torch.equal(a.view(torch.int16), b.view(torch.int16))


@pytest.mark.parametrize("batch", [256, 257, 600])
def test_gather_of_batches_past_one_launch(gpu_device, batch):
    """A launch carries 256 requests' rows; short, empty and long ones on both
    sides of the cuts."""
    nb, bs, kvh, d = 40, 16, 2, 64
    gen = torch.Generator().manual_seed(batch)
    lens = torch.randint(0, 40, (batch,), generator=gen).tolist()
    lens[0] = lens[-1] = 48
    lens[255] = 0
    table = torch.randint(0, nb, (batch, 3), generator=gen, dtype=torch.int32)
    _, _, views = _views(gpu_device, nb, bs, kvh, d)
    rows = [_inputs(nb * bs, kvh, d, torch.bfloat16, seed=s).to(gpu_device) for s in (1, 2)]
    fp8_ops.fp8_per_token_head_store(*rows, torch.arange(nb * bs, device=gpu_device), *views)
    dk, dv = fp8_ops.fp8_per_token_head_dequant_gather(*views, table.to(gpu_device), lens,
                                                       torch.bfloat16)
    wk, wv = ref.fp8_pth_gather(*[v.cpu() for v in views], table, lens, torch.bfloat16)
    assert torch.equal(dk.cpu(), wk) and torch.equal(dv.cpu(), wv)


def test_semantics_object_matches_oracle(gpu_device):
    sem = Fp8PerTokenHeadSemantics(type("Cfg", (), {"head_size": 128})())
    x = _inputs(33, 4, 128, torch.bfloat16, seed=9)
    q, s = sem.quantize(x.to(gpu_device))
    oq, os_ = ref.fp8_pth_quantize(x)
    assert q.dtype == torch.float8_e4m3fn
    assert torch.equal(q.view(torch.uint8).cpu(), oq) and torch.equal(s.cpu(), os_)
    assert torch.equal(sem.compute_scale(x.to(gpu_device)).cpu(), os_)
    back = sem.dequantize(q, s)
    assert torch.equal(back.cpu(), ref.fp8_pth_dequantize(oq, os_))
    fq = sem.fake_quant(x.to(gpu_device))
    assert torch.equal(fq.cpu(), ref.fp8_pth_dequantize(oq, os_).to(torch.bfloat16))
    assert sem.quantize(x[:0].to(gpu_device))[0].shape == (0, 4, 128)


@pytest.mark.parametrize("query_lens", [[1, 1, 1, 1], [5, 1, 17, 40]])
def test_attention_over_paged_codes(gpu_device, query_lens):
    nb, bs, kvh, hq, d = 40, 16, 4, 16, 128
    lens = [150, 33, 97, 300]
    gen = torch.Generator().manual_seed(13)
    perm = torch.randperm(nb, generator=gen)
    maxb = -(-max(lens) // bs)
    table = torch.full((len(lens), maxb), -1, dtype=torch.int64)
    used = 0
    for b, n in enumerate(lens):
        k = -(-n // bs)
        table[b, :k] = perm[used:used + k]
        used += k
    slots = torch.cat([table[b, torch.arange(n) // bs] * bs + torch.arange(n) % bs
                       for b, n in enumerate(lens)])
    x_k = torch.randn((sum(lens), kvh, d), generator=gen).to(torch.bfloat16)
    x_v = torch.randn((sum(lens), kvh, d), generator=gen).to(torch.bfloat16)
    _, _, views = _views(gpu_device, nb, bs, kvh, d)
    fp8_ops.fp8_per_token_head_store(x_k.to(gpu_device), x_v.to(gpu_device),
                                     slots.to(gpu_device), *views)
    q = (torch.randn((sum(query_lens), hq, d), generator=gen)).to(torch.bfloat16)
    out = fp8_ops.fp8_per_token_head_attention(
        q.to(gpu_device), *views, table.to(gpu_device), lens, query_lens, d ** -0.5,
        block_table_host=table.numpy())
    torch.cuda.synchronize()
    dk, dv = ref.fp8_pth_gather(*[v.cpu() for v in views], table, lens, torch.float32)
    want = ref.attention(q.float(), dk, dv, query_lens, lens, d ** -0.5, True)
    torch.testing.assert_close(out.float().cpu(), want, **TOL)


def test_full_size_round_trip_of_grid_values(gpu_device):
    """32 requests x 4096 positions x 8 KV heads x 128: values on the E4M3 grid
    times 2^k, with 448 * 2^k in each row, come back exactly."""
    b, n, kvh, d, bs = 32, 4096, 8, 128, 128
    t = b * n
    gen = torch.Generator(device=gpu_device).manual_seed(21)
    codes = torch.randint(0, 0x7E, (t, kvh, d), generator=gen, device=gpu_device,
                          dtype=torch.int32)
    codes |= torch.randint(0, 2, codes.shape, generator=gen, device=gpu_device,
                           dtype=torch.int32) << 7
    codes[:, :, 5] = 0x7E
    grid = torch.from_numpy(E4M3.astype(np.float32)).to(gpu_device)
    k = torch.randint(-8, 8, (t, kvh, 1), generator=gen, device=gpu_device).float()
    x = (grid[codes.long()] * torch.exp2(k)).to(torch.bfloat16)  # exact in bf16
    del codes
    nb = t // bs + 3
    perm = torch.randperm(nb, generator=gen, device=gpu_device)[: t // bs]
    table = perm.view(b, n // bs)
    slots = (table.view(-1, 1) * bs + torch.arange(bs, device=gpu_device)).view(-1)
    _, _, views = _views(gpu_device, nb, bs, kvh, d)
    fp8_ops.fp8_per_token_head_store(x, x, slots, *views)
    dk, dv = fp8_ops.fp8_per_token_head_dequant_gather(
        *views, table, [n] * b, torch.bfloat16, block_table_host=table.cpu().numpy())
    torch.cuda.synchronize()
    assert torch.equal(dk, x) and torch.equal(dv, x)
    assert torch.equal(views[1].view(-1, kvh)[slots], torch.exp2(k).view(t, kvh))


def _decode_case(dev, lens, *, d, kvh, rep, bs, dtype, index, seed=5, rows=1, causal=True):
    """A decode over pages whose unwritten bytes are NaN codes and scales."""
    gen = torch.Generator().manual_seed(seed)
    need = [-(-n // bs) for n in lens]
    nb = sum(need) + 2
    perm = torch.randperm(nb, generator=gen)
    table = torch.full((len(lens), max(max(need), 1)), -1, dtype=index)
    used = 0
    for b, k in enumerate(need):
        table[b, :k] = perm[used:used + k].to(index)
        used += k
    slots = [table[b, torch.arange(n) // bs].long() * bs + torch.arange(n) % bs
             for b, n in enumerate(lens)]
    _, _, views = _views(dev, nb, bs, kvh, d)
    for i, v in enumerate(views):
        v.fill_(0xFF if i % 2 == 0 else float("nan"))
    x = [(torch.randn((sum(lens), kvh, d), generator=gen) * 10 ** float(e)).to(dtype)
         for e in (0, -3)]  # small values: their scales leave the fp16 range
    fp8_ops.fp8_per_token_head_store(x[0].to(dev), x[1].to(dev), torch.cat(slots).to(dev), *views)
    q = torch.randn((rows * len(lens), kvh * rep, d), generator=gen).to(dtype)
    got = fp8_ops.fp8_per_token_head_attention(
        q.to(dev), *views, table.to(dev), lens, [rows] * len(lens), d ** -0.5, causal=causal,
        block_table_host=table.numpy())
    torch.cuda.synchronize()
    # the rows attended to are the gather's, in the query's dtype
    dk, dv = (x.float() for x in ref.fp8_pth_gather(*[v.cpu() for v in views], table, lens, dtype))
    # only rows with a position to see reach the oracle; the others are zeros
    live = [(b, min(rows, n) if causal else rows) for b, n in enumerate(lens) if n]
    at = torch.cat([torch.arange(rows * b + rows - m, rows * (b + 1)) for b, m in live])
    want = torch.zeros(q.shape)
    want[at] = ref.attention(q[at].float(), dk, dv, [m for _, m in live],
                             [lens[b] for b, _ in live], d ** -0.5, causal)
    # the output's rounding, on values of 1e-3
    rel = 2.0 ** (-8 if dtype == torch.bfloat16 else -11)
    torch.testing.assert_close(got.float().cpu(), want, atol=1e-3 * 2 * rel, rtol=2 * rel)


@pytest.mark.parametrize("d,kvh,rep,bs,dtype,index", [
    (128, 8, 4, 128, torch.bfloat16, torch.int32),   # the item's heads in one workgroup
    (128, 1, 16, 16, torch.float16, torch.int64),
    (128, 3, 7, 48, torch.bfloat16, torch.int64),
    (128, 16, 1, 32, torch.float16, torch.int32),    # one wave per head
    (256, 1, 8, 128, torch.bfloat16, torch.int32),
    (256, 4, 5, 64, torch.float16, torch.int64),
    (256, 8, 2, 16, torch.bfloat16, torch.int32),
])
def test_decode_over_paged_codes(gpu_device, d, kvh, rep, bs, dtype, index):
    """One row per request, straight from the codes: lengths around the tile and
    the 16-token group, an empty request, requests cut into several items."""
    _decode_case(gpu_device, [150, 0, 1, 15, 16, 17, 31, 32, 33, 64, 700], d=d, kvh=kvh, rep=rep,
                 bs=bs, dtype=dtype, index=index)


@pytest.mark.parametrize("d,kvh,rep,bs,dtype,rows", [
    (128, 8, 4, 128, torch.bfloat16, 4),   # a full set of score columns
    (128, 2, 7, 16, torch.float16, 2),     # 14 columns
    (128, 1, 7, 64, torch.bfloat16, 5),    # three passes, the last of one row
    (128, 16, 1, 32, torch.float16, 33),   # one wave per head; 16, 16 and 1 rows
    (256, 1, 8, 128, torch.bfloat16, 3),
    (256, 2, 16, 16, torch.float16, 2),    # a pass per row
])
@pytest.mark.parametrize("causal", [True, False])
def test_decode_of_a_few_rows(gpu_device, d, kvh, rep, bs, dtype, rows, causal):
    """Several rows per request in one pass over its codes, each with its own end:
    ends on both sides of the tiles, requests shorter than their rows."""
    assert fp8_ops._decode_applies(
        torch.empty((rows, kvh * rep, d), dtype=dtype, device=gpu_device),
        torch.empty((1, bs, kvh, d), dtype=torch.uint8, device=gpu_device),
        torch.empty((1, 1), dtype=torch.int32, device=gpu_device), [rows], 0.1)
    _decode_case(gpu_device, [150, 0, 1, 2, 16, 17, 31, 32, 33, 34, 64, 129, 700], d=d, kvh=kvh,
                 rep=rep, bs=bs, dtype=dtype, index=torch.int32, rows=rows, causal=causal)


def test_decode_over_paged_codes_long_request_and_large_batch(gpu_device):
    """More requests than one launch carries, next to one of many items."""
    lens = [9000] + [(37 * i) % 50 for i in range(800)]
    _decode_case(gpu_device, lens, d=128, kvh=2, rep=2, bs=16, dtype=torch.bfloat16,
                 index=torch.int32)


def test_decode_row_forms_agree(gpu_device):
    """Rows whose heads or tokens are strided, and an output of another dtype, give
    the packed rows' result; a batch that is not one row per request and a
    head size the decode does not take run the gathered path."""
    bs, kvh, hq, nb = 16, 2, 4, 12
    gen = torch.Generator().manual_seed(4)
    for d in (128, 64):
        _, _, views = _views(gpu_device, nb, bs, kvh, d)
        x = torch.randn((nb * bs, kvh, d), generator=gen).to(torch.bfloat16).to(gpu_device)
        fp8_ops.fp8_per_token_head_store(x, x, torch.arange(nb * bs, device=gpu_device), *views)
        table = torch.arange(nb, device=gpu_device, dtype=torch.int32).view(3, 4)
        lens = [50, 3, 64]
        wide = torch.randn((3, hq, 2 * d), generator=gen).to(torch.bfloat16).to(gpu_device)
        q = wide[:, :, ::2]
        want = fp8_ops.fp8_per_token_head_attention(q.contiguous(), *views, table, lens, [1] * 3,
                                                    d ** -0.5)
        out = torch.empty((3, hq, d), dtype=torch.float32, device=gpu_device)
        got = fp8_ops.fp8_per_token_head_attention(q, *views, table, lens, [1] * 3, d ** -0.5,
                                                   out=out)
        assert got is out and torch.equal(out.to(torch.bfloat16), want)
        two = fp8_ops.fp8_per_token_head_attention(
            torch.cat([q[:1], q]), *views, table, lens, [2, 1, 1], d ** -0.5)
        torch.testing.assert_close(two[1:].float(), want.float(), **TOL)
    with pytest.raises(RuntimeError, match="does not cover the longest sequence"):
        fp8_ops.fp8_per_token_head_attention(q, *views, table, [65, 3, 64], [1] * 3, 0.1)


@pytest.mark.parametrize("d,rows,dtype", [(128, 1, torch.bfloat16), (256, 1, torch.bfloat16),
                                          (128, 3, torch.bfloat16), (128, 1, torch.float16),
                                          (256, 2, torch.float16)])
def test_decode_attends_to_the_rows_the_gather_leaves(gpu_device, d, rows, dtype):
    """The decode's keys and values are the gather's dense rows in the query's dtype:
    with peaked scores (keys of outlier channels) their rounding shows in the
    output, so a decode of unrounded rows answers otherwise than a gathered one."""
    kvh, rep, bs, lens = 2, 4, 32, [2000, 65, 700, 31]
    gen = torch.Generator().manual_seed(17)
    need = [-(-n // bs) for n in lens]
    table = torch.zeros((len(lens), max(need)), dtype=torch.int32)
    perm = torch.randperm(sum(need), generator=gen).to(torch.int32)
    for b, k in enumerate(need):
        table[b, :k] = perm[sum(need[:b]):sum(need[:b + 1])]
    slots = torch.cat([table[b, torch.arange(n) // bs].long() * bs + torch.arange(n) % bs
                       for b, n in enumerate(lens)]).to(gpu_device)
    _, _, views = _views(gpu_device, sum(need), bs, kvh, d)
    channel = torch.exp(torch.randn((kvh, d), generator=gen))
    key = (torch.randn((sum(lens), kvh, d), generator=gen) * channel).to(dtype)
    value = torch.randn((sum(lens), kvh, d), generator=gen).to(dtype)
    fp8_ops.fp8_per_token_head_store(key.to(gpu_device), value.to(gpu_device), slots, *views)
    q = torch.randn((rows * len(lens), kvh * rep, d), generator=gen).to(dtype)
    args = (*views, table.to(gpu_device), lens)
    got = fp8_ops.fp8_per_token_head_attention(q.to(gpu_device), *args, [rows] * len(lens),
                                               d ** -0.5, block_table_host=table.numpy())
    dk, dv = (x.double().cpu() for x in fp8_ops.fp8_per_token_head_dequant_gather(*args, dtype))
    at = 0
    for b, n in enumerate(lens):
        for j in range(rows):
            k, v = dk[at:at + n - rows + 1 + j], dv[at:at + n - rows + 1 + j]
            for h in range(kvh * rep):
                s = k[:, h // rep] @ q[rows * b + j, h].double() * d ** -0.5
                want = torch.softmax(s, 0) @ v[:, h // rep]
                # the output's rounding (half a unit in the last place) and a part
                # in 2^13 of the largest value for p's parts and the fp32 sums
                ulp = 2.0 ** (-8 if dtype == torch.bfloat16 else -11)
                bound = ulp * want.abs() + v.abs().max() * 2.0 ** -13
                off = (got[rows * b + j, h].double().cpu() - want).abs() - bound
                assert off.max() <= 0, (b, j, h, off.max().item())
        at += n


@pytest.mark.parametrize("where", ["query", "key code", "value code"])
def test_decode_of_nans_is_nan(gpu_device, where):
    """A NaN query row, key or value reaches its heads' outputs and no others, as it
    does over gathered rows (requests cut into several items, and a whole one)."""
    d, kvh, rep, bs, lens = 128, 2, 2, 16, [900, 40]
    gen = torch.Generator().manual_seed(23)
    nb = sum(-(-n // bs) for n in lens)
    table = torch.zeros((2, -(-lens[0] // bs)), dtype=torch.int32)
    table[0] = torch.arange(table.shape[1])
    table[1, :3] = torch.arange(table.shape[1], nb)
    _, _, views = _views(gpu_device, nb, bs, kvh, d)
    x = torch.randn((nb * bs, kvh, d), generator=gen).to(torch.bfloat16).to(gpu_device)
    fp8_ops.fp8_per_token_head_store(x, x, torch.arange(nb * bs, device=gpu_device), *views)
    q = torch.randn((2, kvh * rep, d), generator=gen).to(torch.bfloat16)
    if where == "query":
        q[:, 2, 7] = float("nan")
    else:
        codes = views[0] if where == "key code" else views[2]
        codes[table[:, 2].long(), 5, 1, 9] = 0x7F  # position 37 of both, kv head 1
    args = (q.to(gpu_device), *views, table.to(gpu_device), lens)
    outs = [fp8_ops.fp8_per_token_head_attention(*args, [1, 1], d ** -0.5)]
    k, v = fp8_ops.fp8_per_token_head_dequant_gather(*args[1:], torch.bfloat16)
    from vllm_ascend_quantized_kv_cache.ops.attention import prefill_attention

    outs.append(prefill_attention(args[0], k, v, [1, 1], lens, d ** -0.5, True))
    for out in outs:
        hit = out.isnan().cpu()
        if where == "query":
            assert hit[:, 2].all() and not hit[:, [0, 1, 3]].any()
        elif where == "key code":
            assert hit[:, 2:].all() and not hit[:, :2].any()
        else:
            assert hit[:, 2:, 9].all() and int(hit.sum()) == 4


@pytest.mark.parametrize("lens", [[9000, 3], [100] * 800])
def test_decode_refuses_a_workspace_too_small(gpu_device, lens):
    """A workspace a byte under any launch's partials is refused before a launch."""
    from vllm_ascend_quantized_kv_cache.ops import _native

    d, kvh, hq, bs = 128, 2, 4, 16
    lib, batch = _native.lib(), len(lens)
    lens_np = np.array(lens, dtype=np.int64)
    need = lib.kvq_fp8_pth_decode_workspace_bytes(lens_np.ctypes.data, batch, 1, hq, kvh, d, bs)
    _, _, views = _views(gpu_device, 1, bs, kvh, d)
    q = torch.zeros((batch, hq, d), dtype=torch.bfloat16, device=gpu_device)
    out = torch.full_like(q, 7.0)
    table = torch.zeros((batch, -(-max(lens) // bs)), dtype=torch.int32, device=gpu_device)
    ws = torch.empty(need, dtype=torch.uint8, device=gpu_device)

    def call(nbytes):
        return lib.kvq_fp8_pth_decode_attn(
            q.data_ptr(), _native.dtype_code(q.dtype), batch, 1, 1, hq, kvh, d, 0.1,
            *(v.data_ptr() for v in views), 1, bs, table.data_ptr(), _native.index_code(table.dtype),
            table.shape[1], lens_np.ctypes.data, ws.data_ptr(), nbytes, out.data_ptr(),
            _native.stream_of(q))

    assert call(need - 1) == _native.KVQ_ERR_INVALID
    torch.cuda.synchronize()
    assert (out == 7.0).all()
    assert call(need) == 0
    torch.cuda.synchronize()
    assert not out.any()  # all values are zero
