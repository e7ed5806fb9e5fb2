"""HIP paged decode attention vs the oracle (GPU).

Mirrors section F of reference tests/test_kv_cache_quantization.py:394-545 and
reference tests/test_decode_attention.py:11-42, plus the workload configs:
  * cfg1 against the committed golden output;
  * cfg2 / north star / cfg3 / cfg4 at full size: bit-exact cache bytes for the
    tokens written and every output row against the float64 oracle (tolerance
    2e-2 abs / 1e-2 rel);
  * slot and page reuse through the decode kernel.
"""

from __future__ import annotations

import math
from pathlib import Path

import numpy as np
import pytest
import torch as t

import oracle
from aiproj_amd import workloads
from aiproj_amd.inference.page_allocator import PageAllocator
from aiproj_amd.inference.paged_kv_cache import PagedKVCache
from aiproj_amd.kernals.decode_attention import PagedKVRead, decode_attention_wrapper
from tests.helpers import FP8

pytestmark = pytest.mark.gpu
GOLDEN = Path(__file__).resolve().parent / "golden"

# Lengths cover a single token, a partial page, exactly one page, exactly four
# pages, one past, and several chunks (reference :449-451); 700 and 1300 cross the
# decode kernel's chunk boundaries.
DECODE_LENGTHS = [1, 3, 16, 64, 65, 141, 300, 700, 1300]
OUTPUT_TOLERANCE = {t.float32: 1e-4, t.float16: 2e-3, t.bfloat16: 1.6e-2}
NORTH_STAR_ATOL, NORTH_STAR_RTOL = 2e-2, 1e-2


def fill_decode_batch(caches, lengths, num_kv_heads, head_dim, block_size, kv_dtype, seed):
    """One K/V history per request into every cache (shared manager); context_length == length.

    Same construction as reference tests/test_kv_cache_quantization.py:398-425.
    """
    generator = t.Generator(device="cuda").manual_seed(seed)
    num_blocks = sum(-(-length // block_size) for length in lengths) + 4
    manager = PageAllocator(num_blocks, block_size, len(lengths) + 1, max(lengths) + block_size, "cuda")
    slots, keys, values = [], [], []
    for request_id, length in enumerate(lengths):
        slots.append(manager.allocate_request(request_id, length))
        k = t.randn(length, num_kv_heads, head_dim, device="cuda", generator=generator).to(kv_dtype)
        v = t.randn(length, num_kv_heads, head_dim, device="cuda", generator=generator).to(kv_dtype)
        for cache in caches:
            manager.append_request(request_id, t.arange(length, device="cuda"), k, v, cache)
        manager.advance(request_id, length - 1)
        keys.append(k)
        values.append(v)
    context = manager.create_container(
        t.tensor(slots, device="cuda"),
        t.arange(len(lengths) + 1, dtype=t.int32, device="cuda"),
        t.tensor(lengths, device="cuda") - 1,
    )
    return manager, context, keys, values


def cache_numpy(cache):
    if cache.quantized:
        return (cache.k.view(t.uint8).cpu().numpy(), cache.v.view(t.uint8).cpu().numpy(),
                cache.k_scales.cpu().numpy(), cache.v_scales.cpu().numpy())
    return cache.k.float().cpu().numpy(), cache.v.float().cpu().numpy(), None, None


def oracle_decode(q, cache, block_table, slots, lengths, rows=None):
    kc, vc, ks, vs = cache_numpy(cache)
    rows = range(q.shape[0]) if rows is None else rows
    qn = q.float().cpu().numpy()
    table = block_table.cpu().numpy()
    slots = [int(s) for s in slots.tolist()]
    out = []
    for r in rows:
        k, v = oracle.paged_history(kc, vc, ks, vs, table, slots[r], int(lengths[r]), cache.block_size)
        out.append(oracle.decode_one(qn[r], k, v))
    return np.stack(out)


@t.inference_mode()
@pytest.mark.parametrize("q_dtype", [t.float32, t.float16, t.bfloat16])
@pytest.mark.parametrize("head_dim", [16, 64, 80, 128])
@pytest.mark.parametrize("num_q_heads,num_kv_heads", [(8, 2), (4, 4), (32, 8), (64, 8), (24, 2), (16, 1)])
def test_fp8_decode_matches_attention_over_dequantized_cache(q_dtype, head_dim, num_q_heads, num_kv_heads):
    block_size = 16
    num_blocks = sum(-(-n // 16) for n in DECODE_LENGTHS) + 4
    cache = PagedKVCache(num_blocks, block_size, num_kv_heads, head_dim, "cuda", FP8)
    manager, context, _, _ = fill_decode_batch([cache], DECODE_LENGTHS, num_kv_heads, head_dim, block_size,
                                               t.bfloat16, seed=6)
    q = t.randn(len(DECODE_LENGTHS), num_q_heads, head_dim, device="cuda").to(q_dtype)
    actual = decode_attention_wrapper(q, cache, context)
    assert actual.shape == q.shape and actual.dtype == q_dtype
    expected = oracle_decode(q, cache, manager.block_table, context.cache_slots, DECODE_LENGTHS)
    tol = OUTPUT_TOLERANCE[q_dtype]
    t.testing.assert_close(actual.double().cpu(), t.from_numpy(expected), rtol=tol, atol=tol)


@t.inference_mode()
@pytest.mark.parametrize("head_dim", [16, 128])
def test_fp8_decode_close_to_bf16_decode(head_dim):
    lengths = [5, 64, 200, 300]
    num_q_heads, num_kv_heads, block_size = 8, 2, 16
    bf16_cache = PagedKVCache(64, block_size, num_kv_heads, head_dim, "cuda", t.bfloat16)
    fp8_cache = PagedKVCache(64, block_size, num_kv_heads, head_dim, "cuda", FP8)
    _, context, _, values = fill_decode_batch([bf16_cache, fp8_cache], lengths, num_kv_heads, head_dim,
                                              block_size, t.bfloat16, seed=7)
    q = t.randn(len(lengths), num_q_heads, head_dim, device="cuda", dtype=t.bfloat16)
    bf16_out = decode_attention_wrapper(q, bf16_cache, context).float()
    fp8_out = decode_attention_wrapper(q, fp8_cache, context).float()
    assert t.isfinite(fp8_out).all()
    v_max = max(v.float().abs().max().item() for v in values)
    worst = (fp8_out - bf16_out).abs().max().item()
    assert worst <= 0.06 * v_max, f"max |fp8 - bf16| = {worst:.4f}, limit {0.06 * v_max:.4f}"


@t.inference_mode()
@pytest.mark.parametrize("cache_dtype", [t.bfloat16, FP8])
@pytest.mark.parametrize("head_dim", [32, 128])
def test_decode_ignores_stale_cache_contents(cache_dtype, head_dim):
    lengths = [5, 70, 1, 333]
    num_q_heads, num_kv_heads, block_size = 8, 2, 16
    cache = PagedKVCache(48, block_size, num_kv_heads, head_dim, "cuda", cache_dtype)
    if cache.quantized:
        cache.k.view(t.uint8).fill_(0x7F)      # NaN in float8_e4m3fn
        cache.v.view(t.uint8).fill_(0x7F)
        cache.k_scales.fill_(float("nan"))
        cache.v_scales.fill_(float("nan"))
    else:
        cache.k.fill_(float("nan"))
        cache.v.fill_(float("nan"))
    manager, context, _, _ = fill_decode_batch([cache], lengths, num_kv_heads, head_dim, block_size,
                                               t.bfloat16, seed=8)
    q = t.randn(len(lengths), num_q_heads, head_dim, device="cuda", dtype=t.float32)
    actual = decode_attention_wrapper(q, cache, context)
    assert t.isfinite(actual).all()
    expected = oracle_decode(q, cache, manager.block_table, context.cache_slots, lengths)
    t.testing.assert_close(actual.double().cpu(), t.from_numpy(expected), rtol=1e-4, atol=1e-4)


@t.inference_mode()
@pytest.mark.parametrize("dtype", [t.float32, t.float16, t.bfloat16])
def test_unquantized_decode_matches_dense_reference(dtype):
    # reference tests/test_decode_attention.py:11-42
    t.manual_seed(4)
    lengths = [3, 73, 141]
    hq, hkv, d = 8, 2, 16
    manager = PageAllocator(32, 16, 5, 160, "cuda")
    cache = PagedKVCache(32, 16, hkv, d, "cuda", dtype)
    slots, keys, values = [], [], []
    for request_id, length in enumerate(lengths):
        slots.append(manager.allocate_request(request_id, length))
        k = t.randn(length, hkv, d, dtype=dtype, device="cuda")
        v = t.randn_like(k)
        manager.append_request(request_id, t.arange(length, device="cuda"), k, v, cache)
        manager.advance(request_id, length - 1)
        keys.append(k)
        values.append(v)
    slots = t.tensor(slots, device="cuda")
    context = manager.create_container(slots, t.arange(4, dtype=t.int32, device="cuda"),
                                       t.tensor(lengths, device="cuda") - 1)
    q = t.randn(3, hq, d, dtype=dtype, device="cuda")
    actual = decode_attention_wrapper(q, cache, context)
    expected = []
    for row, (k, v) in enumerate(zip(keys, values)):
        k = k.transpose(0, 1).float().repeat_interleave(hq // hkv, 0).cpu()
        v = v.transpose(0, 1).float().repeat_interleave(hq // hkv, 0).cpu()
        scores = q[row].float().cpu().unsqueeze(1) @ k.transpose(-1, -2) / math.sqrt(d)
        expected.append((scores.softmax(-1) @ v).squeeze(1))
    t.testing.assert_close(actual.float().cpu(), t.stack(expected), rtol=1e-2, atol=1e-2)


@t.inference_mode()
def test_decode_edge_cases_and_calling_forms():
    lengths = [0, 17, 0, 2000]
    hq, hkv, d = 16, 4, 128
    num_blocks = sum(-(-n // 16) for n in lengths) + 8
    cache = PagedKVCache(num_blocks, 16, hkv, d, "cuda", FP8)
    live = [n if n else 1 for n in lengths]
    manager, context, _, _ = fill_decode_batch([cache], live, hkv, d, 16, t.bfloat16, seed=9)
    ctx = t.tensor(lengths, dtype=t.int32, device="cuda")
    q_full = t.randn(4, hq, 2 * d, device="cuda", dtype=t.bfloat16)
    q = q_full[:, :, ::2]                                    # strided last dim -> copied
    q2 = q_full[:, :, :d]                                    # strided rows, contiguous last dim
    for qq in (q, q2):
        for slots in (context.cache_slots.to(t.int32), context.cache_slots.to(t.int64)):
            for lens in (ctx, ctx.long()):
                read = PagedKVRead(cache.k, cache.v, cache.k_scales, cache.v_scales, manager.block_table,
                                   slots, lens, 16)
                out = decode_attention_wrapper(qq, read)
                assert (out[0] == 0).all() and (out[2] == 0).all()
                expected = oracle_decode(qq, cache, manager.block_table, slots, lengths, rows=[1, 3])
                t.testing.assert_close(out[[1, 3]].double().cpu(), t.from_numpy(expected),
                                       rtol=NORTH_STAR_RTOL, atol=NORTH_STAR_ATOL)
    # The cache-object form gives the same result as the PagedKVRead form.
    context.context_lengths = ctx
    a = decode_attention_wrapper(q2, cache, context)
    b = decode_attention_wrapper(q2, PagedKVRead(cache.k, cache.v, cache.k_scales, cache.v_scales,
                                                 manager.block_table, context.cache_slots, ctx, 16))
    assert t.equal(a, b)
    # Every call is deterministic.
    assert t.equal(a, decode_attention_wrapper(q2, cache, context))


@t.inference_mode()
@pytest.mark.parametrize("head_dim", [64, 80])
def test_decode_block_sizes_other_than_16(head_dim):
    # Page sizes under 16 take the grouped VALU kernel, 32 and up the MFMA kernel (D 80 as
    # narrow rows; the grouped kernel's large pages: test_grouped_kernel_at_head_size_80).
    # Pages of 1 and 2 fill the grouped kernel's whole per-wave page list (256 entries
    # for a 256-token chunk), and lengths past 600 cross pages and chunks.
    for block_size in (1, 2, 4, 8, 32, 64, 256, 512):
        lengths = [3, 40, 129, 700]
        cache = PagedKVCache(sum(-(-n // block_size) for n in lengths) + 4, block_size, 2, head_dim, "cuda", FP8)
        manager, context, _, _ = fill_decode_batch([cache], lengths, 2, head_dim, block_size, t.bfloat16, seed=10)
        q = t.randn(len(lengths), 8, head_dim, device="cuda", dtype=t.float32)
        out = decode_attention_wrapper(q, cache, context)
        expected = oracle_decode(q, cache, manager.block_table, context.cache_slots, lengths)
        t.testing.assert_close(out.double().cpu(), t.from_numpy(expected), rtol=1e-4, atol=1e-4)


def _shifted(x, offset):
    """x's bytes copied `offset` bytes past a 16-byte boundary (same shape and dtype)."""
    nbytes = x.numel() * x.element_size()
    raw = t.empty(nbytes + 16, dtype=t.uint8, device=x.device)
    view = raw[offset:offset + nbytes].view(x.dtype).view(x.shape)
    view.view(t.uint8).copy_(x.view(t.uint8))
    return view


# (byte offset, cache dtype, q dtype): a cache tensor starts on a multiple of its
# element size, so byte offset 1 exists for the 1-byte FP8 cache only.
_UNALIGNED_CASES = [
    (offset, cache_dtype, q_dtype)
    for offset in (4, 1)
    for cache_dtype, q_dtype in ((FP8, t.bfloat16), (FP8, t.float32), (t.bfloat16, t.bfloat16),
                                 (t.float16, t.float16), (t.float32, t.float32))
    if offset % t.empty((), dtype=cache_dtype).element_size() == 0
]


@t.inference_mode()
@pytest.mark.parametrize("offset,cache_dtype,q_dtype", _UNALIGNED_CASES)
def test_unaligned_caches_take_the_valu_kernels(offset, cache_dtype, q_dtype):
    # The MFMA kernel needs 16-byte aligned caches. 4-byte aligned caches take the
    # grouped VALU kernel (whole-dword slices), byte-aligned ones the per-element
    # path; both against the oracle on the same bytes, at the north-star head
    # layout (32q/8kv, D 128) with lengths across chunk boundaries.
    lengths = [1, 17, 256, 257, 700, 1300]
    hq, hkv, d = 32, 8, 128
    cache = PagedKVCache(sum(-(-n // 16) for n in lengths) + 4, 16, hkv, d, "cuda", cache_dtype)
    manager, context, _, _ = fill_decode_batch([cache], lengths, hkv, d, 16, t.bfloat16, seed=16)
    q = t.randn(len(lengths), hq, d, device="cuda").to(q_dtype)
    read = PagedKVRead(_shifted(cache.k, offset), _shifted(cache.v, offset), cache.k_scales, cache.v_scales,
                       manager.block_table, context.cache_slots, context.context_lengths, 16)
    actual = decode_attention_wrapper(q, read)
    expected = oracle_decode(q, cache, manager.block_table, context.cache_slots, lengths)
    tol = OUTPUT_TOLERANCE[q_dtype]
    t.testing.assert_close(actual.double().cpu(), t.from_numpy(expected), rtol=tol, atol=tol)
    # Identical to the aligned call within the same tolerance (MFMA or grouped kernel).
    aligned = decode_attention_wrapper(q, cache, context)
    t.testing.assert_close(actual.double().cpu(), aligned.double().cpu(), rtol=2 * tol, atol=2 * tol)


@t.inference_mode()
@pytest.mark.parametrize("num_q_heads,num_kv_heads", [(32, 1), (12, 2), (6, 6)])
def test_valu_kernel_head_groups(num_q_heads, num_kv_heads):
    # D 80: a group of 32 q heads per KV head, which the grouped kernel splits into balanced
    # sets of at most four heads per wave; groups of 6 and 1 on the MFMA kernel's narrow rows
    # (the grouped kernel's: test_grouped_kernel_at_head_size_80).
    lengths = [2, 33, 300, 900]
    d = 80
    cache = PagedKVCache(sum(-(-n // 16) for n in lengths) + 4, 16, num_kv_heads, d, "cuda", FP8)
    manager, context, _, _ = fill_decode_batch([cache], lengths, num_kv_heads, d, 16, t.bfloat16, seed=17)
    q = t.randn(len(lengths), num_q_heads, d, device="cuda", dtype=t.float32)
    actual = decode_attention_wrapper(q, cache, context)
    expected = oracle_decode(q, cache, manager.block_table, context.cache_slots, lengths)
    t.testing.assert_close(actual.double().cpu(), t.from_numpy(expected), rtol=1e-4, atol=1e-4)


@t.inference_mode()
@pytest.mark.parametrize("num_q_heads,num_kv_heads,block_size,lengths", [
    (12, 2, 16, [2, 33, 300, 900]),                     # sets of three and three heads per wave
    (6, 6, 16, [2, 33, 300, 900]),                      # one head per wave
    (8, 2, 32, [3, 40, 129, 700]),
    (8, 2, 256, [3, 40, 129, 700, 1100]),               # a page holds a whole chunk
    (8, 2, 512, [3, 40, 129, 700, 1100]),
])
def test_grouped_kernel_at_head_size_80(num_q_heads, num_kv_heads, block_size, lengths):
    """Caches 4 bytes past a 16-byte boundary, which the MFMA kernel does not take: the grouped kernel's
    slices of 20 at uneven head groups and at pages of a chunk and more."""
    d = 80
    cache = PagedKVCache(sum(-(-n // block_size) for n in lengths) + 4, block_size, num_kv_heads, d, "cuda", FP8)
    manager, context, _, _ = fill_decode_batch([cache], lengths, num_kv_heads, d, block_size, t.bfloat16, seed=17)
    q = t.randn(len(lengths), num_q_heads, d, device="cuda", dtype=t.float32)
    read = PagedKVRead(_shifted(cache.k, 4), _shifted(cache.v, 4), cache.k_scales, cache.v_scales,
                       manager.block_table, context.cache_slots, context.context_lengths, block_size)
    actual = decode_attention_wrapper(q, read)
    expected = oracle_decode(q, cache, manager.block_table, context.cache_slots, lengths)
    t.testing.assert_close(actual.double().cpu(), t.from_numpy(expected), rtol=1e-4, atol=1e-4)


@t.inference_mode()
def test_golden_cfg1_decode():
    g = np.load(GOLDEN / "cfg1_decode.npz")
    nb = int(g["num_blocks"])
    hkv, d = (int(x) for x in g["k_codes"].shape[1:])
    cache = PagedKVCache(nb, 16, hkv, d, "cuda", FP8)
    ks = t.from_numpy(g["ks_bf16_bits"]).view(t.bfloat16).cuda()
    vs = t.from_numpy(g["vs_bf16_bits"]).view(t.bfloat16).cuda()
    cache.append_kv(t.from_numpy(g["blocks"]).cuda(), t.from_numpy(g["offsets"]).cuda(), ks, vs)
    q = t.from_numpy(g["q_bf16_bits"]).view(t.bfloat16).cuda()
    table = t.from_numpy(g["block_table"]).cuda()
    lengths = t.from_numpy(g["lengths"]).cuda()
    read = PagedKVRead(cache.k, cache.v, cache.k_scales, cache.v_scales, table,
                       t.arange(len(lengths), device="cuda"), lengths, 16)
    out = decode_attention_wrapper(q, read)
    t.testing.assert_close(out.double().cpu(), t.from_numpy(g["expected_out"]),
                           rtol=NORTH_STAR_RTOL, atol=NORTH_STAR_ATOL)


def _run_config(name):
    """Fill the cache the workload way (history, then one appended token), decode, and
    check the cache bytes and every output row against the oracle."""
    spec = workloads.spec(name)
    w = workloads.build(spec, "cuda")
    cache = PagedKVCache(w.num_blocks, 16, spec.num_kv_heads, spec.head_dim, "cuda", FP8)
    hist_k, hist_v = workloads.fill_cache(w, cache, "cuda")
    new_k, new_v = workloads.new_kv(w, "cuda")
    cache.append_kv(w.new_blocks, w.new_offsets, new_k, new_v)
    out = decode_attention_wrapper(w.q, cache, workloads.make_context(w))
    assert out.shape == w.q.shape and out.dtype == t.bfloat16
    assert t.isfinite(out.float()).all()

    # Cache bytes of the appended tokens and a sample of history tokens are bit-exact.
    g = t.Generator().manual_seed(0)
    pick = t.randperm(hist_k.shape[0], generator=g)[:4096].cuda()
    for blocks, offsets, k, v in ((w.new_blocks, w.new_offsets, new_k, new_v),
                                  (w.history_blocks[pick], w.history_offsets[pick], hist_k[pick], hist_v[pick])):
        for x, codes, scales in ((k, cache.k, cache.k_scales), (v, cache.v, cache.v_scales)):
            o_codes, o_scales = oracle.quantize(x.float().cpu().numpy())
            assert np.array_equal(codes[blocks, offsets].view(t.uint8).cpu().numpy(), o_codes)
            assert np.array_equal(scales[blocks, offsets].cpu().numpy(), o_scales)
    del hist_k, hist_v

    # Every row against the float64 oracle over the dequantized cache.
    expected = oracle_decode(w.q, cache, w.block_table, w.cache_slots, spec.lengths)
    t.testing.assert_close(out.double().cpu(), t.from_numpy(expected), rtol=NORTH_STAR_RTOL, atol=NORTH_STAR_ATOL)
    return out


@t.inference_mode()
def test_config2_full_size():
    _run_config("cfg2")


@t.inference_mode()
def test_north_star_full_size():
    _run_config("north")


@t.inference_mode()
def test_config3_long_context_outliers():
    _run_config("cfg3")


@t.inference_mode()
def test_config4_heavy_tail():
    _run_config("cfg4")


@t.inference_mode()
def test_reused_slot_never_reads_its_previous_owner():
    """Slot and page reuse through the decode kernel (reference tests/test_inference.py:35-69,
    114-131): a request is freed and a shorter one takes its slot and its pages, whose
    bytes past the new length still hold the old request's tokens. A decode step of the
    new request (its token written by the fused call) must attend over its own history
    only, and the other live request must be unaffected."""
    from aiproj_amd.kernals.decode_attention import append_decode_attention

    hq, hkv, d, bs = 32, 8, 128, 16
    manager = PageAllocator(64, bs, 3, 512, "cuda")
    cache = PagedKVCache(64, bs, hkv, d, "cuda", FP8)
    g = t.Generator(device="cuda").manual_seed(15)

    def fill(rid, n, scale):
        manager.allocate_request(rid, n + 1)
        k = t.randn(n, hkv, d, device="cuda", generator=g, dtype=t.bfloat16) * scale
        v = t.randn(n, hkv, d, device="cuda", generator=g, dtype=t.bfloat16) * scale
        manager.append_request(rid, t.arange(n, device="cuda"), k, v, cache)
        manager.advance(rid, n)

    fill(0, 300, 50.0)        # the old owner: large values, easy to see if they leak
    fill(1, 200, 1.0)
    old_slot = manager.get_slot(0)
    manager.free_request(0)
    fill(2, 37, 1.0)
    assert manager.get_slot(2) == old_slot
    rids = [2, 1]
    slots = t.tensor([manager.get_slot(r) for r in rids], device="cuda")
    positions = t.tensor([manager.get_seq_len(r) for r in rids], device="cuda")
    ctx = manager.create_container(slots, t.arange(3, dtype=t.int32, device="cuda"), positions)
    assert ctx.appends_last_position and ctx.context_lengths.tolist() == [38, 201]
    q = t.randn(2, hq, d, device="cuda", generator=g, dtype=t.bfloat16)
    k = t.randn(2, hkv, d, device="cuda", generator=g, dtype=t.bfloat16)
    v = t.randn(2, hkv, d, device="cuda", generator=g, dtype=t.bfloat16)
    out = append_decode_attention(q, k, v, cache, ctx)
    expected = oracle_decode(q, cache, manager.block_table, slots, [38, 201])
    t.testing.assert_close(out.double().cpu(), t.from_numpy(expected), rtol=NORTH_STAR_RTOL, atol=NORTH_STAR_ATOL)
    assert out.float().abs().max().item() < 8.0       # no trace of the x50 tokens


@t.inference_mode()
def test_decode_split_invariance():
    # One sequence decoded alone and inside a batch of others: the work split moves
    # (workgroups take equal shares of the whole batch's tiles), so only the last
    # bits may change; a repeated call on the same batch is bit-identical.
    lengths = [2500, 40, 900]
    cache = PagedKVCache(sum(-(-n // 16) for n in lengths) + 4, 16, 8, 128, "cuda", FP8)
    manager, context, _, _ = fill_decode_batch([cache], lengths, 8, 128, 16, t.bfloat16, seed=12)
    q = t.randn(3, 32, 128, device="cuda", dtype=t.bfloat16)
    batch = decode_attention_wrapper(q, cache, context)
    assert t.equal(batch, decode_attention_wrapper(q, cache, context))
    for row in range(3):
        read = PagedKVRead(cache.k, cache.v, cache.k_scales, cache.v_scales, manager.block_table,
                           context.cache_slots[row:row + 1], context.context_lengths[row:row + 1], 16)
        alone = decode_attention_wrapper(q[row:row + 1], read)
        t.testing.assert_close(alone[0].float(), batch[row].float(), rtol=1e-2, atol=4e-3)


@t.inference_mode(False)
@pytest.mark.parametrize("hq,hkv,lengths", [
    (32, 8, [2500, 40, 900, 1, 333]),
    (16, 4, [2500, 40, 900, 1, 333, 4000, 3500, 120]),     # replicated heads
])
def test_graph_capture_replays_match_eager(hq, hkv, lengths):
    # The decode step (append + decode + combine) captured once in a HIP graph and
    # replayed several times, with eager work and synchronizations in between,
    # gives the eager bits on every replay.
    cache = PagedKVCache(sum(-(-n // 16) for n in lengths) + 8, 16, hkv, 128, "cuda", FP8)
    manager, context, _, _ = fill_decode_batch([cache], lengths, hkv, 128, 16, t.bfloat16, seed=13)
    q = t.randn(len(lengths), hq, 128, device="cuda", dtype=t.bfloat16)
    blocks = context.physical_blocks[:len(lengths)].clone()
    offsets = context.block_offsets[:len(lengths)].clone()
    new_k = t.randn(len(lengths), hkv, 128, device="cuda", dtype=t.bfloat16)
    new_v = t.randn_like(new_k)

    def step():
        cache.append_kv(blocks, offsets, new_k, new_v)
        return decode_attention_wrapper(q, cache, context)

    eager = step().clone()
    t.cuda.synchronize()
    graph = t.cuda.CUDAGraph()
    with t.cuda.graph(graph):
        out = step()
    for _ in range(4):
        cache.k.view(t.uint8)[blocks, offsets] = 0       # eager work the replay must undo
        graph.replay()
        t.cuda.synchronize()
        assert t.equal(out, eager)
        assert t.equal(eager, step())


@t.inference_mode()
def test_back_to_back_calls_read_fresh_partial_states():
    # Two calls with equal shapes reuse the same workspace block from the caching
    # allocator; the second must merge its own partial states, never the first's.
    lengths = [3000, 2000, 17, 1000]
    cache = PagedKVCache(sum(-(-n // 16) for n in lengths) + 8, 16, 8, 128, "cuda", FP8)
    manager, context, _, _ = fill_decode_batch([cache], lengths, 8, 128, 16, t.bfloat16, seed=14)
    outs, qs = [], []
    for i in range(3):
        q = t.randn(len(lengths), 32, 128, device="cuda", dtype=t.bfloat16) * (1 + i)
        qs.append(q)
        outs.append(decode_attention_wrapper(q, cache, context))
    for q, out in zip(qs, outs):
        expected = oracle_decode(q, cache, manager.block_table, context.cache_slots, lengths)
        t.testing.assert_close(out.double().cpu(), t.from_numpy(expected),
                               rtol=OUTPUT_TOLERANCE[t.bfloat16], atol=OUTPUT_TOLERANCE[t.bfloat16])


@t.inference_mode()
@pytest.mark.parametrize("cache_dtype,head_dim", [(FP8, 128), (FP8, 64), (t.bfloat16, 128), (t.float16, 80)])
def test_split_then_reduce_equals_one_call(cache_dtype, head_dim):
    # kvfp8_paged_decode_split followed by kvfp8_paged_decode_reduce on the same
    # workspace gives the bits of kvfp8_paged_decode (MFMA and generic kernels);
    # sequences the split kernel finishes whole are final before the reduce.
    from aiproj_amd.kernals.decode_attention import prepare_decode

    lengths = [3000, 17, 0, 1000, 1]
    cache = PagedKVCache(sum(-(-n // 16) for n in lengths) + 8, 16, 8, head_dim, "cuda", cache_dtype)
    nonzero = [max(n, 1) for n in lengths]
    manager, context, _, _ = fill_decode_batch([cache], nonzero, 8, head_dim, 16, t.bfloat16, seed=15)
    context.context_lengths.copy_(t.tensor(lengths, dtype=context.context_lengths.dtype))
    q = t.randn(len(lengths), 32, head_dim, device="cuda", dtype=t.bfloat16)
    whole = decode_attention_wrapper(q, cache, context)
    call = prepare_decode(q, cache, context)
    call.output.fill_(float("nan"))
    call.split()
    call.reduce()
    assert t.equal(call.output, whole)
    assert t.equal(whole[2], t.zeros_like(whole[2]))


def test_launches_follow_the_current_stream():
    """The handle passed to the C ABI is torch's current stream, default or not, and a
    decode enqueued under another stream runs there (its output is ready once that
    stream is synchronized)."""
    from aiproj_amd import _native

    dev = t.device("cuda")
    assert _native.stream_handle(dev) == t.cuda.current_stream(dev).cuda_stream
    side = t.cuda.Stream()
    w = workloads.build(workloads.spec("cfg1"), "cuda")
    cache = PagedKVCache(w.num_blocks, 16, w.spec.num_kv_heads, w.spec.head_dim, "cuda", FP8)
    workloads.fill_cache(w, cache, "cuda")
    k_new, v_new = workloads.new_kv(w, "cuda", 0)
    cache.append_kv(w.new_blocks, w.new_offsets, k_new, v_new)
    ctx = workloads.make_context(w)
    want = decode_attention_wrapper(w.q, cache, ctx)
    assert bool(t.isfinite(want).all())
    t.cuda.synchronize()
    side.wait_stream(t.cuda.current_stream())
    with t.cuda.stream(side):
        assert _native.stream_handle(dev) == side.cuda_stream
        assert _native.stream_handle(t.device("cuda", t.cuda.current_device())) == side.cuda_stream
        got = decode_attention_wrapper(w.q, cache, ctx)
    side.synchronize()
    assert t.equal(got, want)
    assert _native.stream_handle(dev) == t.cuda.current_stream(dev).cuda_stream


@t.inference_mode()
def test_large_batch_with_sixteen_kv_heads():
    """4,200 sequences x 16 KV heads (two waves per KV head slot of a workgroup): split
    then reduce equals the single call bit for bit, and sampled rows match the oracle."""
    from aiproj_amd.kernals.decode_attention import prepare_decode

    batch, hkv, hq, d = 4200, 16, 32, 64
    lengths = [(i * 37) % 300 + 1 for i in range(batch)]
    spec = workloads.WorkloadSpec("wide", batch, hq, hkv, d, lengths, seed=16)
    w = workloads.build(spec, "cuda")
    cache = PagedKVCache(w.num_blocks, 16, hkv, d, "cuda", FP8)
    workloads.fill_cache(w, cache, "cuda")
    k, v = workloads.new_kv(w, "cuda")
    cache.append_kv(w.new_blocks, w.new_offsets, k, v)
    ctx = workloads.make_context(w)
    whole = decode_attention_wrapper(w.q, cache, ctx)
    call = prepare_decode(w.q, cache, ctx)
    call.output.fill_(float("nan"))
    call.split()
    call.reduce()
    assert t.equal(call.output.view(t.int16), whole.view(t.int16))
    rows = [0, 1, 777, batch - 1]
    expected = oracle_decode(w.q, cache, w.block_table, w.cache_slots, lengths, rows=rows)
    t.testing.assert_close(whole[rows].double().cpu(), t.from_numpy(expected), rtol=NORTH_STAR_RTOL,
                           atol=NORTH_STAR_ATOL)


@t.inference_mode()
@pytest.mark.parametrize("hq,hkv,d,batch,long_len,cache_dtype,block_size", [
    (16, 4, 128, 3839, 0, FP8, 16),      # the largest batch whose tables leave room for the replicas' merge buffer
    (16, 4, 128, 3841, 0, FP8, 16),      # one table entry over: one wave per head
    (8, 2, 64, 5887, 0, FP8, 16),        # the same boundary at D 64
    (16, 4, 128, 3, 9000, FP8, 16),      # one long sequence cut into many workgroups' pieces
    (8, 1, 128, 12, 6000, FP8, 16),
    (16, 2, 64, 8, 4100, FP8, 16),
    (16, 4, 128, 3, 9000, t.bfloat16, 16),
    (16, 2, 64, 8, 4100, t.bfloat16, 16),
    (16, 4, 128, 40, 3000, FP8, 64),     # pages of 4 tiles
    (8, 2, 128, 24, 5000, t.bfloat16, 32),
    (16, 4, 128, 3, 9000, t.float16, 16),    # f16 cache read with f16 q (f16 products)
])
def test_replicated_heads(hq, hkv, d, batch, long_len, cache_dtype, block_size):
    """Fewer than 8 KV heads (dividing 8) run 8 waves per workgroup, 8 / Hkv replicas
    of each head that merge their softmax states at the end of every segment, when
    the merge buffer fits in LDS beside the batch-sized tables and the batch's tile
    capacity (batch x table width) is at least 2 x 8 / Hkv tiles per CU (every case
    here). Both sides of that LDS boundary, and sequences cut into pieces shorter than
    the replicas' stride (replicas with no step), against float32
    dequantize-then-attend and the oracle; split then reduce equals the single call
    bit for bit."""
    from aiproj_amd.kernals.decode_attention import prepare_decode
    from tests.helpers import torch_paged_decode

    lengths = [(i * 53) % 97 + 1 for i in range(batch)]
    if long_len:
        lengths[1] = long_len
    spec = workloads.WorkloadSpec("replicas", batch, hq, hkv, d, lengths, seed=23, block_size=block_size)
    w = workloads.build(spec, "cuda")
    cache = PagedKVCache(w.num_blocks, block_size, hkv, d, "cuda", cache_dtype)
    workloads.fill_cache(w, cache, "cuda")
    k, v = workloads.new_kv(w, "cuda")
    cache.append_kv(w.new_blocks, w.new_offsets, k, v)
    ctx = workloads.make_context(w)
    q = w.q.to(t.float16) if cache_dtype == t.float16 else w.q
    out = decode_attention_wrapper(q, cache, ctx)
    ref = torch_paged_decode(q, cache, w.cache_slots, ctx.context_lengths, w.block_table)
    t.testing.assert_close(out.float(), ref, rtol=NORTH_STAR_RTOL, atol=NORTH_STAR_ATOL)
    call = prepare_decode(q, cache, ctx)
    call.output.fill_(float("nan"))
    call.split()
    call.reduce()
    assert t.equal(call.output.view(t.int16), out.view(t.int16))
    rows = sorted({0, 1, batch - 1})
    expected = oracle_decode(q, cache, w.block_table, w.cache_slots, lengths, rows=rows)
    t.testing.assert_close(out[rows].double().cpu(), t.from_numpy(expected), rtol=NORTH_STAR_RTOL,
                           atol=NORTH_STAR_ATOL)


@t.inference_mode()
@pytest.mark.parametrize("head_dim", [64, 80])
def test_maximum_batch(head_dim):
    """8,191 sequences, the most the decode kernels' LDS tile prefix holds (8,192 is
    refused on the host, tests/test_native_abi.py): D 64 on the MFMA kernel (its
    prefix and sequence metadata take 64 KB of LDS), D 80 on its narrow rows (and the
    same bytes 4 off a 16-byte boundary on the grouped VALU kernel).
    Every row against float32 dequantize-then-attend, sampled rows against the oracle."""
    from tests.helpers import torch_paged_decode

    batch, hq, hkv = 8191, 8, 2
    lengths = [(i * 29) % 45 + 1 for i in range(batch)]
    spec = workloads.WorkloadSpec("max_batch", batch, hq, hkv, head_dim, lengths, seed=18)
    w = workloads.build(spec, "cuda")
    cache = PagedKVCache(w.num_blocks, 16, hkv, head_dim, "cuda", FP8)
    workloads.fill_cache(w, cache, "cuda")
    k, v = workloads.new_kv(w, "cuda")
    cache.append_kv(w.new_blocks, w.new_offsets, k, v)
    ctx = workloads.make_context(w)
    out = decode_attention_wrapper(w.q, cache, ctx)
    assert t.isfinite(out).all()
    ref = torch_paged_decode(w.q, cache, w.cache_slots, ctx.context_lengths, w.block_table)
    t.testing.assert_close(out.float(), ref, rtol=NORTH_STAR_RTOL, atol=NORTH_STAR_ATOL)
    if head_dim == 80:
        read = PagedKVRead(_shifted(cache.k, 4), _shifted(cache.v, 4), cache.k_scales, cache.v_scales, w.block_table,
                           ctx.cache_slots, ctx.context_lengths, 16)
        t.testing.assert_close(decode_attention_wrapper(w.q, read).float(), ref, rtol=NORTH_STAR_RTOL,
                               atol=NORTH_STAR_ATOL)
    rows = [0, 1, 4095, batch - 1]
    expected = oracle_decode(w.q, cache, w.block_table, w.cache_slots, lengths, rows=rows)
    t.testing.assert_close(out[rows].double().cpu(), t.from_numpy(expected), rtol=NORTH_STAR_RTOL,
                           atol=NORTH_STAR_ATOL)


@t.inference_mode()
@pytest.mark.parametrize("cache_dtype", [FP8, t.bfloat16])
def test_head_dim_512(cache_dtype):
    # The largest head size the library takes (513 is refused on the host). D 512
    # splits into none of the grouped kernel's slice widths, so it runs on the
    # per-q-head VALU kernel; f32 q against the oracle at the reference's tolerance.
    lengths = [1, 17, 300, 700]
    hq, hkv, d = 4, 1, 512
    cache = PagedKVCache(sum(-(-n // 16) for n in lengths) + 4, 16, hkv, d, "cuda", cache_dtype)
    manager, context, _, _ = fill_decode_batch([cache], lengths, hkv, d, 16, t.bfloat16, seed=19)
    q = t.randn(len(lengths), hq, d, device="cuda", dtype=t.float32)
    actual = decode_attention_wrapper(q, cache, context)
    expected = oracle_decode(q, cache, manager.block_table, context.cache_slots, lengths)
    t.testing.assert_close(actual.double().cpu(), t.from_numpy(expected), rtol=1e-4, atol=1e-4)


@t.inference_mode()
@pytest.mark.parametrize("head_dim", [64, 128])
@pytest.mark.parametrize("num_q_heads,num_kv_heads", [(8, 2), (32, 8), (16, 1), (4, 4)])
def test_f16_cache_decode(head_dim, num_q_heads, num_kv_heads):
    # An f16 cache read with f16 q runs on f16 matrix products (both operands exact in
    # f16); with bf16 or f32 q it runs on the VALU kernel. Each against the oracle at
    # the reference's tolerance for its q dtype.
    block_size = 16
    num_blocks = sum(-(-n // 16) for n in DECODE_LENGTHS) + 4
    cache = PagedKVCache(num_blocks, block_size, num_kv_heads, head_dim, "cuda", t.float16)
    manager, context, _, _ = fill_decode_batch([cache], DECODE_LENGTHS, num_kv_heads, head_dim, block_size,
                                               t.float16, seed=20)
    base = t.randn(len(DECODE_LENGTHS), num_q_heads, head_dim, device="cuda")
    for q_dtype in (t.float16, t.bfloat16, t.float32):
        q = base.to(q_dtype)
        actual = decode_attention_wrapper(q, cache, context)
        assert actual.dtype == q_dtype
        expected = oracle_decode(q, cache, manager.block_table, context.cache_slots, DECODE_LENGTHS)
        tol = OUTPUT_TOLERANCE[q_dtype]
        t.testing.assert_close(actual.double().cpu(), t.from_numpy(expected), rtol=tol, atol=tol)
