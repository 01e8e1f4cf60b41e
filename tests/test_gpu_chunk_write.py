"""The single-request KV write (``write_chunk_kv``, slots taken from the block table inside the kernel) and the
slot mapping kernel, bit-exact against the CPU oracle: chunks of one token to several pages, starting on either
side of a page border, with negative (padding) and out-of-range pages, row-strided K / V; and every form of block
table that the native path does not take, which must give the same slots.
"""

from __future__ import annotations

import ctypes

import numpy as np
import pytest
import torch

from oracle import cache as OC
from trianglemix import cache, native


def _tables(table: torch.Tensor) -> dict:
    """The same pages as int32 and in the forms the native ops leave to tensor operations."""
    wide = torch.zeros(1, 2 * table.size(1), dtype=torch.int32, device=table.device)
    wide[:, ::2] = table
    return {"int32": table, "int64": table.to(torch.int64), "strided": wide[:, ::2]}


def test_forms_the_native_path_leaves_to_tensor_operations():
    """On the CPU nothing is native; every form gives the oracle's slots, and bad positions are refused."""
    table = torch.tensor([[4, 0, 2, 9]], dtype=torch.int32)
    for start, n in ((0, 1), (127, 2), (130, 300), (511, 1), (5, 0)):
        want = OC.chunk_slots(table, start, n)
        for name, t in _tables(table).items():
            assert not cache._native_table(t, start, n), name
            assert np.array_equal(cache.chunk_slot_mapping(t, start, n).numpy(), want), (name, start, n)
    for start, n in ((-1, 2), (0, -1), (512, 1), (0, 513)):
        with pytest.raises(ValueError):
            cache.chunk_slot_mapping(table, start, n)
        if n >= 0:
            rows = torch.zeros(n, 8, 128, dtype=torch.bfloat16)
            with pytest.raises(ValueError):
                cache.write_chunk_kv(rows, rows, None, None, table, start)


def test_messages_name_the_index_that_was_passed():
    """The refusals of the C entry points: every check runs before any GPU call."""
    lib = native.load_hip_library()
    raw = ctypes.CDLL(str(native.HIP_LIBRARY))
    p, i64 = ctypes.c_void_p, ctypes.c_int64
    raw.tmi_write_chunk_kv.argtypes = [p] * 5 + [i64] * 6 + [p]
    raw.tm_reshape_and_cache.argtypes = [p] * 5 + [i64] * 4 + [p]
    page = 128 * 8 * 128 * 2
    key, value, kc, vc = 1 << 20, 2 << 20, 3 << 20, (3 << 20) + page
    for index, message in ((None, "must be non-null"), (kc, "must not overlap")):
        assert raw.tmi_write_chunk_kv(key, value, kc, vc, index, 1, 0, 1, 1024, 1024, 1, None) == 1
        error = lib.tm_last_error().decode()
        assert message in error and "block_table" in error and "slot_mapping" not in error
        assert raw.tm_reshape_and_cache(key, value, kc, vc, index, 1, 1024, 1024, 1, None) == 1
        error = lib.tm_last_error().decode()
        assert message in error and "slot_mapping" in error


@pytest.mark.gpu
@pytest.mark.parametrize("start,n", [(0, 1), (127, 1), (128, 1), (127, 2), (1, 127), (64, 129), (300, 513), (0, 1024)])
def test_chunk_write_matches_oracle_bit_exact(gpu, start, n):
    print(f"chunk write start={start} tokens={n}", flush=True)
    native.require_adapter()
    g = torch.Generator().manual_seed(1000 * start + n)
    pages = 12
    table = torch.randperm(pages, generator=g)[:9].to(torch.int32).view(1, -1)
    if n > 300:
        table[0, 3], table[0, 4] = -1, pages  # padding page, page past the cache: neither is written
    qkv = torch.randn(n, 48, 128, generator=g).to(torch.bfloat16)
    key, value = qkv[:, 32:40], qkv[:, 40:48]
    kc = torch.randn(pages, 128, 8, 128, generator=g).to(torch.bfloat16)
    vc = torch.randn(pages, 128, 8, 128, generator=g).to(torch.bfloat16)
    t = np.arange(start, start + n)
    slots = table[0].numpy().astype(np.int64)[t // 128] * 128 + t % 128
    kk, vv = kc.clone(), vc.clone()
    OC.reshape_and_cache(key.contiguous().view(torch.int16).numpy(), value.contiguous().view(torch.int16).numpy(),
                         kk.view(torch.int16).numpy(), vv.view(torch.int16).numpy(), slots)
    qkv_d, table_d = qkv.to(gpu), table.to(gpu)
    assert cache._native_table(table_d, start, n)
    for name, tb in _tables(table_d).items():
        assert np.array_equal(cache.chunk_slot_mapping(tb, start, n).cpu().numpy(), slots), name
        kd, vd = kc.to(gpu), vc.to(gpu)
        cache.write_chunk_kv(qkv_d[:, 32:40], qkv_d[:, 40:48], kd, vd, tb, start)
        torch.cuda.synchronize()
        assert torch.equal(kd.cpu().view(torch.int16), kk.view(torch.int16)), name
        assert torch.equal(vd.cpu().view(torch.int16), vv.view(torch.int16)), name


@pytest.mark.gpu
def test_chunk_write_refuses_what_the_mapped_write_refuses(gpu):
    native.require_adapter()
    table = torch.tensor([[1, 0]], dtype=torch.int32, device=gpu)
    rows = torch.zeros(4, 8, 128, dtype=torch.bfloat16, device=gpu)
    kc = torch.zeros(3, 128, 8, 128, dtype=torch.bfloat16, device=gpu)
    vc = torch.zeros_like(kc)
    with pytest.raises(RuntimeError, match="BF16"):
        cache.write_chunk_kv(rows.half(), rows, kc, vc, table, 0)
    with pytest.raises(RuntimeError, match="num_tokens, 8, 128"):
        cache.write_chunk_kv(rows[:, :4], rows[:, :4], kc, vc, table, 0)
    with pytest.raises(RuntimeError):
        cache.write_chunk_kv(rows, rows, kc, kc, table, 0)  # the caches overlap
    with pytest.raises(RuntimeError, match="and block_table must be GPU tensors"):
        torch.ops.trianglemix.write_chunk_kv(rows, rows, kc, vc, table.cpu(), 0)
    with pytest.raises(RuntimeError, match="lacks logical pages"):
        torch.ops.trianglemix.write_chunk_kv(rows, rows, kc, vc, table, 253)
    cache.write_chunk_kv(rows[:0], rows[:0], kc, vc, table, 256)  # nothing to write
    # a block table inside a cache page that the write overwrites is read before it is
    flat = kc.view(-1).view(torch.int32)
    inner = flat[:2].view(1, 2)
    inner.copy_(table)
    rows.fill_(1.0)
    cache.write_chunk_kv(rows, rows, kc, vc, inner, 126)
    torch.cuda.synchronize()
    slots = torch.tensor([254, 255, 0, 1], device=gpu)
    assert (vc.view(-1, 8, 128)[slots] == 1).all() and vc.sum() == 4 * 1024
