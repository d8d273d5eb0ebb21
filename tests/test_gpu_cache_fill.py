"""pcpa_kv_cache_fill on pools that the caller holds, full of 0xFF.

Whatever the fill does not write it clears: slots past the filled ones, pages
that no table entry names, and whole pages where it does not search the table.
"""

from __future__ import annotations

import ctypes

import pytest
import torch

from aws_training_study_amd import _native
from aws_training_study_amd.pcp_attention import KVCacheWriter, PCPAttentionConfig, owner_and_local_position

pytestmark = pytest.mark.gpu

DTYPES = {"fp8_e4m3fn": torch.float8_e4m3fn, "bfloat16": torch.bfloat16}


def _config(pcp, il, block, blocks, kv_dtype, heads=2):
    bucket = pcp * block * blocks
    return PCPAttentionConfig(pcp_size=pcp, current_len=pcp * il, max_history_len=bucket, actual_history_len=bucket,
                              block_size=block, interleave_size=il, num_q_heads=heads, num_kv_heads=heads,
                              head_dim=64, backend="hip", kv_dtype=kv_dtype).validate()


def _fill(cfg, k, v, table, num_tokens=None, amax=None, scales=(1.0, 1.0)):
    """(pool, lengths) of a fill into 0xFF bytes."""
    writer = KVCacheWriter(cfg)
    pool = torch.empty((cfg.num_pages, cfg.page_elements), dtype=DTYPES[cfg.kv_dtype], device=k.device)
    pool.view(torch.uint8).fill_(255)
    valid = torch.full((cfg.pcp_size, cfg.max_local_blocks), -7, dtype=torch.int32, device=k.device)
    params = _native.PcpaParams(num_pages=cfg.num_pages, k_scale=scales[0], v_scale=scales[1], **writer._static)
    if table.dtype == torch.int64:
        params.flags |= _native.FLAG_TABLE_INT64
    _native.check(_native.load_library().pcpa_kv_cache_fill(
        ctypes.byref(params), cfg.interleave_size, k.shape[1] if num_tokens is None else num_tokens, k.data_ptr(),
        v.data_ptr(), None if amax is None else amax.data_ptr(), table.data_ptr(), pool.data_ptr(), valid.data_ptr(),
        torch.cuda.current_stream().cuda_stream))
    return pool, valid


def _written(cfg, k, v, table, scales=(1.0, 1.0)):
    """The same by zeroing first and writing."""
    pool = torch.zeros((cfg.num_pages, cfg.page_elements), dtype=torch.uint8 if cfg.kv_dtype == "fp8_e4m3fn"
                       else torch.bfloat16, device=k.device).view(DTYPES[cfg.kv_dtype])
    valid = torch.zeros((cfg.pcp_size, cfg.max_local_blocks), dtype=torch.int32, device=k.device)
    KVCacheWriter(cfg)(k, v, pool, table, k_scale=scales[0], v_scale=scales[1], page_valid_len=valid)
    return pool, valid


def _same(a, b):
    return all(torch.equal(x.view(torch.uint8), y.view(torch.uint8)) for x, y in zip(a, b))


@pytest.mark.parametrize("kv_dtype", sorted(DTYPES))
@pytest.mark.parametrize("table_dtype", [torch.int32, torch.int64])
@pytest.mark.parametrize("pcp,il,block", [(4, 16, 128), (1, 64, 64), (3, 48, 192), (5, 32, 64)])
def test_ragged_fills(pcp, il, block, table_dtype, kv_dtype, cuda_device):
    cfg = _config(pcp, il, block, 2, kv_dtype)
    gen = torch.Generator(device=cuda_device).manual_seed(7)
    pages = torch.randperm(cfg.num_pages, generator=torch.Generator().manual_seed(pcp)).reshape(pcp, 2)
    outside = pages.clone()
    outside[0, 0], outside[pcp - 1, 1] = -1, cfg.num_pages
    if table_dtype == torch.int64:
        outside[pcp - 1, 1] = 1 << 32
    for n in (1, block - 1, cfg.max_history_len // 2 + 1, cfg.max_history_len):
        k, v = (torch.randn((2, n, 64), generator=gen, device=cuda_device, dtype=torch.bfloat16) for _ in range(2))
        for table in (pages, outside):
            table = table.to(cuda_device, table_dtype)
            assert _same(_fill(cfg, k, v, table, scales=(0.01, 0.02)), _written(cfg, k, v, table, (0.01, 0.02))), n
    # no token: the pool is cleared
    pool, valid = _fill(cfg, k, v, table, num_tokens=0)
    assert not pool.view(torch.uint8).any() and not valid.any()


@pytest.mark.parametrize("table_dtype", [torch.int32, torch.int64])
def test_pages_that_the_table_names_twice(table_dtype, cuda_device):
    """Such a page keeps the longer prefix (the tokens here are all alike)."""
    cfg = _config(4, 16, 128, 2, "bfloat16")
    table = torch.tensor([[0, 1], [1, 0], [2, 2], [5, 5]], device=cuda_device, dtype=table_dtype)  # 3, 4, 6, 7: none
    k = torch.ones((2, 600, 64), device=cuda_device, dtype=torch.bfloat16)
    lens = torch.zeros((4, 2), dtype=torch.int32)
    for p in range(600):
        rank, local = owner_and_local_position(p, 4, 16)
        lens[rank, local // 128] = local % 128 + 1
    pool, valid = _fill(cfg, k, k, table)
    assert torch.equal(valid.cpu(), lens)
    got = pool.float().cpu().reshape(cfg.num_pages, 4, 128, 64)
    for page in range(cfg.num_pages):
        n = max([int(lens[r, b]) for r in range(4) for b in range(2) if int(table[r, b]) == page], default=0)
        assert (got[page, :, :n] == 1).all() and not got[page, :, n:].any(), page


@pytest.mark.parametrize("kv_dtype", sorted(DTYPES))
@pytest.mark.parametrize("pages", [4096, 4097])
def test_many_pages(pages, kv_dtype, cuda_device):
    """2^24 (page, entry) pairs are searched, beyond that whole pages are cleared."""
    cfg = _config(1, 64, 64, pages, kv_dtype, heads=1)
    table = torch.arange(pages, device=cuda_device, dtype=torch.int32).flip(0).reshape(1, -1).contiguous()
    x = torch.randn((1, 64 * 3 + 5, 64), device=cuda_device, dtype=torch.bfloat16)
    amax = x.float().abs().max().expand(2).contiguous()
    scale = float(amax[0]) / 448.0
    got = _fill(cfg, x, x, table, amax=amax if kv_dtype == "fp8_e4m3fn" else None)
    assert _same(got, _written(cfg, x, x, table, (scale, scale)))
    assert got[1].flatten()[:4].tolist() == [64, 64, 64, 5] and int(got[1].sum()) == 64 * 3 + 5
