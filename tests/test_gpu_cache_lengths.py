"""Valid lengths raised by the cache producer over ragged ranges.

Only an entry's last token of a range raises its page_valid_len; every range
must leave the lengths that raising it for each written token would.
"""

from __future__ import annotations

import pytest
import torch

from aws_training_study_amd.pcp_attention import (
    KVCacheWriter,
    PCPAttentionConfig,
    build_page_pool,
    owner_and_local_position,
)

pytestmark = pytest.mark.gpu

# (pcp, interleave, block): powers of two, one rank, the general index maps
LAYOUTS = [(4, 16, 128), (1, 64, 64), (16, 64, 512), (3, 48, 192), (5, 1, 64)]
# (first position, tokens): one token, chunk and block edges, ragged, everything
RANGES = [(0, 1), (63, 1), (47, 2), (64, 64), (127, 130), (1, 700), (0, None)]


@pytest.mark.parametrize("pcp,il,block", LAYOUTS)
@pytest.mark.parametrize("kv_dtype", ["fp8_e4m3fn", "bfloat16"])
def test_valid_lengths_of_ragged_ranges(pcp, il, block, kv_dtype, cuda_device):
    bucket = pcp * il * max(1, 2 * block // il)
    cfg = PCPAttentionConfig(pcp_size=pcp, current_len=pcp * il, max_history_len=bucket, actual_history_len=bucket,
                             block_size=block, interleave_size=il, num_q_heads=2, num_kv_heads=1, head_dim=64,
                             backend="hip", kv_dtype=kv_dtype).validate()
    writer = KVCacheWriter(cfg)
    table = torch.arange(cfg.num_pages, dtype=torch.int32, device=cuda_device).reshape(pcp, -1)
    table[0, -1] = -1  # an entry without a page: not written, not raised
    dtype = torch.float8_e4m3fn if kv_dtype == "fp8_e4m3fn" else torch.bfloat16
    for first, n in RANGES:
        n = bucket - first if n is None else min(n, bucket - first)
        if n <= 0:
            continue
        pool = torch.zeros((cfg.num_pages, cfg.page_elements), dtype=dtype, device=cuda_device)
        valid = torch.zeros((pcp, cfg.max_local_blocks), dtype=torch.int32, device=cuda_device)
        valid[pcp - 1, 0] = 5  # a longer prefix written before stays
        x = torch.ones((1, n, 64), dtype=torch.bfloat16, device=cuda_device)
        writer(x, x, pool, table, first_pos=first, page_valid_len=valid)
        want = torch.zeros((pcp, cfg.max_local_blocks), dtype=torch.int32)
        want[pcp - 1, 0] = 5
        for p in range(first, first + n):
            rank, local = owner_and_local_position(p, pcp, il)
            blk, slot = divmod(local, block)
            if (rank, blk) != (0, cfg.max_local_blocks - 1):
                want[rank, blk] = max(int(want[rank, blk]), slot + 1)
        assert torch.equal(valid.cpu(), want), (first, n)


@pytest.mark.parametrize("pcp,il,block", LAYOUTS)
@pytest.mark.parametrize("kv_dtype,kv_scale", [("fp8_e4m3fn", "per_tensor"), ("fp8_e4m3fn", "none"), ("bfloat16", "none")])
def test_fresh_pool_equals_a_write_into_zeros(pcp, il, block, kv_dtype, kv_scale, cuda_device):
    """build_page_pool clears only what it does not write: slots past a ragged
    length and the pages of a hole in the table."""
    bucket = pcp * il * max(1, 2 * block // il)
    cfg = PCPAttentionConfig(pcp_size=pcp, current_len=pcp * il, max_history_len=bucket, actual_history_len=bucket,
                             block_size=block, interleave_size=il, num_q_heads=2, num_kv_heads=2, head_dim=64,
                             backend="hip", kv_dtype=kv_dtype).validate()
    dtype = torch.float8_e4m3fn if kv_dtype == "fp8_e4m3fn" else torch.bfloat16
    gen = torch.Generator(device=cuda_device).manual_seed(pcp)
    identity = torch.arange(cfg.num_pages, device=cuda_device).reshape(pcp, -1)
    holes = identity.clone()
    holes[0, -1] = -1
    for n in (1, 63, bucket // 2 + 1, bucket):
        k, v = (torch.randn((2, n, 64), generator=gen, device=cuda_device, dtype=torch.bfloat16) for _ in range(2))
        if n == 63:
            k[0, 5, 5] = float("nan")  # an amax of NaN: unit scale
        for table in (identity, holes.int(), identity.flip(1).cpu()):
            # freed memory that is not zero, for the pool to land in
            torch.full((cfg.num_pages, cfg.page_elements * dtype.itemsize), 255, dtype=torch.uint8, device=cuda_device)
            pool, k_scale, v_scale, valid = build_page_pool(cfg, k, v, table, kv_scale=kv_scale)
            want = torch.zeros((cfg.num_pages, cfg.page_elements), dtype=dtype, device=cuda_device)
            lens = torch.zeros((pcp, cfg.max_local_blocks), dtype=torch.int32, device=cuda_device)
            KVCacheWriter(cfg)(k, v, want, table.to(cuda_device, torch.int32), k_scale=k_scale, v_scale=v_scale,
                               page_valid_len=lens)
            assert torch.equal(pool.view(torch.uint8), want.view(torch.uint8)), n
            assert torch.equal(valid, lens), n
            if kv_scale == "per_tensor":
                for x, scale in ((k, k_scale), (v, v_scale)):
                    amax = float(x.float().abs().max())
                    assert scale == (amax / 448.0 if amax > 0 else 1.0)
    if kv_scale == "per_tensor":
        k[0, 0, 0] = float("inf")
        with pytest.raises(RuntimeError, match="BAD_SCALE"):
            build_page_pool(cfg, k, v, identity)
