"""The e4m3 kernel's workgroup shapes.

Launches of few rows run workgroups of 128 rows and four waves, larger ones
256 rows and eight waves.  A row's arithmetic does not depend on the shape, so
the same rows must come out bit for bit from a small and from a large launch;
both end inside row tiles and key tiles.  (head_dim 256; at 64 and 128 the tile
kernel has one shape, and the launches differ in the tiles that a row shares.)
"""

from __future__ import annotations

import pytest
import torch

from aws_training_study_amd.pcp_attention import PCPAttentionConfig, build_page_pool, make_history_attention_kernel

pytestmark = pytest.mark.gpu


def _launch(cfg, q, pool, table, valid, scales, **kw):
    return make_history_attention_kernel(cfg)(q, pool, table, page_valid_len=valid, return_lse=True, **scales, **kw)


@pytest.mark.parametrize("head_dim", [64, 128, 256])
@pytest.mark.parametrize("tokens,splits", [(1, 1), (64, 1), (65, 1), (449, 1), (704, 3)])
def test_rows_do_not_depend_on_the_workgroup_shape(head_dim, tokens, splits, cuda_device):
    def config(current):
        return PCPAttentionConfig(pcp_size=1, current_len=current, max_history_len=768, actual_history_len=tokens,
                                  block_size=64, interleave_size=32, num_q_heads=4, num_kv_heads=2,
                                  head_dim=head_dim, backend="hip").validate()

    # 2 Q heads per KV head: 192 rows (2 tiles of 128), and 8288 tokens: 130
    # tiles of 128 rows per KV head, more than one a CU over both heads
    few, many = config(96), config(8288)
    gen = torch.Generator(device=cuda_device).manual_seed(tokens + head_dim)
    k, v = (torch.randn((2, tokens, head_dim), generator=gen, device=cuda_device, dtype=torch.bfloat16)
            for _ in range(2))
    table = torch.randperm(few.num_pages, generator=torch.Generator().manual_seed(3)).to(torch.int32)
    table = table.reshape(1, -1).to(cuda_device)
    pool, k_scale, v_scale, valid = build_page_pool(few, k, v, table)
    scales = dict(k_scale=k_scale, v_scale=v_scale)
    q = torch.randn((1, 4, 8288, head_dim), generator=gen, device=cuda_device, dtype=torch.bfloat16)
    q_few = q[:, :, :96].contiguous()
    for exp2 in ("fast", "exact"):
        kw = dict(precision="fp8", splits=splits, exp2=exp2)
        out, lse = _launch(many, q, pool, table, valid, scales, **kw)
        out_few, lse_few = _launch(few, q_few, pool, table, valid, scales, **kw)
        assert torch.equal(out[:, :, :96], out_few) and torch.equal(lse[:, :, :96], lse_few), exp2
        assert torch.isfinite(out.float()).all()
    # guarded: both list the same rows (a short history: every row or nearly),
    # recomputed with ranges that depend on how many were listed
    out, lse = _launch(many, q, pool, table, valid, scales, splits=splits)
    out_few, lse_few = _launch(few, q_few, pool, table, valid, scales, splits=splits)
    # fixups merged from other ranges differ by bf16 roundings of P (2^-9 of
    # max |V| < 6 each) and of the output
    assert (out[:, :, :96].float() - out_few.float()).abs().max() <= 2 * 2**-9 * 6 + 2**-8 * 6
    assert (lse[:, :, :96] - lse_few).abs().max() <= 1e-4
