"""BF16 precision on an FP8 cache at the edges of its key tiles.

The kernel keeps e4m3 tiles in LDS and widens operands as it reads them; at
head_dim 256 the two waves of a SIMD take every other 64-key tile.  Histories
of one tile, of odd and even tile counts and ending inside either wave's tile
are compared with float64 attention on the dequantised cache.
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

from aws_training_study_amd.pcp_attention import PCPAttentionConfig, make_history_attention_kernel
from aws_training_study_amd.pcp_attention.workloads import build_paged_problem
from oracle import pcp_oracle as orc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tokens", [1, 63, 64, 65, 127, 128, 129, 192, 255, 577])
@pytest.mark.parametrize("head_dim,splits", [(64, 1), (128, 1), (256, 1), (256, 3)])
def test_bf16_precision_at_tile_edges(tokens, head_dim, splits, cuda_device):
    cfg = PCPAttentionConfig(pcp_size=1, current_len=96, max_history_len=640, actual_history_len=tokens, block_size=64,
                             interleave_size=32, num_q_heads=4, num_kv_heads=2, head_dim=head_dim,
                             backend="hip").validate()
    problem = build_paged_problem(cfg, seed=tokens, kv_scale="per_tensor")
    gpu = problem.to(cuda_device)
    out, lse = make_history_attention_kernel(cfg)(
        gpu.q_stacked, gpu.kv_pages, gpu.block_table, page_valid_len=gpu.page_valid_len, k_scale=problem.k_scale,
        v_scale=problem.v_scale, precision="bf16", splits=splits, return_lse=True)
    inputs = problem.inputs
    k = orc.decode_e4m3fn(inputs.k.view(torch.uint8).numpy()) * inputs.k_scale
    v = orc.decode_e4m3fn(inputs.v.view(torch.uint8).numpy()) * inputs.v_scale
    q = orc.decode_bfloat16(inputs.q.view(torch.int16).numpy().view(np.uint16))
    want = orc.expected_stacked(q, k, v, orc.OracleShape.from_config(cfg))
    # every P is off by at most 2^-9 of itself (bf16) against an unrounded row
    # sum, and the output by 2^-9 of itself: 2^-8 of the largest |V| in all
    # (5% for the fp32 sums and the exponential)
    assert np.abs(out.float().cpu().numpy() - want).max() <= 1.05 * 2**-8 * np.abs(v).max()
    scores = np.einsum("hqd,hkd->hqk", q.astype(np.float64), np.repeat(k[:, :tokens], 2, axis=0)) / np.sqrt(head_dim)
    want_lse = np.log(np.exp(scores - scores.max(-1, keepdims=True)).sum(-1)) + scores.max(-1)
    # pcp 1: the stacked order is the global one; fp32 scores and sums
    assert np.abs(lse.cpu().numpy()[0] - want_lse).max() <= 2e-5
