"""Host side of a history call, before anything is launched (no GPU needed)."""

from __future__ import annotations

import pytest
import torch

from aws_training_study_amd.pcp_attention import PCPAttentionConfig, make_history_attention_kernel


@pytest.fixture
def kernel():
    return make_history_attention_kernel(PCPAttentionConfig(
        pcp_size=2, current_len=128, max_history_len=512, actual_history_len=512, block_size=128, interleave_size=64,
        num_q_heads=4, num_kv_heads=2, head_dim=64, backend="hip").validate())


def test_workspaces_while_another_thread_makes_plans(kernel):
    """A new workspace makes every plan forget the ones it remembers; dropping
    them may let other threads run, whose calls add plans."""
    forgotten = []

    class Plan:
        def __init__(self, name):
            self.name = name

        def forget(self):
            forgotten.append(self.name)
            kernel._plans[len(kernel._plans)] = Plan("late")

    kernel._plans["a"], kernel._plans["b"] = Plan("a"), Plan("b")
    assert kernel._workspace(64, torch.device("cpu"), 7).numel() == 64
    assert forgotten == ["a", "b"]
