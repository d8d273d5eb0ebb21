"""Host side of a history call, before anything is launched (no GPU needed)."""

from __future__ import annotations

import numpy as np
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


@pytest.mark.parametrize("option,value,message", [
    ("precision", ["auto"], "precision must be one of"),
    ("exp2", {"fast": 1}, "exp2 must be one of"),
    # accepted values that cannot be looked up or kept as they are: on to the next check
    ("splits", np.array(2), "q must be a GPU tensor"),
    ("splits", 2.0, "q must be a GPU tensor"),
    ("splits", -2**40, "q must be a GPU tensor"),
    ("splits", 99, "q must be a GPU tensor"),
])
def test_options_are_checked_by_the_general_path(kernel, option, value, message):
    """Looking up the native call neither refuses an option nor raises ahead
    of the general path's checks, whatever the option's type or range."""

    class OnGpu:  # lengths that say they are on a GPU, so that a plan is made if the options allow one
        is_cuda, device = True, torch.device("cuda", 0)

    kernel.split_count = lambda *_: 1  # (asks the device)
    q = torch.zeros((2, 4, 64, 64), dtype=torch.bfloat16)
    with pytest.raises(ValueError, match=message):
        kernel(q, None, None, page_valid_len=OnGpu(), **{option: value})
