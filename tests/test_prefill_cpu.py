"""What the prompt kernel refuses before anything is launched (no GPU needed): such calls go to torch's routine."""
import types

import pytest
import torch

from kvmix_amd import ops


def on(device):
    return types.SimpleNamespace(dim=lambda: 4, dtype=torch.float16, is_cuda=True, device=torch.device(device), shape=(1, 2, 8, 64))


@pytest.mark.parametrize("other", [(0, 1, 0), (0, 0, 1), (1, 0, 0)])
def test_operands_on_different_gpus_are_not_taken(other):
    assert ops.prefill_attention(*(on(f"cuda:{i}") for i in other)) is None
