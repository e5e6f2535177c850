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


@pytest.mark.parametrize("batch,heads,q_len,mask_batch,mask_heads,taken", [
    (2, 4, 300, 1, 1, True), (2047, 32, 4, 2047, 32, True), (65535, 1, 4, 65535, 1, True),
    (2048, 32, 4, 2048, 32, False), (65536, 1, 4, 65536, 1, False), (2048, 32, 4, 2048, 1, True),  # (slices of the mask: grid.y)
    (1 << 26, 32, 4, 1, 1, False), (1 << 25, 32, 129, 1, 1, False), (1 << 25, 32, 128, 1, 1, True)])  # (blocks: grid.x)
def test_support_query_knows_the_limits_of_a_launch(batch, heads, q_len, mask_batch, mask_heads, taken):
    """A call beyond them is answered by torch's routine as long as the query says so; the launch itself could only fail."""
    import ctypes

    from kvmix_amd import _lib

    st = _lib.PrefillAttn()
    st.batch, st.heads, st.kv_heads, st.q_len, st.kv_len, st.head_dim, st.scale = batch, heads, heads, q_len, q_len, 64, 0.125
    st.mask, st.mask_dtype, st.mask_batch, st.mask_heads = 16, _lib.F16, mask_batch, mask_heads
    assert bool(_lib.load().kvmix_prefill_attention_supported(ctypes.byref(st))) == taken
