"""Calls of the operators that are refused, and what their host side promises beside the results."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def step_operands(dev, slots=5):
    import KVmix

    gen = torch.Generator(device="cpu").manual_seed(2)
    r = lambda *s: torch.randn(*s, generator=gen).to(dev).half()  # noqa: E731
    k, v = (r(2, 2, 64, 128) for _ in range(2))
    keys = KVmix.quantize_pack_last_dim_cuda(k.transpose(2, 3).contiguous(), 32, 4)
    return r(2, 4, 1, 128), keys, KVmix.quantize_pack_last_dim_cuda(v, 32, 2), r(2, 2, slots, 128), r(2, 2, slots, 128)


@pytest.mark.parametrize("single", [False, True])
def test_live_slots_outside_the_window_are_refused(dev, single):
    """A count below zero is a caller's mistake, not a request for the whole window (which is what None asks for)."""
    from kvmix_amd import ops

    q, keys, values, kt, vt = step_operands(dev)

    def step(**kw):
        return ops.decode_attention(q, keys, values, kt, vt, 32, 4, 32, 2, single_pass=single, **kw)[0]

    whole = step()
    assert torch.equal(step(k_tail_len=5, v_tail_len=5), whole) and torch.equal(step(k_tail_len=None, v_tail_len=5), whole)
    assert not torch.equal(step(k_tail_len=4, v_tail_len=4), whole)
    for n in (-1, -2, 6):
        with pytest.raises(RuntimeError):
            step(k_tail_len=n, v_tail_len=n)
        with pytest.raises(RuntimeError):
            step(k_tail_len=n)
        with pytest.raises(RuntimeError):
            step(v_tail_len=n)
