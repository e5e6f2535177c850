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


def test_launches_leave_the_interpreter_to_other_threads(dev):
    """The native host side calls the library without the interpreter's lock.  The library's launches are stood in for by a
    function that tells whether the caller holds it (1) or not (0, which reads as success); nothing is launched."""
    import ctypes

    import KVmix
    from kvmix_amd import _lib, ops

    q, keys, values, kt, vt = step_operands(dev)
    x, w = (torch.zeros(*s, dtype=torch.float16, device=dev) for s in ((2, 256), (512, 256)))
    angles = torch.zeros(1, 1, 128, dtype=torch.float16, device=dev)
    calls = [lambda: KVmix.quantize_pack_last_dim_cuda(kt.transpose(2, 3).repeat(1, 1, 1, 32), 32, 4), lambda: KVmix.quantized_gemm(32, q, *keys, 4),
             lambda: ops.quantize_pack_dense3(vt), lambda: ops.copy_rows([(kt, vt)]),
             lambda: KVmix.process_key_quantization_cuda(kt.transpose(2, 3).repeat(1, 1, 1, 32), *keys, 32, 4),
             lambda: KVmix.process_value_quantization_cuda(vt, *values, 32, 2),
             lambda: ops.grow_tuple((keys[0], kt, *keys[1:], values[0], vt, *values[1:], 69), kt[:, :, :1], vt[:, :, :1], 0, 0, 4, 32, 2),
             lambda: ops.decode_attention(q, keys, values, kt, vt, 32, 4, 32, 2),
             lambda: ops.decode_attention(q, keys, values, kt, vt, 32, 4, 32, 2, single_pass=True),
             lambda: ops.linear_rows(x, w), lambda: ops.swiglu_rows(x, w),
             lambda: ops.qkv_rope_append(x, w, 2, 1, angles, angles, kt[:, :1], vt[:, :1], 0, 0)]
    for call in calls:
        call()
    holds = ctypes.cast(ctypes.pythonapi.PyGILState_Check, ctypes.c_void_p).value
    launches = ("kvmix_quant_pack_last_dim", "kvmix_quant_pack_kv_flush", "kvmix_quantized_gemv", "kvmix_decode_attention",
                "kvmix_decode_attention_fused", "kvmix_copy_rows", "kvmix_linear_rows")
    host = _lib.load_host()
    real = {name: ctypes.cast(getattr(_lib.load(), name), ctypes.c_void_p).value for name in _lib.EXPORTS}
    host.bind({**real, **{name: holds for name in launches}})
    try:
        for i, call in enumerate(calls):
            try:
                call()
            except RuntimeError:
                pytest.fail(f"call {i} holds the interpreter's lock while it launches")
    finally:
        host.bind(real)
    with pytest.raises(RuntimeError, match="torch.float32"):  # (a refusal that asks the interpreter for a type's name)
        ops.linear_rows(x.float(), w)
