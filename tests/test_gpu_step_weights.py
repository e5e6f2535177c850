"""The step that returns its probabilities from the single pass (kvmix_decode_attention_fused_weights): which steps take it, and
its outputs against float64 over the dequantized cache.

Bound: logits are rounded to fp16 (half an ulp, 2^-11 of the logit, scaled by 1 / sqrt(D)) after fp32 sums over D = 128
products; a probability moves by that difference of its logit and of the sum's, relative, and is rounded to fp16
(2^-11, at least 2^-25); the output is their mean of values."""
import math

import pytest
import torch

from helpers import dequantize_torch
from kvmix_amd import _lib


def test_steps_it_is_chosen_for():
    import ctypes

    def chosen(batch, heads, kv_heads, width, kb=4, **kw):
        tokens = width // 352 * 352
        st = _lib.attn_step_descriptor(batch, heads, kv_heads, 128, kb, 0, 11 if kb == 3 else 32, tokens, 2, 0, 32, tokens, width - tokens, width - tokens)
        return _lib.load().kvmix_decode_attention_fused_weights_recommended(ctypes.byref(st))

    assert chosen(1, 32, 8, 1037) and chosen(1, 32, 32, 8000) and chosen(1, 32, 32, 9000, 3)
    assert not chosen(8, 32, 32, 8192) and not chosen(1, 32, 32, 10000, 3) and not chosen(1, 36, 12, 100)  # (three heads per kv head)


@pytest.mark.parametrize("batch,kv_heads,vb,fmt,taken,left", [
    (8, 32, 4, 0, 1360, 1562), (8, 8, 2, 0, 1600, 1750), (8, 32, 3, 1, 976, 1171), (5, 32, 4, 0, 2180, 2500),  # (129 to 256 rows: one round)
    (4, 32, 3, 1, 3400, 3700), (9, 32, 3, 1, 1500, 1700), (32, 32, 2, 0, 430, 450), (1, 8, 4, 0, 14000, 15000)])
def test_sides_of_the_rule(batch, kv_heads, vb, fmt, taken, left):
    import ctypes

    def chosen(width):
        tokens = width // 352 * 352
        st = _lib.attn_step_descriptor(batch, 32, kv_heads, 128, 4, 0, 32, tokens, vb, fmt, 32, tokens, width - tokens, width - tokens)
        return _lib.load().kvmix_decode_attention_fused_weights_recommended(ctypes.byref(st))

    assert chosen(taken) and not chosen(left)


def test_more_blocks_than_a_launch_holds_are_refused():
    """The slabs of a step with probabilities are shorter than the tiles without: 1025 and 2049 a row here.  (No probabilities
    are passed, so that nothing is launched whatever the check says.)"""
    import ctypes

    L = _lib.load()

    def code(samples):
        st = _lib.attn_step_descriptor(samples // 32, 32, 32, 128, 4, 0, 32, 1 << 20, 4, 0, 32, 1 << 20, 16, 16)
        for name in ("q", "out", "k_tail", "v_tail", "k_code", "k_scale", "k_zero", "v_code", "v_scale", "v_zero"):
            setattr(st, name, 4096)
        assert _lib.attn_plan(st)["matrix"]
        return L.kvmix_decode_attention_fused_weights(ctypes.byref(st), None, 0, None)

    null, shape = -7, -8
    assert code(32 * 1000) == null and code(32 * 48000) == shape


@pytest.mark.gpu
# one slab, two with a ragged last, the longest; GQA; no quantized part; left-padded masks; a row masked everywhere
@pytest.mark.parametrize("B,nh,nkv,T,tail", [(2, 4, 4, 40, 40), (1, 8, 2, 512, 32), (1, 8, 2, 1037, 45), (2, 4, 4, 2100, 52), (1, 16, 2, 3000, 24), (1, 32, 32, 8001, 33)])
@pytest.mark.parametrize("kb,vb", [(4, 4), (2, 30), (1, 1), (3, 2)])
@pytest.mark.parametrize("masked", [False, True])
def test_against_float64(dev, B, nh, nkv, T, tail, kb, vb, masked):
    import KVmix
    from kvmix_amd import ops

    gen = torch.Generator(device=dev).manual_seed(T + kb)
    rand = lambda *s: torch.randn(*s, generator=gen, device=dev).half()
    D, g = 128, 11 if kb == 3 else 32
    k, v, q = rand(B, nkv, T, D), rand(B, nkv, T, D), rand(B, nh, 1, D)
    k[..., 5] *= 8
    nk, nv = (T - tail) // g * g, (T - tail) // 32 * 32
    kp = vp = None
    kd, vd = k.double(), v.double()
    if nk:
        kp = KVmix.quantize_pack_last_dim_cuda(k[:, :, :nk].transpose(2, 3).contiguous(), g, kb)
        kd = torch.cat([dequantize_torch(*kp, kb, g).double().transpose(2, 3), kd[:, :, nk:]], 2)
    if nv:
        vp = ops.quantize_pack_dense3(v[:, :, :nv].contiguous(), 32) if vb == 30 else KVmix.quantize_pack_last_dim_cuda(v[:, :, :nv].contiguous(), 32, vb)
        vd = torch.cat([dequantize_torch(*vp, 3 if vb == 30 else vb, 32, vb == 30).double(), vd[:, :, nv:]], 2)
    mask = None
    if masked:
        mask = torch.zeros(B, 1, 1, T, device=dev)
        mask[0, ..., :T // 3] = torch.finfo(torch.float32).min
        mask[-1, ..., T // 2:] = torch.finfo(torch.float32).min if B > 1 else -3.0
    out, probs = ops.decode_attention(q, kp, vp, k[:, :, nk:].contiguous(), v[:, :, nv:].contiguous(), g, kb, 32, 3 if vb == 30 else vb, 0,
                                      1 if vb == 30 else 0, mask, single_pass=True, weights=True)
    assert probs.shape == (B, nh, 1, T) and probs.dtype == torch.float16
    rep = nh // nkv
    logits = torch.matmul(q.double(), kd.repeat_interleave(rep, 1).transpose(2, 3))
    x = logits / math.sqrt(D) + (0 if mask is None else mask.double())
    want = torch.softmax(x.clamp(min=torch.finfo(torch.float32).min), -1)
    # of each logit: its fp16 rounding and 128 products in fp32
    size = torch.matmul(q.double().abs(), kd.abs().repeat_interleave(rep, 1).transpose(2, 3))
    moved = (2.0 ** -11 * logits.abs() + 128 * 2.0 ** -23 * size) / math.sqrt(D) + 2.0 ** -20
    rel = moved + moved.amax(-1, keepdim=True)
    assert ((probs.double() - want).abs() <= want * (1.01 * rel + 2.0 ** -11) + 2.0 ** -25).all()
    vr = vd.repeat_interleave(rep, 1)
    exact = torch.matmul(want, vr)
    bound = torch.matmul(want * 1.01 * rel, vr.abs()) + 2.0 ** -11 * exact.abs() + T * 2.0 ** -23 * torch.matmul(want, vr.abs()) + 2.0 ** -25
    assert ((out.double() - exact).abs() <= bound).all()
    # the launches that round as the reference does return the same probabilities up to one rounding
    _, four = ops.decode_attention(q, kp, vp, k[:, :, nk:].contiguous(), v[:, :, nv:].contiguous(), g, kb, 32, 3 if vb == 30 else vb, 0,
                                   1 if vb == 30 else 0, mask)
    assert ((probs.double() - four.double()).abs() <= four.double() * 2 * (1.01 * rel + 2.0 ** -11) + 2.0 ** -24).all()


@pytest.mark.gpu
def test_lengths_from_the_device_and_windows_past_them(dev):
    """Probabilities past the live positions are zero whatever the windows' unused slots hold."""
    from kvmix_amd import ops

    gen = torch.Generator(device=dev).manual_seed(3)
    q, kt, vt = (torch.randn(2, 4, n, 128, generator=gen, device=dev).half() for n in (1, 96, 96))
    n = torch.tensor([70], device=dev)
    out, probs = ops.decode_attention(q, None, None, kt, vt, 32, 4, 32, 4, k_tail_len=n, v_tail_len=n, single_pass=True, weights=True)
    ref, want = ops.decode_attention(q, None, None, kt[:, :, :70].contiguous(), vt[:, :, :70].contiguous(), 32, 4, 32, 4, single_pass=True, weights=True)
    assert torch.equal(out, ref) and torch.equal(probs[..., :70], want) and not probs[..., 70:].any()
    kt[0, 1, 3, 5] = float("nan")  # a NaN logit reaches its row and no other, as it does through the other launches
    out, probs = ops.decode_attention(q, None, None, kt, vt, 32, 4, 32, 4, k_tail_len=n, v_tail_len=n, single_pass=True, weights=True)
    bad = out.isnan().any(-1).squeeze(-1)
    assert bad.tolist() == [[False, True, False, False], [False] * 4] and probs[0, 1, 0, :70].isnan().all()


@pytest.mark.gpu
@pytest.mark.parametrize("inplace", [False, True])
def test_a_caller_keeps_the_launches_that_round_as_the_reference_does(dev, inplace):
    """forward with its defaults takes the single pass here; with allow_single_pass=False its output is the four launches' bit
    by bit: the halves of the output rounded and added as halves."""
    from kvmix_amd import ops
    from kvmix_amd.attention import KVmixAttention

    gen = torch.Generator(device=dev).manual_seed(11)
    rand = lambda *s: torch.randn(*s, generator=gen, device=dev).half()
    layer = KVmixAttention(4, 2, residual_length=64)
    k, v = rand(2, 2, 501, 128), rand(2, 2, 501, 128)
    past = layer.new_cache(1024) if inplace else None
    *_, past = layer(rand(2, 8, 501, 128), k, v, past, need_weights=False)
    q, k1, v1 = rand(2, 8, 1, 128), rand(2, 2, 1, 128), rand(2, 2, 1, 128)
    out, probs, grown = layer(q, k1, v1, past, allow_single_pass=False)
    kc, kt, ks, km, vc, vt, vs, vm, width = grown.as_tuple() if inplace else grown
    assert ops.prefer_single_pass(2, 8, 2, 128, width, 4, 0, 32, 2, 0, 32, width - kt.shape[2], width - vt.shape[2], True)
    step = lambda single: ops.decode_attention(q, (kc, ks, km), (vc, vs, vm), kt, vt, 32, 4, 32, 2, single_pass=single, weights=single)
    want, wp = step(False)
    assert torch.equal(out, want) and torch.equal(probs, wp)
    tq = width - vt.shape[2]
    halves = ops.quantized_gemm(32, probs[..., :tq], vc, vs, vm, 2).float()
    tail = torch.matmul(probs[..., tq:].double().reshape(2, 2, 4, -1), vt.double()).reshape(out.shape)
    assert ((out.double() - (halves + tail.half().float()).half().double()).abs() <= 2.0 ** -10 * tail.abs() + 2.0 ** -10 * out.double().abs() + 2.0 ** -24).all()
    if inplace:
        assert torch.equal(layer.attend(q, grown, allow_single_pass=False)[0], want)
        assert torch.equal(layer.attend(q, grown)[0], step(True)[0])
