"""Decode steps through the projection kernels on caches that quantize, replayed on the CPU oracle.

The wrappers' and the decoder's step writes keys and values into the cache's slots itself (qkv_rope_append) and goes on with
KVmixAttention.attend.  Objects that stand in for a layer's attention take a step back to the other path, so what is recorded
here is recorded around the functions both share: tokens that enter a cache (append, or the slots behind note_device_append)
and queries, masks and outputs of ops.decode_attention.  The oracle is fed the same tokens and queries: outputs agree within the
attention tolerance at every step, the caches bit for bit at the end, through several flushes."""
import numpy as np
import pytest
import torch

from test_gpu_attention import same_cache
from test_gpu_hf import BITS, build_pair

pytestmark = pytest.mark.gpu


class Trace:
    """tokens[id of cache] = [(k, v, written by the projection kernel)], steps = [(q, mask, out)] over layers, then steps."""

    def __init__(self, monkeypatch):
        from kvmix_amd import ops
        from kvmix_amd.cache import PackedKVCache

        self.tokens, self.steps = {}, []
        append, note, decode = PackedKVCache.append, PackedKVCache.note_device_append, ops.decode_attention

        def host(t):
            return None if t is None else t.contiguous().cpu().numpy()

        def put(cache, k, v, by_kernel):
            self.tokens.setdefault(id(cache), []).append((host(k), host(v), by_kernel))

        def recorded_append(cache, k, v, prompt=False):
            put(cache, k, v, False)
            return append(cache, k, v, prompt)

        def recorded_note(cache):
            note(cache)
            entries = cache.as_tuple()
            put(cache, entries[1][:, :, -1:], entries[5][:, :, -1:], True)

        def recorded_decode(q, *args, **kw):
            out = decode(q, *args, **kw)
            self.steps.append((host(q), host(args[10] if len(args) > 10 else kw.get("attention_mask")), host(out[0])))
            return out

        monkeypatch.setattr(PackedKVCache, "append", recorded_append)
        monkeypatch.setattr(PackedKVCache, "note_device_append", recorded_note)
        monkeypatch.setattr(ops, "decode_attention", recorded_decode)


def after_prompt(o, k, v, k_bits, v_bits, k_ratio, v_ratio, window, v_dense3):
    """The cache the prompt leaves (models/modeling_llama_KVmix.py:213-251)."""
    from kvmix_amd.cache import flush_length

    T, kg = k.shape[2], 11 if k_bits == 3 else 32
    nk, nv = flush_length(T, k_ratio, kg, window, prompt=True), flush_length(T, v_ratio, 32, window, prompt=True)
    keys = values = (None,) * 3
    if nk:
        keys = o.quantize_pack_last_dim(np.ascontiguousarray(k[:, :, :nk].transpose(0, 1, 3, 2)), kg, k_bits)
    if nv:
        values = (o.quantize_pack_dense3(np.ascontiguousarray(v[:, :, :nv]), 32) if v_dense3 else
                  o.quantize_pack_last_dim(np.ascontiguousarray(v[:, :, :nv]), 32, v_bits))
    return keys[0], k[:, :, nk:], keys[1], keys[2], values[0], v[:, :, nv:], values[1], values[2], T


def replay(o, trace, li, layers, cache, entry, window, masked):
    tokens, steps = trace.tokens[id(cache)], trace.steps[li::layers]
    assert len(steps) == len(tokens) - 1 and not tokens[0][2]
    assert all(by_kernel for _, _, by_kernel in tokens[1:]), "a step did not take the projection kernels"
    kb, vb = entry["k_bits"], entry["v_bits"]
    kr, vr = entry["k_residual_ratio"], entry["v_residual_ratio"]
    state = after_prompt(o, *tokens[0][:2], kb, vb, kr, vr, window, vb == 3)
    flushed = (state[0] is not None and state[0].shape[3], state[4] is not None and state[4].shape[2])
    for step, ((k, v, _), (q, mask, out)) in enumerate(zip(tokens[1:], steps)):
        assert (mask is not None) == masked
        want, _, state = o.attention_decode_step(q, k, v, state, kb, vb, kr, vr, group_size=32, fixed_window=window, attention_mask=mask,
                                                 v_dense3=vb == 3)
        np.testing.assert_allclose(out.astype(np.float64), want.astype(np.float64), rtol=5e-3, atol=5e-3, err_msg=f"layer {li} step {step}")
    assert state[0].shape[3] > flushed[0] and state[4].shape[2] > flushed[1]  # (steps have flushed on both sides)
    same_cache(tuple(x.cpu().numpy() if torch.is_tensor(x) else x for x in cache.as_tuple()), state)


@pytest.mark.parametrize("kind,window,padded", [("llama", None, False), ("mistral", 64, True), ("mistral", None, True), ("llama", 64, False)])
def test_wrappers(oracle, dev, monkeypatch, kind, window, padded):
    _, model = build_pair(kind, dev, BITS, residual_length=window)
    B, T, new = 3, 150, 80
    ids = torch.randint(0, 1000, (B, T), generator=torch.Generator().manual_seed(1)).to(dev)
    mask = torch.ones_like(ids)
    if padded:
        mask[1, :17] = 0
        mask[2, :40] = 0
    cache = model.new_cache(capacity=64)  # small on purpose: the packed buffers have to grow
    trace = Trace(monkeypatch)
    out = model.generate(ids, attention_mask=mask, max_new_tokens=new, do_sample=False, past_key_values=cache, pad_token_id=0)
    assert out.shape == (B, T + new)
    for li in range(len(BITS)):
        replay(oracle, trace, li, len(BITS), cache.packed(li), model.quant_bits[li], window, True)


@pytest.mark.parametrize("window", [None, 64])
@pytest.mark.parametrize("heads,kv_heads", [(4, 4), (4, 1)])
def test_eager_decoder(oracle, dev, monkeypatch, window, heads, kv_heads):
    from kvmix_amd.cache import RESIDUAL_RATIO_BY_BITS
    from kvmix_amd.decoder import Decoder, DecoderConfig, init_weights, kvmix_layers

    cfg = DecoderConfig(hidden_size=128 * heads, num_layers=4, num_heads=heads, num_kv_heads=kv_heads, intermediate_size=1024, vocab_size=1000)
    kb, vb, B, T, new = [4, 3, 2, 1], [2, 3, 4, 1], 2, 200, 80
    layers, caches = kvmix_layers(cfg, kb, vb, residual_length=window, capacity=64)
    trace = Trace(monkeypatch)
    prompt = torch.randint(0, 1000, (B, T), generator=torch.Generator().manual_seed(40)).to(dev)
    Decoder(cfg, init_weights(cfg, dev), layers, caches).generate(prompt, new)
    for li in range(4):
        entry = {"k_bits": kb[li], "v_bits": vb[li], "k_residual_ratio": RESIDUAL_RATIO_BY_BITS[kb[li]], "v_residual_ratio": RESIDUAL_RATIO_BY_BITS[vb[li]]}
        replay(oracle, trace, li, 4, caches[li], entry, window, False)
