"""The work that users of this framework have it do, as cases with sizes, for measuring it.

Six kinds of calls, through the public entry points only:

* ``gemv``    the two products of a decode step on the reference's operator, ``KVmix.quantized_gemm``: q.K^T over the
              packed keys and p.V over the packed values;
* ``pack``    the one-shot quantizer, ``KVmix.quantize_pack_last_dim_cuda``, on the keys and values of a prompt;
* ``append``  the append forms, ``KVmix.process_key_quantization_cuda`` / ``process_value_quantization_cuda``: the
              packed cache grown by what one flush brings;
* ``prompt``  the prompt call of one attention layer (``KVmixAttention.forward`` without a past): dense causal attention
              and the quantized cache;
* ``step``    one decode step of one attention layer on the reference's 9-tuple: append, flush if the policy says so,
              attention over packed cache and fp16 tails;
* ``decode``  a Llama-shaped decoder stack: the prompt and then one forward per token, replayed from captured graphs or
              launched by an eager host loop;
* ``hf``      the transformers wrappers: the prompt and then one forward per token on a KVmix cache.

Keys have four channels per head ten times larger than the others, as real key caches do; probabilities are softmax
rows.  The token ids of ``decode`` and ``hf`` are given beforehand (a text is being scored), so that two numerically
different implementations see the same inputs at every step.
"""
from __future__ import annotations

import math

import torch

import KVmix
from kvmix_amd import ops
from kvmix_amd.attention import KVmixAttention
from kvmix_amd.cache import RESIDUAL_RATIO_BY_BITS, flush_length
from kvmix_amd.decoder import Decoder, DecoderConfig, GraphDecoder, init_weights, kvmix_layers

DEV = "cuda"
GROUP = 32
WINDOW = 128  # the fixed fp16 window of the benchmark; 0 in a case: the reference's ratio rule


# ---------------------------------------------------------------------------------------------------------------------
# the cases

def listed():
    return [
        # the smallest useful call: one sequence, one layer, 4k tokens; two launches, bound by latency
        {"name": "gemv_b1_t4096_k4v4", "kind": "gemv", "batch": 1, "heads": 32, "kv_heads": 32, "head_dim": 128,
         "tokens": 4096, "k_bits": 4, "v_bits": 4},
        # serving batch at 8k context, the width most layers get
        {"name": "gemv_b16_t8192_k2v2", "kind": "gemv", "batch": 16, "heads": 32, "kv_heads": 32, "head_dim": 128,
         "tokens": 8192, "k_bits": 2, "v_bits": 2},
        # grouped-query heads at long context, the reference's eleven-per-word 3-bit keys
        {"name": "gemv_gqa_b16_t32768_k3v2", "kind": "gemv", "batch": 16, "heads": 32, "kv_heads": 8, "head_dim": 128,
         "tokens": 32768, "k_bits": 3, "v_bits": 2},
        # the most aggressive compression at a large batch
        {"name": "gemv_b64_t4096_k1v1", "kind": "gemv", "batch": 64, "heads": 32, "kv_heads": 32, "head_dim": 128,
         "tokens": 4096, "k_bits": 1, "v_bits": 1},
        # a long prompt's cache quantized in one go
        {"name": "pack_b8_t8192_k3v4", "kind": "pack", "batch": 8, "kv_heads": 32, "head_dim": 128, "tokens": 8192,
         "k_bits": 3, "v_bits": 4, "dtype": "float16"},
        # a flush onto a mid-sized cache through the append operators
        {"name": "append_b4_t2304_k2v4", "kind": "append", "batch": 4, "kv_heads": 32, "head_dim": 128, "tokens": 2304,
         "new": 32, "k_bits": 2, "v_bits": 4, "dtype": "float16"},
        # the prompt of one layer, causal mask as the decoder builds it
        {"name": "prompt_b4_t2048_k4v2", "kind": "prompt", "batch": 4, "heads": 32, "kv_heads": 32, "head_dim": 128,
         "tokens": 2048, "k_bits": 4, "v_bits": 2, "window": WINDOW, "padded": False},
        # a short-context step that flushes (the tail is one token below the rule's limit), probabilities wanted
        {"name": "step_gqa_b1_t1036_k4v4_flush", "kind": "step", "batch": 1, "heads": 32, "kv_heads": 8, "head_dim": 128,
         "tokens": 1036, "k_bits": 4, "v_bits": 4, "window": 0, "padded": False, "weights": True},
        # an ordinary step of a left-padded batch at an odd context length, probabilities not wanted
        {"name": "step_b8_t8101_k2v4", "kind": "step", "batch": 8, "heads": 32, "kv_heads": 32, "head_dim": 128,
         "tokens": 8101, "k_bits": 2, "v_bits": 4, "window": WINDOW, "padded": True, "weights": False},
        # a generation on the decoder stack at Llama-2-7B width (8 of its layers), steps replayed from graphs
        {"name": "decode_graph_b4_p512_n64", "kind": "decode", "graph": True, "batch": 4, "layers": 8, "heads": 32,
         "kv_heads": 32, "ffn": 11008, "vocab": 32000, "prompt": 512, "steps": 64, "window": WINDOW},
        # a single user's generation on the eager loop, grouped-query heads, the reference's ratio rule
        {"name": "decode_eager_b1_p1001_n16", "kind": "decode", "graph": False, "batch": 1, "layers": 4, "heads": 32,
         "kv_heads": 8, "ffn": 14336, "vocab": 32000, "prompt": 1001, "steps": 16, "window": 0},
        # the transformers wrapper, grouped-query heads, ratio rule
        {"name": "hf_mistral_b2_p333_n16", "kind": "hf", "family": "mistral", "batch": 2, "layers": 4, "heads": 32,
         "kv_heads": 8, "ffn": 14336, "vocab": 32000, "prompt": 333, "steps": 16, "window": 0},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["gemv", "gemv", "gemv", "pack", "append", "prompt", "step", "step", "step", "decode", "hf"])
    heads, kv_heads = rng.choice([(32, 32), (32, 32), (32, 8), (32, 8), (16, 4), (12, 12)])
    dim = 128 if rng.random() < 0.85 else 64
    kb, vb = rng.choice([1, 2, 3, 4]), rng.choice([1, 2, 4])
    window = rng.choice([0, WINDOW])
    if kind == "gemv":
        tokens = _log_int(rng, 256, 32768)
        batch = max(1, min(_log_int(rng, 1, 64), 4194304 // (kv_heads * tokens)))
        return {"kind": kind, "batch": batch, "heads": heads, "kv_heads": kv_heads, "head_dim": dim, "tokens": tokens,
                "k_bits": kb, "v_bits": rng.choice([1, 2, 3, 4])}
    if kind == "pack":
        tokens = _log_int(rng, 64, 8192)
        batch = max(1, min(_log_int(rng, 1, 64), 2097152 // (kv_heads * tokens)))
        return {"kind": kind, "batch": batch, "kv_heads": kv_heads, "head_dim": dim, "tokens": tokens, "k_bits": kb,
                "v_bits": vb, "dtype": rng.choice(["float16", "float16", "float16", "float32"])}
    if kind == "append":
        tokens = _log_int(rng, 64, 8192)
        batch = max(1, min(_log_int(rng, 1, 32), 2097152 // (kv_heads * tokens)))
        return {"kind": kind, "batch": batch, "kv_heads": kv_heads, "head_dim": dim, "tokens": tokens,
                "new": rng.choice([32, 64, 128]), "k_bits": kb, "v_bits": vb,
                "dtype": rng.choice(["float16", "float16", "float16", "float32"])}
    if kind == "prompt":
        tokens = _log_int(rng, 33, 4096)
        batch = max(1, min(_log_int(rng, 1, 16), 16777216 // (tokens * tokens)))
        return {"kind": kind, "batch": batch, "heads": heads, "kv_heads": kv_heads, "head_dim": dim, "tokens": tokens,
                "k_bits": kb, "v_bits": vb, "window": window, "padded": rng.random() < 0.5}
    if kind == "step":
        tokens = _log_int(rng, 150, 16384)
        batch = max(1, min(_log_int(rng, 1, 32), 2097152 // (kv_heads * tokens)))
        return {"kind": kind, "batch": batch, "heads": heads, "kv_heads": kv_heads, "head_dim": dim, "tokens": tokens,
                "k_bits": kb, "v_bits": vb, "window": window, "padded": rng.random() < 0.3, "weights": rng.random() < 0.5}
    if kind == "decode":
        heads, kv_heads = rng.choice([(32, 32), (32, 8), (16, 4)])
        return {"kind": kind, "graph": rng.random() < 0.5, "batch": _log_int(rng, 1, 16), "layers": rng.randint(2, 6),
                "heads": heads, "kv_heads": kv_heads, "ffn": rng.choice([5632, 8192, 11008, 14336]), "vocab": 32000,
                "prompt": _log_int(rng, 40, 1024), "steps": rng.randint(8, 40), "window": window}
    heads, kv_heads = rng.choice([(32, 32), (32, 8), (16, 4)])
    return {"kind": kind, "family": rng.choice(["llama", "mistral"]), "batch": _log_int(rng, 1, 8),
            "layers": rng.randint(2, 4), "heads": heads, "kv_heads": kv_heads, "ffn": rng.choice([5632, 8192, 11008, 14336]),
            "vocab": 32000, "prompt": _log_int(rng, 40, 1024), "steps": rng.randint(8, 24), "window": window}


# ---------------------------------------------------------------------------------------------------------------------
# inputs

def _generator(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _normal(gen, *shape):
    return torch.randn(*shape, generator=gen, device=DEV, dtype=torch.float16)


def _keys(gen, batch, heads, tokens, dim):
    """[B,H,T,D] ~ N(0,1) with four outlier channels per head."""
    k = _normal(gen, batch, heads, tokens, dim)
    outlier = torch.rand(heads, dim, generator=gen, device=DEV).argsort(-1) < 4
    return k.mul_((1.0 + 9.0 * outlier.half())[None, :, None, :])


def _k_group(bits):
    return 11 if bits == 3 else GROUP


def _pack_keys(k, bits):
    """Keys [B,H,n,D] as the cache holds them, quantized along the tokens."""
    return KVmix.quantize_pack_last_dim_cuda(k.transpose(2, 3).contiguous(), _k_group(bits), bits)


def _pack_values(v, bits):
    if bits == 3:  # the reference's 3-bit words cannot hold these head sizes; the dense stream can
        return ops.quantize_pack_dense3(v.contiguous(), GROUP)
    return KVmix.quantize_pack_last_dim_cuda(v.contiguous(), GROUP, bits)


def _tail_length(tokens, ratio, group, window):
    """fp16 tokens a cache of `tokens` tokens holds between two flushes under the policy: the tail is what the packed
    whole groups leave, as long as the rule lets it get."""
    def rests(n):
        return flush_length(n, ratio, group, window or None) == 0
    tail = tokens % group
    if window:
        tail += group * ((tokens // group) % (window // group + 1))
    while not rests(tail):
        tail -= group
    if not window:
        while rests(tail + group):
            tail += group
    return max(tail, 0)


def _padding_mask(gen, batch, width, dtype):
    """[B,1,1,width] additive mask of a left-padded batch."""
    pads = (torch.rand(batch, generator=gen, device=DEV) * (width // 4)).long()
    pads[0] = 0
    dead = torch.arange(width, device=DEV)[None, :] < pads[:, None]
    return torch.zeros(batch, width, dtype=dtype, device=DEV).masked_fill_(dead, torch.finfo(dtype).min)[:, None, None, :]


def _layer_bits(layers):
    """A quarter of the layers 4-bit, half 3-bit, a quarter 2-bit, keys and values in different orders."""
    cycle = [4, 3, 2, 3]
    return [cycle[i % 4] for i in range(layers)], [cycle[(i + 2 * (i // 4) + 1) % 4] for i in range(layers)]


def prepare(case, seed):
    gen = _generator(seed)
    return {"case": case, **globals()["_prepare_" + case["kind"]](case, gen, seed)}


def _prepare_gemv(c, gen, seed):
    B, nh, H, D, T = c["batch"], c["heads"], c["kv_heads"], c["head_dim"], c["tokens"]
    kg = _k_group(c["k_bits"])
    nk, nv = (T - WINDOW) // kg * kg, (T - WINDOW) // GROUP * GROUP
    keys = _pack_keys(_keys(gen, B, H, nk, D), c["k_bits"])
    values = _pack_values(_normal(gen, B, H, nv, D), c["v_bits"])
    q = _normal(gen, B, nh, 1, D)
    p = torch.softmax(1.5 * torch.randn(B, nh, 1, T, generator=gen, device=DEV), -1).half()[..., :nv]
    return {"q": q, "p": p, "keys": keys, "values": values}


def _prepare_pack(c, gen, seed):
    B, H, D, T = c["batch"], c["kv_heads"], c["head_dim"], c["tokens"]
    kg = _k_group(c["k_bits"])
    dt = getattr(torch, c["dtype"])
    k = _keys(gen, B, H, T // kg * kg, D).transpose(2, 3).contiguous().to(dt)
    return {"k": k, "v": _normal(gen, B, H, T, D).to(dt)}


def _prepare_append(c, gen, seed):
    B, H, D, T = c["batch"], c["kv_heads"], c["head_dim"], c["tokens"]
    kg = _k_group(c["k_bits"])
    dt = getattr(torch, c["dtype"])
    nk, new = T // kg * kg, c["new"] // kg * kg
    k = _keys(gen, B, H, nk + new, D).transpose(2, 3).contiguous().to(dt)
    v = _normal(gen, B, H, T + c["new"], D).to(dt)
    return {"k": k[..., nk:].contiguous(), "v": v[:, :, T:].contiguous(),
            "keys": KVmix.quantize_pack_last_dim_cuda(k[..., :nk].contiguous(), kg, c["k_bits"]),
            "values": KVmix.quantize_pack_last_dim_cuda(v[:, :, :T].contiguous(), GROUP, c["v_bits"])}


def _prepare_prompt(c, gen, seed):
    B, nh, H, D, T = c["batch"], c["heads"], c["kv_heads"], c["head_dim"], c["tokens"]
    # the decoder's mask is one fp32 causal matrix; a padded batch's comes in the model's dtype, one per sequence
    dt = torch.float16 if c["padded"] else torch.float32
    mask = torch.triu(torch.full((T, T), torch.finfo(dt).min, dtype=dt, device=DEV), 1)[None, None]
    if c["padded"]:
        mask = torch.minimum(mask, _padding_mask(gen, B, T, dt))
    return {"layer": KVmixAttention(c["k_bits"], c["v_bits"], residual_length=c["window"] or None), "mask": mask,
            "q": _normal(gen, B, nh, T, D), "k": _keys(gen, B, H, T, D), "v": _normal(gen, B, H, T, D)}


def _prepare_step(c, gen, seed):
    B, nh, H, D, T = c["batch"], c["heads"], c["kv_heads"], c["head_dim"], c["tokens"]
    kg = _k_group(c["k_bits"])
    nk = T - _tail_length(T, RESIDUAL_RATIO_BY_BITS[c["k_bits"]], kg, c["window"])
    nv = T - _tail_length(T, RESIDUAL_RATIO_BY_BITS[c["v_bits"]], GROUP, c["window"])
    k, v = _keys(gen, B, H, T, D), _normal(gen, B, H, T, D)
    kc, ks, km = _pack_keys(k[:, :, :nk], c["k_bits"])
    vc, vs, vm = _pack_values(v[:, :, :nv], c["v_bits"])
    past = (kc, k[:, :, nk:].contiguous(), ks, km, vc, v[:, :, nv:].contiguous(), vs, vm, T)
    return {"layer": KVmixAttention(c["k_bits"], c["v_bits"], residual_length=c["window"] or None), "past": past,
            "q": _normal(gen, B, nh, 1, D), "k": _keys(gen, B, H, 1, D), "v": _normal(gen, B, H, 1, D),
            "mask": _padding_mask(gen, B, T + 1, torch.float32) if c["padded"] else None}


def _prepare_decode(c, gen, seed):
    cfg = DecoderConfig(hidden_size=128 * c["heads"], num_layers=c["layers"], num_heads=c["heads"],
                        num_kv_heads=c["kv_heads"], intermediate_size=c["ffn"], vocab_size=c["vocab"])
    layers, caches = kvmix_layers(cfg, *_layer_bits(c["layers"]), residual_length=c["window"] or None,
                                  capacity=c["prompt"] + c["steps"])
    ids = torch.randint(0, c["vocab"], (c["batch"], c["prompt"] + c["steps"]), generator=gen, device=DEV)
    return {"cfg": cfg, "weights": init_weights(cfg, DEV, seed=seed), "layers": layers, "caches": caches, "ids": ids}


def _prepare_hf(c, gen, seed):
    from transformers import LlamaConfig, MistralConfig

    from kvmix_amd import hf

    llama = c["family"] == "llama"
    cfg = (LlamaConfig if llama else MistralConfig)(
        hidden_size=128 * c["heads"], intermediate_size=c["ffn"], num_hidden_layers=c["layers"],
        num_attention_heads=c["heads"], num_key_value_heads=c["kv_heads"], vocab_size=c["vocab"],
        max_position_embeddings=4096)
    cfg._attn_implementation = "eager"
    cfg.residual_length = c["window"] or None
    kb, vb = _layer_bits(c["layers"])
    with torch.device("meta"):
        model = (hf.LlamaForCausalLM_KVmix if llama else hf.MistralForCausalLM_KVmix)(
            cfg, quant_bits={i: {"k_bits": kb[i], "v_bits": vb[i]} for i in range(c["layers"])})
    model = model.to(torch.float16).to_empty(device=DEV).eval()
    with torch.no_grad():
        for w in model.parameters():
            w.fill_(1.0) if w.dim() == 1 else w.normal_(0.0, 0.02, generator=gen)
    model.model.rotary_emb = type(model.model.rotary_emb)(config=cfg).to(DEV)
    ids = torch.randint(0, c["vocab"], (c["batch"], c["prompt"] + c["steps"]), generator=gen, device=DEV)
    return {"model": model, "ids": ids}


# ---------------------------------------------------------------------------------------------------------------------
# one pass

def run(state):
    return globals()["_run_" + state["case"]["kind"]](state, state["case"])


def _run_gemv(s, c):
    fmt = ops.FMT_DENSE3 if c["v_bits"] == 3 else ops.FMT_REF
    logits = KVmix.quantized_gemm(_k_group(c["k_bits"]), s["q"], *s["keys"], c["k_bits"])
    return {"logits": logits, "out": KVmix.quantized_gemm(GROUP, s["p"], *s["values"], c["v_bits"], fmt)}


def _run_pack(s, c):
    return {"k": KVmix.quantize_pack_last_dim_cuda(s["k"], _k_group(c["k_bits"]), c["k_bits"]),
            "v": KVmix.quantize_pack_last_dim_cuda(s["v"], GROUP, c["v_bits"])}


def _run_append(s, c):
    return {"k": KVmix.process_key_quantization_cuda(s["k"], *s["keys"], _k_group(c["k_bits"]), c["k_bits"]),
            "v": KVmix.process_value_quantization_cuda(s["v"], *s["values"], GROUP, c["v_bits"])}


def _run_prompt(s, c):
    out, _, past = s["layer"](s["q"], s["k"], s["v"], None, attention_mask=s["mask"], need_weights=False)
    return {"out": out, "past": past}


def _run_step(s, c):
    out, weights, past = s["layer"](s["q"], s["k"], s["v"], s["past"], attention_mask=s["mask"], need_weights=c["weights"])
    return {"out": out, "weights": weights, "past": past}


def _run_decode(s, c):
    for cache in s["caches"]:
        cache.reset()  # a new sequence on the buffers of the last one
    decoder = (GraphDecoder if c["graph"] else Decoder)(s["cfg"], s["weights"], s["layers"], s["caches"])
    logits = [decoder.forward(s["ids"][:, :c["prompt"]])]
    for t in range(c["prompt"], c["prompt"] + c["steps"]):
        logits.append(decoder.forward(s["ids"][:, t:t + 1]))
    return torch.stack(logits)


@torch.no_grad()
def _run_hf(s, c):
    cache = s["model"].new_cache(c["prompt"] + c["steps"])
    logits = [s["model"](input_ids=s["ids"][:, :c["prompt"]], past_key_values=cache, logits_to_keep=1).logits]
    for t in range(c["prompt"], c["prompt"] + c["steps"]):
        logits.append(s["model"](input_ids=s["ids"][:, t:t + 1], past_key_values=cache).logits)
    return torch.cat(logits, 1)


# ---------------------------------------------------------------------------------------------------------------------
# what a pass cannot do without, and how exact it is

def _packed_bytes(rows, tokens, dim, bits, side, elem=2):
    """Codes, scales and zeros of `rows` (batch, kv-head) slices."""
    if bits == 3 and side == "k":
        return rows * dim * (tokens // 11) * (4 + 2 * elem)
    return rows * dim * tokens * (bits / 8 + 2 * elem / GROUP)


def _model_params(c):
    h, kv = 128 * c["heads"], 128 * c["kv_heads"]
    return c["layers"] * (h * (h + 2 * kv) + h * h + 3 * h * c["ffn"]) + h * c["vocab"]


def work(case):
    c, kind = case, case["kind"]
    if kind in ("decode", "hf"):
        # every forward streams the weights once; a step also reads the cache
        h, kv, params = 128 * c["heads"], 128 * c["kv_heads"], _model_params(c)
        kb, vb = _layer_bits(c["layers"])
        cache = sum(_packed_bytes(c["batch"] * c["kv_heads"], c["prompt"], 128, b, side) for side, bits in (("k", kb), ("v", vb))
                    for b in bits)
        fresh = params - h * c["vocab"]  # the head is applied to one position per forward
        return {"bytes": (c["steps"] + 1) * 2 * params + c["steps"] * cache,
                "flops": 2 * c["batch"] * ((c["prompt"] + c["steps"]) * fresh + (c["steps"] + 1) * h * c["vocab"])
                + 2 * c["batch"] * c["layers"] * h * (c["prompt"] ** 2 + 2 * c["steps"] * c["prompt"])}
    B, H, D, T = c["batch"], c["kv_heads"], c["head_dim"], c["tokens"]
    if kind in ("pack", "append"):
        elem = 2 if c["dtype"] == "float16" else 4
        packed = [_packed_bytes(B * H, T, D, c["k_bits"], "k", elem), _packed_bytes(B * H, T, D, c["v_bits"], "v", elem)]
        if kind == "pack":
            return {"bytes": sum(packed) + 2 * B * H * T * D * elem, "flops": 2 * 4 * B * H * T * D}
        n = c["new"]
        fresh = [_packed_bytes(B * H, n, D, c["k_bits"], "k", elem), _packed_bytes(B * H, n, D, c["v_bits"], "v", elem)]
        return {"bytes": 2 * sum(packed) + sum(fresh) + 2 * B * H * n * D * elem, "flops": 2 * 4 * B * H * n * D}
    nh = c["heads"]
    if kind == "prompt":
        packed = sum(_packed_bytes(B * H, T, D, c[s + "_bits"], s) for s in "kv")
        mask = T * T * (2 * B if c["padded"] else 4)
        return {"bytes": 2 * B * D * T * (2 * nh + 2 * H) + packed + mask, "flops": 2 * B * nh * D * T * T}
    packed = sum(_packed_bytes(B * H, max(T - WINDOW, GROUP), D, c[s + "_bits"], s) for s in "kv")
    if kind == "gemv":
        return {"bytes": packed + 2 * B * nh * (2 * D + 2 * T), "flops": 4 * B * nh * T * D}
    probs = 2 * B * nh * T if c["weights"] else 0
    return {"bytes": packed + 2 * 2 * 2 * B * H * D * min(WINDOW, T) + 2 * 2 * B * nh * D + probs, "flops": 4 * B * nh * T * D}


def tolerance(case):
    """About four times what another order of the sums, or the same path in 64 bits, was measured to change."""
    kind = case["kind"]
    if kind in ("pack", "append"):
        return "exact"  # whole codes; scales and zeros are single roundings of exact minima and maxima
    if kind == "gemv":
        # against sums in 64 bits, both rounded to fp16: up to 1.6e-5, where a rounding falls the other way (largest: 1e-3)
        return {"rel": 1e-4, "max": 4e-3, "differ": 0.0}
    if kind == "prompt":
        return {"rel": 1e-3, "max": 5e-3, "differ": 0.0}  # 2.3e-4 against 64 bits, most of it the output's rounding
    if kind == "step":
        # the step with and without probabilities (fp16 or fp32 after the softmax): 3.5e-4 to 4.7e-4, largest 4.5e-3
        return {"rel": 2e-3, "max": 2e-2, "differ": 0.0}
    # projections summed in fp32 instead of fp16 pieces: 3e-3 to 2e-2 (largest 0.17), because a rounding that differs
    # turns codes of the 2- and 3-bit layers over
    return {"rel": 3e-2, "max": 0.5}
