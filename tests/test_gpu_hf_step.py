"""The wrappers' decode step through the projection kernels against the stock layers' step.

A hook on a module inside a layer takes the step back to the stock modules, which is how the two are compared, teacher
forced, with nothing quantized (no rounding can turn a code over).  Both are fp16 implementations of the same layers:
about nine roundings of 2^-11 per layer on the way, so the logits may differ by 2^-11 times their number, relative to
their norm."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def model_of(family, dev, layers=2, ffn=768, window=512, **kw):
    from transformers import LlamaConfig, MistralConfig

    from kvmix_amd import hf

    llama = family == "llama"
    cfg = (LlamaConfig if llama else MistralConfig)(hidden_size=512, intermediate_size=ffn, num_hidden_layers=layers, num_attention_heads=4,
                                                    num_key_value_heads=2, head_dim=128, vocab_size=999, max_position_embeddings=2048, **kw)
    cfg._attn_implementation = "eager"
    cfg.residual_length = window
    torch.manual_seed(3)
    model = (hf.LlamaForCausalLM_KVmix if llama else hf.MistralForCausalLM_KVmix)(cfg).half().to(dev).eval()
    with torch.no_grad():
        for n, p in model.named_parameters():
            p.uniform_(0.5, 1.5) if "norm" in n else p.normal_(0, 0.05)
    return model


def decode(model, ids, prompt, mask=None, **kw):
    cache, out = model.new_cache(256), []
    for a, b in [(0, prompt)] + [(t, t + 1) for t in range(prompt, ids.shape[1])]:
        out.append(model(input_ids=ids[:, a:b], past_key_values=cache, attention_mask=None if mask is None else mask[:, :b], **kw).logits[:, -1:])
    return torch.cat(out, 1).float(), cache


def close(a, b, layers):
    assert float((a - b).norm()) <= (9 * layers + 2) * 2.0 ** -11 * float(b.norm())


@pytest.mark.parametrize("family,batch,padded,ffn", [("llama", 1, False, 768), ("mistral", 3, True, 768), ("llama", 16, True, 128), ("mistral", 5, False, 11392)])
def test_step_equals_the_stock_layers(dev, family, batch, padded, ffn):
    model = model_of(family, dev, ffn=ffn)
    ids = torch.randint(0, 999, (batch, 40), device=dev)
    mask = None
    if padded:
        mask = torch.ones_like(ids)
        mask[batch // 2:, :7] = 0
    with torch.no_grad():
        fast, cache = decode(model, ids, 33, mask)
        seen = []
        hooks = [layer.mlp.register_forward_hook(lambda *a: seen.append(1)) for layer in model.model.layers]
        stock, cache2 = decode(model, ids, 33, mask)
        assert len(seen) == 2 * 8  # (every layer, the prompt and each step)
        for h in hooks:
            h.remove()
        assert torch.equal(decode(model, ids, 33, mask)[0], fast)
    close(fast, stock, 2)
    for i in range(2):
        a, b = cache.packed(i).as_tuple(), cache2.packed(i).as_tuple()
        assert a[-1] == b[-1] == 40 and a[1].shape == b[1].shape
        close(a[1].float(), b[1].float(), 2)
        close(a[5].float(), b[5].float(), 2)


def test_step_leaves_observers_and_replacements_alone(dev):
    """Hooks see every call, recorded outputs stay complete, gradients flow, replaced projections and autocast are used."""
    model = model_of("mistral", dev)
    ids = torch.randint(0, 999, (2, 21), device=dev)
    with torch.no_grad():
        want, cache = decode(model, ids, 20)
        out = model(input_ids=ids[:, -1:], past_key_values=cache, output_hidden_states=True, output_attentions=True)
        assert len(out.hidden_states) == 3 and len(out.attentions) == 2 and out.attentions[0] is not None
    model = model_of("mistral", dev)
    logits, _ = decode(model, ids, 20)          # (parameters require gradients here: recorded)
    assert logits.requires_grad
    close(logits.detach(), want, 2)
    layer = model.model.layers[1]

    class Doubled(torch.nn.Linear):
        def forward(self, x):
            return 2 * super().forward(x)

    layer.mlp.down_proj.__class__ = Doubled
    with torch.no_grad():
        doubled, _ = decode(model, ids, 20)
        layer.mlp.down_proj.__class__ = torch.nn.Linear
        layer.mlp.down_proj.weight.mul_(2)
        scaled, _ = decode(model, ids, 20)
    close(doubled, scaled, 2)


def test_mask_rows_beyond_the_sliding_window_are_the_stock_ones(dev):
    model = model_of("mistral", dev, sliding_window=24)
    ids = torch.randint(0, 999, (1, 40), device=dev)
    with torch.no_grad():
        long, cache = decode(model, ids, 20)
        model.config.sliding_window = None
        full, _ = decode(model, ids, 20)
        assert model._step_mask(ids[:, :1], None, cache).shape == (1, 1, 1, 41)
        model.config.sliding_window = 24
        assert model._step_mask(ids[:, :1], None, cache) is None
    close(long[:, :4], full[:, :4], 2)
    assert float((long[:, -1] - full[:, -1]).norm()) > 0.02 * float(full[:, -1].norm())  # (the window does cut)


@pytest.mark.parametrize("family", ["llama", "mistral"])
def test_replacements_on_the_class_are_used(dev, family, monkeypatch):
    """A forward replaced on the class of a module inside (not on an instance) is what a step runs, as before a prompt does."""
    from kvmix_amd import hf
    from kvmix_amd.attention import KVmixAttention

    model = model_of(family, dev)
    layer = model.model.layers[0]
    ids = torch.randint(0, 999, (2, 24), device=dev)
    kinds = [type(layer.mlp), type(layer.input_layernorm), type(layer.mlp.act_fn), torch.nn.Linear, type(layer.self_attn), type(layer).__mro__[2],
             KVmixAttention]
    assert kinds[5] in (hf.StockLlamaDecoderLayer, hf.StockMistralDecoderLayer)
    with torch.no_grad():
        want, _ = decode(model, ids, 20)
        for kind in kinds:
            seen, own = [], kind.__call__ if kind is KVmixAttention else kind.forward
            with monkeypatch.context() as m:
                m.setattr(kind, "__call__" if kind is KVmixAttention else "forward", lambda self, *a, **kw: (seen.append(1), own(self, *a, **kw))[1])
                got, _ = decode(model, ids, 20)
            assert len(seen) >= 2 * 5, kind  # (each of the two layers, at the prompt and at four steps)
            close(got, want, 2)
        assert torch.equal(decode(model, ids, 20)[0], want)


def test_modules_of_other_kinds_inside(dev):
    """A weight that is a plain tensor, an attention wrapped in a module of its own: the stock layer runs."""
    model = model_of("llama", dev)
    ids = torch.randint(0, 999, (2, 24), device=dev)

    class Wrapped(torch.nn.Module):
        def __init__(self, inner):
            super().__init__()
            self.inner = inner

        def forward(self, *a, **kw):
            return self.inner(*a, **kw)

    with torch.no_grad():
        want, _ = decode(model, ids, 20)
        lin = model.model.layers[0].mlp.up_proj
        weight = lin.weight.detach().clone()
        del lin.weight
        lin.weight = weight
        norm = model.model.layers[1].post_attention_layernorm
        weight = norm.weight.detach().clone()
        del norm.weight
        norm.weight = weight
        close(decode(model, ids, 20)[0], want, 2)
        model.model.layers[1].self_attn = Wrapped(model.model.layers[1].self_attn)
        close(decode(model, ids, 20)[0], want, 2)
