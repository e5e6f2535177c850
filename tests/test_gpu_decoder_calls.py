"""The decoder stack in calls that something records, and on weights in other layouts than init_weights makes them."""
import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu


def small(dev, window=32, **kw):
    from kvmix_amd.decoder import DecoderConfig, init_weights, kvmix_layers

    cfg = DecoderConfig(hidden_size=512, num_layers=2, num_heads=4, num_kv_heads=2, intermediate_size=1024, vocab_size=500)
    weights = init_weights(cfg, dev, std=0.05, seed=9)
    gen = torch.Generator(device=dev).manual_seed(1)
    for lw in weights["layers"] + [weights]:
        for n in [n for n in lw if "norm" in n]:
            lw[n].uniform_(0.5, 1.5, generator=gen)
    layers, caches = kvmix_layers(cfg, [4, 3], [2, 4], residual_length=window, capacity=256)
    ids = torch.randint(0, 500, (3, 60), generator=gen, device=dev)
    return cfg, weights, layers, caches, ids


def decode(dec, ids, prompt=50):
    out = [dec.forward(ids[:, :prompt])]
    for t in range(prompt, ids.shape[1]):
        out.append(dec.forward(ids[:, t:t + 1]))
    return torch.stack(out)


def test_gradients_of_prompt_and_step(dev):
    """The head's gradient against its formula, and gradients of whatever lies behind the attention, at a prompt and at steps."""
    from kvmix_amd.decoder import Decoder

    cfg, weights, layers, caches, ids = small(dev)
    behind = [weights["lm_head"], weights["norm"]] + [weights["layers"][1][n] for n in ("wo", "post_norm", "w_gate_up", "w_down")]
    for t in behind:
        t.requires_grad_(True)
    dec = Decoder(cfg, weights, layers, caches)
    for a, b in ((0, 50), (50, 51), (51, 52)):
        logits = dec.forward(ids[:, a:b])
        assert logits.requires_grad
        grads = torch.autograd.grad(logits.sum(), behind)
        assert all(g is not None and bool(torch.isfinite(g).all()) and float(g.abs().max()) > 0 for g in grads)
        # d(sum of logits) / d(head row) is the normalised row of x, summed over the sequences, for every token of the vocabulary
        assert torch.equal(grads[0], grads[0][:1].expand_as(grads[0]))
        want = logits.detach() @ torch.ones(cfg.vocab_size, 1, device=dev)
        got = (weights["lm_head"].detach().float() @ grads[0][0].float()).sum()
        assert float((got - want.sum()).abs()) <= 2e-2 * float(logits.detach().abs().sum()) / cfg.vocab_size ** 0.5


def test_forward_mode_and_traces_of_the_pieces(dev):
    from kvmix_amd.decoder import add_mlp, add_projection, head_logits

    cfg, weights, _, _, _ = small(dev)
    lw, eps = weights["layers"][0], cfg.rms_norm_eps
    gen = torch.Generator(device=dev).manual_seed(5)
    x, x2, t = (torch.randn(3, 1, 512, generator=gen, device=dev).half() for _ in range(3))
    head_t = 0.05 * torch.randn(500, 512, generator=gen, device=dev).half()
    _, tangent = torch.func.jvp(lambda w: head_logits(x, {**weights, "lm_head": w}, eps), (weights["lm_head"],), (head_t,))
    want = F.linear(F.rms_norm(x[:, 0], (512,), weights["norm"], eps), head_t).float()
    assert float((tangent - want).norm()) <= 1e-2 * float(want.norm())
    _, tangent = torch.func.jvp(lambda h: add_projection(x, h, lw["wo"]), (x2,), (t,))
    assert float((tangent - F.linear(t, lw["wo"])).norm()) <= 1e-2 * float(tangent.norm())
    for f in (lambda x: head_logits(x, weights, eps), lambda x: add_projection(x, x, lw["wo"]), lambda x: add_mlp(x, lw, eps)):
        traced = torch.jit.trace(f, (x,), check_trace=False)
        want = f(x2).float()
        assert float((traced(x2).float() - want).norm()) <= 1e-2 * float(want.norm())


def misaligned(t):
    buf = torch.empty(t.numel() + 1, dtype=t.dtype, device=t.device)
    buf[1:] = t.reshape(-1)
    return buf[1:].view(t.shape)


def transposed(t):
    return t.t().contiguous().t() if t.dim() == 2 else t


def spread(t):
    return torch.stack([t, t], -1)[..., 0]


def sliced(t):  # (rows of a wider matrix: the kernels take these)
    return torch.cat([t, t[..., :64]], -1)[..., :t.shape[-1]]


@pytest.mark.parametrize("layout", [misaligned, transposed, spread, sliced])
@pytest.mark.parametrize("graph", [False, True])
def test_weights_in_other_layouts(dev, layout, graph):
    """Every projection in turn, then all, on weights that hold the same values in another layout; the steps may differ by
    the order of fp32 sums (nothing is quantized within the window, so no rounding can turn a code over)."""
    from kvmix_amd.decoder import Decoder, GraphDecoder

    cfg, weights, layers, caches, ids = small(dev, window=96)
    names = ["input_norm", "wqkv", "wo", "post_norm", "w_gate_up", "w_down"]
    want = None
    for change in ([], *([n] for n in names), ["lm_head"], ["norm"], names + ["lm_head", "norm"]):
        w = {k: layout(v) if k in change else v for k, v in weights.items() if k != "layers"}
        w["layers"] = [{k: layout(v) if k in change else v for k, v in lw.items()} for lw in weights["layers"]]
        for c in caches:
            c.reset()
        got = decode((GraphDecoder if graph else Decoder)(cfg, w, layers, caches), ids)
        if want is None:
            want = got
        assert float((got - want).norm()) <= (9 * cfg.num_layers + 2) * 2.0 ** -11 * float(want.norm()), change


def test_other_rows_of_x(dev):
    """The functions of a step on an x that is a view: every second row, an odd offset, a transposed one."""
    from kvmix_amd.decoder import add_mlp, add_projection, head_logits

    cfg, weights, _, _, _ = small(dev)
    lw, eps = weights["layers"][0], cfg.rms_norm_eps
    x = torch.randn(3, 1, 512, generator=torch.Generator(device=dev).manual_seed(5), device=dev).half()
    for f in (lambda x: head_logits(x, weights, eps), lambda x: add_projection(x, x, lw["wo"]), lambda x: add_mlp(x, lw, eps)):
        want = f(x).float()
        for view in (misaligned(x), spread(x), torch.cat([x, x], 1)[:, 1:], torch.cat([x, x[..., :1]], -1)[..., :512], x[:1].expand(3, 1, 512)):
            expect = f(view.contiguous()).float()
            assert float((f(view).float() - expect).norm()) <= 1e-2 * float(want.norm())


class Dense:
    """Plain attention over whole keys and values: no limit on head dimensions."""

    def __call__(self, q, k, v, cache, attention_mask=None, need_weights=False):
        if cache is not None:
            k, v = torch.cat([cache[0], k], 2), torch.cat([cache[1], v], 2)
        rep = q.shape[1] // k.shape[1]
        kk, vv = k.float().repeat_interleave(rep, 1), v.float().repeat_interleave(rep, 1)
        logits = torch.matmul(q.float(), kk.transpose(2, 3).contiguous()) / q.shape[3] ** 0.5
        p = torch.softmax(logits if attention_mask is None else logits + attention_mask, -1)
        return torch.matmul(p, vv).to(q.dtype), None, (k, v)


# head dimensions that the projection kernel, rope_append or neither takes
@pytest.mark.parametrize("hidden,heads,kv_heads", [(320, 8, 4), (128, 16, 8), (240, 5, 5), (512, 4, 2), (360, 15, 3)])
def test_steps_with_other_head_dimensions(dev, hidden, heads, kv_heads):
    """Token by token as the prompt of all tokens, on any sizes that torch's products take."""
    from kvmix_amd.decoder import Decoder, DecoderConfig, init_weights

    cfg = DecoderConfig(hidden_size=hidden, num_layers=2, num_heads=heads, num_kv_heads=kv_heads, intermediate_size=384, vocab_size=100)
    weights = init_weights(cfg, dev, std=0.05, seed=2)
    ids = torch.randint(0, 100, (2, 12), generator=torch.Generator().manual_seed(1)).to(dev)
    got = decode(Decoder(cfg, weights, [Dense(), Dense()]), ids, 6)
    want = torch.stack([Decoder(cfg, weights, [Dense(), Dense()]).forward(ids[:, :t]) for t in range(6, 13)])
    assert float((got - want).norm()) <= (9 * cfg.num_layers + 2) * 2.0 ** -11 * float(want.norm())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_autocast_is_torchs(dev, dtype):
    """Under autocast the projections and the prompt's attention are torch's, in the type it casts them to."""
    from kvmix_amd.attention import KVmixAttention
    from kvmix_amd.decoder import add_projection, head_logits

    cfg, weights, _, _, _ = small(dev)
    gen = torch.Generator(device=dev).manual_seed(5)
    x = torch.randn(3, 1, 512, generator=gen, device=dev).half()
    q, k, v = (torch.randn(1, 4, 70, 128, generator=gen, device=dev).half() for _ in range(3))
    mask = torch.full((70, 70), torch.finfo(torch.float32).min, device=dev).triu_(1)[None, None]
    with torch.autocast("cuda", dtype=dtype):
        y, want = add_projection(x, x, weights["layers"][0]["wo"]), x + F.linear(x, weights["layers"][0]["wo"])
        assert y.dtype == want.dtype and torch.equal(y, want)
        logits = head_logits(x, weights, cfg.rms_norm_eps)
        assert torch.equal(logits, F.linear(F.rms_norm(x[:, 0], (512,), weights["norm"], cfg.rms_norm_eps), weights["lm_head"]).float())
        out, _, _ = KVmixAttention(4, 4, residual_length=32)(q, k, v, None, attention_mask=mask, need_weights=False)
        want = F.scaled_dot_product_attention(q, k, v, attn_mask=mask.clamp(min=-65504.0).half())
        assert out.dtype == want.dtype and torch.equal(out, want)
