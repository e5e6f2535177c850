"""ops.prefill_attention (kvmix_prefill_attention) against softmax(q k^T / sqrt(D) + mask) v in float64.

Bound per output: a probability is off by its rounding for the product with v (fp16: 2^-11; grouped heads, two fp16 parts:
2^-22) and by twice the error of a logit (fp32 sums of D products that start from the mask's entry, and the exponent's own
rounding), all weighted with p |v|, and the output by its own rounding to fp16."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu
LOWEST = -65504.0


def operands(dev, B, nh, nkv, Q, T, D, seed=0):
    gen = torch.Generator(device="cpu").manual_seed(seed + 7 * Q + T + D)
    r = lambda *s: torch.randn(*s, generator=gen).half().to(dev)  # noqa: E731
    k = r(B, nkv, T, D)
    k[..., 3] *= 10
    return r(B, nh, Q, D), k, r(B, nkv, T, D)


def reference(q, k, v, mask):
    D, rep = q.shape[3], q.shape[1] // k.shape[1]
    q, k, v = q.double().cpu(), k.double().cpu().repeat_interleave(rep, 1), v.double().cpu().repeat_interleave(rep, 1)
    s = torch.matmul(q, k.transpose(2, 3).contiguous()) / math.sqrt(D)
    size = torch.matmul(q.abs(), k.abs().transpose(2, 3).contiguous()) / math.sqrt(D)
    if mask is not None:
        m = mask.cpu()
        dead = m.amax(-1, keepdim=True) <= (LOWEST if m.dtype == torch.float16 else -1e30)
        m = m.float().clamp(min=LOWEST).half().double()
        s = (s + m).masked_fill(dead, 0.0)
        size = size + m.abs() * (m > LOWEST)
    p = torch.softmax(s, -1)
    delta = ((D + 2) * 2.0 ** -24 * size).amax(-1, keepdim=True) + 2.0 ** -21
    return torch.matmul(p, v), torch.matmul(p, v.abs()), delta


def check(got, q, k, v, mask):
    want, size, delta = reference(q, k, v, mask)
    parts = 2.0 ** -11 if q.shape[1] == k.shape[1] else 2.0 ** -22
    err = (got.double().cpu() - want).abs()
    bound = (parts + 2 * delta) * size + 2.0 ** -11 * want.abs() + 2.0 ** -24
    assert (err <= bound).all(), float((err / bound).max())


def causal(Q, T, dtype, dev):
    return torch.triu(torch.full((Q, T), torch.finfo(dtype).min, dtype=dtype, device=dev), 1 + T - Q)[None, None]


# lengths around the 32 queries of a wave, the 128 of a block, the 64 keys of a tile and the 64 tiles looked up at once
@pytest.mark.parametrize("B,nh,nkv,Q,T,D", [(1, 1, 1, 1, 1, 128), (2, 4, 4, 33, 33, 128), (1, 8, 2, 63, 63, 128), (2, 4, 1, 65, 65, 64),
                                            (1, 3, 3, 128, 128, 64), (1, 2, 1, 129, 257, 128), (3, 6, 6, 200, 200, 128),
                                            (1, 4, 2, 513, 513, 128), (1, 1, 1, 40, 4161, 128), (1, 2, 2, 4160, 4160, 64)])
@pytest.mark.parametrize("kind", ["none", "float", "half", "padded"])
def test_against_float64(dev, B, nh, nkv, Q, T, D, kind):
    from kvmix_amd import ops

    q, k, v = operands(dev, B, nh, nkv, Q, T, D)
    mask = None if kind == "none" else causal(Q, T, torch.float32 if kind == "float" else torch.float16, dev)
    if kind == "padded":  # one mask per sequence; rows before the first token are masked everywhere
        pads = torch.tensor([(37 * b + 5) % max(T // 2, 1) for b in range(B)], device=dev)
        dead = torch.arange(T, device=dev)[None, :] < pads[:, None]
        mask = torch.minimum(mask, torch.zeros(B, T, dtype=torch.float16, device=dev).masked_fill_(dead, LOWEST)[:, None, None, :])
    got = ops.prefill_attention(q, k, v, mask)
    assert got is not None and got.shape == q.shape
    check(got, q, k, v, mask)
    assert torch.equal(got, ops.prefill_attention(q, k, v, mask))


def test_masks_of_every_form(dev):
    """Dense biases, a mask per head, expanded and unaligned masks, entries between the classes, -inf, rows whose every
    entry is low but not lowest (nothing may be skipped there)."""
    from kvmix_amd import ops

    B, nh, Q, T, D = 2, 2, 70, 150, 128
    q, k, v = operands(dev, B, nh, nh, Q, T, D)
    gen = torch.Generator(device="cpu").manual_seed(5)
    bias = 3 * torch.randn(B, nh, Q, T, generator=gen).to(dev)
    low = torch.full((1, 1, Q, T), -65504.0, device=dev)
    low[..., :40] = -65472.0
    low[..., 3:, :] = -1e31
    row = torch.where(torch.arange(T, device=dev) < 90, 0.0, -float("inf"))
    masks = [bias, bias.half(), bias[:1], bias[:, :1].half(), low, low.half(), row.expand(B, nh, Q, T), row.half().expand(1, 1, Q, T),
             torch.zeros(B, 1, Q, T + 3, device=dev, dtype=torch.float16)[..., 3:], bias.transpose(2, 3).contiguous().transpose(2, 3)]
    for m in masks:
        check(ops.prefill_attention(q, k, v, m), q, k, v, m)


def test_views_and_refusals(dev):
    from kvmix_amd import ops

    q, k, v = operands(dev, 2, 4, 2, 50, 50, 128)
    want = ops.prefill_attention(q, k, v)
    tokens_first = [t.transpose(1, 2).contiguous().transpose(1, 2) for t in (q, k, v)]
    assert torch.equal(ops.prefill_attention(*tokens_first), want)
    odd = [torch.empty(t.numel() + 1, dtype=t.dtype, device=dev)[1:].view(t.shape).copy_(t) for t in (q, k, v)]
    assert torch.equal(ops.prefill_attention(*odd), want)
    long_rows = [torch.cat([t, t], -1)[..., :128] for t in (q, k, v)]
    assert torch.equal(ops.prefill_attention(*long_rows), want)
    for bad in ((q[..., :96], k[..., :96], v[..., :96]), (q, k, v[..., :64]), (q[:1], k, v), (q.float(), k, v), (q[:, :3], k, v)):
        assert ops.prefill_attention(*bad) is None
    assert ops.prefill_attention(q, k, v, torch.zeros(50, 50, device=dev)) is None
    assert ops.prefill_attention(q, k, v, torch.zeros(1, 1, 50, 50, device=dev, dtype=torch.bool)) is None


def test_prompt_branch_takes_it_only_for_plain_calls(dev):
    from kvmix_amd import ops
    from kvmix_amd.attention import KVmixAttention

    q, k, v = operands(dev, 1, 4, 2, 96, 96, 128)
    mask = causal(96, 96, torch.float32, dev)
    layer = KVmixAttention(4, 4)
    out, _, _ = layer(q, k, v, None, attention_mask=mask, need_weights=False)
    assert torch.equal(out, ops.prefill_attention(q, k, v, mask))
    qg = q.clone().requires_grad_()
    out_g, _, _ = layer(qg, k, v, None, attention_mask=mask, use_cache=False, need_weights=False)
    out_g.float().sum().backward()
    assert qg.grad is not None and torch.allclose(out_g.float(), out.float(), rtol=2e-3, atol=2e-3)
    tangent = torch.func.jvp(lambda x: layer._prompt_attention(x.float().half(), k, v, mask, 2), (q,), (torch.zeros_like(q),))[0]
    assert torch.allclose(tangent.float(), out.float(), rtol=2e-3, atol=2e-3)


@pytest.mark.parametrize("nh,nkv,T,D", [(2, 2, 70, 128), (4, 1, 129, 64), (2, 2, 64, 128)])
def test_an_infinite_value_at_the_ragged_end(dev, nh, nkv, T, D):
    """A value of the last token that is infinite stays infinite in the outputs that weigh it, without a mask."""
    from kvmix_amd import ops

    q, k, v = operands(dev, 1, nh, nkv, T, T, D)
    v[0, 0, T - 1, 5], v[0, 0, T - 1, 6] = float("inf"), -float("inf")
    q[...] = k[:, :, T - 1:].repeat_interleave(nh // nkv, 1) * 0.1  # (every query weighs it)
    got, want = ops.prefill_attention(q, k, v), reference(q, k, v, None)[0]
    assert torch.isinf(want).any() and not torch.isnan(want).any()
    assert torch.equal(torch.isinf(got).cpu(), torch.isinf(want)) and not torch.isnan(got).any()


@pytest.mark.parametrize("nh,nkv", [(2, 2), (4, 1)])
def test_a_dominant_key_has_a_weight_of_one(dev, nh, nkv):
    """Rows that one late key dominates by less than a factor of 2^8: its probability is not rounded and the sum is that of
    the weights the products see, so that nearly all outputs are the correctly rounded ones (a rounding of that probability
    to eleven bits would move every third)."""
    from kvmix_amd import ops

    T, D = 256, 128
    gen = torch.Generator(device="cpu").manual_seed(3)
    q, k, v = torch.zeros(1, nh, T, D), torch.zeros(1, nkv, T, D), torch.randn(1, nkv, T, D, generator=gen)
    q[..., 0] = 16.0
    q[..., 1] = 16.0 * torch.rand(1, nh, T, generator=gen)
    k[..., 0] = -60.0
    k[:, :, 5, 0] = 0.0                              # logit 0 in the first tile
    k[:, :, 200, 0], k[:, :, 200, 1] = 0.5, 3.3      # up to 5.3 above it in the fourth
    v[:, :, 5] *= 2.0 ** -9
    q, k, v = (t.half().to(dev) for t in (q, k, v))
    got, want = ops.prefill_attention(q, k, v), reference(q, k, v, None)[0]
    assert float((got.cpu() == want.half()).float().mean()) > 0.9


@pytest.mark.parametrize("nh,nkv", [(8, 8), (8, 2)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
def test_large_entries_of_a_mask_round_once(dev, nh, nkv, dtype):
    """A mask of -10000 on everything: the sum of logit and entry is rounded at the size of 10000 sqrt(128), 2^-7 in the last
    place, which is 2.0e-4 (rms) of the logit; with the roundings of probabilities and outputs (2.0 to 2.4e-4) 3.2e-4."""
    from kvmix_amd import ops

    q, k, v = operands(dev, 1, nh, nkv, 700, 700, 128)
    mask = torch.full((1, 1, 700, 700), -10000.0, dtype=dtype, device=dev)
    want = reference(q, k, v, mask)[0]
    got = ops.prefill_attention(q, k, v, mask).double().cpu()
    assert float((got - want).norm()) <= 4.5e-4 * float(want.norm())
