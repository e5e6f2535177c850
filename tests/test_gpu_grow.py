"""A cache grown in one launch (kvmix_grow): the append operators and a step on the 9-tuple against what the separate
quantizers and torch.cat give, bit for bit."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def bits(a, b):
    assert a.shape == b.shape and a.dtype == b.dtype and torch.equal(a.contiguous().view(torch.uint8), b.contiguous().view(torch.uint8))


# rows shorter than a 16-byte piece, odd row lengths (scales at any two bytes), one head, nothing cached, a part of its own launch
@pytest.mark.parametrize("B,H,D,old,new", [(1, 1, 64, 32, 32), (2, 3, 128, 96, 64), (1, 8, 128, 992, 32), (3, 1, 64, 0, 32), (2, 4, 128, 2304, 352), (8, 32, 128, 64, 704)])
@pytest.mark.parametrize("kb,vb", [(1, 4), (2, 1), (4, 2), (3, 2)])
@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
def test_append_operators(dev, B, H, D, old, new, kb, vb, dtype):
    import KVmix

    gen = torch.Generator(device=dev).manual_seed(old + new + kb)
    kg = 11 if kb == 3 else 32
    old_k, new_k = old // kg * kg, new // kg * kg
    k = torch.randn(B, H, D, old_k + new_k, generator=gen, device=dev).to(dtype)
    v = torch.randn(B, H, old + new, D, generator=gen, device=dev).to(dtype)
    for x, dim, group, b, op, n in ((k, 3, kg, kb, KVmix.process_key_quantization_cuda, old_k), (v, 2, 32, vb, KVmix.process_value_quantization_cuda, old)):
        fresh = x.narrow(dim, n, x.shape[dim] - n)
        before = KVmix.quantize_pack_last_dim_cuda(x.narrow(dim, 0, n).contiguous(), group, b)
        alone = op(fresh, *(t.narrow(dim, 0, 0) for t in before), group, b)
        for got, first, second in zip(op(fresh, *before, group, b), before, alone):
            bits(got, torch.cat([first, second], dim))
        # previous parts as views of longer buffers, (batch, head) collapsible and not
        wide = [torch.cat([t, t], dim).narrow(dim, 0, t.shape[dim]) for t in before]
        swapped = [t.transpose(0, 1).contiguous().transpose(0, 1) for t in before]
        for parts in (wide, swapped):
            for got, first, second in zip(op(fresh, *parts, group, b), before, alone):
                bits(got, torch.cat([first, second], dim))


# both sides flush, one side does, none; first flush; key groups of 11; head dimension 64; one (batch, head) slice
@pytest.mark.parametrize("B,H,D", [(1, 8, 128), (2, 3, 64), (1, 1, 128)])
@pytest.mark.parametrize("kb,vb,rk,rv", [(4, 4, 0.3, 0.3), (2, 1, 0.2, 0.1), (3, 2, 0.2, 0.2), (1, 4, 0.1, 0.3)])
def test_steps_on_the_tuple(dev, B, H, D, kb, vb, rk, rv):
    from kvmix_amd.attention import KVmixAttention

    gen = torch.Generator(device=dev).manual_seed(kb)
    layer = KVmixAttention(kb, vb, rk, rv)
    slow = KVmixAttention(kb, vb, rk, rv)
    rand = lambda n: torch.randn(B, H, n, D, generator=gen, device=dev).half()
    got = want = (None,) * 8 + (0,)
    flushed = set()
    for step in range(120):
        k, v = rand(1), rand(1)
        if step % 2:  # (strides of a fused projection)
            k, v = (t.transpose(1, 2).contiguous().transpose(1, 2) for t in (k, v))
        sizes = tuple(0 if t is None else t.shape for t in (got[0], got[4]))
        got = layer._grown(got, k, v) + (step + 1,)
        kt = k if want[1] is None else torch.cat([want[1], k], 2)
        vt = v if want[5] is None else torch.cat([want[5], v], 2)
        kt, kq, vt, vq = slow._flush(kt, (want[0], want[2], want[3]), vt, (want[4], want[6], want[7]))
        want = (kq[0], kt, kq[1], kq[2], vq[0], vt, vq[1], vq[2], step + 1)
        flushed.add(tuple(a != (0 if t is None else t.shape) for a, t in zip(sizes, (got[0], got[4]))))
        for a, b in zip(got[:8], want[:8]):
            assert (a is None) == (b is None)
            if a is not None:
                bits(a, b)
    assert (False, False) in flushed and len(flushed) >= 2


# flush and tails in one launch and, from 2^18 value groups on, in two; nothing to flush on one side; a head dimension of 64
@pytest.mark.parametrize("B,H,T,D,R", [(1, 4, 400, 128, 128), (2, 3, 333, 64, None), (2, 32, 1100, 128, 64), (1, 2, 129, 128, 128), (1, 1, 40, 128, 128)])
@pytest.mark.parametrize("kb,vb", [(4, 2), (3, 4), (1, 1)])
def test_prompts_on_the_tuple(dev, B, H, T, D, R, kb, vb):
    from kvmix_amd.attention import KVmixAttention

    gen = torch.Generator(device=dev).manual_seed(T)
    layer = KVmixAttention(kb, vb, residual_length=R)
    k, v = (torch.randn(B, T, H, D, generator=gen, device=dev).half().transpose(1, 2) for _ in range(2))
    for key, value in ((k, v), (k.contiguous(), v.contiguous())):
        kt, kq, vt, vq = layer._flush(key, (None,) * 3, value, (None,) * 3, prompt=True)
        for a, b in zip(layer._prompt_entries(key, value), (kq[0], kt, kq[1], kq[2], vq[0], vt, vq[1], vq[2])):
            assert (a is None) == (b is None)
            if a is not None:
                bits(a, b)
                assert a.is_contiguous()
