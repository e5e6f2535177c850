"""ops.copy_rows (kvmix_copy_rows) against copy_, and what is built on it against the composition by concatenation, bit for
bit."""
import pytest
import torch

pytestmark = pytest.mark.gpu


# rows around the 16-byte piece, alignments of two bytes, more copies than a launch takes, blocks around 1024 pieces
@pytest.mark.parametrize("B,H,R,S,pad", [(1, 1, 1, 1, 0), (2, 3, 5, 7, 1), (1, 2, 64, 8, 3), (3, 1, 9, 9, 0), (2, 2, 33, 73, 1),
                                         (1, 1, 1, 8191, 5), (2, 4, 128, 64, 0), (1, 1, 1024, 8, 1), (1, 1, 1025, 8, 8)])
def test_copies_match(dev, B, H, R, S, pad):
    from kvmix_amd import ops

    gen = torch.Generator(device="cpu").manual_seed(R + S)
    pairs, wants, wholes = [], [], []
    for i in range(18):
        dtype = (torch.float16, torch.int32, torch.float32)[i % 3]
        src = torch.randint(-30000, 30000, (B, H, R, S + 2 * pad), generator=gen).to(dev).to(dtype)[..., pad:pad + S]
        whole = torch.full((B, H, R + 2, S + pad + i % 2), 7, dtype=dtype, device=dev)
        if i % 4 == 3:
            src = src.transpose(0, 1).contiguous().transpose(0, 1)
        want = whole.clone()
        want[:, :, 1:R + 1, pad:pad + S] = src
        pairs.append((whole[:, :, 1:R + 1, pad:pad + S], src))
        wants.append(want)
        wholes.append(whole)
    ops.copy_rows(pairs)
    for got, want in zip(wholes, wants):
        assert torch.equal(got, want)


def test_copies_refuse_what_they_cannot_do(dev):
    from kvmix_amd import ops

    a, b = torch.zeros(1, 1, 2, 4, device=dev), torch.zeros(1, 1, 2, 5, device=dev)
    for pair in ((a, b), (a, b[..., :4].half()), (a[0], a[0]), (b.transpose(2, 3)[..., :2], a.transpose(2, 3)[:, :, :1].expand(1, 1, 5, 2))):
        with pytest.raises(RuntimeError):
            ops.copy_rows([pair])
    ops.copy_rows([])
    ops.copy_rows([(a[:, :, :0], b[:, :, :0, :4])])


@pytest.mark.parametrize("k_bits,v_bits,window,B,H,D", [(4, 2, None, 2, 3, 128), (3, 4, None, 1, 2, 64), (2, 1, 32, 3, 1, 128),
                                                        (1, 4, 64, 1, 1, 96), (3, 2, 128, 2, 2, 128)])
def test_growing_the_tuple_matches_concatenation(dev, k_bits, v_bits, window, B, H, D):
    from kvmix_amd.attention import KVmixAttention

    layer = KVmixAttention(k_bits, v_bits, residual_length=window)
    gen = torch.Generator(device="cpu").manual_seed(k_bits + D)
    past, flushes = (None,) * 8 + (0,), 0
    for step in range(280):
        n = 3 if step == 40 else 1
        k, v = (torch.randn(B, H, n, D, generator=gen).half().to(dev) for _ in range(2))
        if step % 7 == 0:  # (as projections leave them)
            k = k.transpose(1, 2).contiguous().transpose(1, 2)
        kc, kt, ks, km, vc, vt, vs, vm, length = past
        kt2, vt2 = (k, v) if kt is None else (torch.cat([kt, k], 2), torch.cat([vt, v], 2))
        kt2, (kc, ks, km), vt2, (vc, vs, vm) = layer._flush(kt2, (kc, ks, km), vt2, (vc, vs, vm))
        before = [None if t is None else t.clone() for t in past[:8]]
        got = layer._grown(past, k, v)
        for a, b in zip(got, (kc, kt2, ks, km, vc, vt2, vs, vm)):
            assert (a is None) == (b is None) and (a is None or (a.dtype == b.dtype and torch.equal(a, b)))
        assert all(a is None or torch.equal(a, b) for a, b in zip(past[:8], before))  # (the caller's tuple is left alone)
        flushes += past[0] is None and got[0] is not None or (past[0] is not None and got[0].shape != past[0].shape)
        past = got + (length + n,)
    assert flushes >= 2


def test_more_pieces_than_one_launch_counts(dev):
    """A cache of 2^31 rows (expanded ones here, of one group each) is grown by torch's copies as before: a launch counts
    fewer sixteen-byte pieces than that."""
    import KVmix

    shape = (1 << 11, 1 << 10, 1 << 10, 1)
    code = torch.tensor(0x12345678, dtype=torch.int32, device=dev).expand(shape)
    scale, zero = (torch.tensor(v, dtype=torch.float16, device=dev).expand(shape) for v in (0.5, -2.0))
    nothing = torch.empty(shape[:3] + (0,), dtype=torch.float16, device=dev)
    for got, want in zip(KVmix.process_key_quantization_cuda(nothing, code, scale, zero, 32, 4), (0x12345678, 0.5, -2.0)):
        assert got.shape == shape and got.is_contiguous()
        assert all(bool((part == want).all()) for part in got.view(64, -1))
    del got
    torch.cuda.empty_cache()
