"""q.K^T of gemv_cols_mfma with four query heads of a kv head: the launches whose blocks share a tile, and the sums in two
fp16 parts against float64.

Bound: fp32 sums of K <= 256 products and as many zero terms (a rounding after every four products, and fewer than 16 steps
that bring lanes and waves together: 2^-17 of the sum of magnitudes covers both terms) and the rounding of the output to
fp16; what two parts lose of x * scale has no term of its own."""
import pytest
import torch

from helpers import unpack_codes_torch
from kvmix_amd import _lib


def plan(bits, samples, rep, K, N):
    return _lib.gemv_plan(32, bits, 0, samples, rep, 1, K, N)


def test_launches_of_few_tiles_share_them():
    few, many = plan(4, 32, 4, 128, 1024), plan(4, 512, 4, 128, 8064)
    assert few["kernel"] == many["kernel"] == "gemv_cols_mfma<4,4>"
    assert few["ksplit"] == 4 and few["block"][1] == 4 and few["grid"][:2] == (2, 8)
    assert many["ksplit"] == 1
    assert plan(4, 128, 4, 128, 8192)["ksplit"] == 4 and plan(4, 128, 4, 128, 8704)["ksplit"] == 1  # (512 tiles, 544)
    assert plan(2, 32, 4, 32, 1024)["ksplit"] == 1 and plan(2, 32, 4, 80, 1024)["ksplit"] == 3      # (chunks of 32 rows)


def operands(bits, B, nh, nkv, M, K, N, seed):
    gen = torch.Generator().manual_seed(seed)
    code = torch.randint(-2 ** 31, 2 ** 31, (B, nkv, K, N * bits // 32), generator=gen).int()
    scale = (torch.rand(B, nkv, K, N // 32, generator=gen) + 0.3).half()
    zero = torch.randn(B, nkv, K, N // 32, generator=gen).half()
    return torch.randn(B, nh, M, K, generator=gen).half(), code, scale, zero


def check(dev, bits, x, code, scale, zero):
    import KVmix

    B, nh, M, K = x.shape
    nkv, N = code.shape[1], scale.shape[-1] * 32
    assert plan(bits, B * nh, nh // nkv, K, N)["kernel"] == "gemv_cols_mfma<%d,4>" % bits
    x, code, scale, zero = (t.to(dev) for t in (x, code, scale, zero))
    got = KVmix.quantized_gemm(32, x, code, scale, zero, bits).double()
    s = scale.double().repeat_interleave(32, -1)
    term, z, xd = s * unpack_codes_torch(code, bits, False).double(), zero.double().repeat_interleave(32, -1), x.double().reshape(B, nkv, -1, K)
    want, size = (t.reshape(got.shape) for t in (xd @ (term + z), xd.abs() @ (term.abs() + z.abs())))
    finite = want.abs() < 65504
    assert finite.float().mean() > 0.5
    assert ((got - want).abs() <= 2.0 ** -11 * want.abs() + 2.0 ** -17 * size + 2.0 ** -25)[finite].all()
    return got.cpu()


@pytest.mark.gpu
# one tile and a ragged last one, fewer chunks than waves, chunks that do not divide among them or end past K, two rows of x,
# eight heads of a kv head, the largest launch that shares and the smallest that does not, several tiles per wave
@pytest.mark.parametrize("B,nh,nkv,M,K,N", [(1, 4, 1, 1, 128, 512), (1, 4, 1, 2, 128, 544), (2, 8, 2, 1, 33, 1024), (1, 4, 1, 1, 65, 736), (1, 16, 2, 1, 150, 992),
                                            (1, 4, 1, 1, 224, 512), (4, 32, 8, 1, 128, 8192), (4, 32, 8, 1, 128, 8704), (8, 64, 16, 1, 96, 16384)])
@pytest.mark.parametrize("bits", [1, 2, 4])
def test_against_float64(dev, bits, B, nh, nkv, M, K, N):
    check(dev, bits, *operands(bits, B, nh, nkv, M, K, N, K + N + bits))


@pytest.mark.gpu
# x of any size, heads far apart; scales beyond the first powers, tokens far apart, rows that grow; shared tiles and several
# tiles per wave
@pytest.mark.parametrize("B,nh,nkv,N", [(1, 8, 2, 1056), (8, 64, 16, 16384)])
@pytest.mark.parametrize("kind", ["large", "heads apart", "groups apart", "rising", "tiny"])
@pytest.mark.parametrize("bits", [1, 2, 4])
def test_two_fp16_parts(dev, bits, kind, B, nh, nkv, N):
    x, code, scale, zero = operands(bits, B, nh, nkv, 1, 128, N, 7 * bits)
    if kind == "large":
        x, scale = x * 6, scale * 20
    if kind == "heads apart":
        x = x * (10.0 ** (torch.arange(nh) % 8 - 4)).half()[None, :, None, None]
    if kind == "groups apart":
        scale = scale * torch.tensor([1e-4, 1.0, 30.0, 300.0]).repeat(N // 32)[:N // 32].half()
    if kind == "rising":
        x[..., -1], scale[:, :, -1, ::3] = 30.0, 90.0
        x[..., 40], scale[:, :, 5, 1::5] = 9.0, 20.0
    if kind == "tiny":
        x, scale, zero = x * 2.0 ** -6, scale * 2.0 ** -10, zero * 2.0 ** -10
    check(dev, bits, x, code, scale, zero)


@pytest.mark.gpu
# scales from ordinary ones down to where the outputs are fp16's smallest, the same everywhere or those of normal values; x that
# is all of one size, and so small that only its scales make the outputs
@pytest.mark.parametrize("x_size,size", [(1.0, 2e-3), (1.0, 5e-4), (1.0, 1e-5), (2e-3, 2e-3), (1e-5, 2.0)])
@pytest.mark.parametrize("bits,constant", [(4, True), (2, False)])
def test_small_operands(dev, bits, constant, x_size, size):
    """The code term alone (zeros of zero), and with minima that nearly cancel it."""
    x, code, scale, zero = operands(bits, 1, 8, 2, 1, 128, 1056, bits)
    scale = torch.full_like(scale, size) if constant else (scale.double() * size).half()
    x = torch.full_like(x, x_size) if constant else (x.double() * x_size).half()
    for zeros in (torch.zeros_like(zero), (scale.double() * (-(2.0 ** bits - 1) / 2)).half()):
        check(dev, bits, x, code, scale, zeros)


@pytest.mark.gpu
def test_infinities_stay_with_their_own_tokens(dev):
    x, code, scale, zero = operands(2, 1, 4, 1, 1, 128, 1024, 3)
    clean = check(dev, 2, x, code, scale, zero)
    import KVmix

    scale[0, 0, 70, 3] = float("inf")
    got = KVmix.quantized_gemm(32, x.to(dev), code.to(dev), scale.to(dev), zero.to(dev), 2).double().cpu()
    other = torch.arange(1024) // 32 != 3
    assert torch.equal(got[..., other], clean[..., other]) and not torch.isfinite(got[..., ~other]).any()
