"""q.K^T with four query heads per pass over the reference's 3-bit words (gemv_cols3<1,2,8,4>): the plan that takes it,
and its sums against float64.

Bound: fp32 sums of K products in blocks of four (K * 2^-23 of the sum of magnitudes, the weights themselves being exact)
and the rounding of the output to fp16."""
import pytest
import torch

from kvmix_amd import _lib

KERNEL = "gemv_cols3<1,2,8,4>"


def weights(code, scale, zero):
    w = torch.stack([(code.long() & 0xFFFFFFFF) >> (3 * i) & (3 if i == 10 else 7) for i in range(11)], -1).flatten(-2)
    return scale.double().repeat_interleave(11, -1) * w + zero.double().repeat_interleave(11, -1)


def test_rows_it_is_chosen_for():
    def kernel(units, K=128, rep=4, samples=32):
        return _lib.gemv_plan(11, 3, 0, samples, rep, 1, K, 11 * units)["kernel"]

    for units in (128, 205, 256, 2967):
        assert kernel(units) == KERNEL and kernel(units, rep=8) == KERNEL and kernel(units, K=64) == KERNEL
    for units in (64, 127, 129, 186):
        assert kernel(units) == "gemv_cols3<2,2,4,4>"
    assert kernel(256, K=100) == "gemv_cols3<2,2,4,4>" and kernel(256, K=4096) != KERNEL and kernel(256, rep=2) != KERNEL


@pytest.mark.gpu
# one tile and moved-back last tiles, one wave per tile (many tiles) and four slicing K, two rows of x, eight heads per kv head
@pytest.mark.parametrize("B,nh,nkv,M,K,units", [(1, 4, 1, 1, 128, 128), (1, 8, 2, 2, 64, 205), (2, 16, 2, 1, 32, 333), (16, 32, 8, 1, 128, 1100),
                                                (1, 8, 2, 1, 256, 2967)])
# ordinary scales; outside the exact range of the matrix operands in some rows (tiny, huge, zero); negative and not finite nowhere
@pytest.mark.parametrize("spread", ["ordinary", "mixed", "tiny"])
def test_against_float64(dev, B, nh, nkv, M, K, units, spread):
    import KVmix

    gen = torch.Generator(device="cpu").manual_seed(units + K)
    code = torch.randint(-2 ** 31, 2 ** 31, (B, nkv, K, units), generator=gen).int()
    scale = torch.rand(B, nkv, K, units, generator=gen) + 0.3
    if spread == "tiny":
        scale = scale * 2.0 ** -18
    if spread == "mixed":
        pick = torch.randint(0, 40, scale.shape, generator=gen)
        scale = torch.where(pick == 0, 0.0 * scale, torch.where(pick == 1, 3e-7 + 0 * scale, torch.where(pick == 2, 0.00613 * scale, scale)))
        scale[:, :, 5, ::7] = 9001.0
        scale[:, :, 9, 3] = -scale[:, :, 9, 3]
    zero = (torch.randn(B, nkv, K, units, generator=gen) * (2.0 ** -18 if spread == "tiny" else 1.0)).half()
    scale, x = scale.half(), torch.randn(B, nh, M, K, generator=gen).half()
    x[..., 5] *= 0.01
    got = KVmix.quantized_gemm(11, *(t.to(dev) for t in (x, code, scale, zero)), 3).double().cpu()
    w, xd = weights(code, scale, zero), x.double().reshape(B, nkv, nh // nkv * M, K)
    want = torch.matmul(xd, w).reshape(got.shape)
    size = torch.matmul(xd.abs(), weights(code, scale.abs(), zero.abs())).reshape(got.shape)
    assert ((got - want).abs() <= 2.0 ** -11 * want.abs() + K * 2.0 ** -23 * size + 2.0 ** -25).all()
