"""p.V of gemv_rows_mfma where blocks share the columns of an output row: the grids it is launched with and its sums
against float64.

Bound: fp32 sums of K products and as many zero terms (K * 2^-23 of the sum of magnitudes) and the rounding of the output
to fp16."""
import pytest
import torch

from helpers import unpack_codes_torch
from kvmix_amd import _lib


def plan(bits, samples, rep, K):
    return _lib.gemv_plan(32, 3 if bits == 30 else bits, 1 if bits == 30 else 0, samples, rep, 1, K, 128)


def test_launches_that_leave_cus_idle_are_cut_along_the_columns():
    assert plan(4, 32, 1, 3968)["grid"][:2] == (4, 32) and plan(4, 64, 1, 3968)["grid"][:2] == (4, 64)
    assert plan(2, 128, 1, 2048)["grid"][:2] == (2, 128) and plan(2, 256, 1, 2048)["grid"][:2] == (1, 256)
    long = plan(2, 32, 1, 32640)  # (four blocks along K already, and their reduction)
    assert long["splits"] == 4 and long["grid"][:2] == (8, 32) and long["launches"] == 2
    assert plan(4, 32, 4, 1024)["grid"][:2] == (4, 8)
    assert plan(1, 2048, 1, 4064)["grid"][:2] == (1, 2048)


def operands(bits, B, nh, nkv, M, K, seed):
    gen = torch.Generator().manual_seed(seed)
    words = 12 if bits == 30 else 4 * bits
    code = torch.randint(-2 ** 31, 2 ** 31, (B, nkv, K, words), generator=gen).int()
    scale = (torch.rand(B, nkv, K, 4, generator=gen) + 0.3).half()
    zero = torch.randn(B, nkv, K, 4, generator=gen).half()
    x = torch.softmax(1.5 * torch.randn(B, nh, M, K, generator=gen), -1).half()
    return x, code, scale, zero


def exact(bits, x, code, scale, zero):
    """The sums in float64, and the sums of the terms' magnitudes."""
    q = unpack_codes_torch(code, 3 if bits == 30 else bits, bits == 30).double()
    B, nh, M, K = x.shape
    xd = x.double().reshape(B, code.shape[1], -1, K)
    term = scale.double().repeat_interleave(32, -1) * q
    z = zero.double().repeat_interleave(32, -1)
    return tuple(t.reshape(B, nh, M, 128) for t in (xd @ (term + z), xd.abs() @ (term.abs() + z.abs())))


@pytest.mark.gpu
# quarters and halves of rows, one chunk and less than two, ragged ends, waves without rows, blocks along K, two rows of x
@pytest.mark.parametrize("B,nh,nkv,M,K", [(1, 2, 2, 1, 128), (1, 3, 3, 2, 250), (1, 32, 32, 1, 3968), (4, 32, 32, 1, 1111), (2, 32, 32, 1, 16500),
                                          (1, 4, 1, 1, 131), (1, 32, 8, 1, 1024), (1, 16, 2, 2, 700), (4, 32, 8, 1, 9000), (16, 32, 8, 1, 500)])
@pytest.mark.parametrize("bits", [1, 2, 4, 30])
def test_against_float64(dev, bits, B, nh, nkv, M, K):
    import KVmix

    assert plan(bits, B * nh, nh // nkv, K)["kernel"].startswith("gemv_rows_mfma<")
    ops = operands(bits, B, nh, nkv, M, K, K + bits)
    got = KVmix.quantized_gemm(32, *(t.to(dev) for t in ops), 3 if bits == 30 else bits, *((1,) if bits == 30 else ())).double().cpu()
    want, size = exact(bits, *ops)
    assert ((got - want).abs() <= 2.0 ** -11 * want.abs() + K * 2.0 ** -23 * size + 2.0 ** -25).all()
