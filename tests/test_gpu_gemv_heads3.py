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


def test_operands_are_exact():
    """The arithmetic of the operands over every finite scale, code and offset, in numpy's fp16 (no GPU): below 64 the scale
    itself, from 64 to 8192 scale / 128; both parts times code * 2^o, and their sum, are what they stand for."""
    import numpy as np

    bits = np.arange(0x7C00, dtype=np.uint16)
    bits = np.concatenate([bits, bits | 0x8000])
    scale = bits.view(np.float16)
    for large in (False, True):
        size = np.abs(scale.astype(np.float64))
        s = scale[(size >= 64) & (size < 8192) if large else size < 64]
        if large:
            s = s * np.float16(0.0078125)
        assert np.isfinite(s).all()
        high = (s.view(np.uint16) & 0xFFF8).view(np.float16)
        low = s - high
        assert (low.astype(np.float64) + high.astype(np.float64) == s.astype(np.float64)).all()
        for part in (high, low):
            away = part * np.float16(-1024)
            assert np.isfinite(away).all() and (away.astype(np.float64) == -1024 * part.astype(np.float64)).all()
            for o in range(8):
                for code in range(8):
                    h = np.float64(np.float16(1024 + code * 2 ** o))
                    exact = h * part.astype(np.float64) + away.astype(np.float64)  # (one rounding to fp16 follows)
                    assert (exact.astype(np.float16).astype(np.float64) == exact).all() and (exact == code * 2.0 ** o * part.astype(np.float64)).all()


SPREADS = {
    "uniform": lambda s, r: r,                                                    # [0, 1): small ones everywhere
    "small": lambda s, r: 0.01 * r,
    "subnormal": lambda s, r: 2.0 ** -14 * r,
    "channels": lambda s, r: s * torch.tensor([0.002, 1.0, 0.05, 300.0]).repeat(s.shape[2] // 4)[:, None],  # rows of every size, large ones among them
    "large": lambda s, r: 64 + 8000 * r * r,
    "largest": lambda s, r: 64 + 65000 * r * r,
    "beside": lambda s, r: torch.where(r < 0.02, 900.0 + 0 * s, torch.where(r < 0.04, 0.00613 * s, s)),     # both sizes in one row: plain fp32
}


@pytest.mark.gpu
@pytest.mark.parametrize("spread", list(SPREADS))
@pytest.mark.parametrize("x_scale", [1.0, 700.0])
@pytest.mark.parametrize("B,nh,nkv,M,K,units", [(1, 8, 2, 1, 128, 205), (2, 16, 4, 2, 64, 333)])
def test_scales_of_every_size(dev, spread, x_scale, B, nh, nkv, M, K, units):
    """The zero terms are kept at the size of the code terms, so that both weigh in."""
    import KVmix

    gen = torch.Generator(device="cpu").manual_seed(len(spread) + K)
    code = torch.randint(-2 ** 31, 2 ** 31, (B, nkv, K, units), generator=gen).int()
    r = torch.rand(B, nkv, K, units, generator=gen)
    scale = SPREADS[spread](r * 0.5 + 0.3, torch.rand(B, nkv, K, units, generator=gen)).half()
    zero = (-3.5 * scale.float() * torch.rand(B, nkv, K, units, generator=gen)).clamp(-60000, 60000).half()
    x = (torch.randn(B, nh, M, K, generator=gen) * x_scale).half()
    assert bool(torch.isfinite(zero).all())
    if spread.startswith("larg"):
        x = (x.float() * 2.0 ** -16).half()  # (an output that fp16 can hold)
    elif x_scale > 1 and spread == "channels":
        x[..., 3::4] *= 0.01
    got = KVmix.quantized_gemm(11, *(t.to(dev) for t in (x, code, scale, zero)), 3).double().cpu()
    xd = x.double().reshape(B, nkv, nh // nkv * M, K)
    want = torch.matmul(xd, weights(code, scale, zero)).reshape(got.shape)
    size = torch.matmul(xd.abs(), weights(code, scale.abs(), zero.abs())).reshape(got.shape)
    bound = 2.0 ** -11 * want.abs() + K * 2.0 ** -23 * size + 2.0 ** -25
    fits = want.abs() + bound < 65504
    assert fits.float().mean() > 0.05 and ((got - want).abs() <= bound)[fits].all()


@pytest.mark.gpu
def test_what_is_not_finite(dev):
    """Infinities and NaN among x, scales and zeros end where sums of the separate code and zero terms put them."""
    import KVmix

    gen = torch.Generator(device="cpu").manual_seed(4)
    B, nh, nkv, K, units = 1, 8, 2, 128, 160
    code = torch.randint(-2 ** 31, 2 ** 31, (B, nkv, K, units), generator=gen).int()
    scale = (0.25 * torch.randint(1, 5, (B, nkv, K, units), generator=gen).float()).half()  # (a second part of zero)
    zero, x = torch.randn(B, nkv, K, units, generator=gen).half(), torch.randn(B, nh, 1, K, generator=gen).half()
    inf, nan = float("inf"), float("nan")
    for spots in ({"x": (0, 1, 0, 5, inf)}, {"x": (0, 5, 0, 99, -inf)}, {"x": (0, 2, 0, 0, nan)}, {"scale": (0, 1, 7, 33, inf)},
                  {"scale": (0, 0, 127, 159, nan)}, {"zero": (0, 0, 64, 2, -inf)}, {"x": (0, 1, 0, 5, inf), "zero": (0, 0, 5, 9, nan)}):
        t = {"x": x.clone(), "scale": scale.clone(), "zero": zero.clone()}
        for name, (*at, v) in spots.items():
            t[name][tuple(at)] = v
        got = KVmix.quantized_gemm(11, *(a.to(dev) for a in (t["x"], code, t["scale"], t["zero"])), 3).double().cpu()
        c = torch.stack([(code.long() & 0xFFFFFFFF) >> (3 * i) & (3 if i == 10 else 7) for i in range(11)], -1).flatten(-2).double()
        s, z = (t[n].double().repeat_interleave(11, -1) for n in ("scale", "zero"))
        xd = t["x"].double().reshape(B, nkv, nh // nkv, K, 1)
        want = ((xd * (s * c)[:, :, None]).sum(-2) + (xd * z[:, :, None]).sum(-2)).reshape(got.shape)
        assert torch.equal(torch.isnan(got), torch.isnan(want)) and torch.equal(torch.isinf(got), torch.isinf(want))
        fine = torch.isfinite(want)
        assert torch.equal(got[torch.isinf(want)], want[torch.isinf(want)]) and float((got - want)[fine].abs().max()) < 0.1


@pytest.mark.gpu
def test_time_does_not_depend_on_the_scales(dev):
    """Keys of small, mixed and large channels cost what ordinary ones cost (everything but the exceptions above is one path)."""
    import KVmix

    B, nh, nkv, K, units = 8, 32, 8, 128, 744
    gen = torch.Generator(device=dev).manual_seed(1)
    code = torch.randint(-2 ** 31, 2 ** 31 - 1, (B, nkv, K, units), generator=gen, device=dev).int()
    r = torch.rand(B, nkv, K, units, generator=gen, device=dev)
    zero, x = torch.randn(B, nkv, K, units, generator=gen, device=dev).half(), torch.randn(B, nh, 1, K, generator=gen, device=dev).half()

    def best(scale):
        scale, times = scale.half(), []
        for _ in range(40):
            start, end = (torch.cuda.Event(enable_timing=True) for _ in range(2))
            start.record()
            for _ in range(10):
                KVmix.quantized_gemm(11, x, code, scale, zero, 3)
            end.record()
            end.synchronize()
            times.append(start.elapsed_time(end))
        return min(times)

    ordinary = best(0.5 * r + 0.3)
    for scale in (r, 0.01 * r, torch.where(torch.arange(K, device=dev)[:, None] % 4 == 0, 0.003 * r, r), 100 * r):
        assert best(scale) < 1.6 * ordinary
