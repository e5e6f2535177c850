"""ops.linear_rows / swiglu_rows / qkv_rope_append (kvmix_linear_rows) against the torch modules they stand for.

Reference: the product in float64 of the fp16 operands, rounded to fp16, then the elementwise work in fp16 tensor
arithmetic.  The kernel sums in fp32 (error at most k * 2^-24 of the sum of magnitudes), which can turn a rounding to
fp16 over (2^-10 of the value); with a norm, rms_norm's own fp32 arithmetic can turn over the rounding of an element of
x as well (at worst of every one: 2^-10 of the sum of magnitudes)."""
import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu
ULP = 2.0 ** -10


def operands(dev, m, k, n):
    gen = torch.Generator(device="cpu").manual_seed(1000 * m + k + n)
    r = lambda *s: torch.randn(*s, generator=gen).to(dev).half()  # noqa: E731
    return r(m, k), (0.03 * r(n, k)).half(), (1 + 0.2 * r(k)).half(), r(m, n)


def product(x, w):
    return (x.double() @ w.double().t()).half(), x.double().abs() @ w.double().abs().t()


def within(got, want, bound):
    assert got.shape == want.shape
    err = (got.double() - want.double()).abs()
    assert (err <= bound).all(), float((err - bound).max())
    assert float(err.norm()) <= ULP / 2 * float(want.double().norm())  # (in the mean: the rounding of the output)


# rows of x around the groups of four sequences, k around the chunks of 128 elements and the eight waves, n around the
# tiles of four rows and the blocks
@pytest.mark.parametrize("m,k,n", [(1, 128, 1), (1, 1024, 6), (3, 1152, 255), (4, 2048, 1026), (5, 2176, 61), (8, 4096, 300),
                                   (9, 4096, 130), (16, 4096, 4099), (4, 5632, 513), (16, 6144, 77), (2, 8192, 64),
                                   (8, 11008, 259), (4, 14336, 65)])
def test_plain_float_residual(dev, m, k, n):
    from kvmix_amd import ops

    x, w, _, res = operands(dev, m, k, n)
    assert ops.linear_rows_supported(m, k, n)
    y, mag = product(x, w)
    bound = ULP * y.double().abs() + k * 2.0 ** -24 * mag
    got = ops.linear_rows(x, w)
    within(got, y, bound)
    assert torch.equal(got, ops.linear_rows(x, w))
    f = ops.linear_rows(x, w, fp32=True)
    assert f.dtype == torch.float32 and torch.equal(f, got.float())
    assert torch.equal(ops.linear_rows(x, w, residual=res), res + got)  # the sum in fp16 tensor arithmetic
    wide = torch.zeros(m, k + 64, device=dev, dtype=torch.float16)      # rows of a larger tensor
    wide[:, :k] = x
    assert torch.equal(ops.linear_rows(wide[:, :k], w), got)


@pytest.mark.parametrize("m,k,n", [(1, 256, 4), (4, 4096, 1001), (7, 2048, 129), (16, 4096, 64), (4, 8192, 31), (8, 6144, 10)])
def test_norm_and_swiglu(dev, m, k, n):
    from kvmix_amd import ops

    x, w, nw, _ = operands(dev, m, k, 2 * n)
    xn = F.rms_norm(x, (k,), nw, 1e-5)
    y, mag = product(xn, w)
    got = ops.linear_rows(x, w, nw, 1e-5)
    within(got, y, ULP * (y.double().abs() + mag))
    for norm in (None, nw):
        a = got if norm is not None else ops.linear_rows(x, w)
        want = F.silu(a[:, :n]) * a[:, n:]
        s = ops.swiglu_rows(x, w, norm, 1e-5)
        within(s, want, 4 * ULP * want.double().abs() + 2.0 ** -24)  # expf here and torch's: a rounding of each of two steps
        assert torch.equal(s, ops.swiglu_rows(x, (w[:n], w[n:]), norm, 1e-5))


@pytest.mark.parametrize("m,k,heads,kv,D,per_row", [(1, 256, 2, 1, 64, False), (4, 4096, 32, 8, 128, True), (16, 2048, 3, 3, 128, False),
                                                    (5, 512, 4, 2, 32, True), (3, 1024, 1, 1, 8, False)])
def test_qkv_rope_append_is_the_composition(dev, m, k, heads, kv, D, per_row):
    from kvmix_amd import ops

    x, w, nw, _ = operands(dev, m, k, (heads + 2 * kv) * D)
    gen = torch.Generator(device="cpu").manual_seed(7)
    cos, sin = (torch.randn(m if per_row else 1, 1, D, generator=gen).to(dev).half() for _ in range(2))
    kt, vt = (torch.zeros(m, kv, 6, D, device=dev, dtype=torch.float16) for _ in range(2))
    slot = torch.tensor([3], device=dev)
    q = ops.qkv_rope_append(x, w, heads, kv, cos, sin, kt[:, :, 1:], vt, slot, 2, nw, 1e-5)
    y = ops.linear_rows(x, w, nw, 1e-5).view(m, heads + 2 * kv, D)
    rot = torch.cat([-y[..., D // 2:], y[..., :D // 2]], -1)
    want = y * cos + rot * sin
    assert torch.equal(q[:, :, 0], want[:, :heads])
    assert torch.equal(kt[:, :, 4], want[:, heads:heads + kv]) and torch.equal(vt[:, :, 2], y[:, heads + kv:])
    kt[:, :, 4] = 0
    vt[:, :, 2] = 0
    assert not kt.any() and not vt.any()
    ops.qkv_rope_append(x, w, heads, kv, cos, sin, kt, vt, torch.tensor([6], device=dev), torch.tensor([-1], device=dev), nw, 1e-5)
    assert not kt.any() and not vt.any()  # a device-side slot outside the window writes nothing


def test_refusals(dev):
    from kvmix_amd import ops

    x, w, nw, res = operands(dev, 4, 256, 8)
    assert not ops.linear_rows_supported(17, 256, 8) and not ops.linear_rows_supported(4, 200, 8)
    with pytest.raises(RuntimeError):
        ops.linear_rows(x[:, :200].contiguous(), w[:, :200].contiguous())
    with pytest.raises(RuntimeError):
        ops.linear_rows(x, w, residual=res[:2])
    with pytest.raises(RuntimeError):
        ops.linear_rows(x.float(), w)
    with pytest.raises(RuntimeError):
        ops.qkv_rope_append(x, w, 1, 1, nw[:2], nw[:2], *(torch.zeros(4, 1, 2, 2, device=dev).half() for _ in range(2)), 0, 0)


def test_parts_have_the_rows_of_their_heads(dev):
    """Weights given part by part are held to the heads and to each other before anything is launched: a key weight with
    more rows than kv_heads * D would write past the tails' heads, a query weight with fewer leave outputs unwritten."""
    from kvmix_amd import ops

    D, heads, kv = 32, 4, 2
    x, w, nw, _ = operands(dev, 3, 256, (heads + 2 * kv + 4) * D)
    cos, sin = (torch.ones(1, 1, D, device=dev).half() for _ in range(2))
    kt, vt = (torch.zeros(3, kv, 4, D, device=dev).half() for _ in range(2))

    def rows(*parts):
        return tuple(w[:n * D].contiguous() for n in parts)

    def call(weights):
        return ops.qkv_rope_append(x, weights, heads, kv, cos, sin, kt, vt, 0, 0, nw, 1e-5)

    for parts in ((heads, kv + 1, kv + 1), (heads, 2 * kv, 2 * kv), (heads, kv, kv + 1), (heads - 2, kv, kv), (2 * heads, kv, kv),
                  (heads, kv), (heads + 2 * kv - 1, 1)):
        with pytest.raises(RuntimeError):
            call(rows(*parts))
    assert not kt.any() and not vt.any()
    stacked = torch.cat(rows(heads, kv, kv))
    want, k_want, v_want = call(stacked), kt.clone(), vt.clone()
    assert torch.equal(call(rows(heads, kv, kv)), want) and torch.equal(kt, k_want) and torch.equal(vt, v_want)
    for weights in ((w[:D], w[:2 * D]), (w[:D],) * 3):
        with pytest.raises(RuntimeError):
            ops.swiglu_rows(x, weights)


@pytest.mark.parametrize("left", ["x", "w", "norm", "residual", "cos", "sin", "k_tail", "v_tail", "slot"])
def test_operands_lie_on_one_device(dev, left):
    """One operand left in host memory (a partly offloaded model) is refused before a kernel sees its address."""
    from kvmix_amd import ops

    D, heads, kv = 32, 2, 1
    x, w, nw, res = operands(dev, 2, 256, (heads + 2 * kv) * D)
    t = {"x": x, "w": w, "norm": nw, "residual": res, "cos": torch.ones(1, 1, D, device=dev).half(), "sin": torch.ones(1, 1, D, device=dev).half(),
         "k_tail": torch.zeros(2, kv, 3, D, device=dev).half(), "v_tail": torch.zeros(2, kv, 3, D, device=dev).half(), "slot": torch.tensor([1], device=dev)}
    calls = [(("x", "w", "norm", "cos", "sin", "k_tail", "v_tail", "slot"),
              lambda t: ops.qkv_rope_append(t["x"], t["w"], heads, kv, t["cos"], t["sin"], t["k_tail"], t["v_tail"], t["slot"], t["slot"], t["norm"], 1e-5)),
             (("x", "w", "residual"), lambda t: ops.linear_rows(t["x"], t["w"], residual=t["residual"])),
             (("x", "w", "norm"), lambda t: ops.linear_rows(t["x"], t["w"], t["norm"], 1e-5)),
             (("x", "w", "norm"), lambda t: ops.swiglu_rows(t["x"], t["w"], t["norm"], 1e-5))]
    for reads, call in calls:
        call(t)
        if left in reads:
            with pytest.raises(RuntimeError):
                call({**t, left: t[left].cpu()})


def test_residual_and_fp32_exclude_each_other(dev):
    """(The residual sum is an fp16 one; as fp32 storage its bytes would be no numbers at all.)  Likewise residual and norm."""
    from kvmix_amd import ops

    x, w, nw, res = operands(dev, 4, 256, 24)
    for kw in ({"residual": res, "fp32": True}, {"residual": res, "norm_weight": nw, "eps": 1e-5}):
        with pytest.raises(RuntimeError):
            ops.linear_rows(x, w, **kw)
    assert ops.linear_rows(x, w[:0]).shape == (4, 0) and ops.linear_rows(x[:0], w).shape == (0, 24)


@pytest.mark.parametrize("m,k", [(1, 128), (4, 1152), (3, 4224), (9, 2688), (2, 11008)])
def test_what_is_not_finite(dev, m, k):
    """Infinities and NaN in any chunk of x or w end in the outputs they belong to, as in the plain product: k around waves
    whose last chunks lie past the end."""
    from kvmix_amd import ops

    n = 24
    x, w, nw, _ = operands(dev, m, k, n)
    inf = float("inf")
    for at in (0, k // 2, k - 1):
        xi, wi = x.clone(), w.clone()
        wi[5, at], wi[6, at], wi[7, at] = inf, -inf, float("nan")
        xi[0, k - 1 - at] = -inf
        got, want = ops.linear_rows(xi, wi).double(), xi.double() @ wi.double().t()
        assert torch.equal(torch.isnan(got), torch.isnan(want)) and torch.equal(torch.isinf(got), torch.isinf(want))
        assert torch.equal(torch.sign(got[torch.isinf(want)]), torch.sign(want[torch.isinf(want)]))
        fine = torch.isfinite(want)
        assert float((got - want)[fine].norm()) <= ULP * float(want[fine].norm())


@pytest.mark.parametrize("m,k", [(4, 1152), (2, 4224)])
def test_an_infinite_norm_weight(dev, m, k):
    from kvmix_amd import ops

    x, w, nw, _ = operands(dev, m, k, 8)
    nw[k - 1] = float("inf")
    got, want = ops.linear_rows(x, w, nw, 1e-5), F.rms_norm(x, (k,), nw, 1e-5).double() @ w.double().t()
    assert torch.isinf(want).all() and torch.equal(got.double(), want)


def test_a_weight_of_one_row_with_any_stride(dev):
    from kvmix_amd import ops

    x, w, _, _ = operands(dev, 3, 256, 2)
    wide = torch.cat([w, w[:, :3]], 1)[:1, :256]  # (contiguous as torch counts, a stride of 259)
    assert wide.is_contiguous() and wide.stride(0) == 259
    assert torch.equal(ops.linear_rows(x, wide), ops.linear_rows(x, w[:1]))
