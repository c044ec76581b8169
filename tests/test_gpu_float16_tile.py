"""Float16 rows times float16 tables: weights rounded to float16 on the short-group
kernel.  At the edges of its tiles, over its table windows, and where the weight does
not fit: scales so small that a float16 weight would be a denormal, weights past the
largest float16."""

import pytest
import torch

from metaljax_amd import kernels as K

pytestmark = pytest.mark.gpu

DEV = "cuda"
SHIFT = 64.0                                            # what the weight is multiplied by before it is rounded


def weight(g, lead, n, k, bits, gs, lo, hi):
    w = torch.randint(-2**31, 2**31 - 1, lead + (n, k * bits // 32), dtype=torch.int32, device=DEV, generator=g)
    s = (torch.rand(lead + (n, k // gs), device=DEV, generator=g) * (hi - lo) + lo).half()
    b = (-s.float() * torch.randint(1 << bits - 1, (1 << bits - 1) + 3, s.shape, device=DEV, generator=g)).half()
    return w, s, b


def exact(w, s, b, how):
    return K.dequantize(w, s, b, out_dtype=torch.float32, **how)


def tile(w32):
    return (w32 * SHIFT).half().double() / SHIFT


def off(y, want):
    return ((y.double() - want).norm() / want.norm()).item()


@pytest.mark.parametrize("m,n,k", [(9, 64, 64), (17, 130, 320), (33, 65, 448), (48, 1000, 2112), (65, 300, 4096), (77, 4096, 1088),
                                   (200, 520, 8192)])
@pytest.mark.parametrize("bits,gs", [(4, 64), (4, 128), (8, 64), (8, 128)])
def test_dense(m, n, k, bits, gs):
    if k % gs:
        pytest.skip("no whole groups")
    g = torch.Generator(device=DEV).manual_seed(m + n + k)
    how = dict(group_size=gs, bits=bits)
    x = torch.randn((m, k), device=DEV, generator=g).half()
    for lo, hi in ((0.002, 0.02), (2.0 ** -24, 2.0 ** -20)):       # (ordinary scales; the smallest there are)
        w, s, b = weight(g, (), n, k, bits, gs, lo, hi)
        w32 = exact(w, s, b, how)
        y = K.quantized_matmul(x, w, s, b, out_dtype=torch.float32, **how)
        assert off(y, x.double() @ tile(w32).T) <= 2e-5             # float32 sums, the bound of the bf16 tile's tests
        # never further from the exact weights than a bf16 tile (but for the float32 sums)
        want, bf16 = x.double() @ w32.double().T, x.double() @ w32.bfloat16().double().T
        ours, theirs = off(y, want), off(bf16, want)
        assert ours <= theirs + 1e-6
        # two float16 places: one for the rounding, one where the sum lies on the other side of it
        y16 = K.quantized_matmul(x, w, s, b, **how)
        assert y16.dtype == torch.float16
        torch.testing.assert_close(y16.float(), y, rtol=2.0 ** -10, atol=2.0 ** -24)


@pytest.mark.parametrize("counts", [(0, 1, 16, 0, 17), (40, 0, 3, 70, 64)])
@pytest.mark.parametrize("gathered", [False, True])
def test_groups(counts, gathered):
    g = torch.Generator(device=DEV).manual_seed(sum(counts))
    n, k, how = 200, 1088, dict(group_size=64, bits=4)
    w, s, b = weight(g, (len(counts),), n, k, 4, 64, 0.002, 0.02)
    w32 = exact(w, s, b, how)
    r = sum(counts)
    x = torch.randn((r, k), device=DEV, generator=g).half()
    experts = torch.repeat_interleave(torch.arange(len(counts)), torch.tensor(counts)).to(DEV)
    if gathered:
        order = torch.randperm(r, device=DEV, generator=g)
        y = K.gather_qmm(x, w, s, b, order.int(), experts[order].int(), out_dtype=torch.float32, **how)
        y = torch.empty_like(y).index_copy_(0, order, y)
    else:
        ends = torch.tensor((0,) + counts).cumsum(0).int().to(DEV)
        y = K.grouped_qmm(x, w, s, b, ends, out_dtype=torch.float32, **how)
    want = torch.stack([x[i].double() @ w32[e].double().T for i, e in enumerate(experts.tolist())])
    # 2^-12 of a weight at most, 2^-12 / sqrt(3) on average, of groups whose weights spread evenly over their range; decode
    # kernels (the smaller groups' form) multiply the exact weights
    assert off(y, want) <= 2.0 ** -12


@pytest.mark.parametrize("m,n,k", [(20, 70, 256), (70, 140, 4160)])
@pytest.mark.parametrize("bits", [4, 8])
def test_weights_that_are_no_float16(m, n, k, bits):
    """A few columns' scales are so large that a weight, shifted, overflows
    float16: those columns are multiplied again from the weights themselves."""
    g = torch.Generator(device=DEV).manual_seed(n)
    how = dict(group_size=64, bits=bits)
    w, s, b = weight(g, (), n, k, bits, 64, 0.002, 0.02)
    big = [0, 5, n - 1]
    s[big, -1] = 200.0
    b[big, -1] = -1000.0
    x = torch.randn((m, k), device=DEV, generator=g).half()
    x[3] = 0                                             # (a row of zeros is a row of zeros there too)
    y = K.quantized_matmul(x, w, s, b, out_dtype=torch.float32, **how)
    w32 = exact(w, s, b, how)
    want = x.double() @ w32.double().T
    assert torch.isfinite(y).all() and not y[3].any()
    assert off(y[:, big], want[:, big]) <= 1e-6          # double sums, one float32 rounding (and one a split)
    rest = [i for i in range(n) if i not in big]
    assert off(y[:, rest], x.double() @ tile(w32[rest]).T) <= 2e-5


def test_rows_that_are_not_finite_stay_in_their_rows():
    g = torch.Generator(device=DEV).manual_seed(2)
    w, s, b = weight(g, (), 300, 512, 4, 64, 0.002, 0.02)
    how = dict(group_size=64, bits=4)
    x = torch.randn((50, 512), device=DEV, generator=g).half()
    clean = K.quantized_matmul(x, w, s, b, out_dtype=torch.float32, **how)
    x[7, 100], x[20, 3] = float("inf"), float("nan")
    y = K.quantized_matmul(x, w, s, b, out_dtype=torch.float32, **how)
    keep = [i for i in range(50) if i not in (7, 20)]
    assert torch.equal(y[keep], clean[keep]) and torch.isnan(y[20]).all()
    w100 = exact(w, s, b, how)[:, 100]
    assert torch.equal(y[7] > 0, w100 > 0) and not torch.isfinite(y[7]).any()
