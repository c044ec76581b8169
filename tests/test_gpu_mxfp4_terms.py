"""float16 / float32 rows that the general MXFP4 decode kernel splits into bf16 terms as
they arrive: the same numbers, bit for bit, as the terms multiplied one by one and added
smallest first (every sum meets in the same order), for products of a few rows, batches,
pairs of their own and sorted ones; contractions of less than a chunk of 128 to several a
wavefront, columns that end inside a tile, rows and experts that are out of range, rows
that hold infinities, NaNs and the smallest values.  Rows that start between two 16-byte
addresses take the split as a launch of its own and give the same but for the order of
three terms' sums."""

import pytest
import torch

from metaljax_amd import kernels as K

pytestmark = pytest.mark.gpu

DEV = "cuda"
HOW = dict(group_size=32, bits=4, mode="mxfp4")
ACT = {"f16": torch.float16, "f32": torch.float32}


def weight(g, lead, n, k):
    w = torch.randint(-2**31, 2**31 - 1, lead + (n, k // 8), dtype=torch.int32, device=DEV, generator=g)
    s = torch.randint(118, 130, lead + (n, k // 32), dtype=torch.uint8, device=DEV, generator=g)
    s[..., 0, 0] = 255                                     # (a row whose scale is no number)
    return w, s


def rows(g, shape, act):
    x = torch.randn(shape, device=DEV, generator=g).to(ACT[act])
    x[..., ::5] *= 2.0 ** -14                              # (float16: denormal, float32: not)
    flat = x.view(-1, shape[-1])
    if len(flat) > 2:                                      # (some row stays finite)
        flat[-1, 3], flat[-1, 7], flat[0, 1] = float("inf"), -float("inf"), float("nan")
    return x


def bf16_terms(x):
    v = x.float()
    for _ in range(3 if x.dtype == torch.float32 else 2):
        hi = (v.view(torch.int32) & -65536).view(torch.float32)
        hi = torch.where(v != v, v, hi)
        yield hi.bfloat16()
        v = torch.where(torch.isfinite(hi), v - hi, torch.zeros_like(v))


def total(parts):
    y = None
    for p in reversed(list(parts)):
        y = p if y is None else y + p
    return y


def same(a, b):
    return torch.equal(a.isnan(), b.isnan()) and torch.equal(a.nan_to_num(), b.nan_to_num())


@pytest.mark.parametrize("act", ["f16", "f32"])
@pytest.mark.parametrize("pairs,e,n,k", [(1, 3, 40, 32), (3, 9, 72, 1024), (15, 40, 33, 416), (6, 8, 2048, 1024), (9, 30, 48, 160),
                                         (5, 2, 8200, 96),
                                         # sorted by expert first
                                         (16, 8, 100, 1024), (33, 4, 40, 864), (64, 16, 33, 96), (48, 2, 8200, 288)])
def test_pairs(pairs, e, n, k, act):
    g = torch.Generator(device=DEV).manual_seed(pairs + k)
    w, s = weight(g, (e,), n, k)
    x = rows(g, (11, k), act)
    lhs = torch.randint(0, 11, (pairs,), device=DEV, generator=g, dtype=torch.int32)
    rhs = torch.randint(0, e, (pairs,), device=DEV, generator=g, dtype=torch.int32)
    if pairs > 2:
        lhs[0], lhs[1], rhs[2] = 11, -1, e                 # no rows of x: zeros; no expert: nothing
    live = torch.ones(pairs, dtype=torch.bool, device=DEV)
    live[2:3] = pairs <= 2
    got = K.gather_qmm(x, w, s, None, lhs, rhs, out_dtype=torch.float32, **HOW)
    want = total(K.gather_qmm(t, w, s, None, lhs, rhs, out_dtype=torch.float32, **HOW) for t in bf16_terms(x))
    assert same(got[live], want[live]) and got[live].isfinite().any()
    half = K.gather_qmm(x, w, s, None, lhs, rhs, out_dtype=torch.float16, **HOW)
    assert same(half[live], got[live].half())
    apart = torch.empty(x.numel() + 2, dtype=x.dtype, device=DEV)[2:].view(x.shape).copy_(x)
    apart = K.gather_qmm(apart, w, s, None, lhs, rhs, out_dtype=torch.float32, **HOW)[live]
    sound = got[live].isfinite()
    assert same(apart.masked_fill(sound, 0), got[live].masked_fill(sound, 0))
    apart, there = apart[sound].double(), got[live][sound].double()
    assert (apart - there).norm() <= 2.0 ** -23 * there.norm()           # (two roundings each)
    few = min(pairs, 11)
    own = K.gather_qmm(x[:few], w, s, None, None, rhs[:few], out_dtype=torch.float32, **HOW)
    want = total(K.gather_qmm(t, w, s, None, None, rhs[:few], out_dtype=torch.float32, **HOW) for t in bf16_terms(x[:few]))
    assert same(own[live[:few]], want[live[:few]])


# where the general kernel is the faster one although a staged one serves the shape: sizes on both sides of the rules
@pytest.mark.parametrize("act", ["f16", "f32"])
@pytest.mark.parametrize("pairs,e,n,k", [(1, 2, 4096, 4096), (3, 2, 4096, 4096), (5, 4, 352, 1216), (20, 4, 352, 1216), (30, 8, 2880, 1088),
                                         (40, 16, 1024, 2048), (64, 16, 1024, 2048), (8, 9, 2880, 2880), (9, 9, 2880, 2880),
                                         # past 64 pairs
                                         (65, 8, 512, 288), (78, 8, 384, 576), (128, 8, 600, 288), (129, 8, 600, 288), (200, 16, 1024, 1024), (257, 4, 200, 352), (260, 3, 40, 96)])
def test_pairs_of_staged_shapes(pairs, e, n, k, act):
    g = torch.Generator(device=DEV).manual_seed(pairs + k)
    w, s = weight(g, (e,), n, k)
    s[:, 0, 0] = 120
    x = torch.randn((pairs, k), device=DEV, generator=g).to(ACT[act])
    rhs = torch.randint(0, e, (pairs,), device=DEV, generator=g, dtype=torch.int32)
    y = K.gather_qmm(x, w, s, None, None, rhs, out_dtype=torch.float32, **HOW)
    want = torch.empty((pairs, n), dtype=torch.float64, device=DEV)
    for i in range(e):
        want[rhs == i] = x[rhs == i].double() @ K.dequantize(w[i], s[i], None, out_dtype=torch.float32, **HOW).double().T
    # exact products, a rounding (or cut) of 2^-23 at most an instruction of 32 products, a wavefront and a term
    err = ((y.double() - want).norm() / want.norm()).item()
    assert err <= 2.0 ** -23 * (k / 32 + 11) ** 0.5, err


@pytest.mark.parametrize("act", ["f16", "f32"])
@pytest.mark.parametrize("m,lead,n,k", [(1, (), 40, 32), (5, (), 1024, 1024), (4, (), 8200, 96), (2, (3,), 33, 416), (3, (), 64, 4160)])
def test_rows(m, lead, n, k, act):
    g = torch.Generator(device=DEV).manual_seed(m + k)
    w, s = weight(g, lead, n, k)
    x = rows(g, lead + (m, k), act)
    got = K.quantized_matmul(x, w, s, None, out_dtype=torch.float32, **HOW)
    want = total(K.quantized_matmul(t, w, s, None, out_dtype=torch.float32, **HOW) for t in bf16_terms(x))
    assert same(got, want) and got.isfinite().any()


# Float32 sums of exact products in float32 results: up to some twenty roundings in a row
# (sixteen matrix steps of a wavefront, the wavefronts', the terms') measure 0.94e-7 to 1.08e-7
# from 64 bits, twice as many 1.13e-7 to 1.6e-7 (block scales over ten powers of two).
def even_weight(g, lead, n, k):
    w, s = weight(g, lead, n, k)
    return w, s.random_(118, 128, generator=g)


@pytest.mark.parametrize("m,n,k", [(1, 904, 13504), (1, 3072, 13312), (4, 2088, 8192), (2, 2096, 3968), (3, 4104, 4096), (2, 6000, 2112)])
def test_long_rows_are_no_less_exact(m, n, k):
    g = torch.Generator(device=DEV).manual_seed(m + k)
    w, s = even_weight(g, (), n, k)
    x = torch.randn((m, k), device=DEV, generator=g)
    y = K.quantized_matmul(x, w, s, None, **HOW)
    want = x.double() @ K.dequantize(w, s, None, out_dtype=torch.float32, **HOW).double().T
    assert (y.double() - want).norm() <= 1.1e-7 * want.norm()


def pairs_off(pairs, e, n, k, act):
    g = torch.Generator(device=DEV).manual_seed(pairs + k)
    w, s = even_weight(g, (e,), n, k)
    x = torch.randn((pairs, k), device=DEV, generator=g).to(ACT[act])
    rhs = torch.randint(0, e, (pairs,), device=DEV, generator=g, dtype=torch.int32)
    y = K.gather_qmm(x, w, s, None, None, rhs, out_dtype=torch.float32, **HOW).double()
    want = torch.empty((pairs, n), dtype=torch.float64, device=DEV)
    for i in range(e):
        want[rhs == i] = x[rhs == i].double() @ K.dequantize(w[i], s[i], None, out_dtype=torch.float32, **HOW).double().T
    return ((y - want).norm() / want.norm()).item()


@pytest.mark.parametrize("pairs,e,n,k", [(52, 16, 456, 3968), (12, 8, 552, 3584), (3, 4, 992, 3776), (5, 2, 400, 8192)])
def test_pairs_of_long_rows_are_no_less_exact(pairs, e, n, k):
    assert pairs_off(pairs, e, n, k, "f32") <= 1.1e-7


# Past 64 pairs the row-group kernels' sums over parts of K measure 4.6e-8 to 7.0e-8 in float32
# results, the general kernel's 5.0e-8 to 8.2e-8: it serves 16-bit results alone.
@pytest.mark.parametrize("act", ["f16", "f32"])
@pytest.mark.parametrize("pairs,e,n,k,most", [(134, 16, 352, 1408, 7.1e-8), (126, 8, 664, 1216, 6.9e-8), (188, 16, 424, 1600, 7.5e-8)])
def test_many_pairs_are_no_less_exact(pairs, e, n, k, most, act):
    assert pairs_off(pairs, e, n, k, act) <= most
