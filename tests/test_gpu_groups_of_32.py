"""Decode products of weights in groups of 32 on the loader-wavefront kernel: K any
multiple of 64 -- one pass and several, ragged last slices, a row's last chunk -- bf16
and float16 tables, batches, pairs and pairs sorted by expert, against the exact
weights in double precision."""

import pytest
import torch

from metaljax_amd import kernels as K

pytestmark = pytest.mark.gpu

DEV = "cuda"
TAB = {"bf16": torch.bfloat16, "f16": torch.float16}
# float32 sums of exact products.  A four-bit code goes through the matrix core as 128 + q and the 128 leave before a
# group is added to anything, so a group's sum is up to 136 over the codes' spread of 4.6 times what it leaves; some
# ten roundings of 2^-24 meet in a result
ERR = 136 / 4.6 * 2.0 ** -24 * 10 ** 0.5


def weight(g, lead, n, k, bits, tab):
    w = torch.randint(-2**31, 2**31 - 1, lead + (n, k * bits // 32), dtype=torch.int32, device=DEV, generator=g)
    s = (torch.rand(lead + (n, k // 32), device=DEV, generator=g) * 0.02 + 0.002).to(TAB[tab])
    top = 1 << bits
    b = (-s.float() * torch.randint(top // 2 - 2, top // 2 + 3, s.shape, device=DEV, generator=g)).to(TAB[tab])
    return w, s, b


def exact(w, s, b, bits):
    return K.dequantize(w, s, b, out_dtype=torch.float32, group_size=32, bits=bits).double()


def off(y, want):
    return ((y.double() - want).norm() / want.norm()).item()


@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("tab", ["bf16", "f16"])
@pytest.mark.parametrize("n,k", [(16, 1088), (72, 1536), (4104, 2112), (33, 4096), (300, 4160), (1000, 8192), (520, 11008), (9000, 1152),
                                 # 9, 12 and 10 rows a workgroup (K whole slices), 16 where they are dealt by eights
                                 (2100, 1536), (3070, 4096), (2530, 8192), (2100, 4160)])
def test_dense(n, k, bits, tab):
    g = torch.Generator(device=DEV).manual_seed(n + k)
    w, s, b = weight(g, (), n, k, bits, tab)
    # what a row's last chunk must not read: the next row's entries are infinite, the last row's neighbours NaN
    s[1::2, 0], b[1::2, 0] = float("inf"), float("nan")
    even = exact(w, s, b, bits)[::2]
    for m in (1, 2, 5, 9, 16):
        x = torch.randn((m, k), device=DEV, generator=g).bfloat16()
        y = K.quantized_matmul(x, w, s, b, out_dtype=torch.float32, group_size=32, bits=bits)
        assert off(y[:, ::2], x.double() @ even.T) <= ERR, m
        y16 = K.quantized_matmul(x, w, s, b, group_size=32, bits=bits)
        assert torch.equal(y16[:, ::2], y[:, ::2].bfloat16())
    x = torch.randn((3, k), device=DEV, generator=g)                  # wider activations: nine rows of terms
    y = K.quantized_matmul(x, w, s, b, group_size=32, bits=bits)
    assert off(y[:, ::2], x.double() @ even.T) <= ERR


@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("pairs,e,n,k", [(3, 5, 72, 2112), (20, 4, 200, 4160), (70, 8, 136, 2048), (130, 16, 40, 4288)])
def test_pairs(pairs, e, n, k, bits):
    g = torch.Generator(device=DEV).manual_seed(pairs)
    w, s, b = weight(g, (e,), n, k, bits, "bf16")
    x = torch.randn((11, k), device=DEV, generator=g).bfloat16()
    lhs = torch.randint(0, 11, (pairs,), device=DEV, generator=g, dtype=torch.int32)
    rhs = torch.randint(0, e, (pairs,), device=DEV, generator=g, dtype=torch.int32)
    y = K.gather_qmm(x, w, s, b, lhs, rhs, out_dtype=torch.float32, group_size=32, bits=bits)
    w64 = exact(w, s, b, bits)
    want = torch.stack([w64[r] @ x[i].double() for i, r in zip(lhs.tolist(), rhs.tolist())])
    assert off(y, want) <= ERR


# fewer than sixteen pairs: products of their own up to 16 MB of streamed weights, sorted past that; wider rows as
# the rows of one product a pair, or once a term where the experts are fewer than the pairs
@pytest.mark.parametrize("act", ["bf16", "f16", "f32"])
@pytest.mark.parametrize("pairs,e,n,k,bits", [(13, 4, 296, 3072, 4), (15, 4, 496, 5376, 4), (4, 16, 712, 2048, 4), (15, 4, 2400, 2240, 8),
                                              (12, 4, 2400, 2240, 8), (15, 7, 520, 4160, 8), (16, 4, 296, 3072, 4)])
def test_few_pairs(pairs, e, n, k, bits, act):
    g = torch.Generator(device=DEV).manual_seed(pairs + n)
    w, s, b = weight(g, (e,), n, k, bits, "bf16")
    x = torch.randn((7, k), device=DEV, generator=g).to({"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}[act])
    lhs = torch.randint(0, 7, (pairs,), device=DEV, generator=g, dtype=torch.int32)
    rhs = torch.randint(0, e, (pairs,), device=DEV, generator=g, dtype=torch.int32)
    lhs[0], rhs[1] = 7, e                                 # no such row: zeros; no such expert: nothing is written
    y = K.gather_qmm(x, w, s, b, lhs, rhs, out_dtype=torch.float32, group_size=32, bits=bits)
    w64, x64 = exact(w, s, b, bits), x.double()
    live = [p for p in range(2, pairs)]
    want = torch.stack([w64[rhs[p]] @ x64[lhs[p]] for p in live])
    assert off(y[live], want) <= ERR and not y[0].any()


def test_a_batch_of_weights():
    g = torch.Generator(device=DEV).manual_seed(3)
    w, s, b = weight(g, (3,), 130, 1600, 4, "bf16")
    x = torch.randn((3, 4, 1600), device=DEV, generator=g).bfloat16()
    y = K.quantized_matmul(x, w, s, b, out_dtype=torch.float32, group_size=32, bits=4)
    assert off(y, x.double() @ exact(w, s, b, 4).transpose(1, 2).contiguous()) <= ERR
