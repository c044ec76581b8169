"""Decode products of five rows over three passes of the contraction, whose rows all
lie in the matrix operand at once (and their neighbours of four and six rows, which
do not take that form): the first and the last K of three passes, ragged and whole,
every table type, columns that end inside a tile, rows without end values in the
others' place."""

import pytest
import torch

from metaljax_amd import kernels as K

pytestmark = pytest.mark.gpu

DEV = "cuda"
# float32 sums of exact products: a four-bit code goes through the matrix core as 128 + q, up to 136 over the codes'
# spread of 4.6 times what it leaves; some ten roundings of 2^-24 meet in a result.  (Over several passes of whole
# slices -128 scale stays in the sums of a slice's eight chunks until its end: eight times that.)
ERR = 136 / 4.6 * 2.0 ** -24 * 10 ** 0.5


@pytest.mark.parametrize("bits,gs,mode,tab", [(4, 64, "affine", "bf16"), (4, 128, "affine", "f16"), (4, 64, "affine", "f16"),
                                              (8, 64, "affine", "bf16"), (8, 128, "affine", "f16"), (4, 32, "mxfp4", None)])
@pytest.mark.parametrize("k,n", [(8320, 4500), (8704, 9000), (11008, 72), (12288, 300), (12160, 33)])
def test_five_rows(k, n, bits, gs, mode, tab):
    k = k if bits == 4 else k // 128 * 64
    if k % gs:
        pytest.skip("no whole groups")
    g = torch.Generator(device=DEV).manual_seed(k + n)
    how = dict(group_size=gs, bits=bits, mode=mode)
    w = torch.randint(-2**31, 2**31 - 1, (n, k * bits // 32), dtype=torch.int32, device=DEV, generator=g)
    if mode == "mxfp4":
        s, b = torch.randint(118, 130, (n, k // 32), dtype=torch.uint8, device=DEV, generator=g), None
    else:
        dt = torch.bfloat16 if tab == "bf16" else torch.float16
        s = (torch.rand((n, k // gs), device=DEV, generator=g) * 0.02 + 0.002).to(dt)
        top = 1 << bits
        b = (-s.float() * torch.randint(top // 2 - 2, top // 2 + 3, s.shape, device=DEV, generator=g)).to(dt)
    exact = K.dequantize(w, s, b, out_dtype=torch.float32, **how).double()
    for m in (5, 4, 6):
        x = torch.randn((m, k), device=DEV, generator=g).bfloat16()
        y = K.quantized_matmul(x, w, s, b, out_dtype=torch.float32, **how)
        want = x.double() @ exact.T
        assert ((y.double() - want).norm() / want.norm()).item() <= ERR * (8 if k % 512 == 0 else 1), m
        x[1] = float("inf")                              # one row is not finite: the others are what they were
        again = K.quantized_matmul(x, w, s, b, out_dtype=torch.float32, **how)
        keep = [i for i in range(m) if i != 1]
        assert torch.equal(again[keep], y[keep]) and not torch.isfinite(again[1]).any()
