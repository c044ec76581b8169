"""Sixteen to sixty-four pairs that the general decode kernels sort by expert themselves,
and more of them behind a sort's launch: every pair's row is, bit for bit, the product of
that pair alone (a row's sums do not depend on its neighbours), with all pairs on one
expert, one on each, more than sixteen an expert, experts and rows out of range, columns
that end inside a tile and tiles of two."""

import pytest
import torch

from metaljax_amd import kernels as K

pytestmark = pytest.mark.gpu

DEV = "cuda"


@pytest.mark.parametrize("bits,mode,act", [(4, "affine", "bf16"), (8, "affine", "bf16"), (4, "mxfp4", "bf16"), (4, "mxfp4", "f32"),
                                           (4, "affine", "f32")])
@pytest.mark.parametrize("pairs,e,n,k,spread", [(16, 32, 40, 96, "each"), (17, 5, 33, 352, "random"), (64, 4, 72, 160, "one"),
                                                (63, 16, 100, 992, "random"), (32, 3, 8200, 64, "random"), (64, 64, 48, 288, "each"),
                                                # so many experts and columns that the sort is a launch
                                                (32, 48, 1000, 64, "random"),
                                                # more than they sort, a K that is no multiple of 64
                                                (65, 9, 50, 96, "random"), (140, 9, 33, 288, "random"), (96, 4, 40, 416, "one")])
def test_pairs(pairs, e, n, k, spread, bits, mode, act):
    g = torch.Generator(device=DEV).manual_seed(pairs + k)
    how = dict(group_size=32, bits=bits, mode=mode)
    w = torch.randint(-2**31, 2**31 - 1, (e, n, k * bits // 32), dtype=torch.int32, device=DEV, generator=g)
    if mode == "mxfp4":
        s, b = torch.randint(118, 130, (e, n, k // 32), dtype=torch.uint8, device=DEV, generator=g), None
    else:
        s = (torch.rand((e, n, k // 32), device=DEV, generator=g) * 0.02 + 0.002).bfloat16()
        b = (-s.float() * 7).bfloat16()
    x = torch.randn((9, k), device=DEV, generator=g).to({"bf16": torch.bfloat16, "f32": torch.float32}[act])
    rhs = {"each": torch.arange(pairs, device=DEV).flip(0) % e, "one": torch.full((pairs,), e - 1, device=DEV),
           "random": torch.randint(0, e, (pairs,), device=DEV, generator=g)}[spread].int()
    lhs = torch.randint(0, 9, (pairs,), device=DEV, generator=g, dtype=torch.int32)
    if spread != "one":
        rhs[3], rhs[5] = e, -1                             # no experts: nothing is written
        lhs[0], lhs[1] = 9, -1                             # no rows: zeros
    y = K.gather_qmm(x, w, s, b, lhs, rhs, out_dtype=torch.float32, **how)
    for p in range(0, pairs, 1 if pairs <= 64 else 7):
        if 0 <= int(rhs[p]) < e:
            alone = K.gather_qmm(x, w, s, b, lhs[p:p + 1], rhs[p:p + 1], out_dtype=torch.float32, **how)
            assert torch.equal(y[p], alone[0]), p
    own = K.gather_qmm(x, w, s, b, None, rhs, out_dtype=torch.float32, **how)          # pair p: row p
    for p in (0, 8, 9, pairs - 1):
        if 0 <= int(rhs[p]) < e:
            there = torch.tensor([p], device=DEV, dtype=torch.int32)
            alone = K.gather_qmm(x, w, s, b, there, rhs[p:p + 1], out_dtype=torch.float32, **how)
            assert torch.equal(own[p], alone[0]), p
