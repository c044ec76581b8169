"""Decode products whose K is any multiple of 64: the ragged forms of the
loader-wavefront kernel, one pass over K and several, at the edges where they
can go wrong: one chunk or all but one in the last slice, table rows that start
inside a dword, a pass that ends inside a dword of such a row, rows that end
inside a tile, one activation row to sixteen, a neighbouring row whose table
entries are NaN.  The reference is the product of the exact weight in double
precision; products are exact and sums are float32, so a result is off by at
most a few hundred roundings of 2^-24 of the summed magnitudes (biases of the
size of scale times code cancel up to a factor of about ten)."""

import pytest
import torch

from metaljax_amd import kernels as K

pytestmark = pytest.mark.gpu

DEV = "cuda"
ACT = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}
KINDS = [(4, 64, "affine", "bf16"), (4, 128, "affine", "bf16"), (4, 64, "affine", "f16"), (4, 128, "affine", "f16"),
         (4, 64, "affine", "f32"), (4, 128, "affine", "f32"), (8, 64, "affine", "bf16"), (8, 128, "affine", "f16"),
         (8, 64, "affine", "f32"), (4, 32, "mxfp4", None)]


def weight(g, lead, n, k, bits, gs, mode, tab):
    w = torch.randint(-2**31, 2**31 - 1, lead + (n, k * bits // 32), dtype=torch.int32, device=DEV, generator=g)
    if mode == "mxfp4":
        return w, torch.randint(118, 130, lead + (n, k // 32), dtype=torch.uint8, device=DEV, generator=g), None
    s = torch.rand(lead + (n, k // gs), device=DEV, generator=g) * 0.02 + 0.005
    b = -s * torch.rand(s.shape, device=DEV, generator=g) * (1 << bits)
    return w, s.to(ACT[tab]), b.to(ACT[tab])


def exact(w, s, b, how):
    return K.dequantize(w, s, b, out_dtype=torch.float32, **how).double()


def close(y, want):
    err = ((y.double() - want).norm() / want.norm()).item()
    assert err <= 2e-5, err


@pytest.mark.parametrize("n,k", [(40, 1088), (270, 1984), (1000, 2880), (1001, 4160), (4099, 7616), (333, 11008), (520, 14400)])
@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("m", [1, 2, 3, 5, 8, 9, 16])
def test_dense(m, n, k, kind):
    bits, gs, mode, tab = kind
    if k % gs:
        pytest.skip("not a whole number of groups")
    g = torch.Generator(device=DEV).manual_seed(m + n + k)
    how = dict(group_size=gs, bits=bits, mode=mode)
    w, s, b = weight(g, (), n, k, bits, gs, mode, tab)
    x = torch.randn((m, k), device=DEV, generator=g).bfloat16()
    close(K.quantized_matmul(x, w, s, b, out_dtype=torch.float32, **how), x.double() @ exact(w, s, b, how).T)


@pytest.mark.parametrize("k", [1856, 11072])
@pytest.mark.parametrize("kind", [(4, 64, "affine", "bf16"), (8, 64, "affine", "f32"), (4, 32, "mxfp4", None)])
def test_a_rows_tables_stay_its_own(k, kind):
    bits, gs, mode, tab = kind
    g = torch.Generator(device=DEV).manual_seed(k)
    how = dict(group_size=gs, bits=bits, mode=mode)
    w, s, b = weight(g, (), 64, k, bits, gs, mode, tab)
    x = torch.randn((3, k), device=DEV, generator=g).bfloat16()
    clean = K.quantized_matmul(x, w, s, b, **how)
    odd = torch.arange(64, device=DEV) % 3 == 1
    s[odd] = 255 if mode == "mxfp4" else float("nan")
    y = K.quantized_matmul(x, w, s, b, **how)
    assert torch.equal(y[:, ~odd], clean[:, ~odd]) and bool(y[:, odd].isnan().all())


@pytest.mark.parametrize("k", [1856, 2944, 11072, 11136])
@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("pairs,experts", [(3, 5), (40, 6), (64, 2), (90, 7)])
def test_experts(pairs, experts, k, kind):
    bits, gs, mode, tab = kind
    if k % gs:
        pytest.skip("not a whole number of groups")
    n = 264
    g = torch.Generator(device=DEV).manual_seed(pairs + k)
    how = dict(group_size=gs, bits=bits, mode=mode)
    w, s, b = weight(g, (experts,), n, k, bits, gs, mode, tab)
    x = torch.randn((11, k), device=DEV, generator=g).bfloat16()
    lhs = torch.randint(0, 11, (pairs,), device=DEV, generator=g, dtype=torch.int32)
    rhs = torch.randint(0, experts, (pairs,), device=DEV, generator=g, dtype=torch.int32)
    full = exact(w, s, b, how)
    want = torch.stack([full[rhs[p]] @ x[lhs[p]].double() for p in range(pairs)])
    close(K.gather_qmm(x, w, s, b, lhs, rhs, out_dtype=torch.float32, **how), want)


# How far float32 results are from the product in double precision where zero points
# lie in the middle of the codes' range, as a checkpoint's do: what cancels must be
# gone before a chunk of 64 is added to the others.  In units of scale times the
# activations' deviation, a rounding being 2.5e-8 of the value (2^-23 / sqrt 12,
# averaged over a binade): four-bit codes leave 4.6 * 8 a chunk and one rounding of
# half a chunk's 128 * sqrt 32, together 4.9e-7; eight-bit codes leave 74 * 8 a chunk
# of sums of 148 * 8, rounded four times a chunk, together 1.1e-7.  (Added over a
# slice before the codes are: 1.7e-6 to 2.9e-6, and 1.2e-7 to 1.6e-7 with float32
# tables.)
@pytest.mark.parametrize("m,n,k", [(1, 4104, 1984), (5, 4104, 1088), (3, 4104, 4160), (16, 1032, 11008), (5, 2056, 4096)])
@pytest.mark.parametrize("kind", [kind for kind in KINDS if kind[2] == "affine"])
def test_what_cancels_cancels_early(m, n, k, kind):
    bits, gs, mode, tab = kind
    if k % gs or (bits == 8 and k > 4160):
        pytest.skip("not a whole number of groups, or more chunks than the bound counts")
    g = torch.Generator(device=DEV).manual_seed(m + k)
    how = dict(group_size=gs, bits=bits, mode=mode)
    w, s, _ = weight(g, (), n, k, bits, gs, mode, tab)
    zero = torch.randint(6, 11, s.shape, device=DEV, generator=g) * (1 if bits == 4 else 16)
    b = (-zero * s.float()).to(s.dtype)
    x = torch.randn((m, k), device=DEV, generator=g).bfloat16()
    want = x.double() @ exact(w, s, b, how).T
    err = ((K.quantized_matmul(x, w, s, b, out_dtype=torch.float32, **how).double() - want).norm() / want.norm()).item()
    assert err <= (7e-7 if bits == 4 else 1.3e-7), err
