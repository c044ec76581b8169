"""The prefill products that split K over workgroups or take short row groups,
at the edges of their tiles: rows round the sixteens and the 128 / 256 of a
row tile, columns that end inside a tile, a K that ends inside a step, table
rows that start inside a dword, groups without rows.  The reference is a plain
product of the bf16 weight tile in double precision (MXFP4 tiles are exact)."""

import pytest
import torch

from metaljax_amd import kernels as K

pytestmark = pytest.mark.gpu

DEV = "cuda"
ACT = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}
# (bits, group_size, mode, tables)
KINDS = [(4, 64, "affine", "bf16"), (4, 32, "affine", "f16"), (4, 128, "affine", "f32"), (8, 64, "affine", "bf16"),
         (8, 32, "affine", "f32"), (4, 32, "mxfp4", None)]


def weight(g, lead, n, k, bits, gs, mode, tab):
    w = torch.randint(-2**31, 2**31 - 1, lead + (n, k * bits // 32), dtype=torch.int32, device=DEV, generator=g)
    if mode == "mxfp4":
        return w, torch.randint(118, 130, lead + (n, k // 32), dtype=torch.uint8, device=DEV, generator=g), None
    s = torch.rand(lead + (n, k // gs), device=DEV, generator=g) * 0.02 + 0.005
    b = -s * torch.rand(s.shape, device=DEV, generator=g) * (1 << bits)
    return w, s.to(ACT[tab]), b.to(ACT[tab])


def tile(w, s, b, how):
    return K.dequantize(w, s, b, out_dtype=torch.float32, **how).bfloat16().double()


def close(y, want):
    err = ((y.double() - want).norm() / want.norm()).item()
    assert err <= 2e-5, err


# few rows or few columns: the short-group kernel; many: the prefill kernel with 128- and 256-row tiles, its K split
@pytest.mark.parametrize("m,n,k", [(17, 64, 64), (33, 130, 320), (65, 65, 448), (48, 1000, 2112), (128, 333, 4096),
                                   (200, 4104, 8192), (300, 9208, 2944), (513, 2056, 1088)])
@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("act", ["bf16", "f16", "f32"])
def test_dense(m, n, k, kind, act):
    bits, gs, mode, tab = kind
    if k % gs or (mode == "mxfp4" and k % 512 == 0 and act == "bf16"):     # (the latter: the FP6 kernel's tolerance)
        pytest.skip("not a shape of these kernels")
    g = torch.Generator(device=DEV).manual_seed(m + n + k)
    how = dict(group_size=gs, bits=bits, mode=mode)
    w, s, b = weight(g, (), n, k, bits, gs, mode, tab)
    x = torch.randn((m, k), device=DEV, generator=g).to(ACT[act])
    close(K.quantized_matmul(x, w, s, b, out_dtype=torch.float32, **how), x.double() @ tile(w, s, b, how).T)


# Row tiles of 256 rows (several rounds of workgroups, or a split K: columns of whole lines,
# whose sums are stored wide and read once, of whole sixteen bytes and of neither), the last of
# 188, 76, 130 and 88 rows, dealt row tile first, and eleven of them, the last of 140 rows, column tile first; float32 results and 16-bit ones (one rounding, half a place of eight bits, and the sums).
@pytest.mark.parametrize("m,n,k", [(700, 11992, 256), (1100, 6240, 1088), (642, 1096, 12800), (600, 2048, 12800), (642, 1090, 12800), (2700, 1536, 320)])
@pytest.mark.parametrize("kind", [KINDS[0], KINDS[3]])
def test_tiles_of_256_rows(m, n, k, kind):
    bits, gs, mode, tab = kind
    g = torch.Generator(device=DEV).manual_seed(m + n + k)
    how = dict(group_size=gs, bits=bits, mode=mode)
    w, s, b = weight(g, (), n, k, bits, gs, mode, tab)
    x = torch.randn((m, k), device=DEV, generator=g).bfloat16()
    want = x.double() @ tile(w, s, b, how).T
    close(K.quantized_matmul(x, w, s, b, out_dtype=torch.float32, **how), want)
    y = K.quantized_matmul(x, w, s, b, **how).double()
    assert ((y - want).abs() <= 2.0 ** -8 * want.abs() + 1e-4 * want.std()).all()


@pytest.mark.parametrize("counts", [(0, 1, 16, 0, 17), (22, 0, 3, 31, 17), (40, 0, 3, 70, 64), (90, 129, 0, 161, 300)])
@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("act", ["bf16", "f16"])
@pytest.mark.parametrize("gathered", [False, True])
def test_groups(counts, kind, act, gathered):
    bits, gs, mode, tab = kind
    n, k = 520, 1088 if gs < 128 else 1152
    g = torch.Generator(device=DEV).manual_seed(sum(counts))
    how = dict(group_size=gs, bits=bits, mode=mode)
    w, s, b = weight(g, (len(counts),), n, k, bits, gs, mode, tab)
    x = torch.randn((sum(counts), k), device=DEV, generator=g).to(ACT[act])
    owner = torch.repeat_interleave(torch.arange(len(counts), device=DEV), torch.tensor(counts, device=DEV))
    # up to 64 pairs, and (but for groups of 32) up to sixteen an expert, gathers are decode products: exact weights
    exact = gathered and (sum(counts) <= 64 or (sum(counts) <= 16 * len(counts) and gs > 32))
    full = [K.dequantize(w[e], s[e], None if b is None else b[e], out_dtype=torch.float32, **how) for e in range(len(counts))]
    want = torch.cat([x[owner == e].double() @ (full[e] if exact else full[e].bfloat16()).double().T for e in range(len(counts))])
    if not gathered:
        ro = torch.tensor([sum(counts[:e]) for e in range(len(counts) + 1)], dtype=torch.int32, device=DEV)
        close(K.grouped_qmm(x, w, s, b, ro, out_dtype=torch.float32, **how), want)
    else:
        mix = torch.randperm(sum(counts), device=DEV, generator=g)
        close(K.gather_qmm(x, w, s, b, mix.int(), owner[mix].int(), out_dtype=torch.float32, **how), want[mix])


# One expert is a dense product but for its offsets: rows outside them, and pairs
# that name no expert, are left alone, and nothing is written round the result.
# The sizes are those for which a dense product of as many rows splits its K on the
# prefill kernel (two or three ways), and for which no split is still ahead of the
# short-group kernel.
@pytest.mark.parametrize("r,n,k", [(650, 3080, 6144), (1000, 2056, 6144), (1250, 1544, 8256)])
@pytest.mark.parametrize("kind", [KINDS[0], KINDS[3]])
@pytest.mark.parametrize("gathered", [False, True])
def test_one_expert(r, n, k, kind, gathered):
    bits, gs, mode, tab = kind
    g = torch.Generator(device=DEV).manual_seed(r + n + k)
    how = dict(group_size=gs, bits=bits, mode=mode)
    w, s, b = weight(g, (1,), n, k, bits, gs, mode, tab)
    x = torch.randn((r, k), device=DEV, generator=g).bfloat16()
    guarded = torch.full((r + 128, n), 7.0, device=DEV)
    y = guarded[64:64 + r]
    want = x.double() @ tile(w[0], s[0], b[0], how).T
    if gathered:
        rhs = torch.randint(-1, 2, (r,), dtype=torch.int32, device=DEV, generator=g)
        lhs = torch.randperm(r, device=DEV, generator=g).int()
        K.BoundGather(x, w, s, b, lhs, rhs, y, **how).launch()
        live, want = rhs == 0, want[lhs.long()]
    else:
        live = torch.zeros(r, dtype=torch.bool, device=DEV)
        live[7:r - 13] = True
        K.BoundGrouped(x, w, s, b, torch.tensor([7, r - 13], dtype=torch.int32, device=DEV), y, **how).launch()
    close(y[live], want[live])
    assert bool((y[~live] == 7).all()) and bool((guarded[:64] == 7).all()) and bool((guarded[64 + r:] == 7).all())


# Up to sixteen pairs an expert the grouped decode multiplies float16 / float32
# activations too, term by term: with the exact weights, not their bf16 tile, which
# is 1.5e-3 away (the sums are float32: the bound of the other products).
@pytest.mark.parametrize("pairs,experts", [(65, 8), (128, 8), (200, 16)])
@pytest.mark.parametrize("k,kind", [(4096, KINDS[0]), (4096, KINDS[2]), (2048, KINDS[3]), (2944, KINDS[0])])
@pytest.mark.parametrize("act", ["f16", "f32"])
def test_wide_gathers_keep_their_weights(pairs, experts, k, kind, act):
    bits, gs, mode, tab = kind
    g = torch.Generator(device=DEV).manual_seed(pairs + k)
    how = dict(group_size=gs, bits=bits, mode=mode)
    w, s, b = weight(g, (experts,), 1024, k, bits, gs, mode, tab)
    x = torch.randn((pairs, k), device=DEV, generator=g).to(ACT[act])
    rhs = torch.randint(0, experts, (pairs,), dtype=torch.int32, device=DEV, generator=g)
    full = K.dequantize(w, s, b, out_dtype=torch.float32, **how).double()
    want = torch.stack([full[rhs[p]] @ x[p].double() for p in range(pairs)])
    close(K.gather_qmm(x, w, s, b, None, rhs, out_dtype=torch.float32, **how), want)


# Scales up to the top of bfloat16 / float32: a weight is scale times code plus bias
# whatever the scale's size, and the bias where the code is 0.  (The activations are
# small, so that sums stay in range; one group in five is large, every third column
# has none, and each column is judged by its own size.)
def large_weight(g, lead, n, k, kind):
    bits, gs, mode, tab = kind
    w, s, b = weight(g, lead, n, k, bits, gs, mode, tab)
    grow = torch.rand(s.shape, device=DEV, generator=g) < 0.2
    grow[..., ::3, :] = False
    power = torch.randint(110, 122, s.shape, device=DEV, generator=g).float()        # scales of 2^103 .. 2^116
    return w, torch.where(grow, s.float() * torch.exp2(power), s.float()).to(s.dtype), b


def columns_close(y, want):
    err = (y.double() - want).norm(dim=0) / want.norm(dim=0)
    assert bool((err <= 2e-5).all()), err.max().item()


@pytest.mark.parametrize("m,n,k", [(33, 130, 320), (128, 333, 4096), (300, 2056, 2944), (650, 3080, 6144)])
@pytest.mark.parametrize("kind", [(4, 64, "affine", "bf16"), (4, 32, "affine", "bf16"), (4, 128, "affine", "f32"),
                                  (8, 64, "affine", "bf16"), (8, 32, "affine", "f32"), (4, 32, "affine", "f32")])
def test_large_scales(m, n, k, kind):
    bits, gs, mode, _ = kind
    if k % gs:
        pytest.skip("not a whole number of groups")
    g = torch.Generator(device=DEV).manual_seed(m + n + k)
    how = dict(group_size=gs, bits=bits, mode=mode)
    w, s, b = large_weight(g, (), n, k, kind)
    x = (torch.randn((m, k), device=DEV, generator=g) * 2.0 ** -20).bfloat16()
    columns_close(K.quantized_matmul(x, w, s, b, out_dtype=torch.float32, **how), x.double() @ tile(w, s, b, how).T)


@pytest.mark.parametrize("pairs,n,k", [(100, 130, 576), (700, 1544, 1088)])
@pytest.mark.parametrize("kind", [(4, 32, "affine", "bf16"), (8, 64, "affine", "f32"), (4, 32, "affine", "f32")])
@pytest.mark.parametrize("act", ["bf16", "f16"])
def test_large_scales_of_experts(pairs, n, k, kind, act):
    bits, gs, mode, _ = kind
    g = torch.Generator(device=DEV).manual_seed(pairs + n + k)
    how = dict(group_size=gs, bits=bits, mode=mode)
    w, s, b = large_weight(g, (3,), n, k, kind)
    x = (torch.randn((50, k), device=DEV, generator=g) * 2.0 ** -10).to(ACT[act])
    lhs = torch.randint(-1, 51, (pairs,), dtype=torch.int32, device=DEV, generator=g)      # (outside [0, 50): a zero row)
    rhs = torch.randint(0, 3, (pairs,), dtype=torch.int32, device=DEV, generator=g)
    y = K.gather_qmm(x, w, s, b, lhs, rhs, out_dtype=torch.float32, **how)
    rows = torch.where(((lhs >= 0) & (lhs < 50))[:, None], x[lhs.clamp(0, 49).long()], torch.zeros((), dtype=x.dtype, device=DEV))
    for e in range(3):
        columns_close(y[rhs == e], rows[rhs == e].double() @ tile(w[e], s[e], b[e], how).T)


# A result that is not finite makes a kernel look at its column's scales: where an
# activation is the cause, only its row is touched.
@pytest.mark.parametrize("m,n,k", [(33, 130, 320), (300, 2056, 2944), (650, 3080, 6144)])
@pytest.mark.parametrize("kind", [(4, 64, "affine", "bf16"), (8, 64, "affine", "bf16"), (4, 32, "affine", "f32")])
def test_activations_that_are_not_finite_stay_in_their_rows(m, n, k, kind):
    bits, gs, mode, tab = kind
    g = torch.Generator(device=DEV).manual_seed(m + n + k)
    how = dict(group_size=gs, bits=bits, mode=mode)
    w, s, b = weight(g, (), n, k, bits, gs, mode, tab)
    x = torch.randn((m, k), device=DEV, generator=g).bfloat16()
    clean = K.quantized_matmul(x, w, s, b, **how)
    x[::16, 5], x[1::16, k - 1] = float("nan"), float("inf")
    y = K.quantized_matmul(x, w, s, b, **how)
    odd = torch.arange(m, device=DEV) % 16 < 2
    assert torch.equal(y[~odd], clean[~odd]) and not bool(y[odd].isfinite().any())


# With no room for the sums of a split K -- the least scratch that is taken -- and with
# some of it: fewer splits, or the other kernel, and the same product.
@pytest.mark.parametrize("m,n,k", [(17, 1024, 4096), (48, 4096, 14336), (300, 1000, 8256), (650, 3080, 6144)])
@pytest.mark.parametrize("act", ["bf16", "f16"])
@pytest.mark.parametrize("part", [0.0, 0.3])
def test_scratch_limits(m, n, k, act, part):
    from metaljax_amd import _lib
    lib, code = _lib.load(), {"bf16": _lib.BF16, "f16": _lib.F16}[act]
    g = torch.Generator(device=DEV).manual_seed(m + n + k)
    how = dict(group_size=64, bits=4, mode="affine")
    w, s, b = weight(g, (), n, k, 4, 64, "affine", "bf16")
    x = torch.randn((m, k), device=DEV, generator=g).to(ACT[act])
    y = torch.empty((m, n), device=DEV)

    def relaid(rows):
        return (rows + 256 + 63) // 64 * 64 * k * 2
    least = relaid(m) if act == "bf16" else sum(-(-v // 256) * 256 for v in (2 * m * k * 2, 2 * m * n * 4)) + relaid(2 * m)
    most = int(lib.qmm_workspace_bytes(1, m, n, k, 64, 4, 0, code))
    room = least + int(part * (most - least))
    ws = torch.empty(room, dtype=torch.uint8, device=DEV)

    def call(scratch):
        return lib.qmm_quantized_matmul(x.data_ptr(), code, w.data_ptr(), s.data_ptr(), b.data_ptr(), _lib.BF16, y.data_ptr(),
                                        _lib.F32, 1, m, n, k, 64, 4, 0, ws.data_ptr(), scratch, torch.cuda.current_stream().cuda_stream)
    assert call(least - 1) == 4
    assert call(room) == 0
    close(y, x.double() @ tile(w, s, b, how).T)


# a row group ahead of the offsets, behind them and past the 64 experts a wavefront reads at once; the short-group,
# prefill, block-scaled and LDS-staged kernels, terms of wider activations
@pytest.mark.parametrize("n", [72, 1001])
@pytest.mark.parametrize("r,e,k,kind,act", [(40, 3, 256, 0, "bf16"), (700, 3, 256, 0, "bf16"), (700, 70, 320, 3, "bf16"),
                                            (300, 3, 512, 5, "bf16"), (300, 3, 96, 1, "bf16"), (700, 3, 256, 0, "f16")])
def test_rows_that_no_expert_covers_are_zero(n, r, e, k, kind, act):
    bits, gs, mode, tab = KINDS[kind]
    g = torch.Generator(device=DEV).manual_seed(n + r)
    how = dict(group_size=gs, bits=bits, mode=mode)
    w, s, b = weight(g, (e,), n, k, bits, gs, mode, tab)
    x = torch.randn((r, k), device=DEV, generator=g).to(ACT[act])
    for first, last in ((5, r - 3), (0, r), (r // 2, r // 2)):
        ro = torch.linspace(first, last, e + 1, device=DEV).to(torch.int32)
        given = torch.full((r, n), 7.0, dtype=x.dtype, device=DEV)
        K.grouped_qmm(x, w, s, b, ro, out=given, **how)
        poison = torch.full((r, n), float("nan"), dtype=x.dtype, device=DEV)      # what the next allocation holds
        del poison
        y = K.grouped_qmm(x, w, s, b, ro, **how)
        assert torch.equal(y[first:last], given[first:last])
        assert not y[:first].any() and not y[last:].any()
        assert (given[:first] == 7.0).all() and (given[last:] == 7.0).all()


# float16 / float32 rows of pairs that are decode products of their own: the terms are the rows of one product a pair
# (two K-slices or less, a K that is no multiple of 64, groups of 32; one pair to the last before a sort)
@pytest.mark.parametrize("act", ["f16", "f32"])
@pytest.mark.parametrize("pairs,e,n,k,kind", [(1, 3, 40, 96, 1), (3, 9, 72, 1024, 5), (15, 40, 33, 416, 5), (5, 2, 130, 512, 0),
                                              (47, 4, 200, 1024, 5), (9, 30, 48, 160, 4), (2, 4, 64, 256, 3)])
def test_terms_of_a_pair_are_rows_of_one_product(pairs, e, n, k, kind, act):
    # float32 sums of exact products.  A four-bit code goes through the matrix core as 128 + q, so a sum is up to 136 over
    # the codes' spread of 4.6 (16 / sqrt 12) times its result, and the roundings of some ten sums, 2^-24 each, meet in it
    term_err = 136 / 4.6 * 2.0 ** -24 * 10 ** 0.5
    bits, gs, mode, tab = KINDS[kind]
    if k % gs:
        pytest.skip("no whole groups")
    g = torch.Generator(device=DEV).manual_seed(pairs + k)
    how = dict(group_size=gs, bits=bits, mode=mode)
    w, s, b = weight(g, (e,), n, k, bits, gs, mode, tab)
    exact = K.dequantize(w, s, b, out_dtype=torch.float32, **how).double()
    x = torch.randn((7, k), device=DEV, generator=g).to(ACT[act])
    lhs = torch.randint(0, 7, (pairs,), device=DEV, generator=g, dtype=torch.int32)
    rhs = torch.randint(0, e, (pairs,), device=DEV, generator=g, dtype=torch.int32)
    lhs[0] = 7 if pairs > 1 else lhs[0]                    # no row of x: reads as zeros
    y = K.gather_qmm(x, w, s, b, lhs, rhs, out_dtype=torch.float32, **how)
    rows = torch.cat([x.double(), x.new_zeros((1, k)).double()])[lhs.long()]
    want = torch.einsum("pk,pnk->pn", rows.cpu(), exact.cpu()[rhs.cpu().long()]).to(DEV)
    err = ((y.double() - want).norm() / want.norm()).item()
    assert err <= term_err, err
    y = K.gather_qmm(x[:pairs], w, s, b, None, rhs[:min(pairs, 7)], out_dtype=torch.float32, **how)
    want = torch.einsum("pk,pnk->pn", x[:pairs].double().cpu(), exact.cpu()[rhs[:min(pairs, 7)].cpu().long()]).to(DEV)
    assert ((y.double() - want).norm() / want.norm()).item() <= term_err
