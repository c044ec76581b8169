"""Expert blocks as launches against the same blocks as array operations, on the
GPU: experts past a wavefront, a router wider than a workgroup's share of it, ties
and NaN among the logits, and the two kernels against float64."""

import ctypes
import threading

import numpy as np
import pytest
import stablehlo_text as T
import torch

from metaljax_amd import _lib, engine, interpreter as I, moe, moe_launch as ML, qmm
from test_moe_launch import gemma_inputs, run_rows
from test_recognizer import _moe_inputs

pytestmark = pytest.mark.gpu


def both(text, args, monkeypatch):
    """(launches, results as launches, results as array operations)"""
    out, launches = [], []
    for on in (True, False):
        monkeypatch.setattr(ML, "available", lambda on=on: on)
        moe.reset_stats()
        ex = engine.compile_program(text)
        bufs = engine.execute(ex, args)
        bufs = engine.execute(ex, args)                  # (once more on the packed weights)
        assert moe.stats()["dispatches"] >= 2 and moe.stats()["fallbacks"] == 0
        out.append([engine.to_numpy(b)[0] for b in bufs])
        launches.append([g.launches for g in ex.interp._qmm.moe])
    assert all(g is None for g in launches[1])
    return launches[0], out[0], out[1]


# float32: sums in another order; bf16: the last place of an intermediate that was rounded from such a sum
def close(a, b, el):
    tol = 2e-5 if el == "f32" else 2e-2
    np.testing.assert_allclose(a, b, rtol=tol, atol=tol * np.abs(b[np.isfinite(b)]).max(initial=1e-6))


@pytest.mark.parametrize("el", ["f32", "bf16"])
@pytest.mark.parametrize("E,Tk,H,Ii,K", [(4, 3, 64, 32, 2), (5, 1, 96, 64, 1), (8, 64, 1536, 288, 4), (70, 9, 512, 64, 8), (130, 2, 64, 32, 3)])
def test_gpt_oss_block(E, Tk, H, Ii, K, el, monkeypatch):
    raw, _ = _moe_inputs(E, Tk, H, Ii)
    args = [I.from_numpy(a, el) if a.dtype == np.float32 else I.from_numpy(a) for a in raw]
    (g,), (out,), (plain,) = both(T.moe_block_mxfp4(E, Tk, H, Ii, K, el=el), args, monkeypatch)
    assert g is not None and g.rows is not None and g.rows.dot_k == H
    if el == "bf16":                                     # (two logits that round to one choose either expert)
        same = np.abs(out - plain).max(1) <= 2e-2 * np.abs(plain).max()
        assert same.mean() >= 0.9
        out, plain = out[same], plain[same]
    close(out, plain, el)


@pytest.mark.parametrize("el", ["f32", "bf16"])
@pytest.mark.parametrize("E,Tk,K", [(4, 3, 2), (8, 1, 4), (33, 17, 5)])
def test_gemma4_block(E, Tk, K, el, monkeypatch):
    args = gemma_inputs(E, Tk, 64, 32, el)
    (g,), (out,), (plain,) = both(T.moe_block_gemma4_mxfp4(E, Tk, 64, 32, K, el=el), args, monkeypatch)
    assert g is not None and g.rows is not None
    close(out, plain, el)


def test_ties_and_nan_among_the_logits(monkeypatch):
    E, Tk, H, Ii, K = 6, 4, 32, 32, 3
    raw, _ = _moe_inputs(E, Tk, H, Ii)
    x, wr, br = raw[0].copy(), np.zeros_like(raw[1]), np.array([1, 2, 1, 2, 1, 0], np.float32)
    wr[0, 5] = 1.0
    x[:, 0] = (0, 1, np.nan, np.inf)                    # expert 5: below the ties, among them, NaN, infinite
    (g,), (out,), (plain,) = both(T.moe_block_mxfp4(E, Tk, H, Ii, K), [I.from_numpy(a) for a in (x, wr, br) + raw[3:]], monkeypatch)
    assert g is not None and g.rows is not None
    finite = np.isfinite(plain)
    assert np.array_equal(finite, np.isfinite(out)) and finite[:2].all()
    close(out[finite], plain[finite], "f32")


@pytest.mark.parametrize("special", [False, True])
@pytest.mark.parametrize("xel,wel,k,n,along_k", [
    ("f32", "f32", 1000, 8, False), ("f32", "f32", 7, 1, True), ("bf16", "bf16", 77, 100, True), ("f16", "f16", 2049, 3, False),
    ("f32", "bf16", 300, 33, False), ("bf16", "bf16", 16, 64, False), ("f32", "f32", 3, 300, True)])
def test_a_row_program(xel, wel, k, n, along_k, special):
    """Products of every operand form, of whole and partial turns, of a wavefront's columns and
    more; a leaf past the 256 elements that are held; a top-k over several wavefronts' worth of
    elements, with ties, both zeros, infinities and NaN; reductions over one to 300.  Small
    integers: the sums are exact in any order."""
    from metaljax_amd.kernels import _stream
    types = {"f32": torch.float32, "bf16": torch.bfloat16, "f16": torch.float16}
    g, tokens, top = torch.Generator().manual_seed(k), 3, min(n, 6)
    x = torch.randint(-3, 4, (tokens, k), generator=g).to(types[xel])
    w = torch.randint(-2, 3, (n, k) if along_k else (k, n), generator=g).to(types[wel])
    b = torch.randint(-2, 3, (n,), generator=g).float()
    if special:
        x.zero_()
        b[torch.randperm(n, generator=g)[:7]] = torch.tensor([np.nan, np.inf, -0.0, 0.0, -np.inf, np.nan, np.inf])[:min(n, 7)]
    OP, at = ML.OP, lambda row: 512 * row                # (a row of 512 floats a value)
    code = [(OP["add"], at(2), n, at(0), n, at(1), n), (OP["top_k"], at(3), top, at(2), n, 0, 1, at(4), top),
            (OP["sum"], at(5), 1, at(2), n), (OP["rowmax"], at(5) + 1, 1, at(2), n), (OP["rowmin"], at(5) + 2, 1, at(2), n),
            (OP["sum"], at(5) + 3, 1, at(3), top), (OP["slice"], at(5) + 4, (n + 1) // 2, at(2), n, 0, 1, 2, 1)]

    def program(x, w, b, idx, out):
        p = ML.RowProgram(dot_x=x.data_ptr(), dot_w=w.data_ptr(), dot_x_t=k, dot_x_k=1, dot_w_n=k if along_k else 1, dot_w_k=1 if along_k else n,
                          dot_k=k, dot_n=n, dot_cols=1 << (n - 1).bit_length(), dot_dst=at(0), dot_x_el=ML.ELS[xel], dot_w_el=ML.ELS[wel],
                          dot_el=0, tokens=tokens, reg_floats=at(6), leaves=1, instructions=len(code), outs=2)
        p.leaf[0] = ML.RowLeaf(b.data_ptr(), 0, 0, 1, 0, at(1), n)
        for i, (op, dst, m, *rest) in enumerate(code):
            p.code[i] = ML.RowInstruction(op, 0, dst, m, *(rest + [0, 1] * 3)[:6], 0.0)
        p.out[0] = ML.RowOut(idx.data_ptr(), ML.ELS["i32"], at(4), top, top)
        p.out[1] = ML.RowOut(out.data_ptr(), 0, at(5), 4 + (n + 1) // 2, 4 + (n + 1) // 2)
        return p

    def results(device):
        return torch.zeros((tokens, top), dtype=torch.int32, device=device), torch.zeros((tokens, 4 + (n + 1) // 2), device=device)
    want, host = results("cpu"), [a.contiguous() for a in (x, w, b)]
    with np.errstate(all="ignore"):
        run_rows(program(*host, *want), None)
    got, card = results("cuda"), [a.cuda() for a in host]
    ML.run_rows(program(*card, *got), _stream(got[1]))
    assert torch.equal(got[0].cpu(), want[0])
    np.testing.assert_array_equal(got[1].cpu().numpy(), want[1].numpy())


@pytest.mark.parametrize("op,fn", [("exponential", np.exp), ("logistic", lambda v: 1 / (1 + np.exp(-v))), ("tanh", np.tanh), ("log", np.log),
                                   ("rsqrt", lambda v: 1 / np.sqrt(v)), ("round_nearest_even", np.rint), ("sign", np.sign), ("floor", np.floor)])
def test_an_elementwise_instruction(op, fn):
    """One instruction on a 3 x 5 x 300 result read through swapped axes: two
    float32 places of what numpy gives in float64."""
    from metaljax_amd.kernels import _stream
    v = torch.randn((5, 3, 300), device="cuda", generator=torch.Generator(device="cuda").manual_seed(1)) * 3
    if op in ("log", "rsqrt"):
        v = v.abs() + 0.01
    y, experts = torch.empty((2, 3, 5, 300), device="cuda"), torch.tensor([1, 0], dtype=torch.int32, device="cuda")
    m = ML.PairMap(y=y.data_ptr(), experts_of=experts.data_ptr(), pairs=2, inner=4500, dims=(3, 5, 300), per_token=1, experts=2,
                   rank=3, leaves=1, instructions=1, registers=2, result=1)
    m.leaf[0] = ML.MapLeaf(v.data_ptr(), 0, 0, 0, 0, (300, 900, 1), 0)
    m.code[0] = ML.Instruction(ML.OP[op], 1, 0, 0, 0, 0, 0.0)
    ML.run_map(m, _stream(y))
    want = fn(v.double().cpu().numpy().transpose(1, 0, 2))
    for half in y.cpu().numpy():
        np.testing.assert_allclose(half, want, rtol=4e-7, atol=1e-30)


@pytest.mark.parametrize("pairs,per", [(65535, 1), (65536, 1), (131071, 1), (3 * 65536, 3), (140000, 2)])
@pytest.mark.parametrize("summed", [False, True])
def test_more_pairs_than_a_grid_axis(pairs, per, summed):
    """y[p] = 2 x[p], and its weighted sum over a token's pairs, past the 65535 rows
    that a grid's second axis takes: exact in float32 for small integers."""
    from metaljax_amd.kernels import _stream
    g = torch.Generator(device="cuda").manual_seed(pairs)
    x = torch.randint(-8, 8, (pairs, 3), device="cuda", generator=g).float()
    w = torch.randint(-8, 8, (pairs,), device="cuda", generator=g).float()
    experts = torch.zeros(pairs, dtype=torch.int32, device="cuda")
    y = torch.full((pairs // per if summed else pairs, 3), -99.0, device="cuda")
    m = ML.PairMap(y=y.data_ptr(), experts_of=experts.data_ptr(), pairs=pairs, inner=3, dims=(1, 1, 3), per_token=per, experts=1,
                   rank=1, leaves=1, instructions=1, registers=2, result=1, weights=w.data_ptr() if summed else None)
    m.leaf[0] = ML.MapLeaf(x.data_ptr(), 0, 3, 0, 0, (0, 0, 1), 0)
    m.code[0] = ML.Instruction(ML.OP["add"], 1, 0, 0, 0, 0, 0.0)
    ML.run_map(m, _stream(y))
    want = 2 * x if not summed else (2 * x * w[:, None]).reshape(pairs // per, per, 3).sum(1)
    assert torch.equal(y, want)


def test_a_long_prompt(monkeypatch):
    """65600 pairs of 32800 tokens: as launches what it is as array operations."""
    E, Tk, H, Ii, K = 4, 32800, 32, 32, 2
    raw, _ = _moe_inputs(E, Tk, H, Ii)
    (g,), (out,), (plain,) = both(T.moe_block_mxfp4(E, Tk, H, Ii, K), [I.from_numpy(a) for a in raw], monkeypatch)
    assert g is not None
    same = np.abs(out - plain).max(1) <= 2e-5 * np.abs(plain).max()     # (a logit's last place may choose another expert)
    assert same.mean() >= 0.999


def test_pair_tokens_are_there_for_another_stream():
    """Made by the first call, on whatever stream it runs, behind whatever that
    stream still has to do; the next call's launches may be on another one."""
    g = moe.Dispatch()
    g.T, g.K = 3000, 7
    a, stream = torch.randn((4096, 4096), device="cuda"), torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(stream):
        for _ in range(20):
            a = a @ a * 1e-2
        t32, t64 = g.pair_tokens("cuda")
    seen = t32.clone(), t64.clone()
    want = torch.arange(3000).repeat_interleave(7)
    assert seen[0].dtype == torch.int32 and seen[1].dtype == torch.int64
    assert torch.equal(seen[0].cpu().long(), want) and torch.equal(seen[1].cpu(), want)
    stream.synchronize()


@pytest.mark.parametrize("el", ["f32", "bf16", "f16"])
@pytest.mark.parametrize("E,Tk,H,Ii,K,fused", [
    (1, 1, 32, 32, 1, "222"), (4, 1, 160, 96, 4, "222"), (8, 3, 1024, 1024, 2, "222"), (8, 5, 96, 2080, 2, "222"), (8, 7, 4160, 32, 1, "122"),
    (4, 32, 512, 96, 2, "121"), (8, 64, 288, 64, 1, "121"), (8, 33, 64, 64, 2, "000"), (3, 11, 1056, 544, 3, "121"), (5, 2, 64, 32, 5, "111"),
    (16, 24, 3168, 896, 1, "111"), (4, 12, 320, 96, 2, "222"), (8, 64, 160, 64, 1, "222"), (3, 11, 224, 544, 3, "222")])
def test_a_product_and_its_map_in_one_launch(E, Tk, H, Ii, K, fused, el, monkeypatch):
    # fused: how many of a block's two products are, for float32, bf16 and float16 (the sum over a token's pairs
    # is where its workgroups are a round or two)
    """Pairs of their own, pairs sorted by the kernel, the sum over a token's pairs in two
    to sixteen wavefronts, K of a part of a chunk and of more than 2048, there in one round of
    workgroups and in several: what two launches give.  The sums are the same ones in the
    same order."""
    raw, _ = _moe_inputs(E, Tk, H, Ii)
    args = [I.from_numpy(a, el) if a.dtype == np.float32 else I.from_numpy(a) for a in raw]
    out, all_steps, run_steps = [], ML.Launches._steps, ML.run_steps

    def two_launches(self):
        all_steps(self)
        for s in self.steps:
            if s.kind == ML.PRODUCT:
                s.kind, s.skip = ML.MAP, 0                               # (a map of no pairs: nothing)
                nothing = ML.PairMap(per_token=1, experts=1, rank=1)
                s.bytes, s.patches, s.program = ctypes.sizeof(nothing), 0, ctypes.addressof(nothing)
                self.programs.append(nothing)
    served = []
    monkeypatch.setattr(ML, "run_steps", lambda steps, values, stream: (served.append(which(steps, values, stream)), run_steps(steps, values, stream))[1])
    for on in (True, False):
        if not on:
            monkeypatch.setattr(ML.Launches, "_steps", two_launches)
        ex = engine.compile_program(T.moe_block_mxfp4(E, Tk, H, Ii, K, el=el))
        (buf,) = engine.execute(ex, args)
        assert ex.interp._qmm.moe[0].launches is not None
        out.append(engine.to_numpy(buf)[0])
    assert served == [int(fused["f32 bf16 f16".split().index(el)]), 0]
    assert np.array_equal(*out)


@pytest.mark.parametrize("Tk", [3, 12])
def test_blocks_of_two_threads_on_their_streams(Tk):
    """The steps of a block are shared by its calls: two threads at once, each on a stream of
    its own with activations that the work ahead of them there has yet to write, pairs of
    their own and pairs that the launch sorts; what the calls give one after the other."""
    E, H, Ii, K, calls = 8, 512, 256, 2, 25
    args = [I.from_numpy(a) for a in _moe_inputs(E, Tk, H, Ii)[0]]
    ex = engine.compile_program(T.moe_block_mxfp4(E, Tk, H, Ii, K))
    xs = torch.randn((2, calls, Tk, H), device="cuda") / 8
    want = [torch.stack([engine.execute(ex, [x] + args[1:])[0].data.clone() for x in row]) for row in xs]
    assert ex.interp._qmm.moe[0].launches is not None and not torch.equal(*want)
    got, errors = [None, None], []

    def work(i):
        try:
            stream = torch.cuda.Stream()
            a, late = torch.randn((2048, 2048), device="cuda"), torch.zeros_like(xs[i])
            torch.cuda.synchronize()
            with torch.cuda.stream(stream):
                for _ in range(20):
                    a = a @ a * 1e-2
                late.copy_(xs[i])
                got[i] = torch.stack([engine.execute(ex, [x] + args[1:])[0].data for x in late])
            stream.synchronize()
        except Exception as e:                           # (the thread's; raised below)
            errors.append(e)
    threads = [threading.Thread(target=work, args=(i,)) for i in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join(60)
    assert not errors and all(torch.equal(g, w) for g, w in zip(got, want)), errors


def which(steps, values, stream):
    """How many of the pair products the library serves (each is run once more by the call)."""
    n = 0
    for s in steps:
        if s.kind == ML.PRODUCT:
            p = ML.PairProduct.from_buffer_copy(ctypes.string_at(s.program, s.bytes))
            for q in s.patch[:s.patches]:
                ctypes.c_uint64.from_address(ctypes.addressof(p) + q.at).value = values[q.value] + q.add
            n += _lib.load().qmm_pair_product_run(ctypes.byref(p), stream) == 0
    return n


@pytest.mark.parametrize("el", ["f32", "bf16", "f16"])
@pytest.mark.parametrize("pairs,per,E,n,k,inner,columns,summed", [
    (5, 1, 8, 17, 96, 17, [(0, 1)], False), (6, 2, 3, 2, 32, 1, [(1, 0)], False), (12, 4, 5, 35, 160, 17, [(0, 2), (1, 2)], False),
    (3, 3, 2, 24, 1056, 24, [(0, 1), (5, 0)], False), (40, 4, 8, 33, 96, 33, [(0, 1)], False), (64, 1, 3, 34, 288, 17, [(17, 1), (0, 1)], False),
    (33, 3, 16, 31, 544, 1, [(30, 1), (3, 2)], False), (6, 2, 4, 17, 64, 17, [(0, 1)], True), (4, 4, 8, 40, 96, 20, [(1, 2)], True),
    (48, 3, 6, 18, 1056, 18, [(0, 1)], True)])
def test_a_pair_product(pairs, per, E, n, k, inner, columns, summed, el):
    """The product and its map as one launch against the product, then the map: pairs of their own and (from
    sixteen on, where two share an expert) sorted by the kernel, and a token's sum; results that end inside a
    workgroup's sixteen elements, columns that are one, neighbours or every other one; experts outside the
    weight, whose nearest one is read on every route.  The sums are the same ones in the same order."""
    from metaljax_amd import kernels
    types = {"f32": torch.float32, "bf16": torch.bfloat16, "f16": torch.float16}
    g = torch.Generator(device="cuda").manual_seed(pairs + k)
    w = torch.randint(-2**31, 2**31 - 1, (E, n, k // 8), dtype=torch.int32, device="cuda", generator=g)
    s = torch.randint(120, 128, (E, n, k // 32), dtype=torch.uint8, device="cuda", generator=g)
    x = torch.randn((pairs // per, k), device="cuda", generator=g).to(types[el])
    bias, weights = torch.randn((E, inner), device="cuda", generator=g), torch.rand(pairs, device="cuda", generator=g)
    experts = torch.randint(-2, E + 2, (pairs,), dtype=torch.int32, device="cuda", generator=g)
    experts[0], experts[pairs - 1] = -1, E
    rows = pairs // per if summed else pairs
    token = (torch.arange(pairs, dtype=torch.int32, device="cuda") // per).int()
    stream = kernels._stream(x)

    def program(y, product):
        """(columns or their product) + bias of the expert; `product`: the leaves' address, None for the launch that computes it"""
        m = ML.PairMap(y=y.data_ptr(), experts_of=experts.data_ptr(), pairs=pairs, inner=inner, dims=(1, 1, inner), per_token=per, experts=E,
                       rank=1, leaves=len(columns) + 1, instructions=2, registers=4, result=3, weights=weights.data_ptr() if summed else None)
        for i, (base, step) in enumerate(columns):
            m.leaf[i] = ML.MapLeaf(product, 0, 0, 0, 0, (0, 0, 0), ML.ELS[el]) if product is None else ML.MapLeaf(product, base, n, 0, 0, (0, 0, step), ML.ELS[el])
        m.leaf[len(columns)] = ML.MapLeaf(bias.data_ptr(), 0, 0, inner, 0, (0, 0, 1), 0)
        m.code[0] = ML.Instruction(ML.OP["multiply" if len(columns) == 2 else "copy"], 3, 0, 1, 0, 0, 0.0)
        m.code[1] = ML.Instruction(ML.OP["add"], 3, 3, len(columns), 0, 0, 0.0)
        return m
    got, want = (torch.full((rows, inner), float("nan"), device="cuda") for _ in range(2))
    fused = ML.PairProduct(x=x.data_ptr(), w=w.data_ptr(), s=s.data_ptr(), x_rows=pairs // per, n=n, k=k, mode=_lib.MODE_MXFP4, x_el=ML.ELS[el],
                           x_per=per, product_el=ML.ELS[el], tiles=len(columns), map=program(got, None))
    for t, (base, step) in enumerate(columns):
        fused.col_leaf[t], fused.col_base[t], fused.col_step[t] = t, base, step
    _lib.check(_lib.load().qmm_pair_product_run(ctypes.byref(fused), stream))
    nearest = experts.clamp(0, E - 1)
    y = kernels.gather_qmm(x, w, s, None, token, nearest, group_size=32, bits=4, mode="mxfp4")
    ML.run_map(program(want, y.data_ptr()), stream)
    assert torch.equal(got, want)
    full = kernels.dequantize(w, s, None, group_size=32, bits=4, mode="mxfp4", out_dtype=torch.float32).double().cpu()
    exact = torch.stack([full[e] @ v for e, v in zip(nearest.tolist(), x.double().cpu()[token.long().cpu()])])
    tol = 1e-6 if el == "f32" else 2.0 ** -8 if el == "bf16" else 2.0 ** -11      # (one rounding to the product's type)
    assert ((y.double().cpu() - exact).norm() / exact.norm()).item() <= tol
