"""Dispatches compiled to launches (metaljax_amd.moe_launch): the programs that
the planner writes, run here by a plain reading of their structs on host memory,
give what the dispatch's array operations give -- every form that is compiled, at
one token and several, in float32 and bf16; what is not modelled stays with the
array operations."""

import ctypes

import numpy as np
import pytest
import stablehlo_text as T
import torch

from metaljax_amd import _lib, engine, interpreter as I, moe, moe_launch as ML, qmm
from test_recognizer import _moe_inputs, _oracle_expert_product, _without_a_gpu

pytestmark = pytest.mark.filterwarnings("ignore")
NAMES = {v: k for k, v in ML.OP.items()}
TYPES = {0: (ctypes.c_float, 4), 1: (ctypes.c_uint16, 2), 2: (ctypes.c_uint16, 2), 3: (ctypes.c_uint8, 1), 4: (ctypes.c_int32, 4)}


def load(p, i, el):
    raw = TYPES[el][0].from_address(p + i * TYPES[el][1]).value
    if el == 1:
        return np.uint32(raw << 16).view(np.float32)
    return np.float32(np.uint16(raw).view(np.float16)) if el == 2 else np.float32(raw)


def rounded(v, el):
    v = np.float32(v)
    return I.round_bf16(v.reshape(1))[0] if el == 1 else np.float32(np.float16(v)) if el == 2 else v


def store(p, i, v, el):
    if el == 1:
        v = int(I.f32_to_bf16_bits(np.float32(v).reshape(1))[0])
    elif el == 2:
        v = int(np.float16(v).view(np.uint16))
    TYPES[el][0].from_address(p + i * TYPES[el][1]).value = int(v) if el == 4 else v


def apply(op, a, b, c):
    with np.errstate(all="ignore"):
        one = np.float32(1)
        return {"copy": lambda: a, "add": lambda: a + b, "subtract": lambda: a - b, "multiply": lambda: a * b,
                "divide": lambda: a / b, "maximum": lambda: np.maximum(a, b), "minimum": lambda: np.minimum(a, b),
                "exponential": lambda: np.exp(a), "logistic": lambda: one / (one + np.exp(-a)), "tanh": lambda: np.tanh(a),
                "clamp": lambda: np.minimum(np.maximum(b, a), c), "negate": lambda: -a, "rsqrt": lambda: one / np.sqrt(a),
                "LT": lambda: one * (a < b), "select": lambda: b if a != 0 else c}[NAMES[op]]()


def run_map(m, _stream):
    per = m.per_token if m.weights else 1
    for row in range(m.pairs // per):
        for i in range(m.inner):
            c, total = np.unravel_index(i, tuple(m.dims)), np.float32(0)
            for k in range(per):
                p = row * per + k
                e = ctypes.c_int32.from_address(m.experts_of + 4 * p).value
                regs = [None] * m.registers
                for j in range(m.leaves):
                    f = m.leaf[j]
                    regs[j] = load(f.p, f.base + p * f.pair + e * f.expert + p // m.per_token * f.token +
                                   sum(int(x) * s for x, s in zip(c, f.coef)), f.el)
                for q in m.code[:m.instructions]:
                    v = q.imm if NAMES[q.op] == "imm" else apply(q.op, regs[q.a], regs[q.b], regs[q.c])
                    regs[q.dst] = rounded(v, q.el)
                v = regs[m.result]
                if m.weights:
                    total += rounded(v, m.sum_el) * load(m.weights, p, m.weights_el)
            store(m.y, row * m.inner + i, total if m.weights else v, m.y_el)


def run_rows(r, _stream):
    for t in range(r.tokens):
        regs = np.full(r.reg_floats, np.nan, np.float32)
        if r.dot_x:
            for n in range(r.dot_n):
                regs[r.dot_dst + n] = rounded(sum(
                    load(r.dot_x, t * r.dot_x_t + k * r.dot_x_k, r.dot_x_el) * load(r.dot_w, n * r.dot_w_n + k * r.dot_w_k, r.dot_w_el)
                    for k in range(r.dot_k)), r.dot_el)
        for f in r.leaf[:r.leaves]:
            for i in range(f.n):
                regs[f.dst + i] = load(f.p, f.base + t * f.token + i * f.step, f.el)
        for q in r.code[:r.instructions]:
            name, a = NAMES[q.op], regs[q.a:q.a + q.an].copy()
            if name == "top_k":
                vals, idx = I.top_k(a[None], q.n)
                regs[q.dst:q.dst + q.n], regs[q.c:q.c + q.n] = vals[0], idx[0]
            elif name in ("sum", "rowmax", "rowmin"):
                regs[q.dst] = rounded({"sum": np.sum, "rowmax": np.max, "rowmin": np.min}[name](a), q.el)
            else:
                for i in range(q.n):
                    at = [regs[s + (0 if w == 1 else i)] for s, w in ((q.a, q.an), (q.b, q.bn), (q.c, q.cn))] if name not in ("imm", "slice") else []
                    regs[q.dst + i] = rounded(q.imm if name == "imm" else regs[q.a + q.b + i * q.c] if name == "slice" else apply(q.op, *at), q.el)
        for o in r.out[:r.outs]:
            for i in range(o.n):
                store(o.p, t * o.n + i, regs[o.src + (0 if o.srcn == 1 else i)], o.el)


def run_product(x, el, rows, arrays, match, lhs, rhs, y, y_el, pairs, experts, n, k, like, _stream):
    from oracle import qmm_oracle as O
    assert match.mode == "mxfp4"
    a = np.array([[load(x, i * k + j, ML.ELS[el]) for j in range(k)] for i in range(rows)], np.float32)
    index = [np.array([ctypes.c_int32.from_address(p + 4 * i).value for i in range(pairs)]) if p else np.arange(pairs) for p in (lhs, rhs)]
    w, scales = moe.split_experts([np.asarray(arrays[0]), np.asarray(arrays[1])], experts)
    out = O.gather_qmm(a, w, scales, None, *index, match.gs, match.bits, match.mode)
    for i, v in enumerate(out.reshape(-1)):
        store(y, i, v, ML.ELS[y_el])


def both(text, args, monkeypatch, rows=run_rows):
    """(launches, results as launches, results as array operations)"""
    monkeypatch.setattr(qmm, "DEVICE", "cpu")
    monkeypatch.setattr(moe, "emit_dot", _oracle_expert_product([]))
    plain = [I.host(b.data).a for b in engine.execute(engine.compile_program(text), args)]
    monkeypatch.setattr(ML, "available", lambda: True)
    monkeypatch.setattr(ML, "run_map", run_map)
    monkeypatch.setattr(ML, "run_rows", rows)
    monkeypatch.setattr(ML, "run_product", run_product)
    moe.reset_stats()
    ex = engine.compile_program(text)
    out = [I.host(b.data).a for b in engine.execute(ex, args)]
    assert moe.stats()["dispatches"] >= 1 and moe.stats()["fallbacks"] == 0
    return [g.launches for g in ex.interp._qmm.moe], out, plain


def gemma_inputs(E, Tk, H, Ii, el):
    rng = np.random.default_rng(E + Tk)
    packed = [T.make_mxfp4_experts(r, c, E, seed=i)[:2] for i, (r, c) in enumerate(((Ii, H), (Ii, H), (H, Ii)))]
    raw = [(rng.standard_normal((Tk, H)) / 8).astype(np.float32), rng.standard_normal((H, E)).astype(np.float32),
           (1 + rng.standard_normal(H) / 8).astype(np.float32), *[a for p in packed for a in p],
           (1 + rng.standard_normal(E) / 8).astype(np.float32)]
    return [I.from_numpy(a, el) if a.dtype == np.float32 else I.from_numpy(a) for a in raw]


@_without_a_gpu
@pytest.mark.parametrize("el", ["f32", "bf16"])
@pytest.mark.parametrize("E,Tk,H,Ii,K,composite", [(4, 3, 64, 32, 2, False), (5, 1, 32, 32, 2, True), (4, 4, 32, 64, 4, True), (3, 2, 32, 32, 1, False)])
def test_gpt_oss_block(E, Tk, H, Ii, K, composite, el, monkeypatch):
    raw, _ = _moe_inputs(E, Tk, H, Ii)
    args = [I.from_numpy(a, el) if a.dtype == np.float32 else I.from_numpy(a) for a in raw]
    (g,), (out,), (plain,) = both(T.moe_block_mxfp4(E, Tk, H, Ii, K, el=el, composite=composite), args, monkeypatch)
    assert g is not None and g.rows is not None and g.rows.dot_k == H      # the router's product is part of it
    assert [d.feed is None for d in g.dots] == [True, False]
    # the same roundings in the same places; sums in another order (bf16: a last place of an intermediate)
    np.testing.assert_allclose(out, plain, rtol=2e-5 if el == "f32" else 2e-2, atol=(1e-6 if el == "f32" else 2e-2) * np.abs(plain).max())


@_without_a_gpu
@pytest.mark.parametrize("el", ["f32", "bf16"])
@pytest.mark.parametrize("E,Tk,K", [(4, 3, 2), (8, 1, 4)])
def test_gemma4_block(E, Tk, K, el, monkeypatch):
    args = gemma_inputs(E, Tk, 64, 32, el)
    (g,), (out,), (plain,) = both(T.moe_block_gemma4_mxfp4(E, Tk, 64, 32, K, el=el), args, monkeypatch)
    assert g is not None and g.rows is not None and not g.rows.dot_x       # its product reads computed activations
    assert len(g.dots) == 3
    np.testing.assert_allclose(out, plain, rtol=2e-5 if el == "f32" else 2e-2, atol=(1e-6 if el == "f32" else 2e-2) * np.abs(plain).max())


@_without_a_gpu
def test_blocks_before_and_inside_a_loop(monkeypatch):
    args = gemma_inputs(4, 3, 32, 32, "f32")
    launches, out, plain = both(T.moe_gemma4_decode_loop(4, 3, 32, 32, 2, 2), args, monkeypatch)
    assert len(launches) == 2 and all(g is not None for g in launches)
    for a, b in zip(out, plain):
        np.testing.assert_allclose(a, b, rtol=2e-5, atol=1e-6)


@_without_a_gpu
@pytest.mark.parametrize("shared", ["a conversion", "the largest logit"])
def test_what_router_and_experts_share_is_computed(shared, monkeypatch):
    """A value that the row program computes for itself and that the launches read
    as well: the activations' conversion, and a router's value that the experts' results
    are multiplied by (the program computes the router then)."""
    E, Tk, H, Ii, K = 4, 3, 64, 32, 2
    text, th, eth = T.moe_block_mxfp4(E, Tk, H, Ii, K), f"tensor<{Tk}x{H}xf32>", f"tensor<{E}x{Tk}x{H}xf32>"
    raw, _ = _moe_inputs(E, Tk, H, Ii)
    args = [I.from_numpy(a) for a in raw]
    if shared == "a conversion":
        half = f"tensor<{Tk}x{H}xbf16>"
        new = text.replace(f"%x: {th}", f"%xh: {half}", 1).replace("    %gu0 =", f"    %x = stablehlo.convert %xh : ({half}) -> {th}\n    %gu0 =")
        args[0] = I.from_numpy(raw[0], "bf16")
    else:
        new = text.replace("    %ys = stablehlo.multiply %y, ", f"""    %lb = stablehlo.broadcast_in_dim %mx, dims = [1] : (tensor<{Tk}xf32>) -> {eth}
    %yl = stablehlo.multiply %y, %lb : {eth}
    %ys = stablehlo.multiply %yl, """)
    assert new != text
    (g,), (out,), (plain,) = both(new, args, monkeypatch)
    assert g is not None and (g.rows is not None) == (shared == "a conversion")
    np.testing.assert_allclose(out, plain, rtol=2e-5, atol=1e-6 * np.abs(plain).max())


@_without_a_gpu
@pytest.mark.parametrize("behind", ["the activations", "the logits"])
def test_a_long_program_ahead_of_the_router(behind, monkeypatch):
    """What lies ahead of a block may be a whole model: it is not walked by recursion."""
    E, Tk, H, Ii, K, n = 4, 3, 32, 32, 2, 1500
    text = T.moe_block_mxfp4(E, Tk, H, Ii, K)
    if behind == "the activations":
        ty, first, last, before = f"tensor<{Tk}x{H}xf32>", "%x0", "%x", "    %gu0 ="
        text = text.replace(f"%x: {ty}", f"%x0: {ty}", 1)
    else:
        ty, first, last, before = f"tensor<{Tk}x{E}xf32>", "%raised", "%logits", "    %vals, %idx ="
        text = text.replace("%logits =", "%raised =", 1)
    names = [first] + [f"%neg{i}" for i in range(n - 1)] + [last]
    chain = "".join(f"    {b} = stablehlo.negate {a} : {ty}\n" for a, b in zip(names, names[1:]))
    raw, _ = _moe_inputs(E, Tk, H, Ii)
    (g,), (out,), (plain,) = both(text.replace(before, chain + before), [I.from_numpy(a) for a in raw], monkeypatch)
    assert g is not None and (g.rows is not None or behind == "the logits")     # (a chain may leave no room for the rest)
    np.testing.assert_allclose(out, plain, rtol=2e-5, atol=1e-6 * np.abs(plain).max())


@_without_a_gpu
@pytest.mark.parametrize("draw", [0, 1, 2])
@pytest.mark.parametrize("block", ["gpt-oss", "gpt-oss composite", "gemma4", "sum of a broadcast", "sum of a constant", "slice of a broadcast",
                                   "top-k of a broadcast"])
def test_a_row_program_is_the_programs_router(block, draw, monkeypatch):
    """The compiled router's experts and weights against the program's own evaluation
    of them, on drawn inputs; from the second draw on coarse ones, whose logits tie."""
    from metaljax_amd.packs import evaluate
    E, Tk, H, Ii, K = 6, 5, 32, 32, 3
    rng = np.random.default_rng(draw)
    if block == "gemma4":
        text, args = T.moe_block_gemma4_mxfp4(E, Tk, H, Ii, K), gemma_inputs(E, Tk, H, Ii, "f32")
        drawn = [0, 1]
    else:
        text = T.moe_block_mxfp4(E, Tk, H, Ii, K, composite=block.endswith("composite"))
        if not block.startswith("gpt-oss"):
            old, new = repeated(block, Tk, E, K)
            assert old in text
            text = text.replace(old, new)
        args, drawn = [I.from_numpy(a) for a in _moe_inputs(E, Tk, H, Ii)[0]], [0, 1, 2]
    for i in drawn:
        a = rng.standard_normal(I.host(args[i]).a.shape).astype(np.float32)
        args[i] = I.from_numpy(np.round(2 * a) / 2 if draw else a)
    out = []

    def kept(r, stream):
        run_rows(r, stream)
        out.append([[load(o.p, i, o.el) for i in range(r.tokens * o.n)] for o in r.out[:2]])
    (g,), _, _ = both(text, args, monkeypatch, rows=kept)
    assert len(out) == 1 and g.rows is not None
    env = dict(zip(g.interp._main_block().args, [I.host(a) for a in args]))
    router = g.g.router
    assert out[0][0] == list(I.host(evaluate(g.interp, router.indices, env)).a.reshape(-1))
    np.testing.assert_allclose(out[0][1], I.host(evaluate(g.interp, router.weights, env)).a.reshape(-1), rtol=2e-6, atol=1e-7)


@_without_a_gpu
def test_a_call_changes_nothing_that_another_one_reads(monkeypatch):
    """Threads share a dispatch's launches: what a call reads of them is there when
    the program is compiled, the size of its buffer first of all."""
    seen, run = [], ML.Launches.run
    monkeypatch.setattr(ML.Launches, "run", lambda self, *a: (seen.append(dict(vars(self))), run(self, *a))[1])
    raw, _ = _moe_inputs(4, 3, 32, 32)
    (g,), _, _ = both(T.moe_block_mxfp4(4, 3, 32, 32, 2), [I.from_numpy(a) for a in raw], monkeypatch)
    assert seen and seen[0] == vars(g)


@_without_a_gpu
@pytest.mark.parametrize("elsewhere", [False, True])
def test_emit_reads_names_what_a_call_reads(elsewhere, monkeypatch):
    """Exactly the values that the launches look up, with the router as a row
    program and, where its weights are read elsewhere, with the program's router."""
    E, Tk, H, Ii, K = 4, 3, 32, 32, 2
    text = T.moe_block_mxfp4(E, Tk, H, Ii, K)
    if elsewhere:
        text = text.replace(f"return %out : tensor<{Tk}x{H}xf32>", f"return %out, %w : tensor<{Tk}x{H}xf32>, tensor<{Tk}x{K}xf32>")
        text = text.replace(f"-> tensor<{Tk}x{H}xf32> {{\n", f"-> (tensor<{Tk}x{H}xf32>, tensor<{Tk}x{K}xf32>) {{\n", 1)
    seen, run = set(), ML.Launches.run

    class Looked:
        def __init__(self, env):
            self.env = env

        def __getitem__(self, v):
            seen.add(v)
            return self.env[v]
    monkeypatch.setattr(ML.Launches, "run", lambda self, interp, env: run(self, interp, Looked(env)))
    raw, _ = _moe_inputs(E, Tk, H, Ii)
    (g,), _, _ = both(text, [I.from_numpy(a) for a in raw], monkeypatch)
    assert (g.rows is None) == elsewhere and set(qmm.emit_reads(g.g)) == seen


def repeated(what, Tk, E, K):
    """(old, new) lines of moe_block_mxfp4: a sum, a slice, a top-k over a value that is repeated along the row"""
    tk, tok, te = f"tensor<{Tk}x{K}xf32>", f"tensor<{Tk}xf32>", f"tensor<{Tk}x{E}xf32>"
    down = f"applies stablehlo.add across dimensions = [1] : ({tk}, tensor<f32>) -> {tok}"
    if what == "sum of a broadcast":
        return f"%sm = stablehlo.reduce(%ex init: %z32) {down}", f"%sm = stablehlo.reduce(%mxb init: %z32) {down}"
    if what == "sum of a constant":
        return (f"%sm = stablehlo.reduce(%ex init: %z32) {down}",
                f"%twos = stablehlo.constant dense<2.0> : {tk}\n    %sm = stablehlo.reduce(%twos init: %z32) {down}")
    if what == "slice of a broadcast":
        one = f"tensor<{Tk}x1xf32>"
        return (f"%smb = stablehlo.broadcast_in_dim %sm, dims = [0] : ({tok}) -> {tk}",
                f"%smw = stablehlo.broadcast_in_dim %sm, dims = [0] : ({tok}) -> {tk}\n"
                f"    %sm1 = stablehlo.slice %smw [0:{Tk}, 1:2] : ({tk}) -> {one}\n"
                f"    %smb = stablehlo.broadcast_in_dim %sm1, dims = [0, 1] : ({one}) -> {tk}")
    return (f"%logits = stablehlo.add %lg, %brb : {te}",
            f"%raised = stablehlo.add %lg, %brb : {te}\n"
            f"    %least = stablehlo.reduce(%raised init: %ninf) applies stablehlo.maximum across dimensions = [1] : ({te}, tensor<f32>) -> {tok}\n"
            f"    %logits = stablehlo.broadcast_in_dim %least, dims = [0] : ({tok}) -> {te}")


@_without_a_gpu
@pytest.mark.parametrize("what", ["sum of a broadcast", "sum of a constant", "slice of a broadcast", "top-k of a broadcast"])
def test_instructions_over_repeated_values(what, monkeypatch):
    E, Tk, H, Ii, K = 4, 3, 32, 32, 2
    old, new = repeated(what, Tk, E, K)
    text = T.moe_block_mxfp4(E, Tk, H, Ii, K)
    assert old in text
    raw, _ = _moe_inputs(E, Tk, H, Ii)
    (g,), (out,), (plain,) = both(text.replace(old, new), [I.from_numpy(a) for a in raw], monkeypatch)
    assert g is not None and g.rows is not None
    np.testing.assert_allclose(out, plain, rtol=2e-5, atol=1e-6 * np.abs(plain).max())


@_without_a_gpu
def test_a_router_that_is_read_elsewhere_stays_with_the_program(monkeypatch):
    """The weights are a result of the program too: the router runs as it did,
    the rest of the dispatch as launches."""
    E, Tk, H, Ii, K = 4, 3, 32, 32, 2
    text = T.moe_block_mxfp4(E, Tk, H, Ii, K)
    text = text.replace(f"return %out : tensor<{Tk}x{H}xf32>", f"return %out, %w : tensor<{Tk}x{H}xf32>, tensor<{Tk}x{K}xf32>")
    text = text.replace(f"-> tensor<{Tk}x{H}xf32> {{\n", f"-> (tensor<{Tk}x{H}xf32>, tensor<{Tk}x{K}xf32>) {{\n", 1)
    raw, _ = _moe_inputs(E, Tk, H, Ii)
    (g,), out, plain = both(text, [I.from_numpy(a) for a in raw], monkeypatch)
    assert g is not None and g.rows is None and not g.skip_keys
    for a, b in zip(out, plain):
        np.testing.assert_allclose(a, b, rtol=2e-5, atol=1e-6)


def test_structs_and_instructions_are_the_headers():
    """Sizes as a C compiler lays them out, and the instruction numbers in the
    header's order."""
    import os
    import re
    text = open(os.path.join(os.path.dirname(_lib.__file__), os.pardir, "include", "qmm_hip.h")).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    names = re.findall(r"QMM_OP_([A-Z0-9]+)", re.search(r"enum \{(\s*QMM_OP_.*?)\};", text, re.S)[1])
    mine = {"subtract": "SUB", "multiply": "MUL", "divide": "DIV", "maximum": "MAX", "minimum": "MIN", "power": "POW",
            "negate": "NEG", "exponential": "EXP", "round_nearest_even": "RINT", "top_k": "TOPK"}
    assert names == [mine.get(n, n.upper()) for n in ML._OPS]
    for name, value in (("MAP_LEAVES", ML.LEAVES), ("MAP_CODE", ML.CODE), ("MAP_REGISTERS", ML.REGISTERS), ("ROW_LEAVES", ML.ROW_LEAVES),
                        ("ROW_CODE", ML.ROW_CODE), ("ROW_OUTS", ML.ROW_OUTS), ("ROW_FLOATS", ML.ROW_FLOATS)):
        assert int(re.search(rf"#define QMM_{name} (\d+)", text)[1]) == value
    assert ctypes.sizeof(ML.MapLeaf) == 48 and ctypes.sizeof(ML.Instruction) == 12 and ctypes.sizeof(ML.RowInstruction) == 44


def test_programs_that_point_outside_their_registers_are_refused():
    lib = _lib.load()
    at = 4096                                           # (never read: the call is refused on the host)
    m = ML.PairMap(y=at, experts_of=at, pairs=2, inner=4, dims=(1, 1, 4), per_token=1, experts=2, rank=1, registers=1)
    for field, value in (("result", 1), ("leaves", ML.LEAVES + 1), ("instructions", ML.CODE + 1), ("inner", 5), ("per_token", 0),
                         ("y_el", 3), ("experts", 0)):
        bad = ML._copy(m)
        setattr(bad, field, value)
        assert lib.qmm_pair_map_run(ctypes.byref(bad), None) == 1, field
    bad = ML._copy(m)
    bad.instructions, bad.code[0] = 1, ML.Instruction(ML.OP["add"], 0, 0, 1, 0, 0, 0.0)
    assert lib.qmm_pair_map_run(ctypes.byref(bad), None) == 1
    r = ML.RowProgram(tokens=1, reg_floats=8, instructions=1)
    for q in ((ML.OP["add"], 0, 6, 4, 0, 4, 0, 4, 0, 4, 0.0), (ML.OP["top_k"], 0, 0, 3, 4, 2, 0, 1, 6, 2, 0.0),
              (ML.OP["slice"], 0, 0, 4, 4, 4, 1, 0, 1, 0, 0.0)):
        r.code[0] = ML.RowInstruction(*q)
        assert lib.qmm_row_program_run(ctypes.byref(r), None) == 1, q


def test_a_map_that_leaves_a_product_no_local_memory_is_two_launches():
    """Eight wavefronts' sums of two columns in three terms are 48 KB; a file of 32
    registers besides is more than a launch gets.  Decided on the host, no GPU needed."""
    at = 4096
    m = ML.PairMap(y=at, experts_of=at, pairs=2, inner=16, dims=(1, 1, 16), per_token=1, experts=2, rank=1, registers=ML.REGISTERS, leaves=2)
    p = ML.PairProduct(x=at, w=at, s=at, x_rows=2, n=32, k=2080, mode=_lib.MODE_MXFP4, x_per=1, tiles=2, col_leaf=(0, 1), col_base=(0, 16),
                       col_step=(1, 1), map=m)
    assert _lib.load().qmm_pair_product_run(ctypes.byref(p), None) == 3
    assert b"two launches" in _lib.load().qmm_last_error()


@pytest.mark.parametrize("pairs,inner", [(0, 4), (3, 0)])
def test_a_call_without_pairs_or_elements_launches_nothing(pairs, inner):
    """An array without elements has no address: every step of such a call is taken, not refused."""
    m = ML.PairMap(per_token=1, experts=2, rank=1, pairs=pairs, inner=inner, registers=1)
    p = ML.PairProduct(n=16, k=32, mode=_lib.MODE_MXFP4, x_per=1, tiles=1, map=m)
    lib = _lib.load()
    assert lib.qmm_pair_map_run(ctypes.byref(m), None) == 0
    assert lib.qmm_pair_product_run(ctypes.byref(p), None) == 0
