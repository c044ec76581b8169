"""The quantized-matmul work that a user of this framework times: one pass per
case through the public entry points.

    listed()             the named cases
    draw(rng)            one more case of the same ranges
    prepare(case, seed)  inputs and handles on the GPU
    run(state)           one pass, its outputs
    work(case)           the bytes and operations one pass cannot do without
    tolerance(case)      how far another correct implementation may be off

Kinds of case:

    dense      `kernels.quantized_matmul`: x [m, k] against a packed [n, k]
    bound      the same product as a kept handle (`kernels.BoundQmm`), as a
               decode loop launches it
    gather     `kernels.gather_qmm`: every token against its top-k experts, pairs
               in token order
    grouped    `kernels.grouped_qmm`: the same rows already sorted by expert
    engine     `engine.execute` on a StableHLO program whose one dot the
               recognizer fuses (codes, scales and zero points as a checkpoint
               holds them)
    moe_block  `engine.execute` on a whole top-k expert block with MXFP4 experts
"""

import math

import numpy as np
import torch

from metaljax_amd import engine, kernels, synth
from metaljax_amd.packing import f32_to_bf16_bits

TORCH = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}
SIZE = {"bf16": 2, "f16": 2, "f32": 4}
MOST_FLOPS = 2 * 1024 * 14336 * 4096        # the largest listed case
MOST_CODES = 8 * 14336 * 4096


def _dense(kind, m, n, k, bits=4, group=64, mode="affine", tables="bf16", act="bf16"):
    return {"kind": kind, "m": m, "n": n, "k": k, "bits": bits, "group": group, "mode": mode,
            "tables": tables, "act": act}


def _routed(kind, tokens, experts, topk, n, k, bits=4, group=64, mode="affine", act="bf16"):
    return {"kind": kind, "tokens": tokens, "experts": experts, "topk": topk, "n": n, "k": k, "bits": bits,
            "group": group, "mode": mode, "tables": "bf16", "act": act}


def _block(tokens, experts, topk, hidden, inner):
    return {"kind": "moe_block", "tokens": tokens, "experts": experts, "topk": topk, "hidden": hidden, "inner": inner}


def listed():
    def named(name, case):
        return dict(case, name=name)
    return [
        # one token through an attention projection, launched from a kept handle: the smallest call
        named("decode_m1_4096x4096", _dense("bound", 1, 4096, 4096)),
        # sixteen sequences decoding through the widest projection of an 8B model (bench.py's headline)
        named("decode_m16_14336x4096", _dense("dense", 16, 14336, 4096)),
        # a 7B model's down projection: the contraction is no whole number of 256-byte pieces
        named("decode_m5_4096x11008", _dense("dense", 5, 4096, 11008)),
        # a serving batch, past what the decode kernels take in one product
        named("batch_m48_4096x14336", _dense("dense", 48, 4096, 14336)),
        # a short prompt of a float16 checkpoint: activations, tables and results in float16
        named("prompt_f16_m77_4096x4096", _dense("dense", 77, 4096, 4096, group=128, tables="f16", act="f16")),
        # an ordinary prompt of odd length, groups of 32
        named("prompt_m333_9216x3072_g32", _dense("dense", 333, 9216, 3072, group=32)),
        # a long prompt against eight-bit codes
        named("prefill_m2048_4096x4096_int8", _dense("dense", 2048, 4096, 4096, bits=8)),
        # MXFP4 prefill
        named("prefill_m256_8192x8192_mxfp4", _dense("dense", 256, 8192, 8192, group=32, mode="mxfp4")),
        # 512 tokens, two of eight experts each, rows sorted by expert: the largest
        named("grouped_512tok_8x14336x4096", _routed("grouped", 512, 8, 2, 14336, 4096)),
        # a few sequences decoding through gpt-oss's gate/up projection (K = 2880, top-4 of 32 experts)
        named("gather_4tok_32x5760x2880_mxfp4", _routed("gather", 4, 32, 4, 5760, 2880, group=32, mode="mxfp4")),
        # a recognized program, a few rows: what the interpreter and the call cost on top of the product
        named("engine_m4_4096x4096", dict(_dense("engine", 4, 4096, 4096))),
        # a recognized top-2 expert block with MXFP4 experts, a few tokens
        named("engine_moe_3tok_8x1024x1024", _block(3, 8, 2, 1024, 1024)),
    ]


def _log(rng, lo, hi, step=1):
    """An integer between lo and hi, spread evenly over the logarithm, a multiple of `step`."""
    v = math.exp(rng.uniform(math.log(lo), math.log(hi + 1)))
    return max(-(-lo // step) * step, int(v) // step * step)


def draw(rng):
    kind = rng.choice(["decode", "decode", "batch", "prompt", "prefill", "gather", "grouped", "engine", "moe_block"])
    if kind == "moe_block":
        experts = rng.choice([4, 8, 16])
        hidden, inner = _log(rng, 256, 1536, 32), _log(rng, 256, 1536, 32)
        while experts * hidden * inner > 8 * 1024 * 1024:
            inner = max(32, inner // 2 // 32 * 32)
        return _block(_log(rng, 1, 64), experts, rng.choice([1, 2, 4]), hidden, inner)
    if kind == "engine":
        return _dense("engine", _log(rng, 1, 64), _log(rng, 512, 4096, 8), _log(rng, 512, 4096, 64))
    mode = rng.choice(["affine", "affine", "affine", "mxfp4"])
    bits = 4 if mode == "mxfp4" else rng.choice([4, 4, 8])
    group = 32 if mode == "mxfp4" else rng.choice([32, 64, 64, 128])
    if kind in ("gather", "grouped"):
        experts, topk = rng.choice([8, 16, 32]), rng.choice([1, 2, 4])
        n, k = _log(rng, 1024, 8192, 8), _log(rng, 1024, 4096, max(64, group))
        while experts * n * k > MOST_CODES:
            n = n // 2 // 8 * 8
        tokens = _log(rng, 1, 512) if kind == "gather" else _log(rng, 32, 512)
        return _routed(kind, tokens, experts, topk, n, k, bits=bits, group=group, mode=mode)
    lo, hi = {"decode": (1, 16), "batch": (17, 128), "prompt": (64, 512), "prefill": (512, 2048)}[kind]
    m, n, k = _log(rng, lo, hi), _log(rng, 1024, 16384, 8), _log(rng, 1024, 14336, max(64, group))
    while 2 * m * n * k > MOST_FLOPS:
        n = n // 2 // 8 * 8
    act = rng.choice(["bf16", "bf16", "bf16", "f16", "f32"]) if kind in ("batch", "prompt") else "bf16"
    tables = "f16" if act == "f16" and mode == "affine" else "bf16"
    return _dense(rng.choice(["dense", "bound"]), m, n, k, bits=bits, group=group, mode=mode, tables=tables, act=act)


def _activations(shape, act, g):
    return torch.randn(shape, device="cuda", generator=g).to(TORCH[act])


def _weight(lead, case, g):
    """A packed weight with its tables: uniform codes; affine: one scale and one zero point a group;
    MXFP4: block exponents around one."""
    n, k, bits = case["n"], case["k"], case["bits"]
    w = torch.randint(-2**31, 2**31, lead + (n, k * bits // 32), dtype=torch.int64, device="cuda",
                      generator=g).to(torch.int32)
    groups = lead + (n, k // case["group"])
    if case["mode"] == "mxfp4":
        return w, torch.randint(118, 128, groups, dtype=torch.uint8, device="cuda", generator=g), None
    top = 0.02 if bits == 4 else 0.002
    s = (torch.rand(groups, device="cuda", generator=g) * 0.75 * top + 0.25 * top).to(TORCH[case["tables"]])
    zero = torch.randint(6, 11, groups, device="cuda", generator=g) * (1 if bits == 4 else 16)
    return w, s, (-zero * s.float()).to(TORCH[case["tables"]])


def _routing(case, g):
    """The experts of every token, [tokens, topk] int32."""
    logits = torch.randn((case["tokens"], case["experts"]), device="cuda", generator=g)
    return torch.topk(logits, case["topk"], dim=-1).indices.to(torch.int32)


def prepare(case, seed):
    kind = case["kind"]
    if kind == "engine":
        return _prepare_engine(case, seed)
    if kind == "moe_block":
        return _prepare_block(case, seed)
    g = torch.Generator(device="cuda").manual_seed(seed)
    how = {"group_size": case["group"], "bits": case["bits"], "mode": case["mode"]}
    if kind in ("dense", "bound"):
        x = _activations((case["m"], case["k"]), case["act"], g)
        w, s, b = _weight((), case, g)
        if kind == "bound":
            y = torch.empty((case["m"], case["n"]), dtype=x.dtype, device="cuda")
            return kernels.BoundQmm(x, w, s, b, y, **how).launch
        return lambda: kernels.quantized_matmul(x, w, s, b, **how)
    x = _activations((case["tokens"], case["k"]), case["act"], g)
    w, s, b = _weight((case["experts"],), case, g)
    experts = _routing(case, g)
    if kind == "gather":
        rhs = experts.reshape(-1).contiguous()
        lhs = torch.arange(case["tokens"], device="cuda", dtype=torch.int32).repeat_interleave(case["topk"]).contiguous()
        return lambda: kernels.gather_qmm(x, w, s, b, lhs, rhs, **how)
    order = torch.argsort(experts.reshape(-1), stable=True)
    rows = x[order // case["topk"]].contiguous()
    ends = torch.bincount(experts.reshape(-1), minlength=case["experts"]).cumsum(0)
    offsets = torch.cat([ends.new_zeros(1), ends]).to(torch.int32)
    return lambda: kernels.grouped_qmm(rows, w, s, b, offsets, **how)


def _buffers(pairs):
    return [engine.buffer_from_host(a, engine.PJRT_TYPES.index(el), a.shape) for a, el in pairs]


def _executable(text, buffers):
    """The compiled program; its first execution packs the weights of these buffers."""
    ex = engine.compile_program(text, "mlir")
    engine.execute(ex, buffers)
    return lambda: [out.data for out in engine.execute(ex, buffers)]


def _prepare_engine(case, seed):
    m, n, k, groups = case["m"], case["n"], case["k"], (case["n"], case["k"] // case["group"])
    rng = np.random.default_rng(seed)
    q = rng.integers(-8, 8, (n, k), dtype=np.int8)
    s = f32_to_bf16_bits(rng.uniform(0.005, 0.02, groups).astype(np.float32))
    z = rng.integers(-2, 3, groups, dtype=np.int8)
    x = f32_to_bf16_bits(rng.standard_normal((m, k), dtype=np.float32))
    return _executable(synth.affine_program_text(m, n, k, case["group"]),
                       _buffers([(q, "S8"), (s, "BF16"), (z, "S8"), (x, "BF16")]))


def _prepare_block(case, seed):
    e, t, h, i = case["experts"], case["tokens"], case["hidden"], case["inner"]
    rng = np.random.default_rng(seed)

    def floats(*shape):
        return rng.standard_normal(shape, dtype=np.float32) / 8, "F32"

    def codes(rows, k):
        return rng.integers(0, 256, (e, rows, k // 2), dtype=np.uint8), "U8"

    def scales(rows, k):
        return rng.integers(120, 128, (e, rows, k // 32), dtype=np.uint8), "U8"
    buffers = _buffers([floats(t, h), floats(h, e), floats(e), codes(2 * i, h), scales(2 * i, h), codes(h, i),
                        scales(h, i), floats(e, 2 * i), floats(e, h)])
    return _executable(_block_text(e, t, h, i, case["topk"]), buffers)


def _mxfp4_text(v, e, n, k):
    """Lines that rebuild %<v> [e, n, k] float32 from %<v>c (two E2M1 codes a byte) and %<v>s (E8M0 bytes)."""
    e2m1 = ", ".join(f"{sign * m:.6e}" for sign in (1, -1) for m in (0.0, 0.5, 1.0, 1.5, 2.0, 3.0, 4.0, 6.0))
    with np.errstate(over="ignore"):
        powers = np.ldexp(np.ones(256), np.arange(256) - 127).astype(np.float32)
    powers[255] = np.nan
    half, one, flat = f"tensor<{e}x{n}x{k // 2}xui8>", f"tensor<{e}x{n}x{k // 2}x1xui8>", e * n * k
    blocks, nb = f"tensor<{e}x{n}x{k // 32}x32xf32>", e * n * k // 32
    table = ("<{{dimension_numbers = #stablehlo.gather<collapsed_slice_dims = [0], start_index_map = [0], "
             "index_vector_dim = 1>, slice_sizes = array<i64: 1>}}> : (tensor<{0}xf32>, tensor<{1}x1xi32>) -> tensor<{1}xf32>")
    return f"""
    %{v}grid = stablehlo.constant dense<[{e2m1}]> : tensor<16xf32>
    %{v}pow = stablehlo.constant dense<"0x{powers.tobytes().hex().upper()}"> : tensor<256xf32>
    %{v}k15 = stablehlo.constant dense<15> : tensor<ui8>
    %{v}k4 = stablehlo.constant dense<4> : tensor<ui8>
    %{v}m15 = stablehlo.broadcast_in_dim %{v}k15, dims = [] : (tensor<ui8>) -> {half}
    %{v}m4 = stablehlo.broadcast_in_dim %{v}k4, dims = [] : (tensor<ui8>) -> {half}
    %{v}lo = stablehlo.and %{v}c, %{v}m15 : {half}
    %{v}hi = stablehlo.shift_right_logical %{v}c, %{v}m4 : {half}
    %{v}lo1 = stablehlo.reshape %{v}lo : ({half}) -> {one}
    %{v}hi1 = stablehlo.reshape %{v}hi : ({half}) -> {one}
    %{v}pair = stablehlo.concatenate %{v}lo1, %{v}hi1, dim = 3 : ({one}, {one}) -> tensor<{e}x{n}x{k // 2}x2xui8>
    %{v}nib = stablehlo.reshape %{v}pair : (tensor<{e}x{n}x{k // 2}x2xui8>) -> tensor<{flat}x1xui8>
    %{v}idx = stablehlo.convert %{v}nib : (tensor<{flat}x1xui8>) -> tensor<{flat}x1xi32>
    %{v}val = "stablehlo.gather"(%{v}grid, %{v}idx) {table.format(16, flat)}
    %{v}sb = stablehlo.reshape %{v}s : (tensor<{e}x{n}x{k // 32}xui8>) -> tensor<{nb}x1xui8>
    %{v}si = stablehlo.convert %{v}sb : (tensor<{nb}x1xui8>) -> tensor<{nb}x1xi32>
    %{v}sv = "stablehlo.gather"(%{v}pow, %{v}si) {table.format(256, nb)}
    %{v}s3 = stablehlo.reshape %{v}sv : (tensor<{nb}xf32>) -> tensor<{e}x{n}x{k // 32}xf32>
    %{v}s4 = stablehlo.broadcast_in_dim %{v}s3, dims = [0, 1, 2] : (tensor<{e}x{n}x{k // 32}xf32>) -> {blocks}
    %{v}v4 = stablehlo.reshape %{v}val : (tensor<{flat}xf32>) -> {blocks}
    %{v}w4 = stablehlo.multiply %{v}v4, %{v}s4 : {blocks}
    %{v} = stablehlo.reshape %{v}w4 : ({blocks}) -> tensor<{e}x{n}x{k}xf32>"""


def _block_text(e, t, h, i, topk):
    """out = sum_e S[:, e] * (silu(g) * u . Wd[e]^T + bd[e]) with g, u the even and odd columns of
    x . Wgu[e]^T + bgu[e] and S the softmax over each token's top-k logits, zero elsewhere."""
    def f(*shape, el="f32"):
        return "tensor<" + "x".join([*map(str, shape), el]) + ">"
    th, te, tk, tke, etm, eti, eth = f(t, h), f(t, e), f(t, topk), f(t, topk, e), f(e, t, 2 * i), f(e, t, i), f(e, t, h)
    return f"""
module @jit_expert_block {{
  func.func public @main(%x: {th}, %wr: {f(h, e)}, %br: {f(e)}, %guc: {f(e, 2 * i, h // 2, el="ui8")}, %gus: {f(e, 2 * i, h // 32, el="ui8")}, %dnc: {f(e, h, i // 2, el="ui8")}, %dns: {f(e, h, i // 32, el="ui8")}, %bgu: {f(e, 2 * i)}, %bd: {f(e, h)}) -> {th} {{{_mxfp4_text("gu", e, 2 * i, h)}{_mxfp4_text("dn", e, h, i)}
    %zero = stablehlo.constant dense<0.000000e+00> : tensor<f32>
    %ninf = stablehlo.constant dense<0xFF800000> : tensor<f32>
    %p0 = stablehlo.dot_general %x, %gu, contracting_dims = [1] x [2] : ({th}, {f(e, 2 * i, h)}) -> {f(t, e, 2 * i)}
    %p1 = stablehlo.transpose %p0, dims = [1, 0, 2] : ({f(t, e, 2 * i)}) -> {etm}
    %bgub = stablehlo.broadcast_in_dim %bgu, dims = [0, 2] : ({f(e, 2 * i)}) -> {etm}
    %p = stablehlo.add %p1, %bgub : {etm}
    %g = stablehlo.slice %p [0:{e}, 0:{t}, 0:{2 * i}:2] : ({etm}) -> {eti}
    %u = stablehlo.slice %p [0:{e}, 0:{t}, 1:{2 * i}:2] : ({etm}) -> {eti}
    %sg = stablehlo.logistic %g : {eti}
    %silu = stablehlo.multiply %g, %sg : {eti}
    %act = stablehlo.multiply %silu, %u : {eti}
    %y0 = stablehlo.dot_general %act, %dn, batching_dims = [0] x [0], contracting_dims = [2] x [2] : ({eti}, {f(e, h, i)}) -> {eth}
    %bdb = stablehlo.broadcast_in_dim %bd, dims = [0, 2] : ({f(e, h)}) -> {eth}
    %y = stablehlo.add %y0, %bdb : {eth}
    %lg = stablehlo.dot_general %x, %wr, contracting_dims = [1] x [0] : ({th}, {f(h, e)}) -> {te}
    %brb = stablehlo.broadcast_in_dim %br, dims = [1] : ({f(e)}) -> {te}
    %logits = stablehlo.add %lg, %brb : {te}
    %vals, %idx = chlo.top_k(%logits, k = {topk}) : {te} -> ({tk}, {f(t, topk, el="i32")})
    %mx = stablehlo.reduce(%vals init: %ninf) applies stablehlo.maximum across dimensions = [1] : ({tk}, tensor<f32>) -> {f(t)}
    %mxb = stablehlo.broadcast_in_dim %mx, dims = [0] : ({f(t)}) -> {tk}
    %sh = stablehlo.subtract %vals, %mxb : {tk}
    %ex = stablehlo.exponential %sh : {tk}
    %sm = stablehlo.reduce(%ex init: %zero) applies stablehlo.add across dimensions = [1] : ({tk}, tensor<f32>) -> {f(t)}
    %smb = stablehlo.broadcast_in_dim %sm, dims = [0] : ({f(t)}) -> {tk}
    %w = stablehlo.divide %ex, %smb : {tk}
    %idxb = stablehlo.broadcast_in_dim %idx, dims = [0, 1] : ({f(t, topk, el="i32")}) -> {f(t, topk, e, el="i32")}
    %io = stablehlo.iota dim = 2 : {f(t, topk, e, el="i32")}
    %eq = stablehlo.compare EQ, %idxb, %io, SIGNED : ({f(t, topk, e, el="i32")}, {f(t, topk, e, el="i32")}) -> {f(t, topk, e, el="i1")}
    %hot = stablehlo.convert %eq : ({f(t, topk, e, el="i1")}) -> {tke}
    %wb = stablehlo.broadcast_in_dim %w, dims = [0, 1] : ({tk}) -> {tke}
    %hw = stablehlo.multiply %hot, %wb : {tke}
    %s = stablehlo.reduce(%hw init: %zero) applies stablehlo.add across dimensions = [1] : ({tke}, tensor<f32>) -> {te}
    %st = stablehlo.transpose %s, dims = [1, 0] : ({te}) -> {f(e, t)}
    %sbc = stablehlo.broadcast_in_dim %st, dims = [0, 1] : ({f(e, t)}) -> {eth}
    %ys = stablehlo.multiply %y, %sbc : {eth}
    %out = stablehlo.reduce(%ys init: %zero) applies stablehlo.add across dimensions = [0] : ({eth}, tensor<f32>) -> {th}
    return %out : {th}
  }}
}}
"""


def run(state):
    return state()


def _touched(case):
    """How many experts the tokens' independent choices reach, on average."""
    e = case["experts"]
    return e * (1.0 - (1.0 - case["topk"] / e) ** case["tokens"])


def work(case):
    if case["kind"] == "moe_block":
        t, e, h, i = case["tokens"], case["experts"], case["hidden"], case["inner"]
        codes = 3 * h * i                                   # of one expert: gate, up and down
        expert = codes / 2 + codes / 32 + (2 * i + h) * 4   # codes, scales, biases
        return {"bytes": _touched(case) * expert + (2 * t * h + h * e + e) * 4,
                "flops": 2 * t * (case["topk"] * codes + h * e)}
    n, k, act = case["n"], case["k"], SIZE[case["act"]]
    weight = n * k * case["bits"] / 8
    weight += n * (k // case["group"]) * (1 if case["mode"] == "mxfp4" else 2 * SIZE[case["tables"]])
    if case["kind"] in ("gather", "grouped"):
        pairs = case["tokens"] * case["topk"]
        rows = pairs if case["kind"] == "grouped" else case["tokens"]
        return {"bytes": _touched(case) * weight + (rows * k + pairs * n) * act, "flops": 2 * pairs * n * k}
    return {"bytes": weight + case["m"] * (k + n) * act, "flops": 2 * case["m"] * n * k}


def tolerance(case):
    if case["kind"] == "moe_block":
        return {"rel": 3e-5}                    # exact weights, float32 sums, two products deep
    # bf16 results: one rounding of float32 sums; above the decode sizes affine weights are rounded to a
    # bf16 tile besides, and bf16 activations of MXFP4 products may pass through a narrower split
    if case["act"] == "bf16":
        return {"rel": 6e-3}
    if case["mode"] == "mxfp4":
        return {"rel": 1e-3 if case["act"] == "f16" else 1e-5}
    return {"rel": 4e-3}                        # the bf16 tile again
