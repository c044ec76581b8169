"""A planned expert dispatch as a handful of launches.

`moe.PairPlan` proves that a dense expert block can run over the selected pairs
and runs it as a list of array operations.  Each of those is a launch and its
host work, and the router ahead of them runs on the host.  Where a GPU is
visible the same plan is compiled once more, into

  * one row program: the router from its logits (product included) to the
    experts of every token and their weights,
  * one pair map ahead of every product that does not read the tokens' rows as
    they are, and one behind the last that ends in the routing-weighted sum,
  * the expert-indexed products themselves (reference src/metaljax/moe.py:335-442
    and :1425-1461 are what these launches stand for).

A pair map computes an output element from the elements of its inputs that the
program's slices, broadcasts, transposes and elementwise operations lead to:
`_Map.pull` follows a value down to what is in memory with the output's
coordinates as affine index expressions.  A row program keeps a token's values as
rows of registers: `_Rows.lower`.

Whatever is not modelled raises Reject while compiling, and the dispatch runs as
its array operations (or the router on the host) as before.
"""

from __future__ import annotations

import ctypes

import numpy as np

from . import _lib, ir
from .interpreter import REGISTRY, host
from .packing import Reject
from .recognize import count, dims_of, elem, op_key

ELS = {"f32": 0, "bf16": 1, "f16": 2, "i1": 3, "i32": 4}           # QMM_EL_*
FLOATS = ("f32", "bf16", "f16")
SIZE = {"f32": 4, "bf16": 2, "f16": 2, "i32": 4}
_DT = {"f32": _lib.F32, "bf16": _lib.BF16, "f16": _lib.F16}
_OPS = ("copy add subtract multiply divide maximum minimum power abs negate exponential log logistic tanh sqrt rsqrt "
        "ceil floor round_nearest_even sign EQ NE LT LE GT GE and or xor not select clamp imm sum rowmax rowmin slice "
        "top_k").split()
OP = {name: i for i, name in enumerate(_OPS)}                      # QMM_OP_*, in the header's order
LEAVES, CODE, REGISTERS = 8, 40, 32                                # QMM_MAP_*
ROW_LEAVES, ROW_CODE, ROW_OUTS, ROW_FLOATS = 8, 48, 2, 8192        # QMM_ROW_*
MAX_ROW = 256                   # elements of a row register: a top-k counts, for each, those ahead of it
MAX_DEPTH = 2 * ROW_CODE        # operations followed up from a value (the recursion's depth): shape ops have no instruction
# Products up to this many multiplications ride in the row program, whose workgroups (one a token) each read the
# whole router weight; larger ones stay a library product.
MAX_ROUTER_MACS = 1 << 23

_i32, _i64, _vp, _u8 = ctypes.c_int32, ctypes.c_int64, ctypes.c_void_p, ctypes.c_uint8


class MapLeaf(ctypes.Structure):
    _fields_ = [("p", _vp), ("base", _i64), ("pair", _i32), ("expert", _i32), ("token", _i32), ("coef", _i32 * 3),
                ("el", _i32)]


class Instruction(ctypes.Structure):
    _fields_ = [(n, _u8) for n in ("op", "dst", "a", "b", "c", "el")] + [("imm", ctypes.c_float)]


class PairMap(ctypes.Structure):
    _fields_ = [("y", _vp), ("weights", _vp), ("experts_of", _vp), ("pairs", _i64), ("inner", _i64), ("dims", _i64 * 3)] + \
               [(n, _i32) for n in ("per_token", "experts", "rank", "y_el", "sum_el", "weights_el", "leaves",
                                    "instructions", "registers", "result")] + \
               [("leaf", MapLeaf * LEAVES), ("code", Instruction * CODE)]


class PairProduct(ctypes.Structure):
    _fields_ = [(n, _vp) for n in ("x", "w", "s")] + [(n, _i64) for n in ("x_rows", "n", "k", "mode")] + \
               [(n, _i32) for n in ("x_el", "x_per", "product_el", "tiles")] + \
               [(n, _i32 * 2) for n in ("col_leaf", "col_base", "col_step")] + [("sorted", _i32), ("map", PairMap)]


class PairGather(ctypes.Structure):
    _fields_ = [(n, _vp) for n in ("x", "w", "scales", "biases", "y", "lhs_idx", "rhs_idx", "workspace")] + \
               [(n, _i64) for n in ("workspace_bytes", "table_dtype", "group_size", "bits", "mode", "pairs", "rows", "experts", "n", "k")] + \
               [(n, _i32) for n in ("x_dtype", "y_dtype")]


class Patch(ctypes.Structure):
    _fields_ = [("at", _i32), ("value", _i32), ("add", _i64)]


class Step(ctypes.Structure):
    _fields_ = [(n, _i32) for n in ("kind", "bytes", "patches", "skip")] + [("program", _vp), ("patch", ctypes.POINTER(Patch))]


class RowInstruction(ctypes.Structure):
    _fields_ = [(n, _i32) for n in ("op", "el", "dst", "n", "a", "an", "b", "bn", "c", "cn")] + [("imm", ctypes.c_float)]


class RowLeaf(ctypes.Structure):
    _fields_ = [("p", _vp), ("base", _i64), ("token", _i64), ("step", _i64), ("el", _i32), ("dst", _i32), ("n", _i32)]


class RowOut(ctypes.Structure):
    _fields_ = [("p", _vp), ("el", _i32), ("src", _i32), ("srcn", _i32), ("n", _i32)]


class RowProgram(ctypes.Structure):
    _fields_ = [("dot_x", _vp), ("dot_w", _vp)] + [(n, _i64) for n in ("dot_x_t", "dot_x_k", "dot_w_n", "dot_w_k", "dot_k")] + \
               [(n, _i32) for n in ("dot_n", "dot_cols", "dot_dst", "dot_x_el", "dot_w_el", "dot_el", "tokens",
                                    "reg_floats", "leaves", "instructions", "outs")] + \
               [("leaf", RowLeaf * ROW_LEAVES), ("out", RowOut * ROW_OUTS), ("code", RowInstruction * ROW_CODE)]


def _copy(struct):
    """A call's own program: the pointers of one call are nobody else's."""
    return type(struct).from_buffer_copy(struct)


def run_map(program, stream):
    rc = _lib.load().qmm_pair_map_run(ctypes.byref(program), stream)
    if rc:
        _lib.check(rc)


STEPS = ROWS, PRODUCT, MAP, GATHER = range(4)                      # QMM_STEP_*


def run_steps(steps, values, stream):
    rc = _lib.load().qmm_steps_run(steps, len(steps), (ctypes.c_uint64 * len(values))(*values), len(values), stream)
    if rc:
        _lib.check(rc)


def run_product(x, el, rows, arrays, match, lhs, rhs, y, y_el, pairs, experts, n, k, like, stream):
    """y [pairs, n] = row lhs[p] of x [rows, k] (row p without lhs) times expert
    rhs[p] of a match's packed weight; x, lhs, rhs and y are addresses.  `like`: a
    tensor of the device."""
    from . import kernels
    lib = _lib.load()
    affine = match.mode == "affine"
    arrays = [a if a.is_contiguous() else a.contiguous() for a in arrays[:3 if affine else 2]]
    nbytes = kernels._gather_workspace_bytes(pairs, experts, n, k, _DT[el])
    ws = kernels._scratch(nbytes, like, stream)
    rc = lib.qmm_gather_qmm(x, _DT[el], arrays[0].data_ptr(), arrays[1].data_ptr(), arrays[2].data_ptr() if affine else None,
                            kernels._dt(arrays[1].dtype) if affine else _lib.BF16, y, _DT[y_el], lhs, rhs, pairs, rows, experts,
                            n, k, match.gs, match.bits, kernels._MODE[match.mode], None if ws is None else ws.data_ptr(), nbytes, stream)
    if rc:
        _lib.check(rc)


def run_rows(program, stream):
    rc = _lib.load().qmm_row_program_run(ctypes.byref(program), stream)
    if rc:
        _lib.check(rc)


def available() -> bool:
    """Do dispatches run on a GPU here?"""
    from . import qmm
    if qmm.DEVICE != "cuda":
        return False
    try:
        import torch
        return torch.cuda.is_available()
    except ImportError:
        return False


def _constant(interp, v):
    """The value of a constant, None for anything else."""
    op = None if v.is_block_arg else v.op
    if op is None or op.name != "stablehlo.constant":
        return None
    out = REGISTRY[op.name](interp, op, [], {})
    return host(out[0] if isinstance(out, (list, tuple)) else out)


def _splat(interp, v):
    """The one value of a constant, as a float; None for anything else."""
    h = _constant(interp, v)
    if h is None or h.el not in FLOATS + ("i1",) or not h.a.size:
        return None
    first = h.a.reshape(-1)[0]
    return float(first) if (h.a == first).all() or h.a.size == 1 else None


def _elementwise(op):
    """(instruction, operands) of an elementwise op whose types the programs model."""
    name = op.name[len("stablehlo."):]
    out, ins = elem(op.results[0]), [elem(x) for x in op.operands]
    if name == "compare":
        if not all(e in FLOATS for e in ins):
            raise Reject("a comparison of other than floats")
        return OP[op.attrs["comparison_direction"]], list(op.operands)
    if name in ("and", "or", "xor", "not"):
        if out != "i1":
            raise Reject(f"{name} of integers")
        return OP[name], list(op.operands)
    if name == "select":
        if ins[0] != "i1" or not all(e in FLOATS + ("i1",) for e in ins[1:]):
            raise Reject("a select of other than floats")
        return OP[name], list(op.operands)
    if name == "convert":
        if out not in FLOATS or ins[0] not in FLOATS + ("i1",):
            raise Reject(f"a conversion from {ins[0]} to {out}")
        return OP["copy"], list(op.operands)
    if name not in OP or name in ("copy", "imm", "sum", "rowmax", "rowmin", "slice", "top_k"):
        raise Reject(f"{op.name} is not modelled")
    if out not in FLOATS or not all(e in FLOATS for e in ins):
        raise Reject(f"{op.name} of other than floats")
    return OP[name], list(op.operands)


def _round_el(op):
    el = elem(op.results[0])
    return ELS[el] if el in FLOATS else ELS["f32"]


# ------------------------------------------------------------- pair maps ----

class _Map:
    """One pair map under construction.  An index expression is (constant, c0,
    c1, c2): an affine function of the output's up to three coordinates."""

    def __init__(self, owner, dims, per_token):
        if len(dims) > 3:
            raise Reject("a result of more than three axes a pair")
        self.owner = owner
        self.dims = [1] * (3 - len(dims)) + list(dims)
        self.rank = max(1, len(dims))
        self.leaves = []                 # (source, MapLeaf without its pointer)
        self.code = []                   # (op, operands, round, imm); operand ("leaf", i) or ("code", i)
        self.memo = {}
        self.per_token = per_token

    def coordinate(self, j):
        """The output's axis j as an index expression."""
        at = 3 - self.rank + j
        return (0,) + tuple(1 if i == at else 0 for i in range(3))

    @staticmethod
    def _combine(terms):
        """sum of stride * expression"""
        total = [0, 0, 0, 0]
        for stride, e in terms:
            for i in range(4):
                total[i] += stride * e[i]
        return tuple(total)

    def _leaf(self, source, el, flat, pair=0, expert=0, token=0):
        if el not in ELS or el == "i32":
            raise Reject(f"an input of {el}")
        if any(abs(c) > 0x7FFFFFFF for c in (pair, expert, token) + flat[1:]):
            raise Reject("an input's strides")
        leaf = MapLeaf(None, flat[0], pair, expert, token, (_i32 * 3)(*flat[1:]), ELS[el])
        if len(self.leaves) == LEAVES:
            raise Reject("more inputs than a pair map takes")
        self.leaves.append((source, leaf))
        return "leaf", len(self.leaves) - 1

    def _emit(self, op, operands, rnd, imm=0.0):
        if len(self.code) == CODE:
            raise Reject("a longer program than a pair map takes")
        self.code.append((op, list(operands), rnd, imm))
        return "code", len(self.code) - 1

    def pull(self, v, e, t, index):
        """The element of `v` at the pair's expert (axis `e`) and token (axis
        `t`; None: no such axis) and at `index` on its other axes."""
        at = (v, e, t, tuple(index))
        if at not in self.memo:
            self.memo[at] = self._pull(v, e, t, list(index))
        return self.memo[at]

    def _external(self, v, e, t, index):
        shape = dims_of(v)
        const = _splat(self.owner.interp, v)
        if const is not None:
            return self._emit(OP["imm"], [], ELS["f32"], const)
        if _constant(self.owner.interp, v) is not None:
            raise Reject("a constant that is not one value")
        strides = [1] * len(shape)
        for i in range(len(shape) - 2, -1, -1):
            strides[i] = strides[i + 1] * shape[i + 1]
        flat = self._combine((s, ix) for i, (s, ix) in enumerate(zip(strides, index)) if i not in (e, t))
        self.owner.reads.append(v)
        return self._leaf(("env", v), elem(v), flat, expert=strides[e] if e is not None else 0,
                          token=strides[t] if t is not None else 0)

    def _pull(self, v, e, t, index):
        op = None if v.is_block_arg else v.op
        if op is None or e is None:
            return self._external(v, e, t, index)
        name, shape = op.name, dims_of(v)
        if name == "stablehlo.dot_general":
            return self._dot(v, op, e, t, index)
        if name == "stablehlo.broadcast_in_dim":
            src = op.operands[0]
            sshape, placement = dims_of(src), ir.i64_list(op, "broadcast_dimensions")
            se = st = None
            inner = [(0, 0, 0, 0)] * len(sshape)
            for j, d in enumerate(placement):
                if sshape[j] == 1:
                    continue
                if d == e:
                    se = j
                elif d == t:
                    st = j
                else:
                    inner[j] = index[d]
            return self.pull(src, se, st, inner)
        if name == "stablehlo.transpose":
            perm = ir.i64_list(op, "permutation")
            inner = [None] * len(perm)
            for i, p in enumerate(perm):
                inner[p] = index[i]
            return self.pull(op.operands[0], perm[e], perm[t] if t is not None else None, inner)
        if name == "stablehlo.slice":
            b, s = op.attrs["start_indices"], op.attrs["strides"]
            inner = [None if i in (e, t) else self._combine([(s[i], ix), (1, (b[i], 0, 0, 0))]) for i, ix in enumerate(index)]
            return self.pull(op.operands[0], e, t, inner)
        if name == "stablehlo.reshape":
            return self.pull(op.operands[0], e, t, self._reshaped(op, shape, e, t, index))
        code, operands = _elementwise(op)
        values = []
        for x in operands:
            if dims_of(x) == shape:
                values.append(self.pull(x, e, t, index))
            elif not dims_of(x):
                values.append(self.pull(x, None, None, []))
            else:
                raise Reject("an elementwise op of several shapes")
        return self._emit(code, values, _round_el(op))

    def _reshaped(self, op, shape, e, t, index):
        """The operand's index of a reshape that keeps the axes up to e and t:
        axes may be merged (the operand's is a sum), come and go as units."""
        src = dims_of(op.operands[0])
        head = max(a for a in (e, t) if a is not None) + 1
        if src[:head] != shape[:head]:
            raise Reject("a reshape across the expert / token axes")
        inner = list(index[:head]) + [(0, 0, 0, 0)] * (len(src) - head)
        j = head
        for i in range(head, len(src)):
            if src[i] == 1:
                continue
            extent, terms = 1, []
            while extent < src[i] and j < len(shape):
                terms = [(stride * shape[j], ix) for stride, ix in terms] + [(1, index[j])]
                extent *= shape[j]
                j += 1
            if extent != src[i]:
                raise Reject("a reshape that splits an axis")
            inner[i] = self._combine(terms)
        return inner

    def _dot(self, v, op, e, t, index):
        d = self.owner.dot(v, e, t)
        flat = self._combine((d.strides[i], ix) for i, ix in enumerate(index) if i not in (e, t))
        return self._leaf(("dot", d.number), d.out_el, flat, pair=d.n)

    def finish(self, result, y_el, sum_el=None):
        """The program with its registers: leaves first, a code's register given
        back after its last reader."""
        m = PairMap()
        last = {}
        for i, (_, operands, _, _) in enumerate(self.code):
            for o in operands:
                last[o] = i
        last[result] = len(self.code)
        free, where, used = [], {}, len(self.leaves)
        for i in range(len(self.leaves)):
            where["leaf", i] = i
        for i, (op, operands, rnd, imm) in enumerate(self.code):
            regs = [where[o] for o in operands]
            for o in dict.fromkeys(operands):
                if last[o] == i:
                    free.append(where[o])
            if free:
                dst = free.pop()
            else:
                dst, used = used, used + 1
            if used > REGISTERS:
                raise Reject("more values at once than a pair map holds")
            where["code", i] = dst
            if ("code", i) not in last:
                free.append(dst)
            regs += [dst if not regs else regs[0]] * (3 - len(regs))
            m.code[i] = Instruction(op, dst, *regs, rnd, imm)
        for i, (_, leaf) in enumerate(self.leaves):
            m.leaf[i] = leaf
        m.leaves, m.instructions, m.registers, m.result = len(self.leaves), len(self.code), max(1, used), where[result]
        m.dims = (_i64 * 3)(*self.dims)
        m.rank, m.inner = self.rank, count(self.dims)
        m.per_token, m.y_el = self.per_token, ELS[y_el]
        m.sum_el = ELS[sum_el or y_el]
        return m


# ----------------------------------------------------------- row programs ----

class _Rows:
    """The router under construction: a value is a row of floats a token."""

    def __init__(self, interp, router, block):
        self.interp, self.router = interp, router
        self.inside = set(block.ops)
        self.code, self.leaves, self.memo = [], [], {}
        self.ops = {}                    # key -> op the program replaces
        self.floats = 0
        self.dot = None
        self.depth = 0
        self.below = {router.top_k}      # the ops that depend on the router's top-k
        todo = [router.top_k]
        while todo:
            for user in [u for res in todo.pop().results for u in res.uses if u not in self.below]:
                self.below.add(user)
                todo.append(user)

    def _row(self, n):
        at, self.floats = self.floats, self.floats + n
        if self.floats > ROW_FLOATS:
            raise Reject("more values than a row program holds")
        return at, n

    def _emit(self, op, n, a, b=None, c=None, rnd=0, imm=0.0, dst=None):
        if len(self.code) == ROW_CODE:
            raise Reject("a longer program than a row program takes")
        dst = dst or self._row(n)
        a, b, c = a or dst, b or a or dst, c or a or dst
        self.code.append(RowInstruction(op, rnd, dst[0], n, a[0], a[1], b[0], b[1], c[0], c[1], imm))
        return dst

    def lower(self, v, t, c):
        """The register holding, for a token, `v` along axis `c` at the token
        on axis `t` (None: no such axis); every other axis has one element."""
        shape = dims_of(v)
        t = t if t is not None and shape[t] != 1 else None
        c = c if c is not None and shape[c] != 1 else None
        if t is not None and shape[t] != self.router.T or c is not None and c == t:
            raise Reject("a router value of another number of tokens")
        if any(d != 1 for i, d in enumerate(shape) if i not in (t, c)) or (c is not None and shape[c] > MAX_ROW):
            raise Reject("a router value that is no row a token")
        at = (v, t, c)
        if at not in self.memo:
            op = None if v.is_block_arg else v.op
            splat = _splat(self.interp, v)
            if splat is not None:
                self.memo[at] = self._emit(OP["imm"], 1, None, imm=splat)
            elif op is None or op not in self.inside:
                self.memo[at] = self._leaf(v, t, c)
            elif op in self.below:
                self.memo[at] = self._op(v, op, t, c)
            else:
                was = len(self.code), len(self.leaves), self.floats, self.dot, dict(self.ops), dict(self.memo)
                try:
                    self.memo[at] = self._op(v, op, t, c)
                except Reject:           # read what the program computed ahead of it instead
                    n, m, self.floats, self.dot, self.ops, self.memo = was
                    del self.code[n:], self.leaves[m:]
                    self.memo[at] = self._leaf(v, t, c)
        return self.memo[at]

    def _whole(self, v, t, axis):
        """`lower` with a float an element: a repeated value (a broadcast, a splat)
        is one float for the whole row, which instructions that go through the row's
        elements cannot read."""
        reg, n = self.lower(v, t, axis), dims_of(v)[axis]
        return reg if reg[1] == n else self._emit(OP["copy"], n, reg)

    def _leaf(self, v, t, c):
        if elem(v) not in FLOATS + ("i1",):
            raise Reject(f"a router input of {elem(v)}")
        if len(self.leaves) == ROW_LEAVES:
            raise Reject("more inputs than a row program takes")
        shape = dims_of(v)
        strides = [count(shape[i + 1:]) for i in range(len(shape))]
        reg = self._row(1 if c is None else shape[c])
        self.leaves.append((v, RowLeaf(None, 0, 0 if t is None else strides[t], 0 if c is None else strides[c],
                                       ELS[elem(v)], reg[0], reg[1])))
        return reg

    def _op(self, v, op, t, c):
        if self.depth == MAX_DEPTH:
            raise Reject("a chain of more operations than a row program follows")
        self.depth += 1
        try:
            return self._followed(v, op, t, c)
        finally:
            self.depth -= 1

    def _followed(self, v, op, t, c):
        shape = dims_of(v)
        name = op.name
        from .moe import _splat_value, is_top_k, top_k_width
        if is_top_k(op):
            x = op.operands[0]
            last = len(shape) - 1
            if c not in (None, last) or top_k_width(op) != shape[last] or dims_of(x)[last] > MAX_ROW:
                raise Reject("a top-k along another axis")
            src = self._whole(x, t, last)
            vals, idx = self._row(shape[last]), self._row(shape[last])
            self._emit(OP["top_k"], shape[last], src, src, idx, dst=vals)
            for i, reg in ((0, vals), (1, idx)):
                self.memo[(op.results[i], t, c)] = reg
            self.ops[op_key(op)] = op
            return vals if v is op.results[0] else idx
        reg = self._rule(v, op, name, shape, t, c, _splat_value)
        self.ops[op_key(op)] = op
        return reg

    def _rule(self, v, op, name, shape, t, c, splat_value):
        x = op.operands[0] if op.operands else None
        if name == "stablehlo.broadcast_in_dim":
            sshape, st, sc = dims_of(x), None, None
            for j, d in enumerate(ir.i64_list(op, "broadcast_dimensions")):
                if sshape[j] != 1:
                    st, sc = (j, sc) if d == t else (st, j) if d == c else (st, sc)
            return self.lower(x, st, sc)
        if name == "stablehlo.transpose":
            perm = ir.i64_list(op, "permutation")
            return self.lower(x, None if t is None else perm[t], None if c is None else perm[c])
        if name == "stablehlo.reshape":
            src = dims_of(x)
            if [d for d in src if d != 1] != [d for d in shape if d != 1]:
                raise Reject("a reshape of a router's rows")
            kept = [i for i, d in enumerate(src) if d != 1]
            mine = [i for i, d in enumerate(shape) if d != 1]
            return self.lower(x, None if t is None else kept[mine.index(t)], None if c is None else kept[mine.index(c)])
        if name == "stablehlo.convert" and elem(v) == "i32" and elem(x) == "i32":
            return self.lower(x, t, c)
        if name == "stablehlo.slice":
            b, l, s = op.attrs["start_indices"], op.attrs["limit_indices"], op.attrs["strides"]
            src = dims_of(x)
            axes = [i for i in range(len(src)) if src[i] != shape[i]]
            if not axes:
                return self.lower(x, t, c)
            axis = axes[0]
            if len(axes) != 1 or axis == t or (c is not None and axis != c) or s[axis] < 1:
                raise Reject("a slice of a router's rows")
            reg, n = self._whole(x, t, axis), shape[axis]
            return self._emit(OP["slice"], n, reg, (b[axis], 0), (s[axis], 0))
        if name == "stablehlo.reduce":
            if len(op.operands) != 2 or len(op.attrs["dimensions"]) != 1:
                raise Reject("a reduction over several axes")
            body = op.attrs.get("body")
            if body is None and op.regions:
                inner = [o for o in op.regions[0].ops if o.name != "return"]
                body = inner[0].name if len(inner) == 1 else None
            start = splat_value(op.operands[1])
            how = {"stablehlo.add": ("sum", 0.0), "stablehlo.maximum": ("rowmax", -np.inf),
                   "stablehlo.minimum": ("rowmin", np.inf)}.get(body)
            if how is None or start is None or float(start) != how[1] or c is not None or elem(v) not in FLOATS:
                raise Reject("a reduction a row program does not model")
            axis = op.attrs["dimensions"][0]
            st = None if t is None else t + (1 if axis <= t else 0)
            return self._emit(OP[how[0]], 1, self._whole(x, st, axis), rnd=_round_el(op))
        if name == "stablehlo.dot_general":
            return self._product(v, op, shape, t, c)
        code, operands = _elementwise(op)
        regs = []
        for y in operands:
            if dims_of(y) == shape:
                regs.append(self.lower(y, t, c))
            elif not dims_of(y):
                regs.append(self.lower(y, None, None))
            else:
                raise Reject("an elementwise op of several shapes")
        return self._emit(code, max(r[1] for r in regs), *regs, rnd=_round_el(op))

    def _product(self, v, op, shape, t, c):
        lb, rb, lc, rc = ir.dot_dims(op)
        T = self.router.T
        if lb or rb or len(lc) != 1 or len(rc) != 1 or len(shape) != 2 or self.dot is not None or elem(v) not in FLOATS:
            raise Reject("a router product of another form")
        sides = [self._stored(x) for x in op.operands]
        (lhs, rhs), (ls, rs) = sides, (dims_of(x) for x in op.operands)
        if len(ls) != 2 or len(rs) != 2:
            raise Reject("a router product of another form")
        # the result is [lhs' free axis, rhs' free axis]; the tokens are one of them
        data = 0 if dims_of(v)[0] == T and (t == 0 or (t is None and T == 1)) else 1
        if dims_of(v)[data] != T or (c is not None and c != 1 - data):
            raise Reject("a router product over other than the tokens")
        x, w = (lhs, rhs) if data == 0 else (rhs, lhs)
        xk, wk = (lc[0], rc[0]) if data == 0 else (rc[0], lc[0])
        xs, ws = (ls, rs) if data == 0 else (rs, ls)
        k, n = xs[xk], ws[1 - wk]
        if n > MAX_ROW or T * n * k > MAX_ROUTER_MACS:
            raise Reject("a router product too large for a row program")
        reg = self._row(n)
        p = RowProgram()
        p.dot_x_t, p.dot_x_k = (k, 1) if xk == 1 else (1, xs[1])
        p.dot_w_n, p.dot_w_k = (k, 1) if wk == 1 else (1, ws[1])
        p.dot_k, p.dot_n, p.dot_dst = k, n, reg[0]
        p.dot_cols = 1 << (n - 1).bit_length()
        p.dot_x_el, p.dot_w_el, p.dot_el = ELS[elem(x)], ELS[elem(w)], _round_el(op)
        self.dot = (p, x, w)
        return reg

    def _stored(self, x):
        """What a product's operand is read from: a program input, conversions
        to wider floats looked through (they are exact)."""
        wide = {"f32": 3, "bf16": 1, "f16": 1}
        while not x.is_block_arg and x.op.name == "stablehlo.convert" and x.op in self.inside:
            src = x.op.operands[0]
            if elem(src) not in FLOATS or (elem(src) != elem(x) and wide[elem(x)] <= wide[elem(src)]):
                break
            self.ops[op_key(x.op)] = x.op
            x = src
        if not x.is_block_arg or elem(x) not in FLOATS:
            raise Reject("a router product of computed operands")
        return x

    def finish(self, idx, weights):
        r = self.router
        p = self.dot[0] if self.dot else RowProgram()
        p.tokens, p.reg_floats = r.T, max(1, self.floats)
        p.leaves, p.instructions, p.outs = len(self.leaves), len(self.code), 2
        for i, (_, leaf) in enumerate(self.leaves):
            p.leaf[i] = leaf
        for i, q in enumerate(self.code):
            p.code[i] = q
        p.out[0] = RowOut(None, ELS["i32"], idx[0], idx[1], r.K)
        p.out[1] = RowOut(None, ELS[elem(r.weights)], weights[0], weights[1], r.K)
        return p


# -------------------------------------------------------------- dispatches ----

class _Dot:
    """A per-expert product: `info` (moe.DotInfo), what feeds it, and where its
    result [P, rows.., columns..] keeps the dense result's axes."""
    __slots__ = ("number", "info", "feed", "strides", "n", "out_el")


def _producers(values):
    """The ops that compute `values`, all the way up."""
    ops, todo = set(), list(values)
    while todo:
        v = todo.pop()
        if not v.is_block_arg and v.op not in ops:
            ops.add(v.op)
            todo += v.op.operands
    return ops


class Launches:
    """The launches of one dispatch.  `skip_keys`: ops besides the dispatch's
    own that need not run (the router's); `env_reads`: the program's values that a
    call reads."""

    def __init__(self, interp, g, block):
        self.interp, self.g = interp, g
        self.reads = []
        self.dots, self._dot_of = [], {}
        r = g.router
        rest = [d for i, d in enumerate(dims_of(g.y)) if i not in (g.y_e, g.y_t)]
        final = _Map(self, rest, g.K)
        index, j = [None] * len(dims_of(g.y)), 0
        for i in range(len(index)):
            if i not in (g.y_e, g.y_t):
                index[i], j = final.coordinate(j), j + 1
        result = final.pull(g.y, g.y_e, g.y_t, index)
        if g.out_el not in FLOATS or g.sum_el not in FLOATS or elem(r.weights) not in FLOATS:
            raise Reject("a dispatch of other than floats")
        self.final, self.final_map = final.finish(result, g.out_el, g.sum_el), final
        import torch
        self.result = [g.T] + rest
        self.result_type = {"f32": torch.float32, "bf16": torch.bfloat16, "f16": torch.float16}[g.out_el]
        self.rows = None
        self.skip_keys = frozenset()
        self.env_reads = self.reads + [r.indices, r.weights]
        try:
            self._route(block)
        except Reject:
            self.rows = None
        if any(op_key(op) in g.skip_keys for op in _producers(self.reads)):
            raise Reject("the launches read what the dispatch replaces")
        self._layout()

    def dot(self, v, e, t) -> _Dot:
        at = (v, e, t)
        if at in self._dot_of:
            return self._dot_of[at]
        info = self.g.plan.dot_info.get(at)
        if info is None or info.rows != 1:
            raise Reject("a per-expert product of several rows a pair")
        if info.out_el not in FLOATS:
            raise Reject("a per-expert product of other than floats")
        d = _Dot()
        d.info, d.out_el = info, info.out_el
        d.n = count(info.nshape)
        d.strides = [0] * len(dims_of(v))
        for axis, pos in info.columns.items():
            d.strides[axis] = count(info.nshape[pos + 1:])
        data = info.data
        dshape = dims_of(data)
        if elem(data) not in FLOATS:
            raise Reject("activations of other than floats")
        if info.direct:
            if info.t_dim != 0 or [i for i in range(1, len(dshape)) if dshape[i] != 1] != [i for i in info.contract if dshape[i] != 1]:
                raise Reject("activations that would have to be re-laid")
            self.reads.append(data)
            d.feed = None
        else:
            feed = _Map(self, [dshape[i] for i in info.contract], self.g.K)
            index = [(0, 0, 0, 0)] * len(dshape)
            for j, i in enumerate(info.contract):
                index[i] = feed.coordinate(j)
            el = elem(data)
            result = feed.pull(data, info.data_e, info.t_dim, index)
            d.feed = (feed, feed.finish(result, el), el)
        d.number = len(self.dots)
        self.dots.append(d)
        self._dot_of[at] = d
        return d

    def _route(self, block):
        from . import moe
        g, r = self.g, self.g.router
        rows = _Rows(self.interp, r, block)
        idx = rows.lower(r.indices, 0, 1)
        weights = rows.lower(r.weights, 0, 1)
        keep = self.reads + [v for v, _ in rows.leaves] + ([rows.dot[1], rows.dot[2]] if rows.dot else [])
        for op in _producers(keep):      # what the launches still read is computed as before, whoever else does so
            rows.ops.pop(op_key(op), None)
        if not any(moe.is_top_k(op) for op in rows.ops.values()):
            raise Reject("the top-k is not part of the program")
        skip = moe.sweep_dead(block, set(g.skip_keys) | set(rows.ops), g, keep)
        for key, op in rows.ops.items():
            for res in op.results:
                if any(op_key(u) is not g.key and op_key(u) not in skip for u in res.uses):
                    raise Reject(f"{op.name} of the router is read elsewhere")
        self.rows, self.row_leaves, self.row_dot = rows.finish(idx, weights), rows.leaves, rows.dot
        self.skip_keys, self.env_reads = frozenset(skip), keep

    def _layout(self):
        """Where a call's intermediate results lie in its one buffer, its steps, and the
        modules it needs: looked up once, and ahead of any call -- several threads may
        make the first one, and none of them changes what the others read."""
        import torch
        from . import kernels, moe, qmm
        self.modules = torch, kernels, moe, qmm
        g, r = self.g, self.g.router
        self.buffer = 0

        def place(n, el):
            return place_bytes(n * SIZE[el])

        def place_bytes(n):
            at, self.buffer = self.buffer, (self.buffer + n + 255) // 256 * 256
            return at
        self.at_experts, self.at_weights = place(g.P, "i32"), place(g.P, elem(r.weights))
        self.at_feed = [place(g.P * d.info.k, d.feed[2]) if d.feed else None for d in self.dots]
        self.at_dot = [place(g.P * d.n, d.out_el) for d in self.dots]
        self.workspace = max([kernels._gather_workspace_bytes(g.P, g.E, d.n, d.info.k, _DT[self._rows_of(d)[0]]) for d in self.dots])
        self.at_workspace = place_bytes(self.workspace)
        self.inputs = list(dict.fromkeys(v for v in self.env_reads if self.rows is not None or v is not r.indices))
        self.lhs = any(d.feed is None for d in self.dots)
        self._steps()

    def _rows_of(self, d):
        """(element type, number of rows) of what a product multiplies."""
        return (elem(d.info.data), self.g.T) if d.feed is None else (d.feed[2], self.g.P)

    # A call's values, in this order: its buffer, its result, the pairs' experts,
    # weights and tokens, the inputs, and of every product the packed weight's
    # w, scales, biases, table type, group size, bits and mode.
    BUFFER, RESULT, EXPERTS, WEIGHTS, TOKENS, INPUTS = range(6)
    OF_PRODUCT = 7

    def _steps(self):
        """A call as the library's steps: every launch's program and where a call's
        values go in it.  A product and its map are a step and, behind it, the two
        that take their place where the library says so."""
        g, r = self.g, self.g.router
        steps = []

        def add(kind, program, patches, skip=0, about=None):
            where = (Patch * len(patches))(*[Patch(*p) for p in patches])
            steps.append((kind, program, where, skip, about))

        def of(v):
            return self.INPUTS + self.inputs.index(v)

        def leaf(kind, i):
            struct = MapLeaf if kind is PairMap else RowLeaf
            return kind.leaf.offset + i * ctypes.sizeof(struct) + struct.p.offset

        def map_patches(built, summed, y, fused=False):
            patches = [(PairMap.y.offset, *y), (PairMap.experts_of.offset, self.EXPERTS, 0)]
            if summed:
                patches.append((PairMap.weights.offset, self.WEIGHTS, 0))
            for i, (source, _) in enumerate(built.leaves):
                if source[0] == "env":
                    patches.append((leaf(PairMap, i), of(source[1]), 0))
                elif not fused:
                    patches.append((leaf(PairMap, i), self.BUFFER, self.at_dot[source[1]]))
            return patches

        if self.rows is not None:
            patches = [(leaf(RowProgram, i), of(v), 0) for i, (v, _) in enumerate(self.row_leaves)]
            if self.row_dot:
                patches += [(RowProgram.dot_x.offset, of(self.row_dot[1]), 0), (RowProgram.dot_w.offset, of(self.row_dot[2]), 0)]
            for i, value in enumerate((self.EXPERTS, self.WEIGHTS)):
                patches.append((RowProgram.out.offset + i * ctypes.sizeof(RowOut) + RowOut.p.offset, value, 0))
            add(ROWS, self.rows, patches)
        for m in [d.feed[1] for d in self.dots if d.feed] + [self.final]:
            m.pairs, m.experts = g.P, g.E
        self.final.weights_el = ELS[elem(r.weights)]
        for d in self.dots:                             # (a map ahead of a product is a step of the product before it)
            at = d.number
            behind = self.dots[at + 1] if at + 1 < len(self.dots) else None
            el, rows = self._rows_of(d)
            x = (of(d.info.data), 0) if d.feed is None else (self.BUFFER, self.at_feed[at])
            packed = self.INPUTS + len(self.inputs) + self.OF_PRODUCT * at
            if at == 0 and d.feed is not None:
                add(MAP, d.feed[1], map_patches(d.feed[0], False, x))
            if behind is None:
                after = self.final, map_patches(self.final_map, True, (self.RESULT, 0))
            elif behind.feed is not None:
                after = behind.feed[1], map_patches(behind.feed[0], False, (self.BUFFER, self.at_feed[at + 1]))
            else:
                after = None
            fused = self._fused(d)
            if fused is not None:
                fused.x_rows, fused.x_el, fused.x_per = rows, ELS[el], g.K if d.feed is None else 1
                built = behind.feed[0] if behind else self.final_map
                y = (self.BUFFER, self.at_feed[at + 1]) if behind else (self.RESULT, 0)
                patches = [(PairProduct.map.offset + o, v, plus) for o, v, plus in map_patches(built, behind is None, y, True)]
                patches += [(PairProduct.x.offset, *x), (PairProduct.w.offset, packed, 0), (PairProduct.s.offset, packed + 1, 0),
                            (PairProduct.mode.offset, packed + 6, 0)]
                add(PRODUCT, fused, patches, 2, d)
            p = PairGather(workspace_bytes=self.workspace, pairs=g.P, rows=rows, experts=g.E, n=d.n, k=d.info.k,
                           x_dtype=_DT[el], y_dtype=_DT[d.out_el])
            patches = [(PairGather.x.offset, *x), (PairGather.y.offset, self.BUFFER, self.at_dot[at]),
                       (PairGather.rhs_idx.offset, self.EXPERTS, 0), (PairGather.workspace.offset, self.BUFFER, self.at_workspace)]
            if d.feed is None:
                patches.append((PairGather.lhs_idx.offset, self.TOKENS, 0))
            for i, name in enumerate(("w", "scales", "biases", "table_dtype", "group_size", "bits", "mode")):
                patches.append((getattr(PairGather, name).offset, packed + i, 0))
            add(GATHER, p, patches, 0, d)
            if after is not None:
                add(MAP, *after)
        self.programs = steps                           # (what the library's steps point at)
        self.steps = (Step * len(steps))(*[
            Step(kind, ctypes.sizeof(program), len(where), skip, ctypes.addressof(program), where)
            for kind, program, where, skip, _ in steps])

    def _fused(self, d):
        """A product with the one map that reads it, the next product's activations or
        the result: the launch's program without its addresses.  None: two launches."""
        behind = self.dots[d.number + 1:d.number + 2]
        if behind and behind[0].feed is None:
            return None
        built, program = behind[0].feed[:2] if behind else (self.final_map, self.final)
        maps = [other.feed[0] for other in self.dots if other.feed] + [self.final_map]
        if any(source == ("dot", d.number) for m in maps if m is not built for source, _ in m.leaves):
            return None
        mine = [(i, leaf) for i, (source, leaf) in enumerate(built.leaves) if source[0] == "dot"]
        if not 1 <= len(mine) <= 2 or any(built.leaves[i][0][1] != d.number for i, _ in mine) or program.rank != 1:
            return None
        p = PairProduct(n=d.n, k=d.info.k, product_el=ELS[d.out_el], tiles=len(mine))
        for t, (i, leaf) in enumerate(mine):
            p.col_leaf[t], p.col_base[t], p.col_step[t] = i, leaf.base, leaf.coef[2]
        p.map = program
        return p

    # -- a call

    def run(self, interp, env):
        torch, kernels, moe, qmm = self.modules
        g, r = self.g, self.g.router
        values, keep = [0] * self.INPUTS, []            # of this call (kept until its launches are out)
        for v in self.inputs:
            t = env[v]
            if not isinstance(t, torch.Tensor):
                t = moe.dev(t).t
            elif t.device.type != qmm.DEVICE:
                t = t.to(qmm.DEVICE)
            if not t.is_contiguous():
                t = t.contiguous()
            keep.append(t)
            values.append(t.data_ptr())
        device = keep[0].device
        buffer = torch.empty(self.buffer, dtype=torch.uint8, device=device)
        total = torch.empty(self.result, dtype=self.result_type, device=device)
        base = buffer.data_ptr()
        values[self.BUFFER], values[self.RESULT] = base, total.data_ptr()
        if self.rows is None:
            experts = moe.pair_experts(env, r)
            values[self.EXPERTS], values[self.WEIGHTS] = experts.data_ptr(), keep[self.inputs.index(r.weights)].data_ptr()
        else:
            values[self.EXPERTS], values[self.WEIGHTS] = base + self.at_experts, base + self.at_weights
        if self.lhs:
            values[self.TOKENS] = g.pair_tokens(device)[0].data_ptr()
        moe.STATS["gather_qmm"] += len(self.dots)
        if device.type != "cuda" or any(d.info.match.has_perm for d in self.dots):
            self._one_by_one(interp, values, buffer, keep)
            return total
        for d in self.dots:
            match = d.info.match
            arrays = [a if a.is_contiguous() else a.contiguous() for a in qmm.pack_arrays(interp, match)]
            keep += arrays
            w, scales = arrays[:2]
            if match.mode == "affine":
                values += (w.data_ptr(), scales.data_ptr(), arrays[2].data_ptr(), kernels._dt(scales.dtype), match.gs, match.bits, _lib.MODE_AFFINE)
            else:
                values += (w.data_ptr(), scales.data_ptr(), 0, _lib.BF16, match.gs, match.bits, _lib.MODE_MXFP4)
        run_steps(self.steps, values, kernels._raw_stream(device.index))
        return total

    def _one_by_one(self, interp, values, buffer, keep):
        """The steps by way of this module's functions: a weight packed with its
        contraction axis permuted, whose activations are permuted ahead of a product."""
        _, kernels, _, qmm = self.modules
        stream = kernels._raw_stream(buffer.device.index) if buffer.device.type == "cuda" else 0
        for kind, program, where, _, d in self.programs:
            if kind == PRODUCT:
                continue
            p = _copy(program)
            for q in where:
                if q.value < len(values):               # (what a packed weight adds goes to run_product)
                    ctypes.c_uint64.from_address(ctypes.addressof(p) + q.at).value = values[q.value] + q.add
            if kind == ROWS:
                run_rows(p, stream)
            elif kind == MAP:
                run_map(p, stream)
            else:
                el, rows = self._rows_of(d)
                arrays, x = qmm.pack_arrays(interp, d.info.match), p.x
                if d.info.match.has_perm:
                    at, n = self.at_feed[d.number], rows * d.info.k
                    whole = keep[self.inputs.index(d.info.data)] if at is None else buffer[at:at + n * SIZE[el]].view(qmm._torch_dtype(el))
                    keep.append(kernels.take_k(whole.reshape(rows, d.info.k), arrays[-1]))
                    x = keep[-1].data_ptr()
                run_product(x, el, rows, arrays, d.info.match, p.lhs_idx, p.rhs_idx, p.y, d.out_el, p.pairs, p.experts, p.n, p.k,
                            buffer, stream)


def compile_dispatch(interp, g, block):
    """The dispatch's launches, None where it runs as array operations."""
    try:
        return Launches(interp, g, block)
    except (Reject, RecursionError) as why:
        from .moe import _debug
        _debug(f"{g.name}: array operations ({why})")
        return None
