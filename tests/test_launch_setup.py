"""What the host does ahead of its launches, without a GPU: the library runs in a child
process whose HIP launch calls are recorded and go nowhere (every address it is given is
made up, and never read)."""

import json
import os
import subprocess
import sys

import pytest

from metaljax_amd import _lib

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

RECORDER = r"""
#include <cstddef>
#include <cstdio>
struct Dim { unsigned x, y, z; };
static Dim grid, block;
static size_t lds;
extern "C" {
int __hipPushCallConfiguration(Dim g, Dim b, size_t bytes, void*) { grid = g; block = b; lds = bytes; return 0; }
int __hipPopCallConfiguration(Dim* g, Dim* b, size_t* bytes, void** stream) { *g = grid; *b = block; *bytes = lds; *stream = nullptr; return 0; }
int hipLaunchKernel(const void* f, Dim g, Dim b, void**, size_t bytes, void*) {
  std::printf("launch %zu %u %u %u %zu\n", (size_t)f, g.x, g.y, b.x, bytes);
  return 0;
}
int hipFuncSetAttribute(const void* f, int, int value) { std::printf("limit %zu %d\n", (size_t)f, value); return 0; }
int hipGetLastError() { return 0; }
void next_call() { std::printf("call\n"); std::fflush(stdout); }
}
"""

CALLS = r"""
import ctypes, json, sys
recorder = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)       # ahead of the library: its calls are found first
sys.path.insert(0, sys.argv[2])
from metaljax_amd import _lib, moe_launch as ML
lib, at = _lib.load(), 1 << 20

def dense(m, n, k, bits, x=_lib.BF16):
    room = lib.qmm_workspace_bytes(1, m, n, k, 64, bits, 0, x)
    return lib.qmm_quantized_matmul(at, x, at, at, at, _lib.BF16, at, x, 1, m, n, k, 64, bits, 0, at, room, None)

def gather(pairs, experts, n, k, x):
    room = lib.qmm_gather_workspace_bytes(pairs, experts, n, k, x)
    return lib.qmm_gather_qmm(at, x, at, at, None, _lib.BF16, at, x, at, at, pairs, pairs, experts, n, k, 32, 4, _lib.MODE_MXFP4, at, room, None)

def fused(pairs, experts, n, k, x, per):
    el = {_lib.F32: 0, _lib.BF16: 1, _lib.F16: 2}[x]
    m = ML.PairMap(y=at, experts_of=at, pairs=pairs, inner=n, dims=(1, 1, n), per_token=per or 1, experts=experts, rank=1, leaves=1,
                   registers=1, weights=at if per else None)
    m.leaf[0] = ML.MapLeaf(None, 0, n, 0, 0, (0, 0, 1), el)
    p = ML.PairProduct(x=at, w=at, s=at, x_rows=pairs, n=n, k=k, mode=_lib.MODE_MXFP4, x_el=el, x_per=1, product_el=el, tiles=1, col_step=(1, 0), map=m)
    return lib.qmm_pair_product_run(ctypes.byref(p), None)

def refused(*shape):
    return int(fused(*shape) != 3)                                 # (UNSUPPORTED: two launches)

for name, args in json.loads(sys.argv[3]):
    recorder.next_call()
    assert globals()[name](*args) == 0, (name, args, lib.qmm_last_error())
recorder.next_call()
"""


@pytest.fixture(scope="module")
def record(tmp_path_factory):
    """calls -> what each did: (kernel, grid x, grid y, threads, bytes of LDS) a launch and (kernel, bytes) a raised limit"""
    where = tmp_path_factory.mktemp("recorder")
    (where / "recorder.cc").write_text(RECORDER)
    subprocess.run(["g++", "-shared", "-fPIC", "-O1", "-o", where / "recorder.so", where / "recorder.cc"], check=True)

    def run(calls):
        out = subprocess.run([sys.executable, "-c", CALLS, str(where / "recorder.so"), ROOT, json.dumps(calls)], check=True,
                             capture_output=True, text=True).stdout
        done = []
        for line in out.splitlines():
            what, *numbers = line.split()
            if what == "call":
                done.append(([], []))
            else:
                done[-1][what == "limit"].append(tuple(int(v) for v in numbers))
        assert len(done) == len(calls) + 1 and all(bool(launches) == (name != "refused") for (name, _), (launches, _) in zip(calls, done))
        return done[:-1]
    return run


def test_a_kernels_limit_is_raised_once(record):
    """By its first launch, for all that any later one may ask: calls of one kernel with a whole K and
    with a K that is split need different amounts of local memory, whichever comes first."""
    calls = [["dense", shape] for shape in ([2048, 4096, 8192, 4], [600, 2048, 12800, 4], [600, 2048, 12800, 4], [2048, 4096, 8192, 4],
                                            [450, 8192, 8192, 8], [2048, 4096, 8192, 8], [450, 8192, 8192, 8], [48, 4096, 14336, 4], [48, 4096, 14336, 4])]
    done = record(calls)
    limits, asked = {}, {}
    for launches, raised in done:
        for kernel, value in raised:
            limits.setdefault(kernel, []).append(value)
        for kernel, _, _, _, lds in launches:
            asked.setdefault(kernel, set()).add(lds)
            assert lds <= max(limits.get(kernel, [65536]))
    assert any(len(sizes) > 1 for sizes in asked.values())               # (one kernel, two amounts)
    assert all(len(values) == 1 for values in limits.values()), limits


@pytest.mark.parametrize("pairs,experts,n,k,types", [
    (4, 8, 64, 2048, "f32 f16"), (4, 8, 64, 2016, "f32 bf16 f16"),
    (5, 8, 96, 2080, "f32 bf16 f16"), (6, 8, 1792, 3168, "f32 bf16 f16"), (24, 16, 1792, 3168, "f32 bf16 f16"), (24, 16, 96, 3168, "f32 bf16 f16"),
    (8, 8, 1024, 3072, "f32 f16"), (16, 8, 512, 3072, "f32 f16"), (7, 8, 64, 4160, "f32 bf16 f16"), (40, 8, 96, 4192, "f32 bf16 f16")])
def test_a_product_and_its_map_share_a_contraction_as_the_product_does(record, pairs, experts, n, k, types):
    """As many wavefronts, and so the same sums, and a token's pairs as many each: of four
    and eight, by the contraction, the type and (where the workgroups are several rounds) the
    columns and the pairs; shapes that a staged kernel would take among them."""
    calls = []
    for x in types.split():
        shape = [pairs, experts, n, k, {"f32": _lib.F32, "bf16": _lib.BF16, "f16": _lib.F16}[x]]
        calls += [["gather", shape], ["fused", shape + [0]]]
        if pairs % 2 == 0 and pairs * n * k / 2 <= 16 << 20:
            calls.append(["fused", shape + [2]])
    threads = 0
    for (name, args), (launches, _) in zip(calls, record(calls)):
        (_, _, rows, lanes, _), = launches
        if name == "gather":
            threads, segments = lanes, rows
        else:
            assert lanes == threads * (args[5] or 1)
            assert rows == (pairs // args[5] if args[5] else segments)


@pytest.mark.parametrize("tokens,per,experts,n,k,types", [
    (4, 2, 8, 1024, 1024, "f32 bf16 f16"), (5, 2, 8, 1024, 1024, "bf16 f16"), (7, 2, 8, 1600, 1024, "bf16 f16"), (7, 2, 8, 8192, 256, "bf16"),
    (8, 2, 8, 512, 512, "f32 bf16 f16"), (12, 2, 8, 512, 512, "bf16 f16"), (20, 2, 8, 512, 512, "bf16"), (32, 2, 8, 1024, 256, ""),
    (12, 1, 8, 1024, 256, "f32 bf16 f16"), (13, 1, 8, 1024, 256, "bf16 f16"), (64, 1, 8, 256, 256, "bf16 f16"), (64, 1, 8, 512, 256, "bf16"),
    (4, 4, 8, 1024, 1024, "f32 bf16 f16"), (8, 4, 8, 1024, 1024, "bf16 f16"), (8, 4, 8, 1024, 256, "f32 bf16 f16"), (16, 4, 8, 1024, 256, "bf16"),
    (2, 4, 8, 4096, 512, "f32 bf16 f16"), (3, 4, 8, 4096, 512, "bf16 f16"), (3, 4, 8, 8192, 256, "bf16")])
def test_a_tokens_sum_is_part_of_the_product_for_a_round_or_two(record, tokens, per, experts, n, k, types):
    """On both sides of what a round of the summing workgroups holds, by the type's terms and the pairs a
    token, sorted by the kernel (16 pairs and more) and not; past it a product and a map are the faster."""
    calls = [["fused" if x in types.split() else "refused", [tokens * per, experts, n, k, {"f32": _lib.F32, "bf16": _lib.BF16, "f16": _lib.F16}[x], per]]
             for x in ("f32", "bf16", "f16")]
    for (name, args), (launches, _) in zip(calls, record(calls)):
        if name == "fused":
            (_, columns, rows, lanes, _), = launches
            assert (columns, rows, lanes) == (-(-n // 16), tokens, 64 * 4 * per)


@pytest.mark.parametrize("m,n,k,bits,workgroups", [
    (698, 5432, 7424, 4, 129), (212, 6896, 5376, 4, 4 * 54),           # (in fours none would be a second round of one, or it is worth it)
    (635, 2138, 2560, 8, 170), (855, 1458, 2496, 8, 168),              # columns that are no fours, whose sums leave one by one: short groups
    (6328, 1486, 7552, 8, 2 * 300), (5076, 1920, 7808, 4, 2 * 300),    # more tiles than a round as they are
    (926, 9576, 14080, 8, 3 * 300)])                                   # more sums than caches hold
def test_a_split_K_counts_what_its_sums_take(record, m, n, k, bits, workgroups):
    (launches, _), = record([["dense", [m, n, k, bits]]])
    assert -(-workgroups // 8) * 8 in [x for _, x, _, lanes, _ in launches if lanes == 512]


@pytest.mark.parametrize("m,n,k,bits,x,short", [
    (2387, 168, 11264, 4, "f32", True), (2988, 200, 5760, 8, "f32", True), (1048, 264, 12800, 4, "f32", True),
    (600, 4096, 4096, 4, "f32", False), (2048, 4096, 4096, 4, "f16", False)])
def test_terms_that_are_launches_of_their_own_count(record, m, n, k, bits, x, short):
    """Terms, the product and its sums on the kernel of short groups; terms, their re-laying, the product, its
    sums and the sum over the terms ahead of it on the other, whose terms take twice the time."""
    (launches, _), = record([["dense", [m, n, k, bits, {"f32": _lib.F32, "f16": _lib.F16}[x]]]])
    assert (len(launches) <= 3) == short
