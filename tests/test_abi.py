"""The C-ABI library: it loads, exports every function include/qmm_hip.h
declares, and its host-only entry points (no device work) behave.  Runs
without a GPU; no compute entry point is called here."""

import ctypes
import os
import re

import pytest

from metaljax_amd import _lib

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HEADER = os.path.join(ROOT, "include", "qmm_hip.h")


def declared_functions():
    text = open(HEADER).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    text = re.sub(r"//[^\n]*", "", text)
    return sorted(set(re.findall(r"\b(qmm_[a-z0-9_]+)\s*\(", text)))


@pytest.fixture(scope="module")
def lib():
    if not os.path.exists(_lib.LIB_PATH):
        from metaljax_amd import build
        build.build()
    return _lib.load()


def test_header_and_binding_agree():
    assert declared_functions() == sorted(_lib.SYMBOLS)


def test_library_exports_every_declared_symbol(lib):
    raw = ctypes.CDLL(_lib.LIB_PATH)
    for name in declared_functions():
        assert hasattr(raw, name), name


def test_header_cites_the_reference_for_every_entry_point():
    text = open(HEADER).read()
    # each declaration is preceded by a comment naming the reference call it replaces
    for name in declared_functions():
        if name in ("qmm_abi_version", "qmm_last_error", "qmm_workspace_bytes",
                    "qmm_gather_workspace_bytes", "qmm_plan"):
            continue
        if name == "qmm_gather_qmm_static":      # says that the reference has no such call
            head = text[:text.index(name + "(")]
            assert "No counterpart in the reference" in head[head.rindex("/*"):]
            continue
        head = text[:text.index(name + "(")]
        comment = head[head.rindex("/*"):]
        assert re.search(r"\.py:\d+", comment), f"{name}: no reference citation"


def test_abi_version_and_error_text(lib):
    assert lib.qmm_abi_version() >= 1
    assert isinstance(lib.qmm_last_error(), bytes)


def test_plan_picks_the_regime(lib):
    k, g, b = ctypes.c_int(), ctypes.c_int(), ctypes.c_int()
    assert lib.qmm_plan(1, 4096, 4096, 64, 4, 0, k, g, b) == 0
    assert k.value == _lib.KERNEL_GEMV and g.value > 0 and b.value % 64 == 0
    assert lib.qmm_plan(16, 14336, 4096, 64, 4, 0, k, g, b) == 0
    assert k.value == _lib.KERNEL_GEMV
    assert lib.qmm_plan(2048, 4096, 4096, 64, 8, 0, k, g, b) == 0
    assert k.value == _lib.KERNEL_GEMM and g.value >= 256


def test_plan_of_the_decode_variants(lib):
    """The decode plan follows the kernel choice: 768-thread workgroups (eight
    compute + four loader wavefronts) where the loader-wavefront kernel serves
    the shape, one workgroup per compute unit (256 assumed without a device)
    with up to 128 rows each when the activations are fetched directly."""
    k, g, b = ctypes.c_int(), ctypes.c_int(), ctypes.c_int()
    assert lib.qmm_plan(4, 28672, 4096, 64, 4, 0, k, g, b) == 0
    assert (k.value, b.value) == (_lib.KERNEL_GEMV, 768)
    rows = -(-28672 // g.value)
    assert 16 <= rows <= 128 and g.value * rows >= 28672
    assert lib.qmm_plan(16, 14336, 4096, 64, 4, 0, k, g, b) == 0        # ring variant: at most 64 rows
    assert b.value == 768 and -(-14336 // g.value) <= 64
    assert lib.qmm_plan(4, 4096, 1024, 64, 4, 0, k, g, b) == 0          # two slices: the self-loading kernel
    assert k.value == _lib.KERNEL_GEMV and b.value < 768
    assert lib.qmm_plan(4, 16384, 3072, 64, 4, 0, k, g, b) == 0         # six slices: loader wavefronts again
    assert k.value == _lib.KERNEL_GEMV and b.value == 768
    assert lib.qmm_plan(16, 3072, 3072, 64, 4, 0, k, g, b) == 0         # ... at sixteen rows too
    assert b.value == 768


def test_plan_of_the_decode_in_groups_of_32(lib):
    """Eight rows a workgroup at least, where groups of 64 keep sixteen: fewer than
    4096 weight rows still give every compute unit (256 assumed) a workgroup."""
    k, g, b = ctypes.c_int(), ctypes.c_int(), ctypes.c_int()
    for n, kk, bits, grid in ((1504, 10304, 8, 188), (2000, 7168, 8, 250), (3072, 8192, 4, 256), (14336, 4096, 4, 256)):
        assert lib.qmm_plan(4, n, kk, 32, bits, 0, k, g, b) == 0
        assert (k.value, g.value, b.value) == (_lib.KERNEL_GEMV, grid, 768), (n, kk)
    assert lib.qmm_plan(4, 1504, 10304, 64, 8, 0, k, g, b) == 0
    assert (g.value, b.value) == (94, 768)


def test_plan_of_the_mxfp4_kernels(lib):
    """MXFP4 prefill: the eight-wavefront block-scaled kernel (512 threads, a
    64 x 128 tile a workgroup) when K is a whole number of 2048-code stages,
    the four-wavefront one for the other multiples of 512, the bf16 kernels
    otherwise.  MXFP4 decode: the loader-wavefront kernel (768 threads) from
    three 512-code slices a row on, for a K that is no whole number of slices
    (gpt-oss: 2880) its one-pass form with rows dealt by eights."""
    k, g, b = ctypes.c_int(), ctypes.c_int(), ctypes.c_int()
    assert lib.qmm_plan(256, 8192, 8192, 32, 4, 1, k, g, b) == 0
    assert (k.value, g.value, b.value) == (_lib.KERNEL_MXFP4_MFMA, (8192 // 128) * (256 // 64), 512)
    assert lib.qmm_plan(300, 260, 1536, 32, 4, 1, k, g, b) == 0
    assert (k.value, b.value) == (_lib.KERNEL_MXFP4_MFMA, 256) and g.value == 16      # 3 x 5 tiles, dealt to eight XCDs
    assert lib.qmm_plan(256, 5760, 2880, 32, 4, 1, k, g, b) == 0        # K % 512 != 0: the bf16 prefill kernel
    assert k.value == _lib.KERNEL_GEMM
    for m in (1, 16):
        assert lib.qmm_plan(m, 5760, 2880, 32, 4, 1, k, g, b) == 0
        rows = -(-5760 // g.value)
        assert (k.value, b.value) == (_lib.KERNEL_GEMV, 768) and rows % 8 == 0 and 16 <= rows <= 128
        assert lib.qmm_plan(m, 8192, 8192, 32, 4, 1, k, g, b) == 0
        assert (k.value, b.value) == (_lib.KERNEL_GEMV, 768) and g.value == 256
    assert lib.qmm_plan(4, 4096, 1024, 32, 4, 1, k, g, b) == 0          # two slices: the general decode kernel
    assert k.value == _lib.KERNEL_GEMV and b.value < 768
    assert lib.qmm_plan(4, 4096, 4160, 32, 4, 1, k, g, b) == 0          # ragged beyond eight slices: general again
    assert b.value < 768
    assert lib.qmm_plan(4, 100, 2880, 32, 4, 1, k, g, b) == 0           # an expert's scale table no multiple of 16 bytes
    assert b.value < 768


def test_plan_keeps_exact_mxfp4_products(lib):
    """K a multiple of 512 but not of 2048: where the short-group kernel served, whose
    products are exact, the four-wavefront form (a narrower split of bf16 activations)
    is not taken for the few per cent that it is ahead."""
    k, g, b = ctypes.c_int(), ctypes.c_int(), ctypes.c_int()
    for m, n, kk in ((227, 13264, 1536), (468, 2184, 7680), (820, 3088, 3072), (1821, 8128, 2560), (75, 13272, 5632), (430, 9328, 11264)):
        assert lib.qmm_plan(m, n, kk, 32, 4, 1, k, g, b) == 0
        assert k.value == _lib.KERNEL_GEMM, (m, n, kk)
    assert lib.qmm_plan(256, 8192, 8192, 32, 4, 1, k, g, b) == 0
    assert k.value == _lib.KERNEL_MXFP4_MFMA


def test_gather_workspace_covers_the_grouped_decode(lib):
    """From four pairs up to sixteen an expert the workspace holds the expert
    sort and the segment list; below four pairs nothing is needed."""
    assert lib.qmm_gather_workspace_bytes(2, 8, 14336, 4096, _lib.BF16) == 0
    few = lib.qmm_gather_workspace_bytes(16, 8, 14336, 4096, _lib.BF16)
    sort_only = ((2 * 8 + 1 + 2 * 16) * 4 + 255) // 256 * 256
    assert few >= sort_only and few % 256 == 0
    assert lib.qmm_gather_workspace_bytes(128, 8, 14336, 4096, _lib.BF16) >= lib.qmm_gather_workspace_bytes(16, 8, 14336, 4096, _lib.BF16)


def test_workspace_queries_need_no_device(lib):
    assert lib.qmm_workspace_bytes(1, 16, 14336, 4096, 64, 4, 0, _lib.BF16) == 0
    need = lib.qmm_gather_workspace_bytes(1024, 8, 14336, 4096, _lib.BF16)
    assert need > 0 and need % 4 == 0
    assert lib.qmm_gather_workspace_bytes(0, 8, 64, 64, _lib.BF16) >= 0


def test_argument_errors_are_reported_before_any_launch(lib):
    # null pointers / bad enums are rejected on the host (no GPU needed)
    rc = lib.qmm_quantized_matmul(None, _lib.BF16, None, None, None, _lib.BF16, None, _lib.BF16,
                                  1, 1, 64, 64, 64, 4, 0, None, 0, None)
    assert rc != 0
    assert lib.qmm_last_error()
    rc = lib.qmm_quantized_matmul(None, _lib.BF16, None, None, None, _lib.BF16, None, _lib.BF16,
                                  1, 1, 64, 48, 64, 4, 0, None, 0, None)
    assert rc in (1, 2, 3)


def test_missing_library_fails_loudly(monkeypatch, tmp_path):
    monkeypatch.setattr(_lib, "_lib", None)
    monkeypatch.setattr(_lib, "LIB_PATH", str(tmp_path / "libqmm_hip.so"))
    with pytest.raises(_lib.QmmLibraryError):
        _lib.load()


def test_static_scratch_entry_point_rejects_what_does_not_fit(lib):
    """qmm_gather_qmm_static refuses, on the host and before any device work,
    a product whose scratch need exceeds the array built into the library."""
    text = open(HEADER).read()
    assert re.search(r"#define QMM_STATIC_SCRATCH_BYTES \(16u << 20\)", text)
    assert _lib.STATIC_SCRATCH_BYTES == 16 << 20
    p, e, n, k = 4096, 8, 14336, 4096                 # the re-laid activations alone are 32 MiB
    assert lib.qmm_gather_workspace_bytes(p, e, n, k, _lib.BF16) > _lib.STATIC_SCRATCH_BYTES
    rc = lib.qmm_gather_qmm_static(None, _lib.BF16, None, None, None, _lib.BF16, None, _lib.BF16,
                                   None, None, p, p, e, n, k, 64, 4, 0, None)
    assert rc == 4 and b"static scratch" in lib.qmm_last_error()


def _no_gpu():
    import torch
    return not torch.cuda.is_available()


@pytest.mark.skipif(not _no_gpu(), reason="made-up pointers: only where nothing can be launched with them")
def test_what_is_refused_does_not_depend_on_the_kernel(lib):
    """Too little scratch, or tables that do not start on sixteen bytes, are refused at
    every size, also where the kernel that would run needs less."""
    at = 0x100000

    def dense(m, n, k, act, mode, scratch, scales=at, batch=1):
        return lib.qmm_quantized_matmul(at, act, at, scales, None if mode else at, _lib.BF16, at, _lib.BF16, batch, m, n,
                                        k, 32 if mode else 64, 4, mode, at, scratch, None)
    for m, n, k in ((17, 4096, 4096), (48, 4096, 14336), (77, 1024, 2048), (300, 9216, 2944)):
        for mode in (0, 1):
            for act in (_lib.BF16, _lib.F16, _lib.F32):
                need = lib.qmm_workspace_bytes(1, m, n, k, 64, 4, mode, act)
                assert dense(m, n, k, act, mode, 256) == 4
                if act == _lib.BF16:                                  # (wider ones are told behind a first launch)
                    assert dense(m, n, k, act, mode, need, scales=at + 4) == 1
                assert dense(m, n, k, act, mode, need) == 5           # (nothing wrong with it: the launch fails)
        terms = 2 * m * k * 2 + 256                                   # room for float16 terms, not for their products
        assert dense(m, n, k, _lib.F16, 0, terms) == 4
        assert lib.qmm_grouped_qmm(at, _lib.F16, at, at, at, _lib.BF16, at, _lib.BF16, at, m, 4, n, k, 64, 4, 0, at,
                                   terms, None) == 4
        assert lib.qmm_gather_qmm(at, _lib.F16, at, at, at, _lib.BF16, at, _lib.BF16, at, at, 5 * m, 5 * m, 4, n, k, 64,
                                  4, 0, at, 5 * terms + 8192, None) == 4


@pytest.mark.skipif(not _no_gpu(), reason="made-up pointers: only where nothing can be launched with them")
@pytest.mark.parametrize("act", [_lib.BF16, _lib.F16, _lib.F32])
def test_the_gather_query_tells_what_the_static_entry_takes(lib, act):
    """At sizes round the array's: products that fit it without the sums of a split K
    (and with them would not), that fall a little short, and that do not fit."""
    at = 0x100000
    for p, e, n, k in ((260, 8, 9200, 6848), (672, 16, 4168, 7808), (494, 16, 4808, 6848), (100, 8, 14336, 4096),
                       (1700, 8, 1024, 4096), (2000, 8, 4096, 4096), (512, 32, 2048, 2880), (64, 8, 14336, 14336),
                       (80, 8, 16384, 14336), (4096, 8, 256, 1024)):
        rc = lib.qmm_gather_qmm_static(at, act, at, at, at, _lib.BF16, at, _lib.BF16, at, at, p, p, e, n, k, 64, 4, 0, None)
        want = 4 if lib.qmm_gather_workspace_bytes(p, e, n, k, act) > _lib.STATIC_SCRATCH_BYTES else 5
        assert rc == want, (p, e, n, k)


def test_the_wrappers_import_without_a_gpu_build_of_torch(monkeypatch):
    """torch's stream queries are not there in a build for the CPU alone; packing,
    the interpreter and the recognizer import the wrappers all the same."""
    import importlib.util

    import torch

    from metaljax_amd import kernels
    for name in ("_cuda_getCurrentRawStream", "_cuda_getDevice"):
        monkeypatch.delattr(torch._C, name, raising=False)
    spec = importlib.util.spec_from_file_location("metaljax_amd.kernels_without_a_gpu", kernels.__file__)
    spec.loader.exec_module(importlib.util.module_from_spec(spec))
