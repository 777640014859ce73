"""The C-ABI shared library loads without a GPU, exports every symbol the header
declares, and rejects bad arguments before touching the device."""

import ctypes
import os
import re

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HEADER = os.path.join(ROOT, "include", "fouroversix_hip.h")


@pytest.fixture(scope="module")
def native():
    if not os.path.exists(os.path.join(ROOT, "fouroversix_amd", "libfouroversix_hip.so")):
        # (the build script by path: importing the package needs the libraries it builds)
        import importlib.util

        spec = importlib.util.spec_from_file_location("fos_build", os.path.join(ROOT, "fouroversix_amd", "build.py"))
        fos_build = importlib.util.module_from_spec(spec)
        spec.loader.exec_module(fos_build)
        fos_build.build()
    from fouroversix_amd import _native

    return _native


def declared_functions():
    text = open(HEADER).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(fos_[a-z0-9_]+)\s*\(", text)))


def test_header_symbols_are_exported(native):
    L = native.lib()
    names = declared_functions()
    assert set(names) == set(native.EXPORTS)
    for name in names:
        assert getattr(L, name) is not None


def test_version_and_error_strings(native):
    L = native.lib()
    assert L.fos_version() >= 100
    assert L.fos_error_string(0) == b"success"
    for code in range(-6, 0):
        assert len(L.fos_error_string(code)) > 8
    assert b"unknown" in L.fos_error_string(-99)


def test_padding_and_workspace_queries(native):
    L = native.lib()
    assert (L.fos_padded_rows(1), L.fos_padded_rows(128), L.fos_padded_rows(129)) == (128, 128, 256)
    assert (L.fos_padded_cols(1), L.fos_padded_cols(64), L.fos_padded_cols(80)) == (64, 64, 128)
    assert L.fos_quantize_workspace_bytes(8192, 8192) >= 4


def test_argument_checks_need_no_device(native):
    """Every check below returns before the first HIP call."""
    L = native.lib()
    buf = ctypes.create_string_buffer(1 << 16)
    p = ctypes.addressof(buf)
    p = (p + 255) & ~255
    q = lambda **kw: L.fos_quantize(  # noqa: E731
        kw.get("x", p), kw.get("x_type", 0), kw.get("rows", 128), kw.get("cols", 64), kw.get("ld", 64),
        kw.get("dtype", 0), kw.get("rule", 3), kw.get("round", 0), 0, 0, 0, kw.get("layout", 1),
        kw.get("codes", p), kw.get("sf", p), kw.get("amax", p), 0, kw.get("ws", p), kw.get("ws_bytes", 1 << 15), None)
    assert q(x=None) == -4
    assert q(rows=0) == -1
    assert q(ld=32) == -1
    assert q(x_type=3) == -3
    assert q(x_type=2, x=p + 2) == -2  # fp32 elements: 4-byte aligned
    assert q(x_type=3, dtype=2, rule=0) == -3  # MXFP4: the same three element types
    assert q(x_type=2, dtype=2, rule=0, x=p + 2) == -2
    assert q(dtype=7) == -3
    assert q(rule=9) == -3
    assert q(dtype=1, rule=0) == -3  # IF4 has no static rule
    assert q(layout=5) == -3
    assert q(ws=None) == -5
    assert q(ws_bytes=8) == -5
    assert q(codes=p + 1) == -2
    g = lambda **kw: L.fos_gemm_nvfp4(  # noqa: E731
        kw.get("A", p), p, p, p, p, kw.get("M", 128), kw.get("N", 128), kw.get("K", 64), p, kw.get("out", 0),
        kw.get("ldd", 128), None, 0, None)
    assert g(A=None) == -4
    assert g(M=100) == -1  # fewer than 128 rows need K % 256 == 0
    assert L.fos_gemm_workspace_bytes(100, 128, 64) == 0
    assert L.fos_gemm_workspace_bytes(128, 1024, 8192) == 2 * 128 * 1024 * 4  # two splits of 16 K steps
    assert L.fos_gemm_workspace_bytes(128, 1024, 4096) == 0  # 16 steps: unsplit
    assert L.fos_gemm_workspace_bytes(8192, 8192, 8192) == 0
    assert g(K=32) == -1
    assert g(ldd=64) == -1
    assert g(out=2) == -3
    d = lambda **kw: L.fos_dequantize(  # noqa: E731
        kw.get("codes", p), p, p, kw.get("dtype", 0), 1, 1536.0, kw.get("rows", 128), 64,
        kw.get("rows_p", 128), 64, p, kw.get("out", 0), 64, kw.get("inter", 1), None)
    assert d(codes=None) == -4
    assert d(rows=200) == -1
    assert d(rows_p=100, rows=100) == -1
    assert d(dtype=3) == -3
    assert d(out=9) == -3
    assert d(inter=0) == -3  # value x scale meets in fp16 or fp32 only


def test_linear_layer_checks_all_arguments_before_it_launches(native):
    """What the product refuses is refused before the quantize kernel, which clears the recorded maximum."""
    L = native.lib()
    buf = ctypes.create_string_buffer(1 << 17)
    p = (ctypes.addressof(buf) + 255) & ~255
    f = lambda **kw: L.fos_linear_nvfp4(  # noqa: E731
        kw.get("x", p), 0, kw.get("rows", 129), 64, kw.get("ld", 64), 3, None, kw.get("W", p), p, kw.get("w_amax", p),
        kw.get("den", 2.0), kw.get("N", 128), kw.get("D", p), kw.get("out", 0), kw.get("ldd", 128), kw.get("bias"), kw.get("d_amax", p),
        p, kw.get("bytes", 1 << 16), None)
    assert f(W=None) == f(D=None) == f(w_amax=None) == f(x=None) == -4
    assert f(N=100) == f(ldd=64) == f(den=0.0) == f(rows=0) == f(ld=32) == -1
    assert f(D=p + 2) == f(D=p + 8) == f(bias=p + 2) == f(d_amax=p + 1) == f(ldd=132) == -2
    assert f(out=2) == -3
    assert f(bytes=16) == -5


def test_products_with_padding_check_their_arguments(native):
    """What of M, N and K is padding: only what the kernels leave out, and nothing for NVFP4's N and K."""
    L = native.lib()
    buf = ctypes.create_string_buffer(1 << 16)
    p = (ctypes.addressof(buf) + 255) & ~255
    f = lambda dtype=1, out=9, **kw: L.fos_gemm_linear_rows(  # noqa: E731  (out type 9: refused after the sizes)
        dtype, p, p, p, p, p, p, 2.0, 128, kw.get("rows", 128), 256, kw.get("cols", 256), 256, kw.get("depth", 256), p, out,
        kw.get("ldd", 256), kw.get("bias"), kw.get("d_amax"), None, 0, None)
    assert f(dtype=2) == -3
    for dtype in (0, 1):
        assert f(dtype) == f(dtype, rows=1) == -3
        assert f(dtype, rows=-1) == f(dtype, rows=129) == f(dtype, cols=264) == f(dtype, depth=320) == f(dtype, ldd=128) == -1
    assert f(depth=208) == f(cols=136, ldd=136) == -3
    assert f(depth=200) == f(depth=192) == f(cols=130) == f(cols=128) == -1  # (a whole tile of padding does not exist)
    assert f(cols=136, bias=p) == f(cols=136, d_amax=p) == f(cols=136, ldd=128) == -1
    assert f(0, depth=240) == f(0, cols=136) == -1


@pytest.mark.parametrize("tile", ["1", "128", "129", "256"])
def test_workspace_query_of_a_small_batch_on_forced_tiles(native, monkeypatch, tile):
    """Fewer rows than a tile has, with the weight-streaming kernels switched off: the query answers (the product itself
    is refused)."""
    monkeypatch.setenv("FOS_GEMM_TILE", tile)
    L = native.lib()
    for m in (1, 16, 127, 128):
        assert L.fos_gemm_workspace_bytes(m, 256, 512) >= 0
        assert L.fos_linear_nvfp4_scratch_bytes(m, 512, 256) > 0


def test_scratch_for_converted_operands_is_bounded(native):
    """No more than 8 GiB of operands in fp16, the weight's among them where it is converted too (IF4)."""
    L = native.lib()
    m = n = 1 << 19  # rows of 4096 columns, 8 GiB together
    assert L.fos_gemm_scratch_bytes(1, m, n, 4096) == 8 << 30
    assert L.fos_gemm_scratch_bytes(1, m + 128, n, 4096) == L.fos_gemm_scratch_bytes(1, m, n + 128, 4096) == 0


LAYERS_FROM_CODES = [
    # narrow outputs of many rows: the fragments' bytes; K split on either side; a second workgroup for a few compute units
    (15439, 6912, 128), (12053, 6272, 768), (10225, 12544, 640), (5726, 9600, 1536), (4842, 13568, 128), (174, 11904, 1152), (1272, 16128, 256),
]
LAYERS_FROM_FRAGMENTS = [(1000, 4096, 14336), (2048, 4096, 4096), (16384, 4096, 14336), (8192, 4096, 4096), (8192, 14336, 4096), (515, 15360, 3456)]


@pytest.fixture
def converts(native, monkeypatch):
    """Whether a query answers with room for an operand in fp16: another number than with those kernels switched off."""
    L = native.lib()

    def ask(query, *args):
        by_plan = getattr(L, query)(*args)
        with monkeypatch.context() as m:
            m.setenv("FOS_GEMM_TILE", "64")  # (the packed kernels as they are chosen by themselves)
            L.fos_tuning_reload()
            packed = getattr(L, query)(*args)
        L.fos_tuning_reload()
        return by_plan != packed

    yield ask


@pytest.mark.parametrize("shapes", [LAYERS_FROM_CODES, LAYERS_FROM_FRAGMENTS], ids=["codes", "fragments"])
def test_layers_convert_their_operand_where_it_pays(converts, shapes):
    """Measured on either route, 7 to 50 % apart."""
    for shape in shapes:
        assert converts("fos_linear_nvfp4_scratch_bytes", *shape) == (shapes is LAYERS_FROM_FRAGMENTS), shape


@pytest.mark.parametrize(("dtype", "pays", "shapes"), [
    (1, False, [(512, 11648, 14144), (640, 13056, 12544), (11008, 512, 11776)]),
    (1, True, [(2048, 4096, 4096), (1280, 13184, 7040), (640, 4224, 13184)]),
    (0, False, [(9856, 256, 16256), (8320, 1024, 14848), (4864, 2176, 16000)]),
    (0, True, [(16384, 14336, 4096), (8192, 8192, 8192), (2560, 13952, 10624)]),
])
def test_products_convert_their_operands_where_it_pays(converts, dtype, pays, shapes):
    """(IF4: both; NVFP4: A, by a pass of its own.)  Measured on either route, 8 to 45 % apart."""
    for shape in shapes:
        assert converts("fos_gemm_scratch_bytes", dtype, *shape) == pays, shape


@pytest.mark.parametrize("rows", [65, 96, 128])
def test_layers_of_up_to_128_rows_stream_the_weight_where_it_pays(converts, rows):
    """As above for the form that streams the weight: 5 to 50 % apart, and ties, which stay with the packed kernel."""
    for cols, n in ((8192, 512), (11264, 2048), (11776, 4096), (14336, 4096), (28672, 3072), (53248, 4096), (16384, 2304)):
        assert converts("fos_linear_nvfp4_scratch_bytes", rows, cols, n), (cols, n)
    for cols, n in ((28672, 512), (53248, 128), (16384, 2048), (24576, 1024), (14336, 1024), (8192, 4096), (8192, 4224), (7936, 512)):
        assert not converts("fos_linear_nvfp4_scratch_bytes", rows, cols, n), (cols, n)
