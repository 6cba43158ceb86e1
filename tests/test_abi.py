"""CPU checks of the C-ABI boundary and the host logic (no kernel is launched here)."""
import ctypes
import os
import re
import subprocess
import sys

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HEADER = os.path.join(ROOT, "include", "libtl.h")
PKG = os.path.join(ROOT, "torchless-nn_amd")
LIB = os.path.join(PKG, "libtl.so")

needs_lib = pytest.mark.skipif(not os.path.exists(LIB), reason="libtl.so not built")


def header_functions():
    text = open(HEADER).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(tl_[a-z0-9_]+)\s*\(", text)))


def test_header_declares_the_binding_table():
    import tl_hip
    assert header_functions() == sorted(tl_hip.SIGNATURES)


def _ctype_of(decl):
    """C parameter declaration -> the ctypes type the binding must use."""
    import ctypes as C
    decl = re.sub(r"\bconst\b", "", decl).strip()
    if "*" in decl:
        base = decl.split("*")[0].strip()
        stars = decl.count("*")
        scalar = {"int": C.c_int, "int64_t": C.c_int64, "size_t": C.c_size_t,
                  "float": C.c_float, "double": C.c_double}
        if stars == 1 and base in scalar:
            return ("ptr", scalar[base])
        return ("ptr", None)
    base = decl.rsplit(" ", 1)[0].strip()
    return {"int": C.c_int, "int32_t": C.c_int32, "int64_t": C.c_int64, "uint32_t": C.c_uint32,
            "uint64_t": C.c_uint64, "size_t": C.c_size_t, "float": C.c_float,
            "double": C.c_double}[base]


def test_binding_argument_types_match_the_header():
    """Every prototype's parameter types, position by position, against SIGNATURES."""
    import ctypes as C
    import tl_hip
    text = re.sub(r"/\*.*?\*/", "", open(HEADER).read(), flags=re.S)
    protos = re.findall(r"\b(?:int|const char\*)\s+(tl_[a-z0-9_]+)\s*\(([^)]*)\)\s*;", text)
    assert sorted(n for n, _ in protos) == sorted(tl_hip.SIGNATURES)
    for name, params in protos:
        params = params.strip()
        decls = [] if params in ("", "void") else [p.strip() for p in params.split(",")]
        got = tl_hip.SIGNATURES[name]
        assert len(decls) == len(got), name
        for i, (d, t) in enumerate(zip(decls, got)):
            want = _ctype_of(d)
            if isinstance(want, tuple):
                if want[1] is None:
                    assert t is C.c_void_p or issubclass(t, C._Pointer), (name, i, d)
                else:
                    assert t is C.c_void_p or t == C.POINTER(want[1]), (name, i, d)
            else:
                assert C.sizeof(t) == C.sizeof(want) and (t in (C.c_float, C.c_double)) == \
                    (want in (C.c_float, C.c_double)), (name, i, d, t, want)


@needs_lib
def test_library_exports_every_declared_symbol():
    lib = ctypes.CDLL(LIB)
    missing = [f for f in header_functions() if not hasattr(lib, f)]
    assert not missing, missing


@needs_lib
def test_exported_symbols_are_exactly_the_header():
    out = subprocess.run(["nm", "-D", "--defined-only", LIB], capture_output=True, text=True).stdout
    exported = sorted(set(re.findall(r" T (tl_[a-z0-9_]+)$", out, flags=re.M)))
    assert exported == header_functions()


def test_gemm_desc_layout_matches_header():
    """The ctypes struct must mirror tl_gemm_desc field for field."""
    import tl_hip
    text = open(HEADER).read()
    body = re.search(r"typedef struct tl_gemm_desc \{(.*?)\} tl_gemm_desc;", text, re.S).group(1)
    body = re.sub(r"/\*.*?\*/", "", body, flags=re.S)
    names = []
    for decl in body.split(";"):
        decl = decl.strip()
        if not decl:
            continue
        decl = re.sub(r"^(const\s+)?(void\s*\*|double\s*\*|float\s*\*|int64_t|int32_t|float)\s*",
                      "", decl)
        names += [re.sub(r"[\s*]", "", n) for n in decl.split(",")]
    assert names == [f[0] for f in tl_hip._GemmDesc._fields_]


@needs_lib
def test_no_device_is_a_clean_error():
    """This container has no GPU: tl_init must fail with TL_ERR_NO_DEVICE and a message,
    and the Python runtime must raise rather than fall back to the CPU."""
    code = (
        "import sys; sys.path.insert(0, %r)\n"
        "import tl_hip\n"
        "try:\n"
        "    tl_hip.ctx()\n"
        "except tl_hip.NoDeviceError as e:\n"
        "    print('NODEV', e)\n"
        "else:\n"
        "    print('HAVE_DEVICE')\n" % PKG)
    r = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, timeout=120)
    if "HAVE_DEVICE" in r.stdout:
        pytest.skip("a GPU is present")
    assert "NODEV" in r.stdout, r.stdout + r.stderr
    assert "device" in r.stdout.lower()


@needs_lib
def test_null_arguments_are_rejected_without_a_context():
    lib = ctypes.CDLL(LIB)
    lib.tl_init.argtypes = [ctypes.c_int, ctypes.c_void_p]
    lib.tl_last_error.restype = ctypes.c_char_p
    assert lib.tl_init(0, None) == 1  # TL_ERR_INVALID
    assert b"null" in lib.tl_last_error()
    lib.tl_sync.argtypes = [ctypes.c_void_p]
    assert lib.tl_sync(None) == 1


def test_missing_library_fails_loudly(tmp_path):
    code = (
        "import os, sys; os.environ['TL_LIBRARY'] = %r; sys.path.insert(0, %r)\n"
        "import tl_hip\n"
        "try:\n"
        "    tl_hip.load_library()\n"
        "except ImportError as e:\n"
        "    print('IMPORTERROR', e)\n" % (str(tmp_path / "nope.so"), PKG))
    r = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, timeout=120)
    assert "IMPORTERROR" in r.stdout, r.stdout + r.stderr


def test_other_runtimes_are_refused():
    for value in ("CUDA", "CPU"):
        code = "import os, sys; os.environ['XP_RUNTIME'] = %r; sys.path.insert(0, %r)\nimport backend\n" % (value, PKG)
        r = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, timeout=120)
        assert r.returncode != 0 and "MI355X" in r.stderr


def test_host_bf16_conversion_matches_oracle():
    import tl_hip
    from oracle import numpy_ref as ref
    x = np.random.default_rng(0).standard_normal(10000).astype(np.float32) * 100
    x[:4] = [np.inf, -np.inf, 0.0, -0.0]
    assert np.array_equal(tl_hip.f32_to_bf16_bits(x), ref.bf16_bits(x))
    bits = tl_hip.f32_to_bf16_bits(x)
    assert np.array_equal(tl_hip.bf16_bits_to_f32(bits), ref.from_bf16_bits(bits))


def test_dtype_mapping():
    import tl_hip
    assert tl_hip.as_dtype(np.float64) is tl_hip.float32
    assert tl_hip.as_dtype(np.uint8) is tl_hip.uint8
    assert tl_hip.as_dtype(np.int64) is tl_hip.int64
    assert tl_hip.as_dtype(np.int16) is tl_hip.int32
    assert tl_hip.as_dtype("bf16") is tl_hip.bfloat16
    with pytest.raises(TypeError):
        tl_hip.as_dtype(np.complex64)


SAN_LIB = os.path.join(PKG, "csrc", "_build", "san", "libtl_san.so")


def _asan_runtime():
    r = subprocess.run(["/opt/rocm/bin/hipcc", "-print-file-name=libclang_rt.asan-x86_64.so"],
                       capture_output=True, text=True)
    path = r.stdout.strip()
    return path if r.returncode == 0 and os.path.isabs(path) and os.path.exists(path) else None


def test_abi_host_paths_under_address_and_ub_sanitizers():
    """Every exported entry point, called the way a binding could get it wrong (null context,
    null pointers, zero sizes) and through the no-device path, in a host build instrumented
    with ASan and UBSan: each returns a status with a message and no sanitizer reports."""
    # incremental: rebuilt when a source or header is newer than the instrumented library
    r = subprocess.run(["make", "-C", os.path.join(PKG, "csrc"), "san", "-j8"],
                       capture_output=True, text=True, timeout=600)
    if r.returncode != 0:
        pytest.skip("sanitizer build unavailable: " + r.stderr[-500:])
    rt = _asan_runtime()
    if rt is None:
        pytest.skip("clang ASan runtime not found")
    code = (
        "import ctypes, sys; sys.path.insert(0, %r)\n"
        "import tl_hip\n"
        "lib = tl_hip.load_library()\n"
        "assert lib.tl_version() >= 1\n"
        "n = ctypes.c_int(-1)\n"
        "rc = lib.tl_device_count(ctypes.byref(n)); print('count', rc, n.value)\n"
        "h = ctypes.c_void_p()\n"
        "rc = lib.tl_init(0, ctypes.byref(h)); print('init', rc, lib.tl_last_error())\n"
        "assert rc != 0 and lib.tl_last_error()\n"
        "for name, argtypes in tl_hip.SIGNATURES.items():\n"
        "    if name in ('tl_version', 'tl_last_error'):\n"
        "        continue\n"
        "    args = []\n"
        "    for t in argtypes:\n"
        "        if t is ctypes.c_void_p or hasattr(t, '_type_') and not isinstance(t._type_, str):\n"
        "            args.append(None)\n"
        "        elif t in (ctypes.c_float, ctypes.c_double):\n"
        "            args.append(0.0)\n"
        "        else:\n"
        "            args.append(0)\n"
        "    rc = getattr(lib, name)(*args)\n"
        "    assert 0 <= rc <= 6, (name, rc)\n"
        "    if name != 'tl_event_destroy':\n"
        "        assert rc != 0 and lib.tl_last_error(), name\n"
        "print('SAN_OK')\n" % PKG)
    env = dict(os.environ, TL_LIBRARY=SAN_LIB, LD_PRELOAD=rt,
               ASAN_OPTIONS="detect_leaks=0:abort_on_error=1",
               UBSAN_OPTIONS="halt_on_error=1:print_stacktrace=1")
    r = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, timeout=300,
                       env=env)
    out = r.stdout + r.stderr
    assert r.returncode == 0 and "SAN_OK" in r.stdout, out[-3000:]
    assert "AddressSanitizer" not in out and "runtime error" not in out, out[-3000:]


class _Memory:
    """Stands in for a device buffer where only the geometry of a tensor is looked at."""

    def __init__(self, nbytes):
        self.ptr, self.nbytes, self.version = 1 << 20, nbytes, 0


def test_reshapes_check_sizes():
    """Views of another size are refused, by reshape and by the layers' own reshapes; a residual of
    another size too (its rows would be read past their end)."""
    import layers
    import tl_hip as xp
    t = xp.DeviceTensor((2, 3, 8), "fp32", buf=_Memory(192))
    assert t._rows().shape == (6, 8) and t.reshape(-1, 24).nrows == 2
    for shape, rows, cols in (((2, 3, 4), 6, 4), ((5, 8), 5, 8), ((2, 4, 8), 8, 8)):
        with pytest.raises(ValueError):
            t._reshaped(shape, rows, cols)
        with pytest.raises(ValueError):
            t.reshape(shape)
    assert layers._residual_rows(t, 6, 8).shape == (6, 8)
    assert layers._residual_rows(t, 12, 4).shape == (12, 4)
    for rows, cols in ((7, 8), (5, 8), (6, 16)):
        with pytest.raises(ValueError):
            layers._residual_rows(t, rows, cols)
    padded = xp.DeviceTensor((6, 4), "fp32", pitch=8, buf=_Memory(192))
    with pytest.raises(ValueError):
        layers._residual_rows(padded, 3, 8)


@pytest.mark.parametrize("shape,to,rows", [((0, 5), (0, 3, 5), 0), ((3, 0), (7, 0), 7), ((2, 0), (0,), 1),
                                           ((1, 1), (), 1), ((), (1, 1), 1), ((4, 6), (2, 2, 6), 4)])
def test_reshape_geometry(shape, to, rows):
    import tl_hip as xp
    t = xp.DeviceTensor(shape, "fp32", buf=_Memory(96)).reshape(to)
    assert (t.shape, t.nrows, t.ncols) == (to, rows, to[-1] if to else 1)


class _FakeContext:
    """A context whose graphs launch nothing; `capture` is set as xp.capture sets it."""

    class lib:
        @staticmethod
        def tl_graph_launch(handle, graph):
            return 0

        tl_graph_destroy = tl_graph_launch

    handle, capture = 1, None


def test_graphs_keep_and_remake_the_copies_they_read(monkeypatch):
    """A copy that a captured call found current keeps its address and is made again before a launch
    when a source was written, whether or not an eager call did so first; a copy that it did not
    find current is made inside the capture, once, and leaves the kept one alone."""
    import tl_hip as xp
    c = _FakeContext()
    monkeypatch.setattr(xp, "_ctx", c)
    source, slots, made = xp.DeviceTensor((4, 4), "fp32", buf=_Memory(64)), {}, []

    def make(out):
        made.append(out)
        return out if out is not None else object()

    def copy():
        return xp.derived(slots, None, source._version, (source,), make, copy)

    class Open:
        def __init__(self):
            self._derived, self._recorded = {}, {}

    def captured():
        c.capture = cap = Open()
        first, second = copy(), copy()
        c.capture = None
        assert first is second
        return first, xp.Graph(7, cap._derived.values())

    source._version += 1
    recorded, graph = captured()  # nothing kept yet
    assert made == [None] and not slots
    graph.launch()
    kept = copy()
    assert kept is not recorded and made == [None, None]
    read, graph = captured()
    assert read is kept and len(made) == 2 and [copy_ for _, copy_ in graph._remake] == [kept]
    graph.launch()
    assert len(made) == 2  # still current
    source._version += 1
    graph.launch()
    graph.launch()
    assert made[2:] == [kept]  # in place, once
    source._version += 1
    assert copy() is kept and made[2:] == [kept] * 2
    graph.launch()
    assert len(made) == 4
    source._version += 1
    c.capture = Open()
    assert copy() is not kept  # written since: the capture records the making
    c.capture = None
    graph.launch()
    assert made[-1] is kept and copy() is kept
    graph.destroy()


@needs_lib
def test_few_row_products_of_long_k_keep_the_weight_stream():
    """Up to 16 rows over a wide weight: the streaming kernels where they are the faster ones (K a
    multiple of 2048; one to three rows on K beyond 768), gemm_rows_kernel elsewhere."""
    class Rows(ctypes.Structure):
        _fields_ = [("tile", ctypes.c_int), ("splits", ctypes.c_int), ("us", ctypes.c_float)]

    plan = getattr(ctypes.CDLL(LIB), "_ZN2tl14gemm_rows_planElllib")
    plan.restype, plan.argtypes = Rows, [ctypes.c_int64] * 3 + [ctypes.c_int, ctypes.c_bool]
    for M, N, K, here in ((4, 50257, 2048, False), (1, 256000, 2048, False), (16, 32768, 4096, False),
                          (2, 50257, 1024, False), (3, 256000, 1536, False), (16, 32767, 256, False),
                          (1, 50257, 768, True), (4, 50257, 1024, True), (16, 256000, 1024, True),
                          (17, 50257, 2048, True)):
        assert (plan(M, N, K, 256, True).tile >= 0) == here, (M, N, K)
    assert plan(4, 50257, 4096, 256, False).tile >= 0  # without workspace for the stream's K parts
