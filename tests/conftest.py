import ctypes
import importlib.util
import os
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG_DIR = os.path.join(ROOT, "cudanative.jl_amd")
if ROOT not in sys.path:
    sys.path.insert(0, ROOT)


def load_package():
    """Import the package directory `cudanative.jl_amd` under the module name cudanative_jl_amd."""
    name = "cudanative_jl_amd"
    if name in sys.modules:
        return sys.modules[name]
    spec_b = importlib.util.spec_from_file_location("_miw_build", os.path.join(PKG_DIR, "build.py"))
    b = importlib.util.module_from_spec(spec_b)
    spec_b.loader.exec_module(b)
    # The library carries the hash of the sources it was built from.  It is read from the file, not by
    # loading the library: a binary loaded here would stay this process's libmiwmma.so even after a
    # rebuild at the same path, and the tests would then run against the stale kernels.
    if b.built_id() != b.source_id():
        # nothing built yet, or built from other sources: build once (hipcc cross-compiles without a GPU)
        b.build()
    spec = importlib.util.spec_from_file_location(name, os.path.join(PKG_DIR, "__init__.py"),
                                                  submodule_search_locations=[PKG_DIR])
    mod = importlib.util.module_from_spec(spec)
    sys.modules[name] = mod
    spec.loader.exec_module(mod)
    if not os.environ.get("MIWMMA_LIB"):
        loaded = mod._lib.load().miw_build_id().decode()
        if loaded != b.source_id():
            raise RuntimeError("libmiwmma.so in this process has build id %s, the sources have %s" % (loaded, b.source_id()))
    return mod


def pytest_report_header(config):
    try:
        m = load_package()
        return "libmiwmma build id: %s" % m._lib.load().miw_build_id().decode()
    except Exception as e:  # noqa: BLE001
        return "libmiwmma not loadable: %s" % e


def pytest_configure(config):
    config.addinivalue_line("markers", "gpu: needs a real MI355X (run with -m gpu on the GPU box)")


@pytest.fixture(scope="session")
def miw():
    return load_package()


@pytest.fixture(scope="session")
def gpu(miw):
    """Initialised library on device 0.  GPU tests fail (not skip) when the HIP path cannot run."""
    miw.init(0)
    return miw


@pytest.fixture(scope="session")
def orc():
    from oracle import oracle
    oracle.lib()
    return oracle


class _GemmParams(ctypes.Structure):
    """gemm_params of csrc/kernels.hpp, which the library's own dispatch rules take."""
    _fields_ = ([(x, ctypes.c_void_p) for x in "ABCD"] +
                [(x, ctypes.c_long) for x in ("M", "N", "K", "lda", "ldb", "ldc", "ldd", "sa", "sb", "sc", "sd", "batch")] +
                [(x, ctypes.c_int) for x in ("a_row", "b_row", "c_row", "d_row", "use_c")] +
                [("alpha", ctypes.c_float), ("beta", ctypes.c_float)])


@pytest.fixture(scope="session")
def narrow_kernel(miw):
    """narrow_kernel(rule, M, N, K, ...): what the library's own rule `rule` says of the kernel for D with one
    extent of at most 128 ("fits": it can run the problem; "pays": it is faster there than the fragment-op kernels;
    "beats_tiles": than the LDS tiles)."""
    lib = ctypes.CDLL(miw._lib.LIB_PATH)

    def ask(rule, M, N, K, batch=1, a_row=1, b_row=0, c_row=1, d_row=1, use_c=0, d_type=0, f16acc=False, lda=0, ldb=0, ldd=0, offset=0, offset_b=0):
        name = "skinny_" + rule
        f = getattr(lib, "_ZN3miw%d%sERKNS_11gemm_paramsEib" % (len(name), name))
        f.restype, f.argtypes = ctypes.c_bool, [ctypes.POINTER(_GemmParams), ctypes.c_int, ctypes.c_bool]
        lda, ldb = lda or (K if a_row else M), ldb or (N if b_row else K)
        ldc, ldd = N if c_row else M, ldd or (N if d_row else M)
        base = 1 << 32
        p = _GemmParams(base + offset, base + (1 << 40) + offset_b, base + (2 << 40), base + (3 << 40), M, N, K, lda, ldb, ldc, ldd,
                        lda * (M if a_row else K), ldb * (K if b_row else N), ldc * (M if c_row else N), ldd * (M if d_row else N),
                        batch, a_row, b_row, c_row, d_row, use_c, 1.0, 1.0)
        return f(ctypes.byref(p), d_type, f16acc)

    return ask


class _KwaveTile(ctypes.Structure):
    _fields_ = [("bi", ctypes.c_int), ("bj", ctypes.c_int)]


@pytest.fixture()
def shared_k_tile(miw):
    """shared_k_tile(M, N, K, ...): the tile (along D's contiguous dimension, along the other) with which the library's
    own rule takes the kernel whose wavefronts share K, or None."""
    lib = ctypes.CDLL(miw._lib.LIB_PATH)
    f = lib._ZN3miw10kwave_paysERKNS_11gemm_paramsEiibi
    f.restype, f.argtypes = _KwaveTile, [ctypes.POINTER(_GemmParams), ctypes.c_int, ctypes.c_int, ctypes.c_bool, ctypes.c_int]

    def ask(M, N, K, batch=1, a_row=1, b_row=0, c_row=1, d_row=1, use_c=0, c_type=1, d_type=0, in_place=False, lda=0, ldb=0, ldd=0, offset=0, cus=256):
        lda, ldb = lda or (K if a_row else M), ldb or (N if b_row else K)
        ldc, ldd = N if c_row else M, ldd or (N if d_row else M)
        base = 1 << 32
        p = _GemmParams(base + offset, base + (1 << 40), base + (2 << 40), base + (3 << 40), M, N, K, lda, ldb, ldc, ldd,
                        lda * (M if a_row else K), ldb * (K if b_row else N), ldc * (M if c_row else N), ldd * (M if d_row else N),
                        batch, a_row, b_row, c_row, d_row, use_c, 1.0, 1.0)
        t = f(ctypes.byref(p), c_type, d_type, in_place, cus)
        return (t.bi, t.bj) if t.bi else None

    return ask
