"""CPU checks of the C-ABI library: it builds, loads, and exports every entry
point include/qma_gpu.h declares; without a GPU it reports unavailability
(no compute calls are made here)."""
import os
import re

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HEADER = os.path.join(ROOT, "include", "qma_gpu.h")


def declared_functions():
    src = open(HEADER).read()
    src = re.sub(r"/\*.*?\*/", "", src, flags=re.S)
    names = re.findall(r"\b((?:qmag?_|dequantize_row_|dot_q)[A-Za-z0-9_]+)\s*\(", src)
    return sorted(set(names))


@pytest.fixture(scope="module")
def built():
    import qmag
    if not os.path.exists(qmag.LIB_PATH):
        import build as b
        b.build()
    return qmag


def test_header_declares_reference_entries():
    names = declared_functions()
    for ref in ("qma_q8k_available", "qma_q8k_quant", "qma_q8k_dot", "qma_q8k_gateup",
                "dequantize_row_q4_K", "dequantize_row_q6_K", "dot_q4_K_f32", "dot_q6_K_f32"):
        assert ref in names


def test_library_exports_every_declared_symbol(built):
    import ctypes
    L = ctypes.CDLL(built.LIB_PATH)
    missing = [n for n in declared_functions() if not hasattr(L, n)]
    assert not missing, missing


def test_python_binding_covers_header(built):
    assert sorted(built.SIGNATURES) == declared_functions()


def test_no_gpu_reports_unavailable(built):
    L = built.lib()
    st = L.qmag_init(0)
    if st == 0:
        pytest.skip("a gfx950 GPU is visible")
    assert st == -3
    assert L.qma_q8k_available() == 0
    assert b"gfx950" in L.qmag_last_error() or b"device" in L.qmag_last_error()


def test_no_gpu_q8k_entries_are_the_reference_stubs(built):
    """Without a usable device the q8k entries do what the reference's build
    without dotprod does (q8k.c:280-316): qma_q8k_quant writes nothing,
    qma_q8k_gateup gives 0.0f twice, qma_q8k_dot gives 0.0f -- and the process
    keeps running."""
    import ctypes as C

    import numpy as np
    L = built.lib()
    if L.qmag_init(0) == 0:
        pytest.skip("a gfx950 GPU is visible")
    n = 512
    x = np.ones(n, np.float32)
    xq = np.full(n, 7, np.int8)
    xd = np.full(n // 256, 3.0, np.float32)
    xs = np.full(n // 16, 5, np.int16)
    p = lambda a: a.ctypes.data_as(C.c_void_p)
    L.qma_q8k_quant(p(x), n, p(xq), p(xd), p(xs))
    assert (xq == 7).all() and (xd == 3.0).all() and (xs == 5).all()
    row = np.full(2 * 144, 0x11, np.uint8)
    assert L.qma_q8k_dot(p(row), 12, p(xq), p(xd), p(xs), n) == 0.0
    g, u = C.c_float(9.0), C.c_float(9.0)
    L.qma_q8k_gateup(p(row), p(row), p(xq), p(xd), p(xs), n, C.byref(g), C.byref(u))
    assert g.value == 0.0 and u.value == 0.0


def test_no_gpu_f32_entries_abort_with_a_message(built):
    """The quants.c entries have no unavailable form in the reference (it
    always computes them), so without a device they abort with a message
    rather than return a wrong value (run in a child process)."""
    import subprocess
    import sys
    code = ("import ctypes as C, numpy as np, qmag\n"
            "L = qmag.lib()\n"
            "assert L.qmag_init(0) != 0\n"
            "w = np.zeros(144, np.uint8); x = np.zeros(256, np.float32)\n"
            "L.dot_q4_K_f32(w.ctypes.data_as(C.c_void_p), x.ctypes.data_as(C.c_void_p), 256)\n"
            "print('returned')\n")
    L = built.lib()
    if L.qmag_init(0) == 0:
        pytest.skip("a gfx950 GPU is visible")
    env = dict(os.environ, PYTHONPATH=os.path.join(ROOT, "qwen-mobile-agent_amd"))
    r = subprocess.run([sys.executable, "-c", code], env=env, capture_output=True, text=True, timeout=120)
    assert r.returncode != 0 and "returned" not in r.stdout
    assert "dot_q4_K_f32 called without a usable gfx950 device" in r.stderr


def test_matrix_core_lines_stay_within_a_grid(built):
    """A launch holds fewer than 2^32 threads in x: the fp32 matrix-core kernel
    has a workgroup of up to 512 threads per 16 rows, so from 2^27 rows on the
    one-token kernel (its grid is bounded) has to take the call."""
    import ctypes as C
    L = C.CDLL(built.LIB_PATH)
    line = L["_ZN4qmag13mmf_supportedEiiii"]        # bool qmag::mmf_supported(nb, n_out, T, wtype)
    line.restype = C.c_bool
    for wtype in (12, 14):
        assert line(8, (1 << 27) - 1, 4, wtype)
        assert not line(8, 1 << 27, 4, wtype) and not line(1, (1 << 31) - 1, 65535, wtype)


@pytest.mark.parametrize("lang", ["c", "c++"])
def test_header_compiles_alone(lang, tmp_path):
    """qma_gpu.h is valid C99 and C++ on its own (an engine includes it from
    C; a C++ caller gets extern "C" linkage)."""
    import shutil
    import subprocess
    cc = shutil.which("gcc" if lang == "c" else "g++")
    if not cc:
        pytest.skip("no host compiler")
    src = tmp_path / ("h.c" if lang == "c" else "h.cpp")
    src.write_text('#include "qma_gpu.h"\nint main(void) { return qmag_init(0) == 0 ? 0 : 1; }\n')
    std = "-std=c99" if lang == "c" else "-std=c++17"
    r = subprocess.run([cc, std, "-Wall", "-Wextra", "-Werror", "-fsyntax-only", "-I", os.path.join(ROOT, "include"),
                        str(src)], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr


def test_header_compiles_after_the_engine_header(tmp_path):
    """Included after the engine's own qma.h (where the reference tree is
    present), the header adds no conflicting declaration: the compatible
    entries' prototypes are the engine's, and the quants.c ones are skipped
    in favour of the engine's typed ones."""
    import shutil
    import subprocess
    ref = "/root/reference/src"
    if not os.path.exists(os.path.join(ref, "qma.h")) or not shutil.which("gcc"):
        pytest.skip("the engine's header is not available here")
    src = tmp_path / "both.c"
    src.write_text('#include "qma.h"\n#include "qma_gpu.h"\nint main(void) { return qma_q8k_available(); }\n')
    r = subprocess.run(["gcc", "-std=gnu11", "-Wall", "-Wextra", "-Werror", "-fsyntax-only", "-I", ref, "-I",
                        os.path.join(ROOT, "include"), str(src)], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
