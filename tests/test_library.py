"""The C-ABI library: built, loadable on a CPU-only host, and exporting every
symbol include/axm.h declares (no compute calls here)."""

import ctypes
import os
import re

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HEADER = os.path.join(ROOT, "include", "axm.h")
LIB = os.path.join(ROOT, "axiomlm_amd", "libaxm.so")


def declared_functions():
    text = open(HEADER).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    names = re.findall(r"\b(axm_[a-z0-9_]+)\s*\(", text)
    return sorted(set(names))


def test_header_declares_entry_points():
    names = declared_functions()
    for n in ["axm_qmv_q4_marlin", "axm_gqa_flash_decode", "axm_gqa_tree_verify", "axm_runner_step",
              "axm_runner_create", "axm_kv_cache_write", "axm_pack_q4_marlin_rtn"]:
        assert n in names


def test_library_loads_and_exports_all_declared_symbols():
    if not os.path.exists(LIB):
        pytest.fail(f"{LIB} not built (run __graft_entry__.build())")
    import torch  # noqa: F401  (binds the HIP runtime torch ships)

    lib = ctypes.CDLL(LIB)
    missing = [n for n in declared_functions() if not hasattr(lib, n)]
    assert not missing, f"symbols declared in axm.h but not exported: {missing}"


def test_python_binding_covers_header():
    from axiomlm_amd import _lib

    bound = set(_lib.exported_symbols())
    missing = [n for n in declared_functions() if n not in bound]
    assert not missing, f"declared but not bound in _lib.py: {missing}"


def test_error_path_without_gpu_compute():
    # Argument validation runs on the host: a bad K is rejected before any launch.
    from axiomlm_amd import _lib

    rc = _lib.lib().axm_qmv_q4_marlin(ctypes.c_void_p(16), ctypes.c_void_p(16), ctypes.c_void_p(16), None,
                                      ctypes.c_void_p(16), 1, 100, 8, None)
    assert rc != 0
    assert b"multiple of 64" in _lib.lib().axm_last_error()


def test_many_row_workspace_covers_the_64_row_passes():
    # Rows of x that the many-row GEMM cannot load (not 16-byte aligned) run in passes of 64,
    # which refuse a workspace smaller than their own: the size for M rows is enough for both.
    from axiomlm_amd import _lib

    L = _lib.lib()
    for M, N, K in [(1000, 12288, 4096), (128, 12288, 4096), (100, 4096, 11008), (130, 4096, 1024), (2048, 4096, 4096)]:
        for swiglu in (0, 1):
            one = L.axm_qmm_q4_tile16_workspace_bytes(K, N, swiglu)
            assert L.axm_qmm_q4_tile16_rows_workspace_bytes(M, K, N, swiglu) >= one
            assert L.axm_qmm_q4_tile16_rows_workspace_bytes(64, K, N, swiglu) == one


def test_wrappers_skip_the_several_row_entry_only_where_it_would_run_the_gemv():
    # The Python products call the GEMV entry without a workspace query up to these rows; the rows from
    # which the library takes the several-row kernel are its own (a workspace is asked for only then, and these
    # shapes split K there).
    from axiomlm_amd import _lib

    L = _lib.lib()
    q8, affine, ternary, gguf, marlin = range(5)
    for N, K in [(512, 4096), (1024, 11008), (4096, 4096)]:
        for fmt in (q8, marlin):
            assert L.axm_qmm_codes_workspace_bytes(fmt, 5, K, N) > 0
        for fmt in (q8, affine, ternary, gguf, marlin):
            for M in range(1, 5):
                assert L.axm_qmm_codes_workspace_bytes(fmt, M, K, N) == 0
    for M in range(1, 5):  # MARLIN from 32 Mi weights on: two rows
        assert (L.axm_qmm_codes_workspace_bytes(marlin, M, 32768, 1024) > 0) == (M > 1)
        assert L.axm_qmm_codes_workspace_bytes(marlin, M, 32768, 1016) == 0
