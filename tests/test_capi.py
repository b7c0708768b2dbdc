"""The C-ABI library loads and exports every symbol include/ditk.h declares (no GPU calls)."""
import ctypes
import os
import re

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HEADER = os.path.join(ROOT, "include", "ditk.h")


def declared_symbols():
    text = open(HEADER).read()
    return sorted(set(re.findall(r"^\s*(?:const\s+)?[\w\*]+\s+\**(ditk_\w+)\s*\(", text, re.M)))


def test_header_declares_entry_points():
    syms = declared_symbols()
    assert "ditk_flash_attn_varlen" in syms and "ditk_gemm" in syms and len(syms) >= 15


def test_library_exports_every_declared_symbol():
    from ditserve_amd import _lib
    if not _lib.LIB_PATH.exists():
        pytest.skip("libditk.so not built (run python -m ditserve_amd.build)")
    lib = ctypes.CDLL(str(_lib.LIB_PATH))
    missing = [s for s in declared_symbols() if not hasattr(lib, s)]
    assert not missing, missing
    # and the Python binding table covers exactly the declared ABI
    assert sorted(_lib.SIGNATURES) == declared_symbols()
    assert lib.ditk_version() == 1


def test_ops_reject_cpu_tensors_before_launch():
    import torch
    from ditserve_amd import ops
    x = torch.zeros(4, 64, dtype=torch.bfloat16)
    with pytest.raises(ValueError):
        ops.adaln(x)
    with pytest.raises(ValueError):
        ops.linear(x, torch.zeros(8, 64, dtype=torch.bfloat16))


def test_table_pair_check_refuses_shared_outputs():
    """The two workgroups of ditk_check_cu_seqlens_pair run at once: an output may be no
    input and not the other output (refused before any launch; addresses only)."""
    from ditserve_amd import _lib
    if not _lib.LIB_PATH.exists():
        pytest.skip("libditk.so not built (run python -m ditserve_amd.build)")
    lib = _lib.load()
    a, b, c, d, st = (0x1000 * i for i in range(1, 6))
    for cu0, out0, cu1, out1 in ((a, a, b, c), (a, b, c, c), (a, b, c, b), (a, b, b, c), (a, b, c, a)):
        assert lib.ditk_check_cu_seqlens_pair(cu0, 10, out0, cu1, 10, out1, 2, st, None) == 1
        assert b"tables of their own" in lib.ditk_last_error()
