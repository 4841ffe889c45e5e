"""CPU checks of the C ABI library: it loads without a GPU and exports every
symbol include/hearth_hip.h declares; the product path has no CPU fallback."""
import ctypes as C
import os
import re

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def declared_symbols():
    txt = open(os.path.join(ROOT, "include", "hearth_hip.h")).read()
    txt = re.sub(r"/\*.*?\*/", "", txt, flags=re.S)
    return sorted(set(re.findall(r"\b(hh_[a-z0-9_]+)\s*\(", txt)))


def test_header_declares_the_binding_surface():
    from hearth_amd.lib import exported_symbols
    assert sorted(exported_symbols()) == declared_symbols()


def test_library_exports_every_declared_symbol():
    from hearth_amd.lib import lib_path
    if not os.path.exists(lib_path()):
        pytest.fail("libhearth_hip.so not built (run __graft_entry__.build())")
    lib = C.CDLL(lib_path())
    missing = [s for s in declared_symbols() if not hasattr(lib, s)]
    assert not missing, missing


def test_version_and_error_channel_without_gpu():
    from hearth_amd.lib import load_library
    lib = load_library()
    assert b"gfx950" in lib.hh_version()
    # a null output pointer is rejected before any device call
    rc = lib.hh_ctx_create(0, None)
    assert rc == 1 and b"null" in lib.hh_last_error()
    cfg_rc = lib.hh_model_create(None, None, None)
    assert cfg_rc == 1


def test_operator_pointers():
    """Raw addresses pass through as they are; None is a null pointer; a host tensor
    gives its own address without a device being asked."""
    import torch
    from hearth_amd.lib import _ptrs
    x = torch.zeros(4)
    assert tuple(_ptrs(1 << 40, 2, 3)) == (1 << 40, 2, 3)
    assert tuple(_ptrs(x, None, 7, x)) == (x.data_ptr(), 0, 7, x.data_ptr())


def test_gemm_plan():
    """The GEMM's choice of a form needs no device: shallow products keep away from the
    expanded forms, deep ones with many tokens take them, matrices past the expansion's
    scratch in whole 256-row tiles; what the GEMM refuses is refused."""
    from hearth_amd.lib import HHError, gemm_plan
    for t in (41, 42, 143):
        assert gemm_plan(t, 2048, 2048, 8) == (0, 2048)
        assert gemm_plan(t, 24576, 1024, 64) == (1, 24576)
        assert gemm_plan(t, 24576, 4096, 2048) == (4, 24576)
        form, rows = gemm_plan(t, 34816, 17408, 2048)
        assert form >= 2 and rows < 34816 and rows % 256 == 0
        for seq in (1, 200, 1 << 20):   # the widest matrices and longest rows
            assert gemm_plan(t, 1 << 30, 128, seq)[1] > 0 and gemm_plan(t, 1, (1 << 31) - 128, seq)[1] == 1
    # int8 MFMA took 12.3 us: straight from the blocks 10.4, expanded 13.2
    assert gemm_plan(42, 6144, 1024, 224) == (1, 6144)
    assert gemm_plan(8, 4096, 4096, 512) == (6, 4096)
    for args, status in (((2, 4, 128, 2), 2), ((42, 4, 100, 2), 3), ((42, 0, 128, 2), 3), ((42, 4, 128, 0), 3),
                         ((42, 4, 1 << 32, 300), 3)):
        with pytest.raises(HHError) as e:
            gemm_plan(*args)
        assert e.value.status == status


def test_no_oracle_in_product():
    """The product package never imports or loads the oracle."""
    pkg = os.path.join(ROOT, "hearth_amd")
    for dirpath, _, files in os.walk(pkg):
        for f in files:
            if f.endswith((".py", ".hip", ".h", ".cpp")):
                txt = open(os.path.join(dirpath, f)).read()
                assert "oracle" not in txt.lower(), f
