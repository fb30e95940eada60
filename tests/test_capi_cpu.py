"""CPU-only checks of the C-ABI library: it loads, exports every symbol that
include/inferflow_amd.h declares, and its registry matches the oracle's."""
import os
import re

import pytest

import inferflow_amd as ia
from inferflow_amd import _capi, dtypes as dt
import oracle as o

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _declared(header="inferflow_amd.h"):
    text = open(os.path.join(ROOT, "include", header)).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(ifa_[a-z0-9_]+)\s*\(", text)))


def test_library_exports_every_declared_symbol():
    L = ia.lib()
    names = _declared()
    assert len(names) >= 30
    for n in names:
        assert hasattr(L, n), "missing symbol " + n


def test_ctypes_signatures_cover_header():
    assert sorted(_capi.SIGNATURES) == _declared()


def test_engine_header_is_exported_and_bound():
    names = _declared("inferflow_engine.h")
    assert sorted(_capi.ENGINE_SIGNATURES) == names and len(names) >= 10
    L = ia.lib()
    for n in names:
        assert hasattr(L, n), "missing symbol " + n


def test_registry_matches_oracle():
    L = ia.lib()
    for d in dt.NAMES:
        assert L.ifa_block_capacity(d) == o.block_capacity(d) == dt.block_capacity(d)
        assert L.ifa_block_bytes(d) == o.block_bytes(d) == dt.block_bytes(d)
        for cols in (64, 4096, 11008):
            assert L.ifa_row_bytes(d, cols) == o.row_bytes(d, cols) == dt.row_bytes(d, cols)
    assert L.ifa_block_capacity(99) == 0


@pytest.mark.parametrize("name,expect", [
    ("q4", dt.Q4_B32T1A), ("Q3H", dt.Q3H_B64T1), ("q8", dt.Q8_B32T2), ("q3", dt.Q3_B32T1B),
    ("q2", dt.Q2_B32T1B), ("fp16", dt.F16), ("q6", dt.Q6_B64T1), ("q5", dt.Q5_B64T1),
    ("q4_b32t1", dt.Q4_B32T1A), ("nope", -1)])
def test_dtype_names(name, expect):
    # TensorCommon::InitElementTypeMap, src/tensor/tensor_common.cc:171-205
    assert ia.lib().ifa_dtype_from_name(name.encode()) == expect


@pytest.mark.parametrize("cols", [128, 4096, 20480, 28672])
def test_rows_products_decline_matrices_whose_copies_pass_32_bit_offsets(cols):
    """the layouts' own sizes on both sides of 4 GiB: operand-order copies of 16 rows x 128 columns are a KiB of codes and, by four of them, a KiB of (base, scale) words -- twice
    where products of many rows read them (2) --, tiled rows (0) 20 bytes a block of 32 and room"""
    import ctypes as C
    f = ia.lib().ifa_gemm_rows_offsets_fit
    f.argtypes, f.restype = [C.c_size_t, C.c_size_t, C.c_int], C.c_int
    sup = cols // 128
    for kind in (1, 2):
        tile = 1024 * (sup + kind * ((sup + 3) // 4))
        most = ((1 << 32) - 1) // tile * 16                      # rows of the largest copy below 4 GiB
        assert f(most, cols, kind) == 1 and f(most + 1, cols, kind) == 0
        assert f(16, cols, kind) == 1
    room = ((1 << 32) - 1) // (20 * (cols // 32 + 16)) - 16
    assert f(room, cols, 0) == 1 and f(room + 1, cols, 0) == 0


def test_errors_are_codes_not_exceptions():
    L = ia.lib()
    # argument validation happens before any HIP call, so this is safe without a GPU
    assert L.ifa_quantize(dt.Q4_B32T1A, None, 1, 32, None, None) == -1
    assert b"null" in L.ifa_last_error()
    assert L.ifa_gemv(dt.F32, 1, 1, 32, dt.F16, 1, None, 1, None) == -1
    assert L.ifa_device_count() >= 0


def test_shared_expert_goes_beside_the_experts_where_one_launch_is_no_slower():
    import ctypes as C
    pays = ia.lib().ifa_moe_shared_pays
    pays.restype, pays.argtypes = C.c_bool, [C.c_size_t] * 3
    assert all(pays(t, 1024, 1408) and pays(t, 6144, 4096) for t in range(1, 9))
    assert pays(2, 8192, 8192) and not any(pays(t, 8192, 8192) or pays(t, 4096, 8192) for t in range(3, 9))
