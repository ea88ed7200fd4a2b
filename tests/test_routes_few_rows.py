"""Which kernel a few rows take with nothing tuned: the one that measured faster (cold weights, us)."""
import ctypes

import pytest

import torchlette_amd as T
from torchlette_amd import _lib as L

INT4, INT8, ROW = (L.FMT_INT4_GROUPED, 32), (L.FMT_INT8_GROUPED, 64), (L.FMT_INT8_ROW, 0)


def chosen(fmt, n, k, m, x, cache=None):
    lib = L.load()
    before = T.exportTuningCache()
    buf = ctypes.create_string_buffer(64)
    ptr = ctypes.cast(buf, ctypes.c_void_p).value
    w, c = L.QWeight(*fmt, n, k, ptr, ptr), L.KernelConfig()
    try:
        T.clearTuningCache()
        if cache is not None:
            T.importTuningCache(cache)
        assert lib.tlhip_selected_config(ctypes.byref(w), x, m, x, ctypes.byref(c)) == 0
    finally:
        T.clearTuningCache()
        T.importTuningCache(before)
    return c.as_tuple()


def whole(c):  # all of K in a workgroup
    return c[0] == L.VARIANT_GEMV_MFMA and c[2] == 0 and c[5] > 0


@pytest.mark.parametrize("fmt,n,k,m,all_of_k", [
    # K slices or the VALU kernel / all of K in a workgroup
    (INT4, 4096, 12288, 16, True),    # 12.3 / 13.8, and 1.7 more with the code cold
    (INT8, 2048, 12288, 16, False),   # 10.1 / 13.0
    (ROW, 2048, 12288, 16, False),    # 10.1 / 12.9
    (INT8, 4096, 12288, 16, False),   # 14.2 / 16.9
    (INT4, 24576, 4096, 8, False),    # 16.1 / 18.9
    (INT4, 768, 16384, 16, False),    # 9.8 / 12.1
    (INT4, 1024, 4096, 2, True),      # 3.7 / 4.2, and 1.7 more with the code cold
    (INT4, 24576, 4096, 3, False),    # 15.1 / 17.4
    (ROW, 14336, 3072, 2, False),     # 9.9 / 11.2
    (INT4, 4096, 4096, 16, True),     # 6.7 / 6.6, with a residual 7.6 / 6.5
    (INT4, 1024, 4096, 8, True),      # 6.1 / 4.5
    (INT8, 4096, 4096, 8, True),      # 7.3 / 6.3
    (INT8, 1024, 12288, 8, True),     # 11.0 / 8.1
    (INT8, 12288, 4096, 2, True),     # 13.0 / 11.7
])
def test_up_to_sixteen_f16_rows(fmt, n, k, m, all_of_k):
    assert whole(chosen(fmt, n, k, m, L.F16)) == all_of_k


@pytest.mark.parametrize("n,k,all_of_k", [(4096, 8192, True), (2048, 12288, False)])
def test_a_neighbours_k_slices_are_weighed_at_a_problems_own_prices(n, k, all_of_k):
    """Sixteen rows of int4 beside a winner in K slices at 4096 x 12288 (2048 x 12288: 12.0 us in those, 9.4 in its own)."""
    cache = '{"version":1,"entries":{"16_4096_12288_int4-grouped_g32_f16_f16":[1,8,2,2,4,0,1,0]}}'
    assert chosen(INT4, 4096, 12288, 16, L.F16, cache) == (1, 8, 2, 2, 4, 0, 1, 0)
    c = chosen(INT4, n, k, 16, L.F16, cache)
    assert whole(c) == all_of_k and c == chosen(INT4, n, k, 16, L.F16), c


@pytest.mark.parametrize("fmt,n,k,x,own_kernel", [
    # the VALU kernel / the kernel for one row
    (INT4, 16384, 14336, L.F16, False),   # 28.2 / 32.7
    (INT4, 6144, 14336, L.F16, True),     # 14.9 / 14.1
    (INT4, 12288, 9728, L.F32, False),    # 19.7 / 24.1
    (INT4, 4096, 9728, L.F32, True),      # 9.6 / 9.8
    (INT8, 16384, 7168, L.F32, False),    # 22.6 / 25.5
    (INT8, 8192, 8192, L.F32, True),      # 15.2 / 14.9
    (ROW, 12288, 7168, L.F16, True),      # 17.0 / 16.6
    (INT4, 12288, 4096, L.F16, True),
])
def test_one_row(fmt, n, k, x, own_kernel):
    c = chosen(fmt, n, k, 1, x)
    assert c[0] == L.VARIANT_GEMV and (c[6] == 3) == own_kernel, c


@pytest.mark.parametrize("fmt,n,k,m,form", [
    # all of K in a workgroup on the matrix cores / K slices there / the VALU
    (ROW, 5120, 12288, 6, "slices"),    # 30.1 / 21.4
    (ROW, 4096, 14336, 12, "slices"),   # 31.9 / 24.7
    (INT8, 4096, 8192, 10, "whole"),    # 15.1 / 19.3
    (ROW, 4096, 8192, 8, "whole"),      # 13.3 / 14.1
    (INT4, 768, 9728, 4, "whole"),      # 10.4 / 19.0
    (INT4, 1024, 9728, 2, "valu"),      # 10.0 / - / 8.0
    (INT4, 8192, 3072, 2, "valu"),      # 8.9 in one launch of all of K on the VALU, 7.7
    (INT8, 10240, 1536, 2, "valu"),     # 7.6, 6.0
    (INT8, 4096, 1024, 2, "some"),      # 4.4, 4.4
    (ROW, 1024, 16384, 2, "whole"),     # 13.1 / - / 18.7
])
def test_a_few_f32_rows(fmt, n, k, m, form):
    c = chosen(fmt, n, k, m, L.F32)
    got = ("whole" if c[2] else "slices") if c[0] == L.VARIANT_GEMV_F32 else ("some" if c[6] == 4 else "valu")
    assert got == form, c


@pytest.mark.parametrize("fmt,n,k,m,all_of_k", [
    # K slices (or none) of the skinny kernel / all of K in a workgroup
    (INT4, 24576, 2048, 32, False),   # 14.0 / 20.9
    (ROW, 768, 16384, 32, False),     # 12.2 / 16.4
    (INT4, 20480, 1024, 32, False),   # 9.8 / 12.6
    (INT8, 28672, 1024, 24, False),   # 13.0 / 16.5
    (INT8, 1024, 16384, 32, False),   # 13.8 / 16.9
    (INT4, 20480, 11008, 24, True),   # three blocks of columns 50.5, one 69.3
    (INT4, 4096, 8192, 17, True),     # 13.2 / 10.6
    (ROW, 5120, 1536, 40, True),      # 9.3 / 7.4
    (INT4, 14336, 1536, 17, True),    # 9.8 / 8.3
])
def test_17_to_64_f16_rows(fmt, n, k, m, all_of_k):
    lib = L.load()
    before = T.exportTuningCache()
    buf = ctypes.create_string_buffer(64)
    ptr = ctypes.cast(buf, ctypes.c_void_p).value
    w, rows, first, last = L.QWeight(*fmt, n, k, ptr, ptr), ctypes.c_int64(), L.KernelConfig(), L.KernelConfig()
    try:
        T.clearTuningCache()
        assert lib.tlhip_selected_route(ctypes.byref(w), L.F16, m, L.F16, ctypes.byref(rows), ctypes.byref(first), ctypes.byref(last)) == 0
    finally:
        T.clearTuningCache()
        T.importTuningCache(before)
    c = last.as_tuple()
    assert c[0] == L.VARIANT_GEMV_MFMA and whole(c) == all_of_k, c
    assert (n, k) != (20480, 11008) or c[5] == 3, c
