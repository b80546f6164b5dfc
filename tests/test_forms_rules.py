"""The rules that choose a kernel form by a call's sizes (CPU: the library's own functions, no launch), at sizes where both
forms were measured on the GPU and one of them is slower."""
import ctypes

import pytest

from rustingstrata_amd import backend

CUS = 256


def rule(name, *argtypes):
    f = getattr(backend.lib(), name)
    f.argtypes, f.restype = argtypes, ctypes.c_int
    return f


@pytest.mark.parametrize("n,rows,form", [
    # few positions of a tall matrix: the ring forms take whole blocks of 64 positions (176 us against 56)
    (2, 16384, 0), (5, 16384, 0), (8, 16384, 0), (17, 16384, 4), (64, 16384, 4),
    # a position over a block of 64, a CU's second round of waves or blocks
    (64, 2048, 1), (65, 2048, 2), (100, 512, 0), (64, 512, 0), (130, 512, 1),
    # the router of 128 experts
    (27, 128, 0), (256, 128, 0), (1024, 128, 1), (1501, 128, 1), (4096, 128, 4), (1501, 512, 4)])
def test_f32_gemm_form(n, rows, form):
    f = rule("_ZN6strata13gemm_f32_formEiii", ctypes.c_int, ctypes.c_int, ctypes.c_int)
    assert f(n, rows, CUS) == form


def test_f32_gemm_form_of_any_size():
    f = rule("_ZN6strata13gemm_f32_formEiii", ctypes.c_int, ctypes.c_int, ctypes.c_int)
    for n in (1, 2, 63, 64, 65, 4097, 1 << 20, 1 << 30):
        for rows in (1, 3, 16, 17, 151936, 1 << 20, 1 << 30):
            assert f(n, rows, CUS) in (0, 1, 2, 4)
