"""The rules that choose a kernel form by a call's sizes (CPU: the library's own functions, no launch), at sizes where both
forms were measured on the GPU and one of them is slower."""
import ctypes

import pytest

from rustingstrata_amd import backend, ggml

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
    """A form for every size, and its blocks of rows within what HIP takes along y up to the rows that one form of 16 rows a
    block took."""
    f = rule("_ZN6strata13gemm_f32_formEiii", ctypes.c_int, ctypes.c_int, ctypes.c_int)
    for n in (1, 2, 63, 64, 65, 4097, 1 << 20, 1 << 30):
        for rows in (1, 3, 16, 17, 151936, 1 << 20, 1 << 30):
            assert f(n, rows, CUS) in (0, 1, 2, 4)
    for n in (1, 2, 3, 8, 17, 33, 64, 65, 128, 129, 1000, 4096):
        for rows in (262140, 262141, 524280, 524281, 1000003, 16 * 65535):
            assert -(-rows // (4 * (f(n, rows, CUS) or 4))) <= 65535


@pytest.mark.parametrize("ty,nt,cols,tiles,pads", [
    (ggml.Q8_0, 3, 2048, 40000, 1), (ggml.Q4_K, 4, 4096, 4096, 1),  # the same blocks a CU
    (ggml.Q8_0, 2, 20480, 4096, 0), (ggml.Q2_K, 2, 20480, 4096, 0),  # one block a CU instead of two (119 us against 203)
    (ggml.Q8_0, 1, 20480, 4096, 0), (ggml.Q5_K, 1, 20480, 20480, 0),  # two instead of three (51 against 60)
    (ggml.Q2_K, 1, 20480, 6000, 1), (ggml.IQ3_S, 3, 6144, 5000, 1),   # worth it for these
    (ggml.Q2_K, 1, 20480, 768, 0), (ggml.Q5_K, 1, 20480, 512, 1),     # a round of tiles
    (ggml.Q6_K, 1, 18432, 512, 0)])
def test_gemv_padding(ty, nt, cols, tiles, pads):
    f = rule("_ZN6strata9gemv_padsEiiixi", ctypes.c_int, ctypes.c_int, ctypes.c_int, ctypes.c_longlong, ctypes.c_int)
    f.restype = ctypes.c_bool
    assert f(ty, nt, cols, tiles, CUS) == bool(pads)


@pytest.mark.parametrize("ty,nt,rows,cols,few", [
    # one input of more columns than the register kernel takes: from 2048 rows (512 rows of Q6_K 14 us against 29)
    (ggml.Q6_K, 1, 4096, 4096, 0), (ggml.Q6_K, 1, 512, 20480, 0), (ggml.Q4_K, 1, 2048, 20480, 1), (ggml.Q3_K, 1, 2048, 20480, 0),
    (ggml.Q3_K, 1, 4096, 20480, 1),
    # two: not few long rows
    (ggml.Q6_K, 2, 64, 2048, 1), (ggml.Q6_K, 2, 512, 8192, 0), (ggml.Q6_K, 2, 1000, 8192, 1), (ggml.Q6_K, 2, 512, 14336, 0),
    (ggml.Q6_K, 2, 640, 14336, 1),
    (ggml.Q4_K, 3, 256, 28672, 0), (ggml.Q4_K, 3, 512, 28672, 1), (ggml.Q4_K, 4, 64, 28672, 1),
    # more x than LDS holds otherwise
    (ggml.Q2_K, 2, 64, 71680, 1), (ggml.Q2_K, 3, 64, 40960, 1)])
def test_gemv_of_few_positions(ty, nt, rows, cols, few):
    f = rule("_ZN6strata14gemv_takes_fewEiiii", ctypes.c_int, ctypes.c_int, ctypes.c_int, ctypes.c_int)
    f.restype = ctypes.c_bool
    assert f(ty, nt, rows, cols) == bool(few)


@pytest.mark.parametrize("ty,nt,rows,cols,splits", [
    (ggml.Q6_K, 1, 6144, 2048, 0), (ggml.Q8_0, 4, 6144, 2048, 0),
    (ggml.Q6_K, 2, 6144, 2048, 0), (ggml.Q4_K, 2, 512, 4096, 0), (ggml.Q4_K, 2, 8192, 6144, 1),  # (11.3 us against 17)
    (ggml.Q6_K, 3, 4096, 4096, 0), (ggml.Q4_K, 3, 1024, 6144, 1),
    (ggml.Q6_K, 4, 256, 768, 0), (ggml.Q6_K, 4, 512, 2048, 1), (ggml.Q6_K, 4, 1024, 4096, 0), (ggml.Q6_K, 4, 256, 14336, 1)])
def test_gemvq2_split(ty, nt, rows, cols, splits):
    f = rule("_ZN6strata13gemvq2_splitsEiiii", ctypes.c_int, ctypes.c_int, ctypes.c_int, ctypes.c_int)
    f.restype = ctypes.c_bool
    assert f(ty, nt, rows, cols) == bool(splits)


# (tile slots: 128 experts of 768 x 2048 and 2048 x 768, 64 of 1024 x 2048 and 2048 x 1024, 32 of 512 x 1024 and 1024 x 512, 8 of
# 1024 x 2048 and 2048 x 1024)
@pytest.mark.parametrize("ty,rows,cols,n_tiles,gathered,n_x,few", [
    # gathered: by the tokens (128 tokens of Q3_K over 64 experts, skewed: 1.24 times the time)
    (ggml.Q3_K, 1024, 2048, 73, 1, 100, 1), (ggml.Q3_K, 1024, 2048, 76, 1, 128, 0), (ggml.Q6_K, 768, 2048, 144, 1, 128, 1),
    (ggml.Q6_K, 512, 1024, 38, 1, 100, 0), (ggml.Q4_K, 768, 2048, 132, 1, 33, 0), (ggml.Q8_0, 768, 2048, 132, 1, 8, 0),
    # rows in order: by the rows, and by the rows a slot
    (ggml.Q2_K, 2048, 768, 134, 0, 384, 1), (ggml.Q2_K, 2048, 1024, 70, 0, 384, 0), (ggml.Q2_K, 2048, 1024, 66, 0, 192, 1),
    (ggml.IQ4_XS, 2048, 1024, 68, 0, 294, 0), (ggml.IQ4_XS, 2048, 768, 133, 0, 320, 1), (ggml.Q6_K, 2048, 1024, 76, 0, 768, 1),
    (ggml.Q4_K, 2048, 768, 130, 0, 128, 1), (ggml.Q4_K, 2048, 768, 131, 0, 216, 0),
    # less than an item, and than half an item, a wave
    (ggml.IQ4_XS, 1024, 512, 36, 0, 256, 1), (ggml.Q6_K, 1024, 512, 38, 0, 400, 0), (ggml.Q4_K, 2048, 1024, 9, 0, 98, 1),
    (ggml.Q4_K, 2048, 1024, 10, 0, 128, 0)])
def test_tile_lists_of_few_positions(ty, rows, cols, n_tiles, gathered, n_x, few):
    f = rule("_ZN6strata20gemm_few_takes_tilesEiiiibi", ctypes.c_int, ctypes.c_int, ctypes.c_int, ctypes.c_int, ctypes.c_bool,
             ctypes.c_int)
    f.restype = ctypes.c_bool
    assert f(ty, rows, cols, n_tiles, bool(gathered), n_x) == bool(few)


@pytest.mark.parametrize("total", [1, 7, 8, 1000, 1 << 23, (1 << 23) + 1, 1 << 24, (1 << 24) + 8, (1 << 18) * 65535])
def test_q8_0_grid(total):
    """Every item has a block, and HIP takes the grid (fewer than 2^32 threads along x, 65536 blocks along y)."""
    class Dim3(ctypes.Structure):
        _fields_ = [("x", ctypes.c_uint), ("y", ctypes.c_uint), ("z", ctypes.c_uint)]
    f = rule("_ZN6strata14gemm_q8_0_gridEx", ctypes.c_longlong)
    f.restype = Dim3
    g = f(total)
    assert g.x % 8 == 0 and g.x * 256 < 1 << 32 and 0 < g.y < 1 << 16 and g.z == 1
    assert g.x * g.y >= total


@pytest.mark.parametrize("heads,staged", [(256, 1), (128 * 40, 1), (64 * 512, 1), (64 * 512 + 1, 0), (1501 * 36, 0)])
def test_norm_rope_staged_values(heads, staged):
    f = rule("_ZN6strata9nr_stagedEii", ctypes.c_int, ctypes.c_int)
    f.restype = ctypes.c_bool
    assert f(heads, CUS) == bool(staged)
