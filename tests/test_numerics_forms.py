"""Why the grouped GEMM keeps exact integer digit planes: cheaper MFMA forms miss the 1e-3 parity bound.

The bound for fp32 outputs is a max relative error of 1e-3 (tests/helpers.py max_rel_err: element-wise,
with a floor of 1e-3 of the largest output). These CPU checks take K-quant rows (random blocks, the reference's
random_tensor design), Q8_K activations (cpu_moe::quantize_q8k), and the exact product of the dequantized values
(what src/cpu_moe.rs computes, up to f32 rounding). They then apply the number formats a faster GEMM would feed the
MFMA:
  * one int8 plane per 256-value super-block (symmetric, a float scale per row and super-block);
  * bf16 weights;
  * OCP MX fp8 (e4m3 values, a power-of-two scale per 32) for weights and activations, the gfx950 block-scaled MFMA
    path.
Each lands far outside the bound (element-wise errors of 0.7 to 20; 0.2% to 4% of the largest output). f32 arithmetic
in another summation order stays inside it (2e-4 to 3e-4). Even 16 bits of weight sit at or past the bound: a form
within 1e-3 feeds the MFMA as many planes as the exact digit-plane form does.
"""
import numpy as np
import pytest

from oracle import oracle as O
from rustingstrata_amd import ggml
from tests.helpers import max_rel_err, normal, random_blocks

R, K, P = 192, 2048, 24
TOL = 1e-3


def q8k_rows(x):
    out = []
    for row in x:
        d, qs, _ = O.quantize_q8k(row)
        out.append((qs.astype(np.float64) * d.astype(np.float64)[:, None]).reshape(-1))
    return np.stack(out)


def bf16(a):
    """Round to bf16 (nearest, ties to even), back as float64."""
    u = np.asarray(a, np.float32).view(np.uint32).astype(np.uint64)
    u = (u + 0x7FFF + ((u >> 16) & 1)) >> 16 << 16
    return u.astype(np.uint32).view(np.float32).astype(np.float64)


def e4m3(a):
    """Round to fp8 e4m3 (3 mantissa bits, nearest even; subnormals from 2^-6), no overflow in range."""
    m = np.abs(a)
    e = np.maximum(np.floor(np.log2(np.maximum(m, 1e-30))), -6.0)
    q = 2.0 ** (e - 3)
    return np.sign(a) * np.round(m / q) * q


def mx_fp8(a):
    """OCP MX: a power-of-two scale per 32 values, 2^(floor(log2 max) - 8), e4m3 elements (e4m3's emax is 8)."""
    b = a.reshape(a.shape[0], -1, 32)
    mx = np.abs(b).max(-1, keepdims=True)
    sc = 2.0 ** (np.floor(np.log2(np.maximum(mx, 1e-30))) - 8)
    return (e4m3(b / sc) * sc).reshape(a.shape)


def int_plane(a, bits):
    """Symmetric integers of the given width per row and 256-value super-block, times a float scale."""
    b = a.reshape(a.shape[0], -1, 256)
    s = np.abs(b).max(-1, keepdims=True) / (2 ** (bits - 1) - 1)
    s = np.where(s == 0, 1.0, s)
    return (np.round(b / s) * s).reshape(a.shape)


@pytest.fixture(scope="module", params=[ggml.Q4_K, ggml.Q5_K, ggml.Q6_K], ids=["Q4_K", "Q5_K", "Q6_K"])
def case(request):
    ty = request.param
    blocks = random_blocks(ty, R, K, seed=31 + ty)
    w = O.dequant(ty, blocks.reshape(-1), R * K).astype(np.float64).reshape(R, K)
    x = normal((P, K), seed=7)
    xq = q8k_rows(x)
    return w, x, xq, xq @ w.T


def test_f32_in_another_order_is_inside_the_bound(case):
    w, _, xq, ref = case
    got = xq.astype(np.float32) @ w.astype(np.float32).T
    assert max_rel_err(got, ref) <= TOL


def test_sixteen_bit_weights_sit_at_the_bound(case):
    """bf16 hi + lo (16 significant bits a weight) lands about at 1e-3; 16-bit integers per super-block (two int8
    planes) miss it: a form inside the bound feeds the MFMA as many planes as the exact digit-plane form."""
    w, _, xq, ref = case
    hi = bf16(w)
    assert 2e-4 < max_rel_err(xq @ (hi + bf16(w - hi)).T, ref) < 5 * TOL
    assert max_rel_err(xq @ int_plane(w, 16).T, ref) > TOL


@pytest.mark.parametrize("form", ["int8_plane", "bf16", "mx_fp8"])
def test_one_plane_forms_miss_the_bound(case, form):
    w, x, xq, ref = case
    if form == "int8_plane":
        got = xq @ int_plane(w, 8).T
    elif form == "bf16":
        got = xq @ bf16(w).T
    else:
        got = mx_fp8(x.astype(np.float64)) @ mx_fp8(w).T
    assert max_rel_err(got, ref) > 100 * TOL
    # also against the largest output alone: above the bound
    assert np.abs(got - ref).max() / np.abs(ref).max() > TOL
