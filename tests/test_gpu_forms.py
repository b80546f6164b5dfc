"""The kernels that a call may take by its size, each at the sizes where its tiles, remainders and dispatch lines lie,
against the CPU oracle (GPU, through the C ABI)."""
import numpy as np
import pytest

import rustingstrata_amd as S
from oracle import oracle as O
from rustingstrata_amd import ggml
from rustingstrata_amd.backend import F32_TYPE
from tests.helpers import normal, random_blocks, rel_l2

pytestmark = pytest.mark.gpu


def up(hip, a):
    return hip.upload(np.ascontiguousarray(a))


# the quad form, and the ring form of 1, 2 and 4 rows a wave (1536, 1537 and 777 positions; rings of 6 and 5 steps of 32 columns)
@pytest.mark.parametrize("n,rows,cols,off", [
    (1, 1, 4, 0), (5, 17, 36, 0), (8, 128, 256, 0), (63, 130, 100, 0), (512, 128, 516, 0), (513, 128, 516, 0),
    (600, 129, 28, 4), (1536, 128, 132, 0), (1537, 128, 100, 0), (2048, 128, 32, 0), (2049, 128, 164, 0),
    (777, 515, 12, 0), (777, 515, 228, 0), (1501, 509, 292, 0), (5, 16385, 164, 0)])
def test_f32_gemm_forms_are_the_sequential_sum(hip, n, rows, cols, off):
    """gemm_dense of a float matrix: every form gives the index-order float32 sum bit for bit (np.add over the columns
    one by one), for ragged rows, positions and columns, and for weights that are only float-aligned."""
    w, x = normal((rows, cols), seed=n + rows), normal((n, cols), seed=cols)
    wb, xb, yb = hip.alloc(w.nbytes + 16), up(hip, x), hip.alloc(n * rows * 4)
    hip.htod(w, wb, off)
    hip.gemm_dense(S.GpuTensor(F32_TYPE, rows, cols, wb, off), n, xb, cols, yb, rows, S.ACT_STORE)
    want = np.zeros((n, rows), np.float32)
    for k in range(cols):
        want += x[:, k:k + 1] * w[None, :, k]
    got = hip.get(yb, np.float32, n * rows).reshape(n, rows)
    assert np.array_equal(got.view(np.uint32), want.view(np.uint32))


# dense GEMMs by items of 16 rows x 16 positions: a block each up to 1280, a wave each up to 2048, the 256-position
# blocks beyond; rows and positions that do not fill a unit, 1 to 17 super-blocks (terms of 8 at a time)
# (Q8_0: blocks of 64 rows x 64 positions)
@pytest.mark.parametrize("ty", ggml.TYPES)
@pytest.mark.parametrize("n,rows,cols", [(1, 1, 256), (64, 64, 512), (129, 63, 768), (17, 33, 2304), (40, 130, 4352), (64, 5120, 256), (65, 4097, 512),
                                         (33, 10912, 256), (33, 10913, 256)])
def test_dense_gemm_few_positions(hip, ty, n, rows, cols):
    """gemm_dense against the CPU dots (bit-equal; IQ4_XS sums in float on the CPU: within 1e-5 rel-L2), store and add."""
    w, x = random_blocks(ty, rows, cols, seed=ty + n), normal((n, cols), seed=rows)
    t, xb, yb = hip.upload_tensor(ty, w), up(hip, x), hip.alloc(n * rows * 4)
    hip.gemm_dense(t, n, xb, cols, yb, rows, S.ACT_STORE)
    got = hip.get(yb, np.float32, n * rows).reshape(n, rows)
    for m in sorted({0, n // 2, n - 1}):
        want = O.matvec(ty, w, rows, cols, x[m])
        if ty == ggml.IQ4_XS:
            assert rel_l2(got[m], want) <= 1e-5
        else:
            assert np.array_equal(got[m].view(np.uint32), want.view(np.uint32)), m
    hip.gemm_dense(t, n, xb, cols, yb, rows, S.ACT_ADD)
    assert np.array_equal(hip.get(yb, np.float32, n * rows).reshape(n, rows), got + got)


def test_q8_0_grid_in_slices(hip):
    """More items than one slice of the grid holds (65535 tiles of one position x 129 row blocks): the items at the slices'
    ends on every XCD, and the first and last ones, against the same rows of X as one dense GEMM."""
    ty, rows, cols, nt = ggml.Q8_0, 64 * 129, 256, 65535
    w, x = random_blocks(ty, rows, cols, seed=5), normal((5, cols), seed=6)
    t, xb, y = hip.upload_tensor(ty, w), up(hip, x), hip.alloc(nt * rows * 4)
    i = np.arange(nt, dtype=np.uint64)
    tiles = up(hip, np.stack([np.full(nt, t.ptr, np.uint64), i | np.uint64(1 << 32)], axis=1))
    xrow, yd = up(hip, (i % 5).astype(np.int32)), hip.alloc(5 * rows * 4)
    hip.memset(y)
    hip.gemm(ty, rows, cols, tiles, nt, xb, cols, 5, xrow, y, rows, S.ACT_STORE)
    hip.gemm_dense(t, 5, xb, cols, yd, rows, S.ACT_STORE)
    want = hip.get(yd, np.uint32, 5 * rows).reshape(5, rows)
    total, per = 129 * nt, -(-129 * nt // 8)
    assert total > 1 << 23
    for xcd in range(8):
        for at in (0, 1, (1 << 20) - 1, 1 << 20, (1 << 20) + 1, per - 2, per - 1):
            item = min(xcd * per + at, total - 1)
            rb, tile = divmod(item, nt)
            got = hip.get(y, np.uint32, 64, at=tile * rows + 64 * rb)
            assert np.array_equal(got, want[tile % 5, 64 * rb:64 * rb + 64]), (xcd, at)


# tile lists of few positions: gathered gate/up and down rows on both sides of the dispatch lines of each kind of type
@pytest.mark.parametrize("ty", [ggml.Q2_K, ggml.Q3_K, ggml.Q5_K, ggml.Q6_K, ggml.IQ4_XS, ggml.IQ2_XXS])
@pytest.mark.parametrize("t,cols", [(3, 512), (32, 2048), (33, 2048), (48, 768), (49, 512), (128, 1536), (129, 256)])
def test_grouped_gemm_few_positions(hip, ty, t, cols):
    """The 64-position tile list's GEMMs (SMALL_TILES) give the bits of the plain forms over the same tiles: the
    paired gate/up, a gathered store, and the rows of X in order (as a down GEMM reads them)."""
    E, k, rows = 8, 2, 64
    x, st = normal((t, cols), seed=t), ggml.row_bytes(ty, cols) * rows
    w = up(hip, random_blocks(ty, 2 * E * rows, cols, seed=ty))
    ids = up(hip, np.stack([np.random.default_rng(m).choice([0, 1, 2, 5, 7], k, replace=False) for m in range(t)]).astype(np.int32))
    mt = t * k // 64 + E
    off, xrow, inv, ntd, tiles = (hip.alloc(b) for b in (4 * (E + 1), 4 * t * k, 4 * t * k, 4, 16 * mt))
    hip.moe_sort(ids, t, k, E, off, xrow, inv, [(int(w), st)], tiles, mt, ntd, chunk=64)
    xb, y = up(hip, x), hip.alloc(t * k * rows * 4)
    xs = up(hip, np.repeat(x, k, axis=0))
    res = {}
    for flag in (0, S.SMALL_TILES):
        out = []
        hip.gemm_grouped_gate_up(ty, rows, cols, tiles, mt, ntd, xb, cols, t, xrow, y, rows, E * st, flags=flag)
        out.append(hip.get(y, np.uint32, t * k * rows))
        for act in (S.ACT_STORE, S.ACT_SWIGLU, S.ACT_ADD):
            hip.gemm_grouped(ty, rows, cols, tiles, mt, ntd, xb, cols, t, xrow, y, rows, act | flag)
            out.append(hip.get(y, np.uint32, t * k * rows))
        hip.gemm_grouped(ty, rows, cols, tiles, mt, ntd, xs, cols, t * k, 0, y, rows, S.ACT_STORE | flag)
        out.append(hip.get(y, np.uint32, t * k * rows))
        res[flag] = out
    for i, (a, b) in enumerate(zip(res[0], res[S.SMALL_TILES])):
        assert np.array_equal(a, b), i


# (empty tiles: slots that keep the rows a slot under the rule's line)
@pytest.mark.parametrize("ty", [ggml.Q2_K, ggml.Q3_K, ggml.IQ4_XS, ggml.IQ3_S])
@pytest.mark.parametrize("sizes,rows", [([1, 16, 17, 63, 64, 65, 0, 2] + [0] * 21, 33), ([0] * 15 + [200] + [0] * 9, 64),
                                        ([130, 3, 1] + [0] * 14, 2000), ([5] * 40, 1600)])
def test_grouped_gemm_chunks_side_by_side(hip, ty, sizes, rows):
    """Tile lists of less than an item a wave, whose tiles' chunks of 16 positions run side by side (and past 64 positions one
    after the other again), against the plain form: the same bits, no row left out or written twice (act add)."""
    cols, n = 512, sum(sizes)
    st = ggml.row_bytes(ty, cols) * rows
    w, x = up(hip, random_blocks(ty, rows * min(len(sizes), 8), cols, seed=ty)), up(hip, normal((n, cols), seed=n))
    m0 = np.concatenate([[0], np.cumsum(sizes)[:-1]])
    tiles = np.array([[int(w) + (i % 8) * st, int(m) | (c << 32)] for i, (m, c) in enumerate(zip(m0, sizes))], np.uint64)
    tb, y, out = up(hip, tiles), hip.alloc(n * rows * 4), []
    for flag in (0, S.SMALL_TILES):
        hip.memset(y)
        for act in (S.ACT_STORE, S.ACT_ADD):
            hip.gemm(ty, rows, cols, tb, len(sizes), x, cols, n, 0, y, rows, act | flag)
        out.append(hip.get(y, np.uint32, n * rows))
    assert np.array_equal(out[0], out[1])


@pytest.mark.parametrize("ty", ggml.TYPES)
@pytest.mark.parametrize("rows,cols", [(3, 256), (33, 2304), (4097, 512), (20500, 256), (40, 20480), (512, 12288), (513, 12288),
                                       (2048, 16640)])
def test_gemvn_few_positions_is_gemv(hip, ty, rows, cols):
    """2 to 4 inputs (and two matrices, gemvq2) give gemv's bits per input, under both numerics, whatever form takes
    them; rows over the 16384 columns of the register kernel against the CPU dots."""
    if ggml.row_bytes(ty, cols) > 24512:
        pytest.skip("row exceeds the GEMV tile")
    w, x = random_blocks(ty, rows, cols, seed=ty), normal((4, cols), seed=rows)
    t, xb, y, y2 = hip.upload_tensor(ty, w), up(hip, x), hip.alloc(4 * rows * 4), hip.alloc(4 * rows * 4)
    y1 = hip.alloc(rows * 4)
    try:
        for numerics in (S.NUM_Q8K, S.NUM_Q8_32):
            hip.set_numerics(numerics)
            one = []
            for m in range(4):
                hip.gemv(t, int(xb) + 4 * m * cols, y1)
                one.append(hip.get(y1, np.uint32, rows))
            if numerics == S.NUM_Q8K:
                assert rel_l2(one[0].view(np.float32), O.matvec(ty, w, rows, cols, x[0])) <= 1e-5
            for nt in (2, 3, 4):
                hip.gemvn(t, xb, cols, y, rows, nt)
                got = hip.get(y, np.uint32, nt * rows).reshape(nt, rows)
                assert all(np.array_equal(got[m], one[m]) for m in range(nt)), (numerics, nt)
                if cols <= 16384:
                    hip.gemvq2(t, t, xb, cols, 0, y, y2, nt)
                    for yy in (y, y2):
                        got = hip.get(yy, np.uint32, nt * rows).reshape(nt, rows)
                        assert all(np.array_equal(got[m], one[m]) for m in range(nt)), (numerics, nt)
    finally:
        hip.set_numerics(S.NUM_Q8K)


@pytest.mark.parametrize("nh,nkv,hd", [(8, 8, 128), (8, 4, 64), (8, 2, 128), (8, 1, 64)])
@pytest.mark.parametrize("t,pos,win", [(1, 0, 0), (31, 63, 0), (33, 100, 0), (130, 1, 48), (257, 64, 64)])
def test_attn_prefill_rows_and_chunks(hip, nh, nkv, hd, t, pos, win):
    """Rows at the edges of the 32-row tiles, the 64-key tiles and the window, per GQA group (heads and row tiles share a
    block differently), against the f64 attention; the same rows computed as chunks of other sizes give the same bits. One
    query row is large, so that the running maximum jumps between tiles. Tolerance: a float32 score s is off by 2^-24 |s| in
    its sum and again in the exponent, which is the weight's relative error; the exps, the splits (2^-22) and the two sums add
    eight times 2^-23 at most (8.8e-7 seen in ordinary rows, 8.9e-6 in the large one, whose scores reach 120)."""
    n = pos + t
    q, k, v = normal((t, nh * hd), seed=1), normal((n, nkv * hd), seed=2).astype(np.float16), normal((n, nkv * hd), seed=3).astype(np.float16)
    q[t // 2] *= 30.0
    kb, vb, out = up(hip, k), up(hip, v), hip.alloc(t * nh * hd * 4)

    def run(chunks):
        got, i = [], 0
        for c in chunks:
            step, qb = up(hip, np.array([pos + i, 0], np.int32)), up(hip, q[i:i + c])
            hip.attn_prefill(qb, kb, vb, 0, out, step, c, nh, nkv, hd, 1.0 / np.sqrt(hd), win=win)
            got.append(hip.get(out, np.float32, c * nh * hd).reshape(c, nh, hd))
            i += c
        return np.concatenate(got)

    one = run([t])
    for i in sorted({0, t // 2, t - 1}):
        lo = max(pos + i + 1 - win, 0) if win else 0
        for h in range(nh):
            g = h // (nh // nkv)
            kk, vv = (a[lo:pos + i + 1, g * hd:(g + 1) * hd].astype(np.float64) for a in (k, v))
            s = kk @ q[i, h * hd:(h + 1) * hd].astype(np.float64) / np.sqrt(hd)
            w = np.exp(s - s.max())
            assert rel_l2(one[i, h], w @ vv / w.sum()) <= 2.0 ** -23 * (8 + np.abs(s).max()), (i, h)
    if t > 1:
        assert np.array_equal(one.view(np.uint32), run([t // 3 + 1, t - t // 3 - 1]).view(np.uint32))


@pytest.mark.parametrize("hd", [64, 128])
@pytest.mark.parametrize("gap", [16, 18, 20])
def test_attn_prefill_small_weights_beside_a_sink(hip, hd, gap):
    """The first key takes weight 1 (and has value 0), every other 2^-gap .. 2^(1 - gap): the running maximum never lags, so
    the small weights are as far below the split's scale as they can be. Scores are exact (one dimension, a scale of
    1 / log2 e), so what is left is the split, at most half an f16 subnormal (2^-25) of weights scaled by 2^14, that is
    2^(gap - 39) of a weight, and the exps (1 ulp) and float32 sums: 5e-7."""
    nh, nkv, t, pos = 8, 4, 33, 1000
    n, rng = pos + t, np.random.default_rng(gap)
    q, k = np.zeros((t, nh * hd), np.float32), np.zeros((n, nkv * hd), np.float16)
    v = normal((n, nkv * hd), seed=gap + 1).astype(np.float16)
    q[:, ::hd] = 1.0
    k[:, ::hd] = rng.uniform(0.0, 1.0, (n, nkv)).astype(np.float16)
    k[0, ::hd], v[0] = gap, 0.0
    scale = float(np.float32(1.0 / 1.44269504088896341))
    step, out = up(hip, np.array([pos, 0], np.int32)), hip.alloc(t * nh * hd * 4)
    hip.attn_prefill(up(hip, q), up(hip, k), up(hip, v), 0, out, step, t, nh, nkv, hd, scale)
    got = hip.get(out, np.float32, t * nh * hd).reshape(t, nh, hd)
    for i in (0, t - 1):
        for h in range(nh):
            g = h // (nh // nkv)
            w = np.exp(k[:pos + i + 1, g * hd].astype(np.float64) * scale)
            want = w @ v[:pos + i + 1, g * hd:(g + 1) * hd].astype(np.float64) / w.sum()
            assert rel_l2(got[i, h], want) <= 2.0 ** (gap - 39) + 5e-7, (i, h)


@pytest.mark.parametrize("nh,nkv,hd", [(8, 8, 128), (8, 2, 64)])
def test_attn_prefill_non_finite(hip, nh, nkv, hd):
    """A query row that is not finite spoils its own row of its head and no other; a key that is not a number spoils every row
    that sees it (in the heads of its group) and no row before it."""
    t, pos, j, d = 100, 60, 131, 5
    n, G = pos + t, nh // nkv
    q, k, v = normal((t, nh * hd), seed=1), normal((n, nkv * hd), seed=2).astype(np.float16), normal((n, nkv * hd), seed=3).astype(np.float16)
    step, out = up(hip, np.array([pos, 0], np.int32)), hip.alloc(t * nh * hd * 4)

    def run(q, k, v):
        hip.attn_prefill(up(hip, q), up(hip, k), up(hip, v), 0, out, step, t, nh, nkv, hd, 1.0 / np.sqrt(hd))
        return hip.get(out, np.float32, t * nh * hd).reshape(t, nh, hd)

    def same(a, b):
        return np.array_equal(a.view(np.uint32), b.view(np.uint32))

    clean = run(q, k, v)
    for bad in (np.nan, np.inf, -np.inf):
        q1 = q.copy()
        q1[40, 3 * hd + d] = bad
        got = run(q1, k, v)
        assert not np.isfinite(got[40, 3]).any()
        got[40, 3] = clean[40, 3]
        assert same(got, clean)
    k1 = k.copy()
    k1[j, hd + d] = np.nan
    got = run(q, k1, v)
    assert not np.isfinite(got[j - pos:, G:2 * G]).any() and same(got[:j - pos], clean[:j - pos])
    got[:, G:2 * G] = clean[:, G:2 * G]
    assert same(got, clean)


@pytest.mark.parametrize("nh,nkv,hd,win,extra", [(8, 8, 128, 0, False), (8, 2, 64, 0, True), (8, 1, 128, 40, True), (4, 2, 64, 150, False)])
@pytest.mark.parametrize("bad", [np.nan, np.inf, -np.inf])
def test_attn_prefill_non_finite_values(hip, nh, nkv, hd, win, extra, bad):
    """A value row's element that is not finite: the rows that see its key get it in that column and nowhere else, the rows that
    do not (masked, in its tile of 64 keys or not) are finite; all as the f64 attention over the keys that a row sees, with a
    window, an attention sink and a gate too. Rows done again add up to 190 float32 terms in order: 190 x 2^-24 at most."""
    t, pos, j, d = 130, 60, 131, 5
    n, G = pos + t, nh // nkv
    rng = np.random.default_rng(7)
    q, k, v = normal((t, nh * hd), seed=1), normal((n, nkv * hd), seed=2).astype(np.float16), normal((n, nkv * hd), seed=3).astype(np.float16)
    g = nkv - 1
    v[j, g * hd + d] = bad
    sink, qg = rng.standard_normal(nh).astype(np.float32), rng.standard_normal((t, nh, 2, hd)).astype(np.float32)
    out = hip.alloc(t * nh * hd * 4)
    hip.attn_prefill(up(hip, q), up(hip, k), up(hip, v), up(hip, qg) if extra else 0, out, up(hip, np.array([pos, 0], np.int32)), t, nh,
                     nkv, hd, 1.0 / np.sqrt(hd), sink=up(hip, sink) if extra else 0, win=win)
    got = hip.get(out, np.float32, t * nh * hd).reshape(t, nh, hd)
    for i in range(t):
        lo = max(pos + i + 1 - win, 0) if win else 0
        for h in range(nh):
            c = h // G
            kk, vv = (a[lo:pos + i + 1, c * hd:(c + 1) * hd].astype(np.float64) for a in (k, v))
            s = kk @ q[i, h * hd:(h + 1) * hd].astype(np.float64) / np.sqrt(hd)
            top = max(s.max(), float(sink[h])) if extra else s.max()
            w = np.exp(s - top)
            want = (w[:, None] * vv).sum(0) / (w.sum() + (np.exp(float(sink[h]) - top) if extra else 0.0))
            if extra:
                want = want / (1.0 + np.exp(-qg[i, h, 1].astype(np.float64)))
            sees = c == g and lo <= j <= pos + i
            assert (not np.isfinite(want[d])) == sees
            if sees:
                np.testing.assert_array_equal(got[i, h, d], np.float32(want[d]))
                got[i, h, d] = want[d] = 0.0
            assert rel_l2(got[i, h], want) <= 190 * 2.0 ** -24, (i, h)


@pytest.mark.parametrize("n,rows,cols", [(8, 128, 256), (1536, 128, 132), (1537, 128, 100), (777, 515, 228)])
def test_f32_gemm_non_finite(hip, n, rows, cols):
    """Infinities and NaN in x or the weights come out where the index-order float32 sum has them, in every form."""
    w, x = normal((rows, cols), seed=n + rows), normal((n, cols), seed=cols)
    x[n // 2, 3], x[n - 1, cols - 1], w[rows - 1, 0], w[rows // 2, cols - 2] = np.inf, np.nan, -np.inf, np.inf
    x[0, cols - 2] = 0.0  # (times the infinite weight: not a number)
    y = hip.alloc(n * rows * 4)
    hip.gemm_dense(S.GpuTensor(F32_TYPE, rows, cols, up(hip, w)), n, up(hip, x), cols, y, rows, S.ACT_STORE)
    want = np.zeros((n, rows), np.float32)
    with np.errstate(invalid="ignore"):
        for k in range(cols):
            want += x[:, k:k + 1] * w[None, :, k]
    np.testing.assert_array_equal(hip.get(y, np.float32, n * rows).reshape(n, rows), want)


@pytest.mark.parametrize("ty", ggml.TYPES)
def test_few_positions_non_finite_scales(hip, ty):
    """Super-blocks whose f16 scales are infinite or not a number: the forms for few positions (GEMM, tile list, several
    inputs) give what gemm_kernel gives, in the affected rows as in the others."""
    rows, cols, n = 40, 768, 9
    w, x = random_blocks(ty, rows, cols, seed=ty), normal((n, cols), seed=3)
    bb, off = ggml.block_bytes(ty), ggml.F16_FIELDS[ty][0]
    for r, b, bits in ((3, 1, 0x7C00), (17, 0, 0xFC00), (39, 2, 0x7E00)):
        w[r, b * bb + off:b * bb + off + 2] = np.frombuffer(np.uint16(bits).tobytes(), np.uint8)
    t, xb, y = hip.upload_tensor(ty, w), up(hip, x), hip.alloc(n * rows * 4)
    st = up(hip, np.array([[t.ptr, n << 32]], np.uint64))

    def get():
        return hip.get(y, np.float32, n * rows).reshape(n, rows)

    hip.gemm(ty, rows, cols, st, 1, xb, cols, n, 0, y, rows, S.ACT_STORE)
    want = get()
    assert not np.isfinite(want[:, [3, 17, 39]]).any() and np.isfinite(np.delete(want, [3, 17, 39], axis=1)).all()
    hip.gemm(ty, rows, cols, st, 1, xb, cols, n, 0, y, rows, S.ACT_STORE | S.SMALL_TILES)
    np.testing.assert_array_equal(get(), want)
    hip.gemm_dense(t, n, xb, cols, y, rows, S.ACT_STORE)
    np.testing.assert_array_equal(get(), want)
    if ty != ggml.Q8_0:  # (its GEMV adds a row's blocks in another order)
        hip.gemvn(t, xb, cols, y, rows, 4)
        np.testing.assert_array_equal(get()[:4], want[:4])


# 64 heads a block: 512 blocks stage the value rows, more read them where they are stored
@pytest.mark.parametrize("t", [910, 911, 1501])
def test_norm_rope_many_heads_in_chunks(hip, t):
    """A prefill chunk's normed and rotated heads and its KV rows have the bits that the same tokens get as a chunk of 600 (value
    rows staged), one of 5 (a wave a head) and the rest; the value rows are the f16 roundings."""
    nh, nkv, hd, pos = 32, 4, 128, 7
    w = (nh + 2 * nkv) * hd
    qkv = normal((t, w), seed=t)
    qw, kw = normal((hd,), seed=1), normal((hd,), seed=2)
    xb, qwb, kwb = up(hip, qkv), up(hip, qw), up(hip, kw)
    n = pos + t

    def run(chunks):
        q, k, kc, vc = (hip.alloc(b) for b in (t * nh * hd * 4, t * nkv * hd * 4, n * nkv * hd * 2, n * nkv * hd * 2))
        hip.memset(kc), hip.memset(vc)
        i = 0
        for c in chunks:
            x = int(xb) + 4 * w * i
            hip.rms_norm_rope_qk_t(x, w, hd, qwb, int(q) + 4 * nh * hd * i, c * nh, nh, x + 4 * nh * hd, w, kwb,
                                   int(k) + 4 * nkv * hd * i, c * nkv, nkv, hd, 1e-6, hd, up(hip, np.array([pos + i, 0], np.int32)),
                                   1e6, x + 4 * (nh + nkv) * hd, w, kc, vc)
            i += c
        return (hip.get(q, np.uint32, t * nh * hd), hip.get(k, np.uint32, t * nkv * hd), hip.get(kc, np.uint16, n * nkv * hd),
                hip.get(vc, np.uint16, n * nkv * hd))

    one = run([t])
    assert all(np.array_equal(a, b) for a, b in zip(one, run([600, 5, t - 605])))
    v = qkv[:, (nh + nkv) * hd:].astype(np.float16).view(np.uint16).reshape(-1)
    assert np.array_equal(one[3], np.concatenate([np.zeros(pos * nkv * hd, np.uint16), v]))


# one block up to 4096 pairs, three launches beyond
@pytest.mark.parametrize("t,k,E,chunk", [(1, 1, 1, 64), (3, 2, 512, 64), (512, 8, 128, 64), (512, 8, 512, 256), (513, 8, 128, 64)])
def test_moe_sort_forms(hip, t, k, E, chunk):
    """The device sort on both sides of its one-block form against numpy's stable sort: off, xrow, inv, the tiles and the
    count of ids out of range (which get no slot)."""
    rng = np.random.default_rng(t + E)
    ids = rng.integers(0, E, (t, k)).astype(np.int32)
    ids.reshape(-1)[:: 37] = E // 2
    bad = rng.random(t * k) < 0.02
    flat = ids.reshape(-1)
    flat[bad] = np.where(rng.random(int(bad.sum())) < 0.5, -1, E)
    mt = t * k // chunk + E
    off, xrow, inv, ntd, err, tiles = (hip.alloc(b) for b in (4 * (E + 1), 4 * t * k, 4 * t * k, 4, 4, 16 * mt))
    hip.moe_sort(up(hip, flat), t, k, E, off, xrow, inv, [(1 << 20, 4096)], tiles, mt, ntd, err_dev=err, chunk=chunk)
    good = np.flatnonzero(~bad)
    order = good[np.argsort(flat[good], kind="stable")]
    want_inv = np.full(t * k, -1, np.int32)
    want_inv[order] = np.arange(len(order))
    cnt = np.bincount(flat[good], minlength=E)
    want_off = np.concatenate([[0], np.cumsum(cnt)])
    assert np.array_equal(hip.get(off, np.int32, E + 1), want_off)
    assert np.array_equal(hip.get(inv, np.int32, t * k), want_inv)
    assert np.array_equal(hip.get(xrow, np.int32, t * k)[:len(order)], order // k)
    assert hip.get(err, np.int32, 1)[0] == bad.sum()
    want = [((1 << 20) + 4096 * e, (want_off[e] + j) | min(chunk, int(cnt[e]) - j) << 32) for e in range(E) for j in range(0, int(cnt[e]), chunk)]
    assert hip.get(ntd, np.int32, 1)[0] == len(want)
    assert [tuple(r) for r in hip.get(tiles, np.uint64, 2 * len(want)).reshape(-1, 2).tolist()] == [(int(a), int(b)) for a, b in want]
