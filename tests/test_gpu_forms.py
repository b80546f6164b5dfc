"""The kernels that a call may take by its size, each at the sizes where its tiles, remainders and dispatch lines lie,
against the CPU oracle (GPU, through the C ABI)."""
import numpy as np
import pytest

import rustingstrata_amd as S
from rustingstrata_amd.backend import F32_TYPE
from tests.helpers import normal

pytestmark = pytest.mark.gpu


def up(hip, a):
    return hip.upload(np.ascontiguousarray(a))


# outputs n * rows: the quad form up to 65536, then 1, 2 and 4 rows a wave (lines at 196608 and 262144)
@pytest.mark.parametrize("n,rows,cols,off", [
    (1, 1, 4, 0), (5, 17, 36, 0), (8, 128, 256, 0), (63, 130, 100, 0), (512, 128, 516, 0), (513, 128, 516, 0),
    (600, 129, 28, 4), (1536, 128, 132, 0), (1537, 128, 100, 0), (2048, 128, 32, 0), (2049, 128, 164, 0),
    (777, 515, 12, 0)])
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
