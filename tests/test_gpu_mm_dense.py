"""The prompt GEMM through weights decoded once (mixed classes, many tokens): against fp64 products of the oracle's
dequantized weights at the edges of its tiles, and bitwise against k_mm, which the no-allocation entry point runs with
the same K split when the decoded weights do not fit its scratch."""
import numpy as np
import pytest

import oracle as O
import p8x

pytestmark = pytest.mark.gpu

MIX = (0, 0, 1, 8, 1, 0, 0, 0)
ALL17 = (0, 1, 1, 2, 1, 1, 1, 1)
REL_L2 = 1e-3   # fp16 activations and weights (2^-11 each, independent), fp32 sums


# rows: 256-row tiles full and not, a row-tile band of 8 and one more; N: the ends of 128-, 160- and 192-token tiles
@pytest.mark.parametrize("rows,K,N,cls", [(32, 256, 200, MIX), (288, 1024, 129, MIX), (2304, 2560, 192, ALL17), (2336, 1280, 385, MIX),
                                          (4096, 4096, 320, ALL17), (1024, 8448, 577, MIX)])
def test_mm_dense(rows, K, N, cls):
    slot = p8x.synth_random(rows + K + N, rows, K, class_p=cls, nd=6)
    t = p8x.Tensor(slot, rows, K)
    X = np.random.default_rng(N).standard_normal((N, K)).astype(np.float32)
    Y = t.mul_mat(X)
    tok = sorted({0, 1, 31, 32, 127, 128, N // 2, N - 2, N - 1} & set(range(N)))
    ref = O.dense_f64(O.Oracle(slot, rows, K).dequant(), np.ascontiguousarray(X[tok]))
    assert np.linalg.norm(Y[tok] - ref) <= REL_L2 * np.linalg.norm(ref)
    assert np.isfinite(Y).all()


def test_mm_dense_equals_k_mm():
    """4096 x 14336, 700 tokens: the decoded weights (117 MB) exceed the no-allocation scratch, so that entry point runs
    k_mm on the same K split"""
    rows, K, N = 4096, 14336, 700
    t = p8x.Tensor(p8x.synth_random(3, rows, K, class_p=MIX, nd=5), rows, K)
    xd = p8x.DeviceBuffer.from_numpy(np.random.default_rng(3).standard_normal((N, K)).astype(np.float32))
    a, b = p8x.DeviceBuffer(4 * N * rows), p8x.DeviceBuffer(4 * N * rows)
    t.mul_mat_dev(xd, p8x.F32, N, a)
    t.mul_mat_noalloc_dev(xd, p8x.F32, N, b)
    p8x.synchronize()
    assert np.array_equal(a.to_numpy(np.uint32, (N, rows)), b.to_numpy(np.uint32, (N, rows)))
