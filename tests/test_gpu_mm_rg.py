"""The prompt GEMM of few tokens (row-group kernel, 1..64 tokens) against fp64 products of the oracle's dequantized
weights, at the edges of its token tiles, K ranges and row-group rounds."""
import numpy as np
import pytest

import oracle as O
import p8x

pytestmark = pytest.mark.gpu

C3 = (0, 0, 0, 1, 0, 0, 0, 0)
C03 = (1, 0, 0, 3, 0, 0, 0, 0)
ALL = (1, 1, 1, 2, 1, 1, 1, 1)
REL_L2 = 1e-3   # fp16 activations and weights (2^-11 each, independent), fp32 sums


# rows: one row group; fewer groups than CUs; 257 groups (two per workgroup, the last workgroup half empty); 1025
# groups (five per workgroup: teams of waves take four, then one). K: one block (most waves idle) to an odd count
# above every wave count. N: the ends of each 32-token tile.
@pytest.mark.parametrize("cls", [C3, C03, ALL])
@pytest.mark.parametrize("rows,K,N", [(32, 256, 1), (96, 4352, 31), (288, 768, 32), (288, 2816, 33), (8224, 512, 9),
                                      (8224, 768, 64), (32736, 256, 17), (32736, 512, 40), (64, 8448, 64)])
def test_mm_rg(rows, K, N, cls):
    slot = p8x.synth_random(rows + K + N, rows, K, class_p=cls, nd=6)
    t = p8x.Tensor(slot, rows, K)
    X = np.random.default_rng(N).standard_normal((N, K)).astype(np.float32)
    ref = O.dense_f64(O.Oracle(slot, rows, K).dequant(), X)
    Y = t.mul_mat(X)
    assert np.linalg.norm(Y - ref) <= REL_L2 * np.linalg.norm(ref)
    assert np.abs(Y - ref).max() <= 2e-2 * np.sqrt(np.mean(ref ** 2))
    assert np.array_equal(Y.view(np.uint32), t.mul_mat(X).view(np.uint32))


def test_mm_rg_strides_bf16():
    """padded strides of x and y (the columns between stay as they were), bf16 activations, 33 tokens"""
    rows, K, N, ldx, ldy = 416, 1280, 33, 1296, 421
    slot = p8x.synth_random(8, rows, K, class_p=ALL, nd=9)
    t = p8x.Tensor(slot, rows, K)
    X = np.random.default_rng(3).standard_normal((N, ldx)).astype(np.float32).view(np.uint32) >> 16
    X = X.astype(np.uint16)
    ref = O.dense_f64(O.Oracle(slot, rows, K).dequant(), np.ascontiguousarray((X[:, :K].astype(np.uint32) << 16).view(np.float32)))
    y = p8x.DeviceBuffer.from_numpy(np.full((N, ldy), 7.0, np.float32))
    xd = p8x.DeviceBuffer.from_numpy(X)
    t.mul_mat_dev(xd, p8x.BF16, N, y, ldx=ldx, ldy=ldy)
    p8x.synchronize()
    Y = y.to_numpy(np.float32, (N, ldy))
    assert np.linalg.norm(Y[:, :rows] - ref) <= REL_L2 * np.linalg.norm(ref)
    assert (Y[:, rows:] == 7.0).all()
