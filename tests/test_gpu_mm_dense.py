"""The prompt GEMM of mixed classes and many tokens, weights decoded once into operands and then multiplied (or k_mm, where
the plan has it): against fp64 products of the oracle's dequantized weights, each tile shape of the dense kernel at its
edges, and bitwise between the entry points and against k_mm on the same K split."""
import numpy as np
import pytest

import oracle as O
import p8x

pytestmark = pytest.mark.gpu

MIX = (0, 0, 1, 8, 1, 0, 0, 0)
ALL17 = (0, 1, 1, 2, 1, 1, 1, 1)
REL_L2 = 1e-3   # fp16 activations and weights (2^-11 each, independent), fp32 sums


# the plan's choices as N and the shape vary: k_mm for the first and third, 128-token tiles of decoded operands for the others
# (the tiles' edges: test_mm_dense_tiles)
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
    """4096 x 14336, 700 tokens: the no-allocation entry point, whose operands (117 MB) are in a buffer of its own (k_mm itself:
    test_busy_buffer_runs_k_mm)"""
    rows, K, N = 4096, 14336, 700
    t = p8x.Tensor(p8x.synth_random(3, rows, K, class_p=MIX, nd=5), rows, K)
    xd = p8x.DeviceBuffer.from_numpy(np.random.default_rng(3).standard_normal((N, K)).astype(np.float32))
    a, b = p8x.DeviceBuffer(4 * N * rows), p8x.DeviceBuffer(4 * N * rows)
    t.mul_mat_dev(xd, p8x.F32, N, a)
    t.mul_mat_noalloc_dev(xd, p8x.F32, N, b)
    p8x.synchronize()
    assert np.array_equal(a.to_numpy(np.uint32, (N, rows)), b.to_numpy(np.uint32, (N, rows)))


# token tiles of 128, 160 and 192, each ending at N and running one token into the next; one and two K ranges; whole row
# tiles, and one short of a row group; two bands of 8 row tiles in the XCD order and one more; output through planes and
# direct (identity rows, one K range)
@pytest.mark.parametrize("rows,K,N,tile,nsplit,permute", [
    (8192, 1024, 640, 128, 1, True), (8160, 1024, 641, 128, 1, True), (8192, 1024, 257, 128, 2, True), (8192, 1024, 1280, 160, 1, True),
    (8160, 1024, 1121, 160, 1, True), (4096, 4096, 1121, 160, 2, True), (8192, 1024, 1344, 192, 1, True), (8160, 1024, 1345, 192, 1, True),
    (4096, 4096, 1345, 192, 2, True), (8192, 1024, 1345, 192, 1, False), (8160, 1024, 1121, 160, 1, False), (8192, 1024, 641, 128, 1, False)])
def test_mm_dense_tiles(rows, K, N, tile, nsplit, permute):
    slot = p8x.synth_random(rows + K + N, rows, K, class_p=ALL17, nd=6, permute=permute)
    t = p8x.Tensor(slot, rows, K)
    plan = t.mul_mat_plan(N)
    assert plan["kernel"] == p8x.MM_DECODED
    assert (plan["token_tile"], plan["nsplit"], plan["direct"]) == (tile, nsplit, 0 if permute else 1)
    X = np.random.default_rng(N).standard_normal((N, K)).astype(np.float32)
    Y = t.mul_mat(X)
    tok = sorted({0, 31, 32, tile - 1, tile, N // tile * tile - 1, N - 1} & set(range(N)))
    ref = O.dense_f64(O.Oracle(slot, rows, K).dequant(), np.ascontiguousarray(X[tok]))
    assert np.linalg.norm(Y[tok] - ref) <= REL_L2 * np.linalg.norm(ref)
    for g in range(0, rows, 1024):   # and each quarter row-tile band by itself
        assert np.linalg.norm(Y[tok, g:g + 1024] - ref[:, g:g + 1024]) <= REL_L2 * np.linalg.norm(ref[:, g:g + 1024])
    assert np.isfinite(Y).all()
