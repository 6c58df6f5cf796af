"""Single calls on the matrix cores (several q8/128 columns, x16, block_q8_1) against the oracle's fp64 GEMV of the same
quantized activations, at the edges of the launch: one row group, more row groups than CUs (teams of waves), K in
one block, K in counted and in paired chunks, quantized in the launch and before it."""
import ctypes

import numpy as np
import pytest

import oracle as O
import p8x

pytestmark = pytest.mark.gpu

C3 = (0, 0, 0, 1, 0, 0, 0, 0)
C6 = (0, 0, 0, 0, 0, 0, 1, 0)
MIX = (0, 0, 1, 6, 1, 0, 0, 0)
ALL = (1, 1, 1, 2, 1, 1, 1, 1)
ACT = {"q8": (p8x.ACT_Q8_128, "q8_128"), "x16": (p8x.ACT_X16, "x16"), "q81": (p8x.ACT_Q8_1, "q8_1")}
# exact integer dots; f32 products and sums of 2 (block_q8_1: 8) terms per block: n terms of equal size in random order
# stay within sqrt(n) 2^-24 of the sum's size, 1e-5 holds to n = 28,000
REL = 1e-5


def check(t, slot, rows, K, act, n, seed):
    orc = O.Oracle(slot, rows, K)
    X = np.random.default_rng(seed).standard_normal((n, K)).astype(np.float32)
    Y = t.mul_mat_vec(X, act=ACT[act][0])
    R = np.stack([orc.gemv_f64(x, act=ACT[act][1]) for x in X])
    for c in range(n):
        assert np.linalg.norm(Y[c] - R[c]) <= REL * np.linalg.norm(R[c])
    assert np.array_equal(Y.view(np.uint32), t.mul_mat_vec(X, act=ACT[act][0]).view(np.uint32))


MODES = [("q8", 2), ("q8", 3), ("q8", 8), ("x16", 1), ("x16", 4), ("q81", 1), ("q81", 2), ("q81", 7)]
SMALL = [(r, K, a, n) for r, K in ((32, 256), (96, 4352), (288, 8448)) for a, n in MODES]
LARGE = [(r, K, a, n) for r, K in ((8224, 512), (24608, 256)) for a, n in (("q8", 3), ("x16", 1), ("q81", 2))]   # teams of waves


@pytest.mark.parametrize("cls", [C3, C6, MIX, ALL], ids=["c3", "c6", "mix", "all"])
@pytest.mark.parametrize("rows,K,act,n", SMALL + LARGE)
def test_gemv_mx(rows, K, cls, act, n):
    slot = p8x.synth_random(rows + K + n, rows, K, class_p=cls, nd=6)
    check(p8x.Tensor(slot, rows, K), slot, rows, K, act, n, n)


@pytest.mark.parametrize("act,n", [("q8", 5), ("x16", 1), ("x16", 3), ("q81", 1), ("q81", 8)])
def test_gemv_mx_long_k(act, n):
    """K = 17408 (68 blocks): three counted chunks at eight columns, two paired ones at one"""
    rows, K = 160, 17408
    slot = p8x.synth_random(n, rows, K, class_p=MIX, nd=3)
    check(p8x.Tensor(slot, rows, K), slot, rows, K, act, n, 7)


def test_gemv_mx_padded_strides():
    """padded column strides of x and y; the columns between stay as they were"""
    rows, K, n, ldx, ldy = 416, 1280, 6, 1284, 423
    slot = p8x.synth_random(4, rows, K, class_p=MIX, nd=9)
    t = p8x.Tensor(slot, rows, K)
    X = np.random.default_rng(2).standard_normal((n, ldx)).astype(np.float32)
    y = p8x.DeviceBuffer.from_numpy(np.full((n, ldy), 7.0, np.float32))
    xd = p8x.DeviceBuffer.from_numpy(X)
    t.mul_mat_vec_dev(xd, y, ncols=n, ldx=ldx, ldy=ldy)
    p8x.synchronize()
    Y = y.to_numpy(np.float32, (n, ldy))
    assert (Y[:, rows:] == 7.0).all()
    assert np.array_equal(Y[:, :rows], t.mul_mat_vec(np.ascontiguousarray(X[:, :K])))


@pytest.mark.parametrize("act,n", [("x16", 2), ("q81", 2), ("q8", 2)])
def test_gemv_mx_strides_past_32_bits(act, n):
    """columns 2^32 + 64 elements apart (a stride cut to 32 bits lands inside the buffers): each column's own call"""
    rows, K, ld = 288, 1024, (1 << 32) + 64
    t = p8x.Tensor(p8x.synth_random(1, rows, K, class_p=MIX, nd=6), rows, K)
    X = np.random.default_rng(n).standard_normal((n, K)).astype(np.float32)
    ref = np.concatenate([t.mul_mat_vec(c, act=ACT[act][0]).reshape(1, rows) for c in X])
    x, y = p8x.DeviceBuffer(4 * ((n - 1) * ld + K)), p8x.DeviceBuffer(4 * ((n - 1) * ld + rows))

    def copy(dst, src, nbytes, kind):
        p8x.hip_check(p8x.hip().hipMemcpy(ctypes.c_void_p(dst), ctypes.c_void_p(src), nbytes, kind), "hipMemcpy")
    for c in range(n):
        copy(x.ptr.value + 4 * c * ld, X[c].ctypes.data, 4 * K, p8x.H2D)
    t.mul_mat_vec_dev(x, y, ncols=n, ldx=ld, ldy=ld, act=ACT[act][0])
    p8x.synchronize()
    Y = np.empty((n, rows), np.float32)
    for c in range(n):
        copy(Y[c].ctypes.data, y.ptr.value + 4 * c * ld, 4 * rows, p8x.D2H)
    assert np.array_equal(Y, ref)
