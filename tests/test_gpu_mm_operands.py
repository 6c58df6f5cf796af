"""The decoded operands of the prompt GEMM (mixed classes, many tokens) in the buffer that a GPU's tensors share: what it
holds and gives back, calls on two streams, captured calls beside eager ones, and tensors larger than the buffer."""
import ctypes
import gc

import numpy as np
import pytest

import p8x

pytestmark = pytest.mark.gpu

MIX = (0, 0, 1, 8, 1, 0, 0, 0)
MIB = 1 << 20


def free_bytes():
    p8x.synchronize()
    f, t = ctypes.c_size_t(), ctypes.c_size_t()
    p8x.hip_check(p8x.hip().hipMemGetInfo(ctypes.byref(f), ctypes.byref(t)), "hipMemGetInfo")
    return f.value


def tensor(seed, rows=4096, K=4096):
    return p8x.Tensor(p8x.synth_random(seed, rows, K, class_p=MIX, nd=5), rows, K)


def test_tensors_share_the_operands():
    """4096 x 4096, 300 tokens: 32 MiB of operands, held once and not per tensor (each has 2.4 MiB of x' and up to 39 MiB of
    planes of its own), and given back with the last tensor"""
    N = 300
    gc.collect()
    x = p8x.DeviceBuffer.from_numpy(np.random.default_rng(0).standard_normal((N, 4096)).astype(np.float32))
    y = p8x.DeviceBuffer(4 * N * 4096)
    t = tensor(9)   # the library's fixed arrays are there from the first tensor on
    t.mul_mat_dev(x, p8x.F32, N, y)
    p8x.synchronize()
    t.release()
    base = free_bytes()
    ts = [tensor(i) for i in range(4)]
    grew = []
    for t in ts:
        before = free_bytes()
        t.mul_mat_dev(x, p8x.F32, N, y)
        grew.append(before - free_bytes())
    assert grew[0] - max(grew[1:]) >= 32 * MIB
    for t in ts:
        t.release()
    assert free_bytes() >= base - 4 * MIB


@pytest.mark.parametrize("rows,K,N", [(1024, 4096, 300), (4096, 14336, 300), (4096, 14336, 700), (5120, 17408, 900)])
def test_noalloc_decodes_first_too(rows, K, N):
    """p8x_mul_mat_noalloc runs p8x_mul_mat's plan on operand buffers of its own, whatever the operands' size, eager and
    captured (three replays with new inputs), and allocates nothing"""
    t = tensor(rows + N, rows, K)
    p = t.mul_mat_plan(N)
    assert p["kernel"] == p["noalloc_kernel"] == p8x.MM_DECODED
    rng = np.random.default_rng(N)
    x = p8x.DeviceBuffer(4 * N * K)
    ya, yb = p8x.DeviceBuffer(4 * N * rows), p8x.DeviceBuffer(4 * N * rows)
    t.mul_mat_reserve(N)
    st = p8x.Stream()
    g = None
    for _ in range(3):
        x.copy_from(p8x.DeviceBuffer.from_numpy(rng.standard_normal((N, K)).astype(np.float32)))
        ya.fill(0xFF)
        yb.fill(0xFF)
        p8x.synchronize()
        t.mul_mat_dev(x, p8x.F32, N, ya)
        before = free_bytes()
        t.mul_mat_noalloc_dev(x, p8x.F32, N, yb)
        assert free_bytes() == before
        ref = ya.to_numpy(np.uint32, (N, rows)).copy()
        assert np.array_equal(yb.to_numpy(np.uint32, (N, rows)), ref)
        yb.fill(0xFF)
        p8x.synchronize()
        g = g or p8x.Graph(lambda s: t.mul_mat_noalloc_dev(x, p8x.F32, N, yb, stream=s), st)
        g.launch(st)
        st.sync()
        assert np.array_equal(yb.to_numpy(np.uint32, (N, rows)), ref)
    g.release()


def test_streams_bitwise():
    """three tensors' calls in turn on three streams, without waiting"""
    N = 1500
    ts = [tensor(i) for i in range(3)]
    xs = [p8x.DeviceBuffer.from_numpy(np.random.default_rng(i).standard_normal((N, 4096)).astype(np.float32)) for i in range(3)]
    ys = [p8x.DeviceBuffer(4 * N * 4096) for _ in ts]
    ref = []
    for t, x, y in zip(ts, xs, ys):
        t.mul_mat_reserve(N)
        t.mul_mat_dev(x, p8x.F32, N, y)
        p8x.synchronize()
        ref.append(y.to_numpy(np.uint32, (N, 4096)).copy())
        y.fill(0xFF)
    p8x.synchronize()
    sts = [p8x.Stream(), p8x.Stream(), p8x.Stream()]
    for _ in range(6):
        for i in (0, 1, 2):
            ts[i].mul_mat_dev(xs[i], p8x.F32, N, ys[i], stream=sts[i])
    p8x.synchronize()
    for y, r in zip(ys, ref):
        assert np.array_equal(y.to_numpy(np.uint32, (N, 4096)), r)


@pytest.mark.parametrize("rows,K,N,permute", [(4096, 4096, 1345, True), (8192, 1024, 641, False)])
def test_busy_buffer_runs_k_mm(rows, K, N, permute):
    """a call that finds every buffer in use on other streams (milliseconds of calls are queued there) decodes in the GEMM, on
    the K ranges of the decoded plan: the same bits; afterwards a buffer is free for this stream too"""
    t = p8x.Tensor(p8x.synth_random(N, rows, K, class_p=MIX, nd=5, permute=permute), rows, K)
    others = [tensor(i) for i in range(4)]
    assert t.mul_mat_plan(N)["kernel"] == p8x.MM_DECODED
    x, xa = (p8x.DeviceBuffer.from_numpy(np.random.default_rng(i).standard_normal(s).astype(np.float32)) for i, s in enumerate(((N, K), (1500, 4096))))
    y, ys = p8x.DeviceBuffer(4 * N * rows), [p8x.DeviceBuffer(4 * 1500 * 4096) for _ in others]
    t.mul_mat_reserve(N)
    for a in others:
        a.mul_mat_reserve(1500)
    t.mul_mat_dev(x, p8x.F32, N, y)
    p8x.synchronize()
    ref = y.to_numpy(np.uint32, (N, rows)).copy()
    st, sts = p8x.Stream(), [p8x.Stream() for _ in others]
    for busy in (True, False):
        y.fill(0xFF)
        p8x.synchronize()
        if busy:
            for _ in range(30):
                for a, ya, s in zip(others, ys, sts):
                    a.mul_mat_dev(xa, p8x.F32, 1500, ya, stream=s)
        t.mul_mat_dev(x, p8x.F32, N, y, stream=st)
        p8x.synchronize()
        assert np.array_equal(y.to_numpy(np.uint32, (N, rows)), ref)


def test_captured_beside_eager():
    """a captured call replayed on one stream while another tensor's eager calls use the shared buffer on a second one"""
    N, rows, K = 640, 2048, 4096
    a, b = tensor(1, rows, K), tensor(2, rows, K)
    xa, xb = (p8x.DeviceBuffer.from_numpy(np.random.default_rng(i).standard_normal((N, K)).astype(np.float32)) for i in (1, 2))
    ya, yb = p8x.DeviceBuffer(4 * N * rows), p8x.DeviceBuffer(4 * N * rows)
    ref = []
    for t, x, y in ((a, xa, ya), (b, xb, yb)):
        t.mul_mat_reserve(N)
        t.mul_mat_dev(x, p8x.F32, N, y)
        p8x.synchronize()
        ref.append(y.to_numpy(np.uint32, (N, rows)).copy())
    s1, s2 = p8x.Stream(), p8x.Stream()
    g = p8x.Graph(lambda s: a.mul_mat_dev(xa, p8x.F32, N, ya, stream=s), s1)
    try:
        for _ in range(3):
            ya.fill(0xFF)
            yb.fill(0xFF)
            p8x.synchronize()
            for _ in range(4):
                g.launch(s1)
                b.mul_mat_dev(xb, p8x.F32, N, yb, stream=s2)
            p8x.synchronize()
            assert np.array_equal(ya.to_numpy(np.uint32, (N, rows)), ref[0])
            assert np.array_equal(yb.to_numpy(np.uint32, (N, rows)), ref[1])
    finally:
        g.release()


@pytest.mark.parametrize("rows,K,N", [(8192, 14336, 257), (9760, 12288, 513)])
def test_bands(rows, K, N):
    """more operands than the buffer holds (224 and 228.75 MiB of 192): two bands of row groups, the second a partial row
    tile shorter in the second case"""
    t = tensor(3, rows, K)
    X = np.random.default_rng(4).standard_normal((N, K)).astype(np.float32)
    Y = t.mul_mat(X)
    tok = [0, 127, 128, N - 1]
    for r0 in (0, rows // 2 - 64, rows - 256):
        W = t.dequantize_rows(r0, 256, p8x.F32).astype(np.float64)
        ref = X[tok].astype(np.float64) @ W.T
        assert np.linalg.norm(Y[tok, r0:r0 + 256] - ref) <= 1e-3 * np.linalg.norm(ref)   # fp16 operands, as test_gpu_mm_dense
    assert np.isfinite(Y).all()
