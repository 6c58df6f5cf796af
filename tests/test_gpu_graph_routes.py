"""HIP graph capture of the matrix-core calls (several columns, x16, block_q8_1, prompts of one row-group pass and of
decoded weights) and of the 16-bit dequantize: three replays with new inputs, each with eager work before it, against
the eager call on the same inputs, bit for bit."""
import numpy as np
import pytest

import p8x

pytestmark = pytest.mark.gpu

C3, MIX = (0, 0, 0, 1, 0, 0, 0, 0), (0, 0, 1, 6, 1, 0, 0, 0)
CALLS = [("vec", C3, 4, p8x.ACT_Q8_128), ("vec", MIX, 7, p8x.ACT_Q8_128), ("vec", MIX, 1, p8x.ACT_X16), ("vec", C3, 2, p8x.ACT_Q8_1),
         ("mm", C3, 19, None), ("mm", MIX, 50, None), ("mm", MIX, 300, None), ("dequant", MIX, 1, None)]


@pytest.mark.parametrize("op,cls,n,act", CALLS)
def test_captured_route_replays_bitwise(op, cls, n, act):
    rows, K = 416, 4608
    t = p8x.Tensor(p8x.synth_random(n, rows, K, class_p=cls, nd=5), rows, K)
    rng = np.random.default_rng(n)
    x = p8x.DeviceBuffer(4 * n * K)
    nout = rows * K if op == "dequant" else 2 * n * rows
    y = p8x.DeviceBuffer(2 * nout)
    if op == "mm":
        t.mul_mat_reserve(n)
    st = p8x.Stream()

    def enqueue(s):
        if op == "vec":
            t.mul_mat_vec_dev(x, y, ncols=n, act=act, stream=s)
        elif op == "mm":
            t.mul_mat_dev(x, p8x.F32, n, y, stream=s)
        else:
            t.dequantize_dev(p8x.F16, y, stream=s)

    def eager():
        y.fill(0xFF)
        p8x.synchronize()
        enqueue(st)
        st.sync()
        return y.to_numpy(np.uint16, (nout,)).copy()

    def fill():
        x.copy_from(p8x.DeviceBuffer.from_numpy(rng.standard_normal((n, K)).astype(np.float32)))
        p8x.synchronize()

    fill()
    eager()
    g = p8x.Graph(enqueue, st)
    try:
        for _ in range(3):
            fill()
            ref = eager()
            y.fill(0xFF)
            p8x.synchronize()
            g.launch(st)
            st.sync()
            assert np.array_equal(y.to_numpy(np.uint16, (nout,)), ref)
    finally:
        g.release()
