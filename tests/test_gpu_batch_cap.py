"""Grouped launches whose longest linear is cut into units of the launch's average length: every row against the
oracle's fp64 GEMV, with K cut at and off a whole number of chunks, one and several columns, x16."""
import numpy as np
import pytest

import oracle as O
import p8x

pytestmark = pytest.mark.gpu

MIX = (0, 0, 1, 6, 1, 0, 0, 0)
REL = 1e-5   # exact integer dots, f32 sums


@pytest.mark.parametrize("ncols,act", [(1, "q8"), (5, "q8"), (2, "x16")])
def test_batch_capped_units(ncols, act):
    # 8 x 8192 rows of 16 blocks (enough units for two rounds of the launch's waves) and two long linears of 55 and 68
    # blocks, which alone would be one unit per row group
    shapes = [(8192, 4096)] * 8 + [(96, 14080), (160, 17408)]
    slots = [p8x.synth_random(60 + i, r, K, class_p=MIX, nd=4) for i, (r, K) in enumerate(shapes)]
    ts = [p8x.Tensor(s, r, K) for s, (r, K) in zip(slots, shapes)]
    rng = np.random.default_rng(ncols)
    X = [rng.standard_normal((ncols, K)).astype(np.float32) for _, K in shapes]
    ys = [p8x.DeviceBuffer.from_numpy(np.full((ncols, r), np.nan, np.float32)) for r, _ in shapes]
    b = p8x.GemvBatch(ts, [p8x.DeviceBuffer.from_numpy(x) for x in X], ys, ncols=ncols, act=p8x.ACT_X16 if act == "x16" else p8x.ACT_Q8_128)
    info = b.info()
    assert info["small_launch"] == 0
    b.run()
    p8x.synchronize()
    for i, (r, K) in enumerate(shapes):
        if 1 <= i < 7:
            continue   # eight alike: the first and the last
        orc = O.Oracle(slots[i], r, K)
        Y = ys[i].to_numpy(np.float32, (ncols, r))
        for c in range(ncols):
            R = orc.gemv_f64(X[i][c], act="x16" if act == "x16" else "q8_128")
            assert np.linalg.norm(Y[c] - R) <= REL * np.linalg.norm(R)
    assert info["split_jobs"] >= 2
