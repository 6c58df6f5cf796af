"""One column of a tensor of mixed classes (the row-group kernel's class-agnostic tile body) against the oracle's fp64
GEMV of the same quantized activations: each class by itself, the class sets with an instantiation of their own and all
of them, at the edges of the launch: one tile, waves without a tile, K in paired and in counted chunks, more row groups
than CUs (teams of waves)."""
import numpy as np
import pytest

import oracle as O
import p8x

pytestmark = pytest.mark.gpu

CLS = {"c1": (0, 1, 0, 0, 0, 0, 0, 0), "c2": (0, 0, 1, 0, 0, 0, 0, 0), "c4": (0, 0, 0, 0, 1, 0, 0, 0), "c5": (0, 0, 0, 0, 0, 1, 0, 0),
       "c6": (0, 0, 0, 0, 0, 0, 1, 0), "c7": (0, 0, 0, 0, 0, 0, 0, 1), "c0234": (1, 0, 1, 4, 1, 0, 0, 0),
       "c02346": (1, 0, 1, 2, 1, 0, 2, 0), "all": (1, 1, 1, 2, 1, 1, 1, 1)}
# exact integer dots; two f32 products and sums per block: n terms of equal size in random order stay within
# sqrt(n) 2^-24 of the sum's size, 1e-5 holds to n = 28,000
REL = 1e-5


@pytest.mark.parametrize("cls", sorted(CLS))
@pytest.mark.parametrize("rows,K", [(32, 256), (96, 4352), (288, 8448), (8224, 512), (24608, 256), (64, 28928)])
def test_gemv_any_class(rows, K, cls):
    slot = p8x.synth_random(rows + K, rows, K, class_p=CLS[cls], nd=6)
    t, orc = p8x.Tensor(slot, rows, K), O.Oracle(slot, rows, K)
    x = np.random.default_rng(K).standard_normal(K).astype(np.float32)
    y, r = t.mul_mat_vec(x).reshape(-1), orc.gemv_f64(x, act="q8_128")
    assert np.linalg.norm(y - r) <= REL * np.linalg.norm(r)
    assert np.array_equal(y.view(np.uint32), t.mul_mat_vec(x).reshape(-1).view(np.uint32))
