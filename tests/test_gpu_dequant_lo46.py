"""fp16 / bf16 dequantize of tensors with tiles of classes 4 and 6 beside 0-3 (integer stages up to 16 columns, then the
reference's f32 additions; calls of fewer tiles than CUs and tensors with negative or infinite scales take the general
kernel): bitwise the round-to-nearest-even of the f32 dequantize, whose bits the oracle pins."""
import numpy as np
import pytest

import oracle as O
import p8x

pytestmark = pytest.mark.gpu

MIXES = {"c4": (0, 0, 0, 0, 1, 0, 0, 0), "c6": (0, 0, 0, 0, 0, 0, 1, 0), "c234": (0, 0, 1, 4, 2, 0, 0, 0), "c012346": (1, 1, 1, 1, 2, 0, 2, 0)}


def rne(W, dtype):
    if dtype == p8x.F16:
        with np.errstate(over="ignore"):
            return W.astype(np.float16).view(np.uint16)
    u = W.view(np.uint32).astype(np.uint64)
    r = ((u + 0x7FFF + ((u >> 16) & 1)) >> 16).astype(np.uint16)
    nan = np.isnan(W)
    r[nan] = ((u[nan] >> 16) | 0x40).astype(np.uint16)
    return r


@pytest.mark.parametrize("dtype", [p8x.F16, p8x.BF16])
@pytest.mark.parametrize("mix", sorted(MIXES))
@pytest.mark.parametrize("rows,K,codebook", [(32, 256, 0), (992, 2048, 1), (1056, 2816, 0), (8224, 256, 0)])
def test_dequant_lo46(rows, K, codebook, mix, dtype):
    slot = p8x.synth_random(rows + K, rows, K, class_p=MIXES[mix], codebook=codebook, nd=40)
    t = p8x.Tensor(slot, rows, K)
    W = O.Oracle(slot, rows, K).dequant()
    assert np.array_equal(t.dequantize(dtype), rne(W, dtype))
    part = t.dequantize_rows(rows // 3, rows // 2, dtype, ld=K + 8)
    assert np.array_equal(part[:, :K], rne(W, dtype)[rows // 3:rows // 3 + rows // 2])


def scales(slot, rows, K):
    nt = rows // 32 * (K // 256)
    return slot[2064 + 4 * nt:2064 + 4 * nt + 2 * rows * (K // 256)].view(np.uint16)


def test_dequant_lo46_extreme_scales():
    """full 11-bit scale mantissas, the largest and the subnormal ones, a negative one among them, which takes the general
    kernel (without it, the exactness bound's edge: test_dequant_lo46_extreme_positive_scales)"""
    rows, K = 1024, 2048
    slot = p8x.synth_random(5, rows, K, class_p=MIXES["c012346"], nd=6).copy()
    s = scales(slot, rows, K)
    nz = np.nonzero(s)[0]
    s[nz] = np.random.default_rng(1).choice(np.array([0x7BFF, 0x1FFF, 0x03FF, 0x0001, 0x83FF, 0x3FFF, 0x2AAB], np.uint16), nz.size)
    W = O.Oracle(slot, rows, K).dequant()
    t = p8x.Tensor(slot, rows, K)
    for dtype in (p8x.F16, p8x.BF16):
        assert np.array_equal(t.dequantize(dtype), rne(W, dtype))


@pytest.mark.parametrize("bad", [0x7C00, 0xFC00])
def test_dequant_lo46_infinite_scale(bad):
    """an infinite row scale: inf and NaN land where the f32 dequantize has them"""
    rows, K = 1024, 2048
    slot = p8x.synth_random(6, rows, K, class_p=MIXES["c234"], nd=2).copy()
    s = scales(slot, rows, K)
    s[np.nonzero(s)[0][[3, 4000]]] = bad
    t = p8x.Tensor(slot, rows, K)
    W = t.dequantize(p8x.F32)
    assert not np.isfinite(W).all()
    H = t.dequantize(p8x.F16)
    nan = np.isnan(W)
    assert np.array_equal(np.isnan(H.view(np.float16)), nan) and np.array_equal(H[~nan], rne(W, p8x.F16)[~nan])


@pytest.mark.parametrize("mix", ["c1", "c3", "c4", "c6", "c012346"])   # also classes 0-3 alone (k_dequant_lo's)
def test_dequant_lo46_negative_scales(mix):
    """negative row scales over constant tiles: 255 of 256 rotated sums cancel, and the zeros keep the sign that the f32
    dequantize gives them (-0 only where every term is -0)"""
    rows, K = 1024, 2048
    p = {"c1": (0, 1, 0, 0, 0, 0, 0, 0), "c3": (0, 0, 0, 1, 0, 0, 0, 0)}.get(mix) or MIXES[mix]
    slot = p8x.synth_random(7, rows, K, class_p=p, nd=0).copy()
    nt = rows // 32 * (K // 256)
    M = slot[2064:2064 + 4 * nt].view(np.uint32)
    doff = (2064 + 68 * nt + 15) // 16 * 16
    slot[doff:doff + 256 * int(np.array((0, 4, 6, 8, 10, 12, 16, 24))[M >> 29].sum())] = 0
    s = scales(slot, rows, K)
    s[s != 0] |= 0x8000
    W = O.Oracle(slot, rows, K).dequant()
    assert (W == 0).any()
    t = p8x.Tensor(slot, rows, K)
    for dtype in (p8x.F16, p8x.BF16):
        assert np.array_equal(t.dequantize(dtype), rne(W, dtype))


def test_dequant_lo46_extreme_positive_scales():
    """the extreme scales without the negative one, which would send the tensor to the general kernel"""
    rows, K = 1024, 2048
    slot = p8x.synth_random(5, rows, K, class_p=MIXES["c012346"], nd=6).copy()
    s = scales(slot, rows, K)
    nz = np.nonzero(s)[0]
    s[nz] = np.random.default_rng(1).choice(np.array([0x7BFF, 0x1FFF, 0x03FF, 0x0001, 0x3FFF, 0x2AAB], np.uint16), nz.size)
    W = O.Oracle(slot, rows, K).dequant()
    t = p8x.Tensor(slot, rows, K)
    for dtype in (p8x.F16, p8x.BF16):
        assert np.array_equal(t.dequantize(dtype), rne(W, dtype))


def test_dequant_classes_0_to_3_infinite_scale():
    rows, K = 256, 2048
    slot = p8x.synth_random(6, rows, K, class_p=(0, 1, 1, 1, 0, 0, 0, 0), nd=2).copy()
    s = scales(slot, rows, K)
    s[np.nonzero(s)[0][[3, 400]]] = 0x7C00
    t = p8x.Tensor(slot, rows, K)
    W = t.dequantize(p8x.F32)
    H = t.dequantize(p8x.F16)
    nan = np.isnan(W)
    assert nan.any()
    assert np.array_equal(np.isnan(H.view(np.float16)), nan) and np.array_equal(H[~nan], rne(W, p8x.F16)[~nan])
