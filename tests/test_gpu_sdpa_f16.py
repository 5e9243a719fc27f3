"""The strict SDPA's fp16 products (csrc/sdpa_f16.hip, from 64 keys on) where
they can go wrong: ragged tiles around the key tile and both workgroup sizes,
the scales of q, k and v, references that move, huge scores and masks, and
infinities.  Against the float64 formula; the fp32 oracle's own error is the
yardstick where the inputs are plain."""
from __future__ import annotations

import math

import numpy as np
import pytest

from _parity import sdpa_f64, stats
from test_gpu_sdpa import _qkv, _run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("packed", [False, True])
@pytest.mark.parametrize("H,Lq,Lk,bias", [(2, 1, 64, None), (2, 33, 65, "one"), (3, 129, 127, None),
                                          (1, 128, 1023, "uniform"), (2, 65, 1025, None), (1, 31, 2111, "one"),
                                          (16, 8200, 130, "uniform"), (16, 4100, 1090, None)])
def test_sizes(oracle, cuda, H, Lq, Lk, bias, packed):
    import torch

    print(f"sdpa f16 H={H} Lq={Lq} Lk={Lk} bias={bias} packed={packed}", flush=True)
    q, k, v = _qkv(Lq + Lk, 1, H, Lq, Lk)
    b = None
    if bias == "one":
        b = np.zeros(Lk, np.float32)
        b[Lk - 1] = math.log(Lk)
    elif bias == "uniform":
        b = np.random.default_rng(3).uniform(-2, 0, Lk).astype(np.float32)
    got = _run(torch, cuda, q, k, v, b, packed=packed)
    rows = np.unique(np.r_[0:min(Lq, 24), max(0, Lq - 24):Lq])
    exact = sdpa_f64(q[:, :, rows], k, v, b)
    ref = oracle.sdpa_q8t512(np.ascontiguousarray(q[:, :, rows]), k, v, b)
    got = got[:, :, rows]
    assert np.all(np.isfinite(got))
    assert stats(got, exact)["rmse"] <= 1.1 * stats(ref, exact)["rmse"] + 2.0 ** -24 * float(np.abs(v).max())


@pytest.mark.parametrize("Lk", [200, 1100])
def test_scales(cuda, Lk):
    """q rows, heads of k and of v at any magnitude; tokens far below their head's largest."""
    import torch

    q, k, v = _qkv(9, 1, 4, 70, Lk)
    plain = _run(torch, cuda, q, k, v)
    # powers of two that cancel in the scores change no bit
    q2, k2 = q.copy(), k.copy()
    q2[:, 1] *= np.float32(2.0 ** -40)
    k2[:, 1] *= np.float32(2.0 ** 40)
    q2[:, 2] *= np.float32(2.0 ** 30)
    k2[:, 2] *= np.float32(2.0 ** -30)
    assert np.array_equal(_run(torch, cuda, q2, k2, v).view(np.uint32), plain.view(np.uint32))
    v2 = v * np.float32(2.0 ** -60)
    assert np.array_equal(_run(torch, cuda, q, k, v2) * np.float32(2.0 ** 60), plain)
    k2, v2 = k.copy(), v.copy()
    k2[:, :, 5::7] *= np.float32(1e-4)
    v2[:, :, 3::5] *= np.float32(1e3)
    got, exact = _run(torch, cuda, q, k2, v2), sdpa_f64(q, k2, v2)
    assert stats(got, exact)["rel_rmse"] < 2e-6
    z = np.zeros_like(k)
    assert stats(_run(torch, cuda, q, z, v), sdpa_f64(q, z, v))["rel_rmse"] < 1e-6
    assert np.all(_run(torch, cuda, q, k, np.zeros_like(v)) == 0)


@pytest.mark.parametrize("scale", [30.0, 1e3, 1e5, 1e7])
def test_huge_scores(cuda, scale):
    """One key holds all the weight: its value, whatever the scores' size."""
    import torch

    q, k, v = _qkv(11, 1, 2, 70, 300)
    q, k = (q * np.float32(scale)).astype(np.float32), (k * np.float32(scale)).astype(np.float32)
    top = np.argsort(np.einsum("bhqd,bhkd->bhqk", q.astype(np.float64), k.astype(np.float64)), -1)
    got = _run(torch, cuda, q, k, v)
    exact = sdpa_f64(q, k, v)
    assert np.all(np.isfinite(got)) and top.shape[-1] == 300
    assert stats(got, exact)["rel_rmse"] < (1e-4 if scale < 100 else 1e-6)


@pytest.mark.parametrize("value", [-1e4, -1e8, -1e30])
@pytest.mark.parametrize("Lq", [70, 8200])
def test_masks(oracle, cuda, value, Lq):
    """Additive masks over leading, trailing and all keys, on both workgroup sizes."""
    import torch

    H, Lk = (2, 300) if Lq < 100 else (16, 300)
    q, k, v = _qkv(13, 1, H, Lq, Lk)
    rows = np.arange(0, 70)
    for cols in (slice(0, 100), slice(100, 300), slice(0, 299), slice(0, 300)):
        b = np.zeros(Lk, np.float32)
        b[cols] = value
        got = _run(torch, cuda, q, k, v, b)
        assert np.all(np.isfinite(got))
        if cols != slice(0, 300) or value != -1e8:  # (there fp32 holds the scores to 8)
            exact = sdpa_f64(q[:, :, rows], k, v, b)
            assert stats(got[:, :, rows], exact)["max_abs"] < (2e-3 if cols == slice(0, 300) and value == -1e4 else 1e-5)


def test_not_finite(cuda):
    """An infinite k makes the scores it should (no weight, or NaN); an infinite
    or NaN v reaches the outputs of its dim and no others; a NaN q its row."""
    import torch

    q, k, v = _qkv(15, 1, 2, 66, 130)
    base = _run(torch, cuda, q, k, v)
    v2 = v.copy()
    v2[0, 0, 100, 7] = np.inf
    v2[0, 0, 3, 9] = np.nan
    got = _run(torch, cuda, q, k, v2)
    assert np.all(got[0, 0, :, 7] == np.inf) and np.all(np.isnan(got[0, 0, :, 9]))
    keep = np.setdiff1d(np.arange(64), [7, 9])
    assert np.array_equal(got[0, 0][:, keep], base[0, 0][:, keep]) and np.array_equal(got[0, 1], base[0, 1])
    k2 = k.copy()
    k2[0, 1, 77, 5] = -np.inf
    got = _run(torch, cuda, q, k2, v)
    drop = np.setdiff1d(np.arange(130), [77])
    exact = sdpa_f64(q, k[:, :, drop], v[:, :, drop])
    up = q[0, 1, :, 5] > 0                                  # score -inf: the key has no weight
    assert stats(got[0, 1][up], exact[0, 1][up])["max_abs"] < 1e-5
    assert np.all(np.isnan(got[0, 1][~up]))                 # score +inf
    assert np.array_equal(got[0, 0], base[0, 0])
    q2 = q.copy()
    q2[0, 0, 4, 60] = np.nan
    got = _run(torch, cuda, q2, k, v)
    assert np.all(np.isnan(got[0, 0, 4]))
    rest = np.setdiff1d(np.arange(66), [4])
    assert np.array_equal(got[0, 0][rest], base[0, 0][rest])


@pytest.mark.parametrize("packed", [False, True])
@pytest.mark.parametrize("biased", [False, True])
@pytest.mark.parametrize("Lq,Lk", [(40, 16384), (8200, 4096)])
@pytest.mark.parametrize("bits", [26, 29, 31])
def test_many_small_weights(cuda, Lq, Lk, biased, packed, bits):
    """One key 2^(bits + 0.4) above all others, which are alike and whose values
    share a mean: together they weigh Lk 2^-(bits + 0.4), and that has to reach
    the result."""
    import torch

    H = 2 if Lq < 100 else 16
    q, k, v = _qkv(bits, 1, H, Lq, Lk)
    v = (1.0 + 0.05 * v).astype(np.float32)
    v[:, :, 77] = 0.0
    gap = np.float32((bits + 0.4) * math.log(2.0))
    k[:] = 0.0
    b = None
    if biased:
        b = np.full(Lk, -gap, np.float32)
        b[77] = 0.0
    else:
        q[:] = 1.0
        k[:, :, 77] = gap / 8.0
    rows = np.arange(0, min(Lq, 64))
    got = _run(torch, cuda, q, k, v, b, packed=packed)[:, :, rows]
    exact = sdpa_f64(q[:, :, rows], k, v, b)
    # exponents of up to 32 in log2 units, rounded twice, and fp32 sums over at
    # most 512 blocks of 32 like keys: (2 * 32 + 512) * 2^-24 of the small weights;
    # and a weight is held to 2^-36 of the largest (|v| < 1.3)
    err = float(np.abs(got - exact).max())
    rest = Lk * 2.0 ** -(bits + 0.4)
    assert err <= 1.3 * (576 * 2.0 ** -24 * rest + Lk * 2.0 ** -36), err / rest


@pytest.mark.parametrize("packed", [False, True])
@pytest.mark.parametrize("H,Lq,Lk", [(2, 70, 300), (2, 70, 1200), (16, 8200, 300)])
@pytest.mark.parametrize("size", [1e4, 1e8, 1e12, 1e30, 1e36])
@pytest.mark.parametrize("mask", [-math.inf, -1e30])
def test_masked_keys_of_any_size(cuda, H, Lq, Lk, size, mask, packed):
    """What a masked key holds, in k or in v, changes nothing (a finite mask: as
    long as its scores stay below the others)."""
    import torch

    q, k, v = _qkv(int(math.log10(size)) + Lk, 1, H, Lq, Lk)
    print(f"sdpa masked H={H} Lq={Lq} Lk={Lk} size={size} mask={mask} packed={packed}", flush=True)
    cols = np.r_[0:3, 40:90, Lk - 50:Lk]
    live = np.setdiff1d(np.arange(Lk), cols)
    b = np.zeros(Lk, np.float32)
    b[cols] = mask
    rows = np.arange(0, 64)
    exact = sdpa_f64(q[:, :, rows], k[:, :, live], v[:, :, live])
    sign = np.sign(v[:, :, cols]).astype(np.float32)
    v2 = v.copy()
    v2[:, :, cols] = sign * np.float32(size)
    got = _run(torch, cuda, q, k, v2, b, packed=packed)[:, :, rows]
    assert stats(got, exact)["rel_rmse"] < 2e-6
    if math.isinf(mask) or size < 1e29:  # (q k below the finite mask)
        k2 = k.copy()
        k2[:, :, cols] = sign * np.float32(size)
        got = _run(torch, cuda, q, k2, v2, b, packed=packed)[:, :, rows]
        assert stats(got, exact)["rel_rmse"] < 2e-6


@pytest.mark.parametrize("packed", [False, True])
@pytest.mark.parametrize("H,Lq,Lk,bias", [(2, 70, 300, False), (2, 70, 1200, True), (16, 8200, 300, False),
                                          (16, 8200, 300, True)])
@pytest.mark.parametrize("dims", [[5], [0, 17, 63]])
def test_outlier_dims(cuda, H, Lq, Lk, bias, dims, packed):
    """Dims of v far larger than the rest cost the rest nothing; dims of k far
    larger than the rest, where q is zero, cost the scores nothing."""
    import torch

    q, k, v = _qkv(5 + Lk, 1, H, Lq, Lk)
    print(f"sdpa outlier dims H={H} Lq={Lq} Lk={Lk} bias={bias} dims={dims} packed={packed}", flush=True)
    b = np.random.default_rng(1).uniform(-2, 0, Lk).astype(np.float32) if bias else None
    rows = np.arange(0, 64)
    keep = np.setdiff1d(np.arange(64), dims)
    q[:, :, :, dims] = 0.0
    exact = sdpa_f64(q[:, :, rows], k, v, b)
    for size in (1e6, 1e12, 1e25):
        v2, k2 = v.copy(), k.copy()
        v2[:, :, :, dims] *= np.float32(size)
        got = _run(torch, cuda, q, k, v2, b, packed=packed)[:, :, rows]
        assert stats(got[..., keep], exact[..., keep])["rel_rmse"] < 2e-6, size
        assert stats(got[..., dims], exact[..., dims] * size)["rel_rmse"] < 2e-6, size
        k2[:, :, :, dims] *= np.float32(size)
        got = _run(torch, cuda, q, k2, v, b, packed=packed)[:, :, rows]
        assert stats(got, exact)["rel_rmse"] < 2e-6, size


@pytest.mark.parametrize("Lq", [40, 8200])
def test_tokens_of_any_size(cuda, Lq):
    """Key tiles whose values of v differ by any power: each query's weight lies
    on the keys of one tile, and its result has that tile's precision."""
    import torch

    H, Lk = (1, 320) if Lq < 100 else (16, 320)
    q, k, v = _qkv(21, 1, H, Lq, Lk)
    size = np.float32([1.0, 1e-25, 1e12, 3e-10, 1e30])
    tile = np.repeat(np.arange(5), 64)
    v = (v * size[tile][:, None]).astype(np.float32)
    k = 0.01 * k
    k[:, :, np.arange(Lk), tile] += 1.0
    q[:] = 0.0
    want = np.arange(Lq) % 5
    q[:, :, np.arange(Lq), want] = 3000.0                 # 375 above the keys of the other tiles
    got = _run(torch, cuda, q, k, v)
    exact = sdpa_f64(q[:, :, :64], k, v)
    for i in range(5):
        r = np.nonzero(want[:64] == i)[0]
        # scores of about 375, fp32's last place of which is 2^-16
        assert stats(got[:, :, r] / size[i], exact[:, :, r] / size[i])["rel_rmse"] < 1e-4, i


@pytest.mark.parametrize("packed", [False, True])
@pytest.mark.parametrize("Lq", [40, 8200])
def test_masked_first_block_of_few_keys(cuda, Lq, packed):
    """Fewer keys than a key tile (the fp32 tiles), the first 32 of them masked
    by -inf: the block adds nothing, and the others are the result."""
    import torch

    H, Lk = (2, 50) if Lq < 100 else (16, 50)
    q, k, v = _qkv(31, 1, H, Lq, Lk)
    b = np.zeros(Lk, np.float32)
    b[:34] = -np.inf
    got = _run(torch, cuda, q, k, v, b, packed=packed)[:, :, :64]
    assert stats(got, sdpa_f64(q[:, :, :64], k[:, :, 34:], v[:, :, 34:]))["rel_rmse"] < 2e-6


@pytest.mark.parametrize("packed", [False, True])
@pytest.mark.parametrize("H,Lq,Lk", [(2, 70, 300), (2, 70, 1200), (16, 8200, 300)])
@pytest.mark.parametrize("mask", [-1e9, -1e30])
@pytest.mark.parametrize("level", [-30.0, -60.0])
def test_first_keys_under_a_finite_mask(cuda, H, Lq, Lk, mask, level, packed):
    """The reference starts at a mask of many digits and then has to be the live
    keys', however low they lie.  (Scores of up to 100 log2 units are held to 2^-18:
    2.6e-6 of a weight, beside the 2e-6 of the other cases.)"""
    import torch

    q, k, v = _qkv(int(-level) + Lk, 1, H, Lq, Lk)
    print(f"sdpa first keys masked H={H} Lq={Lq} Lk={Lk} mask={mask} level={level} packed={packed}", flush=True)
    b = np.full(Lk, level, np.float32)
    b[:70] = mask
    got = _run(torch, cuda, q, k, v, b, packed=packed)[:, :, :64]
    exact = sdpa_f64(q[:, :, :64], k[:, :, 70:], v[:, :, 70:])
    assert stats(got, exact)["rel_rmse"] < 4.6e-6


@pytest.mark.parametrize("packed", [False, True])
@pytest.mark.parametrize("H,Lq,Lk,masked", [(2, 70, 300, 0), (2, 70, 300, 70), (2, 70, 1200, 1030),
                                            (16, 8200, 300, 0), (16, 8200, 300, 70)])
@pytest.mark.parametrize("log2_level", [-2.9e38, -3.0e38, -3.3e38])
def test_bias_at_the_end_of_the_range(cuda, H, Lq, Lk, masked, log2_level, packed):
    """A bias that leaves every live key the same score near fp32's lowest: all of
    them weigh the same, in one part or merged with parts that are masked whole."""
    import torch

    level = np.float32(log2_level / math.log2(math.e))
    print(f"sdpa bias {level} H={H} Lq={Lq} Lk={Lk} masked={masked} packed={packed}", flush=True)
    q, k, v = _qkv(masked + Lk, 1, H, Lq, Lk)
    b = np.full(Lk, level, np.float32)
    b[:masked] = -np.inf
    got = _run(torch, cuda, q, k, v, b, packed=packed)[:, :, :64]
    exact = np.broadcast_to(v[:, :, masked:].astype(np.float64).mean(axis=2, keepdims=True), got.shape)
    assert np.abs(got - exact).max() <= 2.0 ** -20 * np.abs(v).max()


@pytest.mark.parametrize("Lq,Lk", [(70, 300), (70, 1200), (8200, 300)])
def test_scores_that_a_bias_takes_back(cuda, Lq, Lk):
    """Scores and a bias of 2^30 each, one above the other by a few hundred log2
    units: equal keys keep equal weights."""
    import torch

    H = 2 if Lq < 100 else 16
    q, k, v = _qkv(3, 1, H, Lq, Lk)
    print(f"sdpa bias takes scores back Lq={Lq} Lk={Lk}", flush=True)
    q[:], k[:] = 0.0, 0.0
    q[..., 0] = np.float32(2.0 ** 15)
    k[..., 0] = np.float32(2.0 ** 18 * (1 + 2.0 ** -22))
    b = np.full(Lk, -(2.0 ** 30), np.float32)
    got = _run(torch, cuda, q, k, v, b)[:, :, :64]
    exact = np.broadcast_to(v.astype(np.float64).mean(axis=2, keepdims=True), got.shape)
    assert np.abs(got - exact).max() <= 2.0 ** -20 * np.abs(v).max()
