"""The strict GEMM's fp16 products (csrc/nf24_gemm_f16.hip, calls of more than
32 rows) where they can go wrong: tile edges, the row scale (outliers beyond
its headroom, rows that begin with zeros, tiny and huge rows), infinities and
NaNs, and codes over the format's whole range.

Bound.  Each operand is carried as two fp16 values that hold it to one unit of
fp32's last place, the dropped product of the low parts is below 2^-22 of the
term, and the sums are fp32: within _parity.gemm_order_bound for K >= 64.  A
value of x is held to 2^-36 in the unit in which the largest of the values the
scale was set from (the row's first 32, or all of them when those are zero or the
row is taken again) is at least 2^3: 2^-39 * max|x_row| * sum_k |w_k| covers it.
"""
from __future__ import annotations

import numpy as np
import pytest

from _parity import gemm_f64, gemm_order_bound, seeded_linear, stats

pytestmark = pytest.mark.gpu


def _run(torch, x, c01, q2, s, b):
    from tsplat.nf24 import nf24_linear

    t = [torch.from_numpy(np.ascontiguousarray(a)).cuda() for a in (x, c01, q2, s, b)]
    return nf24_linear(*t).cpu().numpy()


def _check(oracle, x, c01, q2, s, b, got):
    w = oracle.decode_nf24(c01, q2, s)
    floor = 2.0 ** -39 * np.abs(x.astype(np.float64)).max(1)[:, None] * np.abs(w.astype(np.float64)).sum(0)[None]
    exact = gemm_f64(x, w, b)
    assert np.all(np.isfinite(got))
    assert np.all(np.abs(got - exact) <= gemm_order_bound(x, w, b) + floor), float(np.abs(got - exact).max())
    return stats(got, exact)


@pytest.mark.parametrize("M,K,N", [(33, 64, 4), (64, 1024, 1024), (127, 96, 68), (129, 100, 132), (255, 1024, 260),
                                   (257, 68, 1028), (300, 1024, 3072), (511, 1056, 576), (2100, 1024, 1024),
                                   (4100, 1000, 3072), (6500, 256, 2048), (8200, 64, 4096)])
def test_tile_edges(oracle, cuda, hiplib, M, K, N):
    import torch

    print(f"gemm f16 M={M} K={K} N={N}", flush=True)
    x, w, b = seeded_linear(M + K + N, M, K, N, w_scale=0.02)
    c01, q2, s = oracle.quantize_nf24_i16(w)
    got = _run(torch, x, c01, q2, s, b)
    e = _check(oracle, x, c01, q2, s, b, got)
    # against the sequential fp32 chain on some of the rows: no less exact
    rows = np.random.default_rng(M).choice(M, min(M, 24), replace=False)
    ref = oracle.nf24_gemm(x[rows], c01, q2, s, b)
    exact = gemm_f64(x[rows], oracle.decode_nf24(c01, q2, s), b)
    assert stats(got[rows], exact)["rmse"] <= 1.05 * stats(ref, exact)["rmse"] + 1e-12, e


@pytest.mark.parametrize("M,N", [(40, 64), (300, 1024), (700, 576)])
def test_row_scale(oracle, cuda, hiplib, M, N):
    """Rows of every kind beside plain ones; the plain rows keep their bits."""
    import torch

    K = 160
    x, w, b = seeded_linear(M + N, M, K, N, w_scale=0.02)
    c01, q2, s = oracle.quantize_nf24_i16(w)
    plain = _run(torch, x, c01, q2, s, b)
    y = x.copy()
    y[1, 40] = 3.0e5                      # beyond the headroom of the first 32 values
    y[5, 159] = -7.0e9
    y[9, :32] = 0.0                       # the scale comes from the rest
    y[12, :] = 0.0
    y[17] *= np.float32(1e-30)
    y[21] *= np.float32(1e30)
    y[25, :32] = 1e-20                    # the first values say nothing about the row
    y[30] *= np.exp2(np.random.default_rng(3).integers(-20, 20, K)).astype(np.float32)
    y[33, 0] = 1.0e6                      # large among the first 32
    y[35, 100] = 3000.0                   # scaled, between fp16's largest value and twice that
    changed = [1, 5, 9, 12, 17, 21, 25, 30, 33, 35]
    got = _run(torch, y, c01, q2, s, b)
    _check(oracle, y, c01, q2, s, b, got)
    keep = np.setdiff1d(np.arange(M), changed)
    assert np.array_equal(got[keep].view(np.uint32), plain[keep].view(np.uint32))
    w64 = oracle.decode_nf24(c01, q2, s)
    for r in (9, 17, 21, 25):             # rows of one magnitude: as exact as any other
        zero = np.zeros_like(b)
        one = _run(torch, y, c01, q2, s, zero)[r:r + 1]
        assert stats(one, gemm_f64(y[r:r + 1], w64, zero))["rel_rmse"] < 1e-6


@pytest.mark.parametrize("M,N", [(40, 64), (300, 1024)])
def test_not_finite(oracle, cuda, hiplib, M, N):
    """Infinities and NaNs of x give what the fp32 chain gives; other rows keep their bits."""
    import torch

    K = 96
    x, w, b = seeded_linear(M + N + 1, M, K, N, w_scale=0.02)
    c01, q2, s = oracle.quantize_nf24_i16(w)
    c01[50, ::3], q2[50, ::3] = 0, 0      # inf * 0
    plain = _run(torch, x, c01, q2, s, b)
    y = x.copy()
    y[2, 7] = np.inf
    y[3, 50] = -np.inf
    y[8, 95] = np.nan
    y[11, [4, 60]] = np.inf, -np.inf
    y[20, [3, 80]] = np.inf, 2.0e38
    got = _run(torch, y, c01, q2, s, b)
    ref = oracle.nf24_gemm(y, c01, q2, s, b)
    bad = [2, 3, 8, 11, 20]
    assert np.array_equal(np.isnan(got[bad]), np.isnan(ref[bad]))
    inf = np.isinf(ref[bad])
    assert np.array_equal(got[bad][inf], ref[bad][inf])
    keep = np.setdiff1d(np.arange(M), bad)
    assert np.array_equal(got[keep].view(np.uint32), plain[keep].view(np.uint32))


def test_whole_code_range(oracle, cuda, hiplib):
    """Any int16 / int8 code, not only the packer's."""
    import torch

    M, K, N = 64, 128, 64
    r = np.random.default_rng(5)
    c01 = r.integers(-32768, 32768, (K, N)).astype(np.int16)
    q2 = r.integers(-128, 128, (K, N)).astype(np.int8)
    c01[0, :4], q2[0, :4] = (32767, -32768, 32767, 0), (127, -128, -128, 1)
    s = (r.random(N) * 1e-6).astype(np.float32)
    x = r.standard_normal((M, K)).astype(np.float32)
    b = r.standard_normal(N).astype(np.float32)
    _check(oracle, x, c01, q2, s, b, _run(torch, x, c01, q2, s, b))


def _dead_features(oracle, seed, M, K, N, dead):
    """x, weights and bias with the features `dead` (a list of k) at zero weight."""
    x, w, b = seeded_linear(seed, M, K, N, w_scale=0.02)
    w[:, dead] = 0.0
    c01, q2, s = oracle.quantize_nf24_i16(w)
    assert not oracle.decode_nf24(c01, q2, s)[dead].any()
    return x, c01, q2, s, b


@pytest.mark.parametrize("M,N", [(40, 64), (300, 1028), (700, 576)])
@pytest.mark.parametrize("dead", [[5], [40], [159], list(range(32)), list(range(3, 160, 7)), [6, 130],
                                  list(range(1, 160, 4))])
def test_large_values_without_weight(oracle, cuda, hiplib, M, N, dead):
    """A feature of any size whose weights are zero costs the row's other
    features nothing: each result within the fp32 bound of its own terms."""
    import torch

    x, c01, q2, s, b = _dead_features(oracle, M + N, M, 160, N, dead)
    plain = _run(torch, x, c01, q2, s, b)
    rows = {1: 1e4, 2: 1e6, 8: 1e8, 17: 1e10, 30: 1e20, 33: -3e38}
    y = x.copy()
    for r, value in rows.items():
        y[r, dead] = value
    print(f"gemm f16 M={M} N={N} dead={dead[:4]}", flush=True)
    got = _run(torch, y, c01, q2, s, b)
    w = oracle.decode_nf24(c01, q2, s)
    pick = list(rows)
    if dead[:2] != [1, 5]:
        assert np.all(np.abs(got[pick] - gemm_f64(y[pick], w, b)) <= gemm_order_bound(y[pick], w, b))
    else:
        # every four values hold such a feature: the others are held to 2^-40
        # of the largest of the row's first 32
        floor = 2.0 ** -40 * np.abs(y[pick].astype(np.float64)).max(1)[:, None] * np.abs(w).sum(0)[None]
        assert np.all(np.abs(got[pick] - gemm_f64(y[pick], w, b)) <= gemm_order_bound(y[pick], w, b) + floor)
    keep = np.setdiff1d(np.arange(M), pick)
    assert np.array_equal(got[keep].view(np.uint32), plain[keep].view(np.uint32))


@pytest.mark.parametrize("M,N", [(40, 64), (300, 1028)])
@pytest.mark.parametrize("dead", [[5], [40]])
def test_values_that_the_row_scale_takes_to_zero(oracle, cuda, hiplib, M, N, dead):
    """A value times its row's scale may be zero in fp32 and still be all that the
    results consist of."""
    import torch

    x, c01, q2, s, b = _dead_features(oracle, M + N, M, 160, N, dead)
    b[:] = 0.0
    print(f"gemm f16 to zero M={M} N={N} dead={dead}", flush=True)
    y = x.copy()
    rows = {1: (1e30, 1e-18), 8: (3e38, 1e-9), 33: (-3e38, 1e-25)}
    for r, (large, f) in rows.items():
        y[r] *= np.float32(f)
        y[r, dead] = large
    got = _run(torch, y, c01, q2, s, b)
    w = oracle.decode_nf24(c01, q2, s)
    pick = list(rows)
    assert np.all(np.abs(got[pick] - gemm_f64(y[pick], w, b)) <= gemm_order_bound(y[pick], w, b))


@pytest.mark.parametrize("M,N", [(40, 64), (300, 1024)])
def test_ends_of_the_range(oracle, cuda, hiplib, M, N):
    """Finite results of huge and tiny rows (the decoded weights are small) stay finite and exact."""
    import torch

    K = 96
    x, w, _ = seeded_linear(M, M, K, N, w_scale=0.02)
    b = np.zeros(N, np.float32)
    c01, q2, s = oracle.quantize_nf24_i16(w)
    w64 = oracle.decode_nf24(c01, q2, s)
    y = x.copy()
    scales = {0: 1e36, 3: 3e37, 9: 1e-30, 20: 1e-33, 35: 6e37}
    for r, f in scales.items():
        y[r] *= np.float32(f)
    y[5] = 0.0
    y[5, 50] = 3.4e38
    got = _run(torch, y, c01, q2, s, b)
    assert np.all(np.isfinite(got))
    for r in [*scales, 5]:
        assert stats(got[r:r + 1], gemm_f64(y[r:r + 1], w64, b))["rel_rmse"] < 1e-6, r
    # any scale of the weights: x w stays at 0.02 N(0, 1)
    for f in (2.0 ** 100, 2.0 ** -100):
        got = _run(torch, x * np.float32(1.0 / f), c01, q2, s * np.float32(f), b)
        assert stats(got, gemm_f64(x, w64, b))["rel_rmse"] < 1e-6, f


@pytest.mark.parametrize("M", [37, 300])
@pytest.mark.parametrize("K,N", [(96, 130), (100, 131), (98, 132), (96, 252)])
def test_ranges_of_any_alignment(oracle, cuda, hiplib, M, K, N):
    """A column range of a small call holds the bits of the whole call, whichever
    kernel the weight's sizes send it to."""
    import torch
    from tsplat.nf24 import nf24_linear

    x, w, b = seeded_linear(M + K + N, M, K, N, w_scale=0.02)
    c01, q2, s = oracle.quantize_nf24_i16(w)
    _check(oracle, x, c01, q2, s, b, _run(torch, x, c01, q2, s, b))
    t = [torch.from_numpy(np.ascontiguousarray(a)).cuda() for a in (x, c01, q2, s, b)]
    full = nf24_linear(*t)
    for start, count in ((0, 2), (2, 6), (5, 7), (4, 100), (N - 1, 1), (1, N - 1)):
        got = nf24_linear(*t, output_start=start, output_count=count)
        assert torch.equal(got, full[:, start:start + count]), (start, count)


def test_capture_before_any_eager_call(oracle, cuda, hiplib):
    """A row tail that only the fp16 tiles split off: a capture on a stream
    without a workspace keeps it in the tiles."""
    import torch
    from tsplat.nf24 import nf24_linear

    M, K, N = 6913, 1024, 1664
    x, w, b = seeded_linear(3, M, K, N, w_scale=0.02)
    c01, q2, s = oracle.quantize_nf24_i16(w)
    t = [torch.from_numpy(np.ascontiguousarray(a)).cuda() for a in (x, c01, q2, s, b)]
    want = nf24_linear(*t)
    out = torch.empty_like(want)
    stream = torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=stream, capture_error_mode="relaxed"):
        nf24_linear(*t, out=out)
    for _ in range(3):
        out.fill_(float("nan"))
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(out[:-1], want[:-1])
        rows = slice(M - 1, M)
        _check(oracle, x[rows], c01, q2, s, b, out[rows].cpu().numpy())
        assert torch.equal(nf24_linear(*t), want)
