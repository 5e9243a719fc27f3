"""The strict SDPA's 128-query tiles split along the keys (few queries, at
least 1024 keys): ragged query and key tiles, ranges of unequal length, a range
that holds masked keys alone, and an unsplit call of the same rows.  Against
the float64 formula, as closely as the fp32 oracle is."""
from __future__ import annotations

import math

import numpy as np
import pytest

from _parity import sdpa_f64, stats
from test_gpu_sdpa import _qkv, _run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("packed", [False, True])
@pytest.mark.parametrize("H,Lq,Lk,bias", [(1, 1, 1024, None), (2, 127, 1025, "one"), (2, 128, 4097, None),
                                          (3, 129, 2111, "mask"), (16, 300, 1100, "one"), (16, 2050, 2562, None)])
def test_key_ranges(oracle, cuda, H, Lq, Lk, bias, packed):
    import torch

    print(f"sdpa key ranges H={H} Lq={Lq} Lk={Lk} bias={bias} packed={packed}", flush=True)
    q, k, v = _qkv(Lq + Lk, 1, H, Lq, Lk)
    b = None
    if bias == "one":
        b = np.zeros(Lk, np.float32)
        b[Lk - 1] = math.log(Lk)
    elif bias == "mask":  # the first and the last 300 keys
        b = np.zeros(Lk, np.float32)
        b[:300] = b[-300:] = -np.inf
    got = _run(torch, cuda, q, k, v, b, packed=packed)
    rows = np.unique(np.r_[0:min(Lq, 24), max(0, Lq - 24):Lq])
    sub = slice(300, Lk - 300) if bias == "mask" else slice(0, Lk)
    ks, vs = np.ascontiguousarray(k[:, :, sub]), np.ascontiguousarray(v[:, :, sub])
    bs = None if b is None else np.ascontiguousarray(b[sub])
    exact = sdpa_f64(q[:, :, rows], ks, vs, bs)
    ref = oracle.sdpa_q8t512(np.ascontiguousarray(q[:, :, rows]), ks, vs, bs)
    got = got[:, :, rows]
    assert np.all(np.isfinite(got))
    assert stats(got, exact)["rmse"] <= 1.1 * stats(ref, exact)["rmse"] + 2.0 ** -24 * float(np.abs(v).max())
