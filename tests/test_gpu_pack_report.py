"""The packer's error report against the same fp32 steps in torch on the CPU.

The digits and residuals are the same fp32 operations on both sides, so the
maxima and the clamp counts are equal; the sums of squares are fp64 sums of
the same fp32 squares, and only their order differs (1e-12 is 2^-52 times the
largest count here, rounded up).
"""
from __future__ import annotations

import math
import sys
from pathlib import Path

import pytest
import torch

sys.path.insert(0, str(Path(__file__).resolve().parents[1] / "triposplat-cpu-avx512_amd"))

pytestmark = pytest.mark.gpu


def _report(w, alphabet):
    base = torch.clamp_min(w.abs().amax(1), torch.finfo(torch.float32).tiny)[:, None] / 127.0
    mid = ((alphabet[:-1] + alphabet[1:]) * 0.5).contiguous()
    r1 = w - alphabet[torch.bucketize(w / base, mid)] * base
    s1, s2 = base / 4.0, base / 1024.0
    q1 = torch.floor(r1 / s1 + 0.5)
    r2 = r1 - q1.clamp(-128, 127) * s1
    q2 = torch.floor(r2 / s2 + 0.5)
    r3 = r2 - q2.clamp(-128, 127) * s2
    rms = [math.sqrt(float((r * r).double().mean())) for r in (r1, r2, r3, w)]
    top = [float(r.abs().max()) for r in (r1, r2, r3)]
    clamped = [0] + [int(((q < -128) | (q > 127)).sum()) for q in (q1, q2)]
    return rms, top, clamped


def _same(a, b):
    return math.isclose(a, b, rel_tol=1e-12) or (math.isnan(a) and math.isnan(b))


# one value, one row, one column, the edges of the 32 x 64 tile, many blocks
@pytest.mark.parametrize("out_f,in_f,kind", [
    (1, 1, "normal"), (1, 200, "normal"), (200, 1, "normal"), (32, 64, "normal"), (33, 65, "normal"),
    (31, 63, "steps"), (1024, 5, "normal"), (517, 1030, "steps"), (7, 70, "zero"), (40, 70, "nan"), (40, 70, "inf")])
def test_error_report(out_f, in_f, kind):
    from tsplat.nf24 import nf24_alphabet, quantize_nf24_i16_per_output_channel

    w = torch.randn((out_f, in_f), generator=torch.Generator().manual_seed(out_f * 1000 + in_f)) * 0.02
    if kind == "steps":  # a value of 127 a row and half steps of q2: its upper end is clamped
        w = torch.round(w * 50000.0) / 2048.0
        w[:, 0] = 127.0
    elif kind == "zero":
        w.zero_()
    elif kind in ("nan", "inf"):
        w[3, 4] = float(kind)
    rms, top, clamped = _report(w, nf24_alphabet(torch))
    _, _, got = quantize_nf24_i16_per_output_channel(w.cuda())
    for i, s in enumerate(got["stages"]):
        assert _same(s["residual_rmse"], rms[i]), (i, s, rms)
        assert _same(s["residual_max_abs"], top[i]), (i, s, top)
        assert s["saturated_values"] == clamped[i], (i, s, clamped)
    assert _same(got["weight_rmse"], rms[2]) and _same(got["weight_max_abs"], top[2])
    assert _same(got["weight_rms"], rms[3])
