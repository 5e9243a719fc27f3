"""Calls of several host threads on one stream: each call's launches, and the
workspace they share, stay together.  On the host with fake streams, and on the
GPU against the results of the same calls one after another."""
from __future__ import annotations

import shutil
import subprocess
import threading
from pathlib import Path

import pytest

HERE = Path(__file__).resolve().parent
CSRC = HERE.parent / "triposplat-cpu-avx512_amd" / "csrc"


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs a host C++ compiler")
def test_enqueue_locks(tmp_path):
    exe = tmp_path / "workspace_threads_check"
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-pthread", "-I", str(CSRC),
                    str(HERE / "workspace_threads_check.cpp"), "-o", str(exe)], check=True, timeout=120)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout + r.stderr
    assert r.stdout.strip() == "ok"


@pytest.mark.gpu
def test_threads_on_one_stream(cuda, hiplib):
    """Presplit images, key ranges, a split last round, few-row sums and row
    tails from four threads on the default stream."""
    import torch
    from tsplat.native_sdpa_ctypes import native_sdpa_f32_ex
    from tsplat.nf24 import nf24_linear, quantize_nf24_i16_per_output_channel

    g = torch.Generator(device=cuda).manual_seed(5)

    def randn(*shape):
        return torch.randn(shape, generator=g, device=cuda)

    calls = []
    for h, lq, lk, precision in ((16, 300, 2100, "fp32"), (64, 2050, 300, "fp32"), (64, 2100, 700, "fp32"),
                                 (2, 70, 4000, "fp32"), (64, 6200, 130, "bf16x3")):
        q, k, v = randn(1, h, lq, 64), randn(1, h, lk, 64), randn(1, h, lk, 64)
        calls.append(lambda q=q, k=k, v=v, p=precision: native_sdpa_f32_ex(q, k, v, out_layout="blhd", precision=p))
    codes, scales, _ = quantize_nf24_i16_per_output_channel(randn(1024, 1024) * 0.02)
    w = (codes[0], codes[1], scales[0], randn(1024))
    for m in (2, 12, 16385):
        x = randn(m, 1024)
        calls.append(lambda x=x: nf24_linear(x, *w))
    want = [f() for f in calls]
    torch.cuda.synchronize()
    wrong = []

    def work(t):
        with torch.cuda.device(cuda):
            for i in range(24):
                j = (i * (2 * t + 1) + t) % len(calls)
                got = calls[j]()
                if not torch.equal(got, want[j]):
                    wrong.append((t, i, j))

    threads = [threading.Thread(target=work, args=(t,)) for t in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong
