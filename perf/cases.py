"""The performance cases of this repository: what a flow-model program has it do.

One case is one call (or one sampler step) through the public entry points:
the NF24 Linears at the timestep's few rows, at the bench's 4096 rows and at
the reference model's ragged lengths (8192 latent + 4101 condition + 1 camera
row), the fused QKV projection, the exact attention in its self, key-bias,
cross and selected-rows forms, LayerNorm with modulation, the packer, and a
whole CFG Euler step of the single-stream graph.  Inputs follow the model:
activations after LayerNorm ~ N(0, 1), weights 0.02 N(0, 1), q and k after
the per-head RMSNorm (norm 8 each).
"""
import math
import sys
from pathlib import Path

import torch

sys.path.insert(0, str(Path(__file__).resolve().parents[1] / "triposplat-cpu-avx512_amd"))

from tsplat import block_ops as bo  # noqa: E402
from tsplat.flow import FlowConfig  # noqa: E402
from tsplat.flow_joint import JointFlowModel  # noqa: E402
from tsplat.native_sdpa_ctypes import native_sdpa_f32_ex  # noqa: E402
from tsplat.nf24 import (bf16_planes, nf24_linear,  # noqa: E402
                         quantize_nf24_i16_per_output_channel)
from tsplat.qkv import gemm_nf24_qkv_direct  # noqa: E402

DEV = torch.device("cuda", 0)
HEADS, CHANNELS = 16, 1024


def linear(name, m, k, n, epilogue="none", precision="fp32"):
    return {"name": name, "kind": "linear", "m": m, "k": k, "n": n, "epilogue": epilogue, "precision": precision}


def sdpa(name, b, lq, lk, bias="none", packed=False, precision="fp32"):
    return {"name": name, "kind": "sdpa", "b": b, "lq": lq, "lk": lk, "bias": bias, "packed": packed,
            "precision": precision}


def listed():
    return [
        # the shared modulation of a CFG pair: two timestep rows, once per model call
        linear("adaln_2x1024x6144", 2, 1024, 6144),
        # the QKV-sized Linear of the reference's own GEMM benchmark
        linear("linear_4096x1024x3072", 4096, 1024, 3072),
        # the MLP's second Linear with its gated residual, positive branch at the model's real length
        linear("fc2_gated_12294x4096x1024", 12294, 4096, 1024, "gated"),
        # the MLP's first Linear of the selected-rows final block, opt-in products
        linear("fc1_gelu_bf16x3_8193", 8193, 1024, 4096, "gelu", "bf16x3"),
        # the fused QKV projection of the compressed negative branch
        {"name": "qkv_8194", "kind": "qkv", "b": 1, "l": 8194, "kv": "bhld", "precision": "fp32"},
        # dense self attention, the headline benchmark's length: the largest case
        sdpa("sdpa_self_16384", 1, 16384, 16384),
        # self attention of the compressed negative branch: log(4101) on one key
        sdpa("sdpa_key_bias_8194", 1, 8194, 8194, "shared"),
        # cross attention of a CFG pair at a small latent
        sdpa("sdpa_cross_2x1025x513", 2, 1025, 513),
        # the selected-rows final block's attention on packed K/V, opt-in products
        sdpa("sdpa_bf16x3_8193x12294", 1, 8193, 12294, "none", True, "bf16x3"),
        # LayerNorm + modulation of a CFG pair
        {"name": "layernorm_2x8192", "kind": "layernorm", "b": 2, "rows": 8192, "affine": False},
        # packing one MLP weight when a model is loaded from fp32
        {"name": "pack_4096x1024", "kind": "pack", "n": 4096, "k": 1024},
        # one CFG Euler step of the single-stream graph, four blocks, short sequence
        {"name": "step_2048_513_4blocks", "kind": "step", "l": 2048, "lc": 513, "blocks": 4, "precision": "fp32"},
    ]


def _log_uniform(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    kind = rng.choice(["few", "linear", "linear", "linear", "qkv", "sdpa", "sdpa", "sdpa", "layernorm", "pack", "step"])
    precision = rng.choice(["fp32", "fp32", "fp32", "bf16x3", "bf16"])
    if kind == "few":  # timestep, modulation and camera rows
        k, n = rng.choice([(256, 1024), (1024, 1024), (1024, 6144), (1024, 5), (5, 1024), (4096, 1024)])
        c = linear("", rng.randint(1, 32), k, n)
    elif kind == "linear":
        k, n = rng.choice([(1024, 1024), (1024, 2048), (1024, 3072), (1024, 4096), (4096, 1024)])
        c = linear("", _log_uniform(rng, 33, 12294), k, n, rng.choice(["none", "gelu", "gated", "add"]), precision)
    elif kind == "qkv":
        b = rng.choice([1, 2])
        c = {"kind": "qkv", "b": b, "l": _log_uniform(rng, 33, 12294 // b), "kv": rng.choice(["bhld", "packed"]),
             "precision": precision}
    elif kind == "sdpa":
        b = rng.choice([1, 2])
        lq, lk = _log_uniform(rng, 65, 12294 // b), _log_uniform(rng, 65, 12294)
        c = sdpa("", b, lq, lk, rng.choice(["none", "none", "shared", "per_head"]), rng.choice([False, True]), precision)
    elif kind == "layernorm":
        b = rng.choice([1, 2])
        c = {"kind": "layernorm", "b": b, "rows": _log_uniform(rng, 2, 16385), "affine": rng.choice([False, True])}
    elif kind == "pack":
        k, n = rng.choice([(256, 1024), (1024, 1024), (1024, 3072), (1024, 6144), (4096, 1024), (5, 1024), (1024, 5)])
        c = {"kind": "pack", "n": n, "k": k}
    else:
        c = {"kind": "step", "l": _log_uniform(rng, 64, 2048), "lc": _log_uniform(rng, 16, 513),
             "blocks": rng.randint(1, 4), "precision": rng.choice(["fp32", "fp32", "bf16x3"])}
    c.pop("name", None)
    return c


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _randn(g, *shape, std=1.0, mean=0.0):
    return torch.randn(shape, generator=g, device=DEV, dtype=torch.float32) * std + mean


def _packed_weight(g, k, n):
    codes, scales, _ = quantize_nf24_i16_per_output_channel(_randn(g, n, k, std=0.02))
    return codes[0], codes[1], scales[0], _randn(g, n, std=0.01)


def _heads(g, *shape):
    """Vectors of 64 with norm 8: q or k after the per-head RMSNorm."""
    x = _randn(g, *shape, 64)
    return x * (8.0 / x.norm(dim=-1, keepdim=True))


def _frequencies(length):
    i = torch.arange(32, dtype=torch.float64, device=DEV)
    ang = torch.arange(length, dtype=torch.float64, device=DEV)[:, None] * 10000.0 ** (-2.0 * i / 64.0)[None, :]
    f = torch.stack((torch.cos(ang), torch.sin(ang)), dim=-1).reshape(length, 64).to(torch.float32)
    return f[None, :, None, :].expand(1, length, HEADS, 64).contiguous()


def prepare(case, seed):
    g, kind = _gen(seed), case["kind"]
    s = {"case": case}
    if kind == "linear":
        m, k, n = case["m"], case["k"], case["n"]
        s["x"], s["w"] = _randn(g, m, k), _packed_weight(g, k, n)
        s["planes"] = None if case["precision"] == "fp32" else bf16_planes(*s["w"][:3], case["precision"])
        s["out"] = _randn(g, m, n) if case["epilogue"] in ("gated", "add") else None
        s["gate"] = _randn(g, 1, n, std=0.5) if case["epilogue"] == "gated" else None
    elif kind == "qkv":
        rows = case["b"] * case["l"]
        s["x"], s["w"] = _randn(g, rows, CHANNELS), _packed_weight(g, CHANNELS, 3 * CHANNELS)
        s["planes"] = None if case["precision"] == "fp32" else bf16_planes(*s["w"][:3], case["precision"])
        s["freqs"] = _frequencies(case["l"])
        s["q_gamma"], s["k_gamma"] = (_randn(g, HEADS, 64, std=0.05, mean=1.0) for _ in range(2))
    elif kind == "sdpa":
        b, lq, lk = case["b"], case["lq"], case["lk"]
        s["q"], k, v = _heads(g, b, HEADS, lq), _heads(g, b, HEADS, lk), _randn(g, b, HEADS, lk, 64, std=0.64)
        if case["packed"]:  # [B, H, 64, Lkp], zeros past Lk: what the QKV postprocess writes
            pad = (0, -lk % 16)
            k, v = (torch.nn.functional.pad(t.transpose(2, 3), pad).contiguous() for t in (k, v))
        s["k"], s["v"], s["bias"], s["head_bias"] = k, v, None, None
        if case["bias"] == "shared":  # one key stands for lk identical ones
            s["bias"] = torch.zeros(lk, device=DEV)
            s["bias"][lk - 1] = math.log(lk)
        elif case["bias"] == "per_head":
            s["head_bias"] = torch.rand((HEADS, lk), generator=g, device=DEV) * 2.0 - 2.0
    elif kind == "layernorm":
        b, rows = case["b"], case["rows"]
        s["x"] = _randn(g, b, rows, CHANNELS, std=1.5, mean=0.1)
        s["weight"] = s["bias"] = s["scale"] = s["shift"] = None
        if case["affine"]:
            s["weight"], s["bias"] = _randn(g, CHANNELS, std=0.05, mean=1.0), _randn(g, CHANNELS, std=0.02)
        else:
            mod = _randn(g, b, 6 * CHANNELS, std=0.3)
            s["shift"], s["scale"] = mod[:, :CHANNELS], mod[:, CHANNELS:2 * CHANNELS]
    elif kind == "pack":
        s["w"] = _randn(g, case["n"], case["k"], std=0.02)
    else:
        cfg = FlowConfig(blocks=case["blocks"], latent_tokens=case["l"], cond_tokens=case["lc"])
        s["model"] = JointFlowModel(cfg, DEV)
        if case["precision"] != "fp32":
            s["model"].set_precision(case["precision"], include=("blocks", "attention"))
        s["z"], s["cond"] = _randn(g, case["l"], CHANNELS), _randn(g, case["lc"], CHANNELS)
        s["cam"] = _randn(g, 1, cfg.cam_channels)
        s["step"] = int(seed) % 20
        # the model's per-length tables (rotations, selected rows, key bias) are laid out once per sampler run
        l, lc = case["l"], case["lc"]
        for rows in (lc + 1, 2):
            s["model"].freqs(l, rows)
            s["model"].selected(l, l + rows)
        s["model"].key_bias(l, lc)
    return s


EPILOGUES = {"gelu": bo.EPILOGUE_GELU, "gated": bo.EPILOGUE_GATED, "add": bo.EPILOGUE_ADD}


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "linear":
        if case["epilogue"] == "none":
            return nf24_linear(s["x"], *s["w"], precision=case["precision"], planes=s["planes"])
        return bo.nf24_linear_epilogue(s["x"], *s["w"], EPILOGUES[case["epilogue"]], out=s["out"], gate=s["gate"],
                                       precision=case["precision"], planes=s["planes"])
    if kind == "qkv":
        return gemm_nf24_qkv_direct(s["x"], *s["w"], s["freqs"], s["q_gamma"], s["k_gamma"], case["b"], case["l"],
                                    HEADS, kv_layout=case["kv"], precision=case["precision"], planes=s["planes"])
    if kind == "sdpa":
        return native_sdpa_f32_ex(s["q"], s["k"], s["v"], key_bias=s["bias"], key_bias_per_head=s["head_bias"],
                                  kv_packed=case["packed"], key_count=case["lk"] if case["packed"] else None,
                                  out_layout="blhd", precision=case["precision"])
    if kind == "layernorm":
        return bo.layer_norm(s["x"], 1e-6, s["weight"], s["bias"], scale=s["scale"], shift=s["shift"])
    if kind == "pack":
        codes, scales, error = quantize_nf24_i16_per_output_channel(s["w"])
        return {"code01_t": codes[0], "q2_t": codes[1], "scale": scales[0], "weight_rmse": error["weight_rmse"],
                "weight_max_abs": error["weight_max_abs"], "weight_rms": error["weight_rms"]}
    return s["model"].euler_cfg_step(s["z"], s["cond"], s["cam"], step=s["step"])


def _linear_work(m, k, n, extra=0):
    return {"bytes": 4 * m * k + 3 * k * n + 8 * n + 4 * m * n + extra, "flops": 2 * m * k * n}


def work(case):
    kind = case["kind"]
    if kind == "linear":
        m, n = case["m"], case["n"]
        return _linear_work(m, case["k"], n, 4 * m * n if case["epilogue"] in ("gated", "add") else 0)
    if kind == "qkv":
        rows = case["b"] * case["l"]
        return _linear_work(rows, CHANNELS, 3 * CHANNELS, 4 * case["l"] * CHANNELS)
    if kind == "sdpa":
        bh, lq, lk = case["b"] * HEADS, case["lq"], case["lk"]
        bias = {"none": 0, "shared": 4 * lk, "per_head": 4 * HEADS * lk}[case["bias"]]
        return {"bytes": 4 * 64 * bh * (2 * lq + 2 * lk) + bias, "flops": 4 * 64 * bh * lq * lk}
    if kind == "layernorm":
        n = case["b"] * case["rows"] * CHANNELS
        return {"bytes": 8 * n + 8 * CHANNELS * (1 if case["affine"] else case["b"]), "flops": 8 * n}
    if kind == "pack":
        n = case["n"] * case["k"]
        return {"bytes": 7 * n + 4 * case["n"], "flops": 0}
    # a step: both branches' Linears and attention; weights, states and each block's hidden rows once
    l, lc, c, total = case["l"], case["lc"], CHANNELS, {"bytes": 0, "flops": 0}
    for rows in (l + lc + 1, l + 2):
        for i in range(case["blocks"]):
            out = l + 1 if i == case["blocks"] - 1 else rows
            total["flops"] += 2 * c * c * (2 * rows + 10 * out) + 4 * c * out * rows
            total["bytes"] += 36 * c * c + 4 * c * (rows + out)
        total["flops"] += 4 * l * c * c
        total["bytes"] += 6 * c * c + 12 * l * c
    return total


def tolerance(case):
    """About four times the error against 64 bits that the products and sums of each type show."""
    kind, precision = case["kind"], case.get("precision", "fp32")
    if kind == "pack":
        return {"rel": 2e-6}
    if kind == "layernorm":
        return {"rel": 1e-6}
    if precision == "bf16":
        return {"rel": 1e-2}
    if precision == "bf16x3":
        return {"rel": 2.5e-5}
    return {"rel": 3e-6 if kind in ("linear", "qkv") else 1e-5}


# ---- the same results in 64 bits, from torch alone -------------------------

def _weight64(w):
    """The packed weight as the format defines it (an fp32 product), and its bias."""
    p = w[0].to(torch.int32) * 256 + w[1].to(torch.int32)
    return (p.to(torch.float32) * w[2]).double(), w[3].double()


def _linear64(x, w):
    wt, bias = _weight64(w)
    return x.double() @ wt + bias


def _gelu64(x):
    return 0.5 * x * (1.0 + torch.tanh(math.sqrt(2.0 / math.pi) * (x + 0.044715 * x * x * x)))


def _layernorm64(x, eps):
    x = x.double()
    mean = x.mean(-1, keepdim=True)
    return (x - mean) * torch.rsqrt(((x - mean) ** 2).mean(-1, keepdim=True) + eps)


def _rope64(x, freqs):
    """x [..., 64] rotated in (even, odd) pairs by freqs (cos, sin) pairs."""
    f = freqs.double()
    c, s, a, b = f[..., 0::2], f[..., 1::2], x[..., 0::2], x[..., 1::2]
    return torch.stack((a * c - b * s, a * s + b * c), -1).flatten(-2)


def _rms64(x, gamma):
    return x * 8.0 / x.norm(dim=-1, keepdim=True).clamp_min(1e-12) * gamma.double()


def _sdpa64(q, k, v, bias=None):
    """q [B, H, Lq, 64], k and v [B, H, Lk, 64], bias [H, Lk] or [1, Lk] -> [B, Lq, H, 64]."""
    b, h, lq, _ = q.shape
    out = torch.empty((b, lq, h, 64), dtype=torch.float64, device=q.device)
    for i in range(b):
        for j in range(h):
            kt, vt = k[i, j].double().t().contiguous(), v[i, j].double()
            for r in range(0, lq, 4096):
                score = q[i, j, r:r + 4096].double() @ kt / 8.0
                if bias is not None:
                    score += bias[j % bias.shape[0]].double()
                out[i, r:r + 4096, j] = torch.softmax(score, -1) @ vt
    return out


def _lin(lin):
    return lin.code01_t, lin.q2_t, lin.scale, lin.bias


def _step64(s):
    model, z, cond, cam = s["model"], s["z"], s["cond"], s["cam"]
    cfg, l, lc = model.cfg, s["case"]["l"], s["case"]["lc"]
    ts = [cfg.shift * u / (1.0 + (cfg.shift - 1.0) * u) for u in (1.0 - i / cfg.steps for i in range(cfg.steps + 1))]
    # the embedding's arguments are fp32 in the model: their cosine is part of its definition
    t = torch.full((1,), ts[s["step"]] * 1000.0, dtype=torch.float32, device=DEV)
    half = cfg.freq_dim // 2
    f = torch.exp(-math.log(10000.0) * torch.arange(half, dtype=torch.float32, device=DEV) / half)
    a = t[:, None] * f[None, :]
    silu = torch.nn.functional.silu
    temb = _linear64(silu(_linear64(torch.cat((torch.cos(a), torch.sin(a)), -1), _lin(model.t_fc1))), _lin(model.t_fc2))
    tmod = _linear64(silu(temb), _lin(model.adaln))

    def heads(x):
        return x.view(1, -1, HEADS, 64)

    def velocity(rows, bias):
        x = torch.cat((_linear64(z, _lin(model.input_layer)), rows.double(), _linear64(cam, _lin(model.cam_refiner))), 0)
        total = x.shape[0]
        ang = torch.zeros((total, 64), dtype=torch.float64, device=DEV)
        ang[:, 0::2] = 1.0
        ang[:l] = _frequencies(l)[0, :, 0].double()
        keep = torch.cat((torch.arange(l, device=DEV), torch.tensor([total - 1], device=DEV)))
        for i, blk in enumerate(model.blocks):
            mod = (tmod[0] + blk.shift_table.double()).view(6, CHANNELS)
            qkv = _linear64(_layernorm64(x, cfg.ln_eps) * (1.0 + mod[1]) + mod[0], _lin(blk.lin["qkv"]))
            q, k, v = (heads(qkv[:, j * CHANNELS:(j + 1) * CHANNELS]) for j in range(3))
            rot = ang[None, :, None, :]
            q, k = _rms64(_rope64(q, rot), blk.q_gamma), _rms64(_rope64(k, rot), blk.k_gamma)
            if i == len(model.blocks) - 1:  # only the latent and camera rows leave the model
                q, x = q[:, keep], x[keep]
            att = _sdpa64(*(t.transpose(1, 2) for t in (q, k, v)), bias=bias).reshape(-1, CHANNELS)
            x = x + _linear64(att, _lin(blk.lin["out"])) * mod[2]
            h = _layernorm64(x, cfg.ln_eps) * (1.0 + mod[4]) + mod[3]
            x = x + _linear64(_gelu64(_linear64(h, _lin(blk.lin["fc1"]))), _lin(blk.lin["fc2"])) * mod[5]
        fs = temb + model.final_shift_table.double()
        h = _layernorm64(x, cfg.final_ln_eps) * (1.0 + fs[1]) + fs[0]
        return _linear64(h[:l], _lin(model.out_layer)), _linear64(h[l:], _lin(model.cam_out_layer))

    bias = torch.zeros((1, l + 2), device=DEV)
    bias[0, l] = math.log(float(lc))
    pos, neg = velocity(cond, None), velocity(torch.zeros_like(cond[:1]), bias)
    dt, out = ts[s["step"]] - ts[s["step"] + 1], []
    for vp, vn, state in zip(pos, neg, (z, cam)):
        v = cfg.guidance * vp - (cfg.guidance - 1.0) * vn
        out += [state.double() - dt * v, v]
    return tuple(out)


def exact(case, seed):
    s, kind = prepare(case, seed), case["kind"]
    if kind == "linear":
        y = _linear64(s["x"], s["w"])
        if case["epilogue"] == "gelu":
            return _gelu64(y)
        if case["epilogue"] == "gated":
            return s["out"].double() + y * s["gate"].double()
        return y if s["out"] is None else s["out"].double() + y
    if kind == "qkv":
        b, l = case["b"], case["l"]
        y = _linear64(s["x"], s["w"]).view(b, l, 3, HEADS, 64)
        q = _rms64(_rope64(y[:, :, 0], s["freqs"]), s["q_gamma"])
        k = _rms64(_rope64(y[:, :, 1], s["freqs"]), s["k_gamma"])
        q, k, v = (t.transpose(1, 2).contiguous() for t in (q, k, y[:, :, 2]))
        if case["kv"] == "packed":
            k, v = (torch.nn.functional.pad(t.transpose(2, 3), (0, -l % 16)).contiguous() for t in (k, v))
        return q, k, v
    if kind == "sdpa":
        k, v = s["k"], s["v"]
        if case["packed"]:
            k, v = (t[..., :case["lk"]].transpose(2, 3) for t in (k, v))
        return _sdpa64(s["q"], k, v, s["bias"][None] if s["bias"] is not None else s["head_bias"])
    if kind == "layernorm":
        y = _layernorm64(s["x"], 1e-6)
        if case["affine"]:
            return y * s["weight"].double() + s["bias"].double()
        return y * (1.0 + s["scale"].double()[:, None]) + s["shift"].double()[:, None]
    if kind == "pack":
        w = s["w"].double()
        return {"code01_t": None, "q2_t": None, "scale": w.abs().amax(1) / 127.0 / 1024.0, "weight_rmse": None,
                "weight_max_abs": None, "weight_rms": float(w.square().mean().sqrt())}
    return _step64(s)
