"""The performance cases of the quantized-inference library: what its users run, through the public Python binding.

A case is a dict of plain values with an "op":
  quant   AscendQuant per-token dynamic (x -> int8 + fp32 scale per row), then AscendDequant back to x's type
  w8a8    the int8 Matmul with int32 bias and per-channel dequant (f16 / bf16 C) or requant (int8 C)
  fp8     the fp8 e4m3 Matmul with per-channel QF322BF16 -> bf16
  mxfp4   the MX block-scaled E2M1 Matmul -> bf16
  wo      the weight-only antiquant matmul (W4A16 / W8A16, group-wise f16 scale + offset) -> f16
  moe     the quantized group matmul (int8, per-token and per-channel scales) -> bf16
Sizes are those of the repository's benchmark and tests: K = 4096 / 11008 and N = 11008 / 4096 projections at decode
batches (1-64 rows) and prefill batches (512-4096 rows), 8192 x 8192 (x 8192), 16 experts of 4096 x 1408.
"""
from __future__ import annotations

import math
import sys
from pathlib import Path

import torch

sys.path.insert(0, str(Path(__file__).resolve().parents[1] / "asc-devkit_clone_amd"))
import ascq  # noqa: E402

DEV = "cuda"
FLOAT = {"f16": torch.float16, "bf16": torch.bfloat16}
CUBE = 8192 ** 3  # M N K of the largest listed Matmuls


def listed():
    return [
        # one decode step's activations of 16 sequences, quantised for a W8A8 layer and back: the smallest call, latency
        dict(name="quant_decode", op="quant", m=16, n=4096, dtype="f16"),
        # the headline: a large prefill activation, HBM-bound
        dict(name="quant_8192", op="quant", m=8192, n=8192, dtype="f16"),
        # up projection at a decode batch, weights laid out [N, K]: the weight stream
        dict(name="w8a8_decode", op="w8a8", m=16, n=11008, k=4096, trans_b=True, out="f16"),
        # the same projection at a prefill chunk of 512 tokens, weights [K, N] as the reference's default has them
        dict(name="w8a8_prefill_512", op="w8a8", m=512, n=11008, k=4096, trans_b=False, out="f16"),
        # the largest int8 Matmul
        dict(name="w8a8_8192", op="w8a8", m=8192, n=8192, k=8192, trans_b=False, out="f16"),
        # sizes that divide nothing (an odd batch, a K and an N that were never padded)
        dict(name="w8a8_ragged", op="w8a8", m=1030, n=4100, k=4095, trans_b=False, out="f16"),
        # fp8 down projection at a decode batch: long K
        dict(name="fp8_decode_64", op="fp8", m=64, n=4096, k=11008, trans_b=True),
        # fp8 up projection at a prefill batch
        dict(name="fp8_prefill_2048", op="fp8", m=2048, n=11008, k=4096, trans_b=True),
        # the largest MX-FP4 Matmul
        dict(name="mxfp4_8192", op="mxfp4", m=8192, n=8192, k=8192, pair_scales=False),
        # weight-only int4, one sequence: the decode GEMV
        dict(name="w4_decode", op="wo", m=1, n=11008, k=4096, bits=4, group=128),
        # weight-only int4 at a prefill chunk
        dict(name="w4_prefill_512", op="wo", m=512, n=11008, k=4096, bits=4, group=128),
        # a mixture-of-experts layer: 4096 routed tokens over 16 experts of uneven load, weights [G, K, N]
        dict(name="moe_4096", op="moe", m=4096, n=1408, k=4096, experts=16, trans_b=False),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _size(rng, lo, hi, step):
    return max(lo, _log(rng, lo, hi) // step * step)


def draw(rng):
    op = rng.choice(["quant", "w8a8", "w8a8", "fp8", "fp8", "mxfp4", "wo", "wo", "moe"])
    ragged = rng.random() < 0.25
    while True:
        m = _log(rng, 1, 8192)
        k = _size(rng, 512, 14336, 128)
        n = _size(rng, 512, 14336, 64)
        if op == "quant":
            m, n = _log(rng, 1, 16384), _size(rng, 512, 16384, 1 if ragged else 64)
            c = dict(op=op, m=m, n=n, dtype=rng.choice(["f16", "bf16"]))
            cost, most = m * n, 8192 * 8192
        elif op in ("w8a8", "fp8"):
            if ragged:
                n = _size(rng, 512, 8192, 1)
            if ragged and op == "w8a8":
                k = _size(rng, 512, 8192, 1)
            c = dict(op=op, m=m, n=n, k=k, trans_b=(op == "fp8" and ragged) or rng.random() < 0.5)
            if op == "w8a8":
                c["out"] = rng.choice(["f16", "f16", "bf16", "int8"])
            cost, most = m * n * k, CUBE // (8 if ragged else 1)
        elif op == "mxfp4":
            c = dict(op=op, m=m, n=n, k=k, pair_scales=rng.random() < 0.5)
            cost, most = m * n * k, CUBE
        elif op == "wo":
            m = rng.choice([_log(rng, 1, 64), _log(rng, 65, 4096)])
            c = dict(op=op, m=m, n=n, k=k, bits=rng.choice([4, 8]), group=rng.choice([128, 128, 64]))
            cost, most = m * n * k, 4096 * 11008 * 2048
        else:
            m = _log(rng, 16, 16384)
            n, k = _size(rng, 512, 8192, 64), _size(rng, 512, 8192, 128)
            c = dict(op=op, m=m, n=n, k=k, experts=rng.choice([8, 16, 64]), trans_b=rng.random() < 0.5)
            cost, most = max(m * n * k, c["experts"] * n * k * 32), CUBE // 2
        if cost <= most:
            return c


# ------------------------------------------------------------------------------------------------
# inputs
# ------------------------------------------------------------------------------------------------
def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    return g


def _codes(g, shape, std, lo, hi):
    """integer codes of absmax-quantised normal data"""
    return (torch.randn(shape, generator=g, device=DEV) * std).round_().clamp_(lo, hi).to(torch.int8)


def _e2m1(g, rows, k):
    """[rows, k / 2] bytes of nearest E2M1 codes of N(0, 2) data, even element in the low nibble"""
    x = torch.randn((rows, k), generator=g, device=DEV) * 2
    mid = torch.tensor([0.25, 0.75, 1.25, 1.75, 2.5, 3.5, 5.0], device=DEV)
    code = torch.bucketize(x.abs(), mid).to(torch.uint8) | ((x < 0).to(torch.uint8) << 3)
    return (code[:, 0::2] | (code[:, 1::2] << 4)).contiguous()


def _channel_scales(g, n, typical):
    """per-channel multipliers within a factor of two of `typical`, representable in QUANT_PRE's 19 bits"""
    s = typical * (0.5 + 1.5 * torch.rand(n, generator=g, device=DEV))
    return s.to(torch.bfloat16).float()


def _words(scale):
    return scale.view(torch.int32).to(torch.int64) & 0xFFFFFFFF


def _inputs(c, seed):
    g, op = _gen(seed), c["op"]
    if op == "quant":
        x = torch.randn((c["m"], c["n"]), generator=g, device=DEV)
        x = torch.where(torch.rand(x.shape, generator=g, device=DEV) < 0.001, x * 50, x)
        return dict(x=x.to(FLOAT[c["dtype"]]))
    m, n, k = c["m"], c["n"], c["k"]
    if op == "w8a8":
        typical = (20.0 if c["out"] == "int8" else 1.0) / (32 * 32 * math.sqrt(k))
        return dict(a=_codes(g, (m, k), 32, -127, 127),
                    b=_codes(g, (n, k) if c["trans_b"] else (k, n), 32, -127, 127),
                    bias=torch.randint(-30000, 30001, (n,), generator=g, device=DEV, dtype=torch.int32),
                    scale=_channel_scales(g, n, typical))
    if op == "fp8":
        e4m3 = lambda shape: torch.randn(shape, generator=g, device=DEV).to(torch.float8_e4m3fn)  # noqa: E731
        return dict(a=e4m3((m, k)), b=e4m3((n, k) if c["trans_b"] else (k, n)),
                    scale=_channel_scales(g, n, 1 / math.sqrt(k)))
    if op == "mxfp4":
        e8m0 = lambda shape: torch.randint(125, 130, shape, generator=g, device=DEV, dtype=torch.uint8)  # noqa: E731
        return dict(a=_e2m1(g, m, k), b=_e2m1(g, n, k), sa=e8m0((m, k // 32)),
                    sb=e8m0((k // 64, n, 2) if c["pair_scales"] else (n, k // 32)))
    if op == "wo":
        lim = 8 if c["bits"] == 4 else 128
        w = _codes(g, (k, n), lim / 4, -lim, lim - 1)
        rows = k // c["group"]
        scale = (1 / (lim / 4 * math.sqrt(k))) * (0.5 + torch.rand((rows, n), generator=g, device=DEV))
        offset = torch.randint(-lim // 4, lim // 4 + 1, (rows, n), generator=g, device=DEV)
        return dict(x=torch.randn((m, k), generator=g, device=DEV).half(), w=w, scale=scale.half(), offset=offset.half())
    share = torch.rand(c["experts"], generator=g, device=DEV) + 0.25
    edges = (share.cumsum(0) / share.sum() * m).round().long()
    edges[-1] = m
    counts = torch.diff(edges, prepend=torch.zeros(1, dtype=torch.int64, device=DEV))
    return dict(x=_codes(g, (m, k), 32, -127, 127),
                w=_codes(g, (c["experts"], n, k) if c["trans_b"] else (c["experts"], k, n), 32, -127, 127),
                pts=0.01 + 0.02 * torch.rand(m, generator=g, device=DEV),
                scale=(1 / (20 * math.sqrt(k))) * (0.5 + torch.rand((c["experts"], n), generator=g, device=DEV)),
                counts=counts)


def prepare(case, seed):
    """weights, activations and output buffers on the GPU, and the handle (or packed weight) a serving program keeps"""
    c, t, op = case, _inputs(case, seed), case["op"]
    state = dict(c=c, **t)
    if op == "quant":
        x = t["x"]
        state.update(q=torch.empty(x.shape, dtype=torch.int8, device=DEV),
                     s=torch.empty(c["m"], dtype=torch.float32, device=DEV), y=torch.empty_like(x))
    elif op in ("w8a8", "fp8", "mxfp4"):
        m, n, k = c["m"], c["n"], c["k"]
        if op == "w8a8":
            out = {"f16": ascq.F16, "bf16": ascq.BF16, "int8": ascq.INT8}[c["out"]]
            mm = ascq.Matmul(ascq.INT8, ascq.INT8, out, ascq.INT32)
            mm.SetBias(t["bias"])
        elif op == "fp8":
            mm = ascq.Matmul(ascq.FP8_E4M3, ascq.FP8_E4M3, ascq.BF16)
        else:
            mm = ascq.Matmul(ascq.FP4_E2M1, ascq.FP4_E2M1, ascq.BF16, 0, ascq.E8M0)
        mm.SetOrgShape(m, n, k)
        mm.SetTensorB(t["b"], c.get("trans_b", True))
        if op == "mxfp4":
            mm.SetTensorScaleB(t["sb"], not c["pair_scales"])
        else:
            if op == "w8a8" and c["out"] == "int8":
                words = _words(t["scale"]) | (1 << 46)  # signed int8 saturation
            else:
                words = _words(t["scale"])
            state["words"] = words
            mm.SetQuantVector(words)
        dtype = {"f16": torch.float16, "int8": torch.int8}.get(c.get("out"), torch.bfloat16)
        state.update(mm=mm, y=torch.empty((m, n), dtype=dtype, device=DEV))
    elif op == "wo":
        w, w_type = t["w"], ascq.INT8
        if c["bits"] == 4:
            u = (w & 15).to(torch.uint8)
            w, w_type = (u[:, 0::2] | (u[:, 1::2] << 4)).contiguous(), ascq.INT4
        state.update(w=None, w_type=w_type, packed=ascq.weight_pack(w, w_type, c["k"], c["n"]),
                     y=torch.empty((c["m"], c["n"]), dtype=torch.float16, device=DEV))
    else:
        state["y"] = torch.empty((c["m"], c["n"]), dtype=torch.bfloat16, device=DEV)
    return state


def run(state):
    s, c, op = state, state["c"], state["c"]["op"]
    if op == "quant":
        q, sc = ascq.quant_dynamic_per_token(s["x"], out=s["q"], scale_out=s["s"])
        y = ascq.ascend_dequant_policy(q, sc, ascq.PER_TOKEN, FLOAT[c["dtype"]], out=s["y"])
        return dict(q=q, s=sc, y=y)
    if op in ("w8a8", "fp8", "mxfp4"):
        mm = s["mm"]
        mm.SetTensorA(s["a"])
        if op == "mxfp4":
            mm.SetTensorScaleA(s["sa"])
        mm.IterateAll(s["y"])
        return s["y"]
    if op == "wo":
        return ascq.antiquant_matmul(s["x"], s["packed"], s["w_type"], s["scale"], s["offset"], c["group"], c["n"],
                                     out=s["y"])
    return ascq.quant_group_matmul(s["x"], s["pts"], s["w"], s["scale"], s["counts"], 1, c["trans_b"], torch.bfloat16,
                                   out=s["y"])


def work(case):
    c, op, m, n = case, case["op"], case["m"], case["n"]
    if op == "quant":
        # quant reads x and writes q and the scales; dequant reads them and writes y
        return dict(bytes=6 * m * n + 8 * m, flops=3 * m * n)
    k, mnk = c["k"], 2 * m * n * c["k"]
    if op == "w8a8":
        return dict(bytes=m * k + k * n + m * n * (1 if c["out"] == "int8" else 2) + 12 * n, flops=mnk)
    if op == "fp8":
        return dict(bytes=m * k + k * n + 2 * m * n + 8 * n, flops=mnk)
    if op == "mxfp4":
        return dict(bytes=(m + n) * (k // 2 + k // 32) + 2 * m * n, flops=mnk)
    if op == "wo":
        return dict(bytes=k * n * c["bits"] // 8 + 4 * (k // c["group"]) * n + 2 * m * k + 2 * m * n, flops=mnk)
    # the experts that get tokens stream their weights once
    used = min(c["experts"], m)
    return dict(bytes=m * k + 4 * m + used * (k * n + 4 * n) + 2 * m * n, flops=mnk)


def tolerance(case):
    """quant and the int8 paths are pinned bit for bit (integer sums, one fp32 product, one rounding).  fp8 and MX-FP4:
    fp32 sums of up to 14336 products (fp8: the matrix unit aligns each group of 16 to its largest) and one rounding to
    bf16, 1.7e-3 off the 64-bit result; weight-only: the same with f16, 2e-4 off."""
    if case["op"] in ("fp8", "mxfp4"):
        return dict(rel=5e-3)
    if case["op"] == "wo":
        return dict(rel=8e-4)
    return "exact"


# ------------------------------------------------------------------------------------------------
# the same in 64 bits, plain torch
# ------------------------------------------------------------------------------------------------
def _decode_e2m1(b, scales):
    """[rows, k / 2] bytes and [rows, k / 32] E8M0 scales -> float64 [rows, k]"""
    table = torch.tensor([0, 0.5, 1, 1.5, 2, 3, 4, 6, -0.0, -0.5, -1, -1.5, -2, -3, -4, -6], dtype=torch.float64,
                         device=DEV)
    v = torch.stack([table[(b & 15).long()], table[(b >> 4).long()]], dim=-1).reshape(b.shape[0], -1)
    return v * torch.exp2(scales.double() - 127).repeat_interleave(32, dim=1)


def exact(case, seed):
    c, t, op = case, _inputs(case, seed), case["op"]
    if op == "quant":
        x = t["x"].double()
        top = x.abs().amax(dim=1, keepdim=True)
        q = torch.where(top > 0, (x * (127 / top)).round(), torch.zeros_like(x))
        return dict(q=None, s=(top / 127).reshape(-1), y=q * (top / 127))
    if op == "w8a8":
        if c["out"] == "int8":
            return None
        b = t["b"].double()
        acc = t["a"].double() @ (b.t() if c["trans_b"] else b) + t["bias"].double()
        return acc * t["scale"].double()
    if op == "fp8":
        b = t["b"].float().double()
        return (t["a"].float().double() @ (b.t() if c["trans_b"] else b)) * t["scale"].double()
    if op == "mxfp4":
        sb = t["sb"].permute(1, 0, 2).reshape(c["n"], -1) if c["pair_scales"] else t["sb"]
        return _decode_e2m1(t["a"], t["sa"]) @ _decode_e2m1(t["b"], sb).t()
    if op == "wo":
        # the dequantised weight is an f16 value by definition: (q + offset) and its product are half operations
        rep = lambda v: v.repeat_interleave(c["group"], dim=0)  # noqa: E731
        w = (t["w"].half() + rep(t["offset"])) * rep(t["scale"])
        return t["x"].double() @ w.double()
    y = torch.zeros((c["m"], c["n"]), dtype=torch.float64, device=DEV)
    at = 0
    for e, rows in enumerate(t["counts"].tolist()):
        w = t["w"][e].double()
        part = t["x"][at:at + rows].double() @ (w.t() if c["trans_b"] else w)
        y[at:at + rows] = part * t["scale"][e].double() * t["pts"][at:at + rows, None].double()
        at += rows
    return y
