"""The work that programs give this package, as cases that can be timed and checked.

Five kinds of call, each through the public ``op_plugin_amd`` entry points:

* ``rows``   the per-token quantizers in front of a W8A8 layer: ``npu_dynamic_quant``, and RMSNorm / SwiGLU fused
             with it;
* ``w8a8``   a W8A8 linear layer: ``npu_dynamic_quant`` of the activations, then ``npu_quant_matmul``;
* ``w4a16``  a weight-only int4 linear layer (``npu_weight_quant_batchmatmul``);
* ``w8a16``  the same with int8 weights;
* ``mlp``    the quantized Llama-style MLP block (``op_plugin_amd.mlp.quant_mlp``).

The row count of a call is the number of tokens a server has in hand: 1 to a few dozen in decode, anything up to
4096 in prefill, so odd counts are the rule.  The weight shapes are those of the benchmark configurations, the
shapes the tests and the shape sweep use, the way back of each MLP projection ([in, out] swapped), and the halves
and eighths that a tensor-parallel rank holds.  A weight is laid out once, outside the pass: FRACTAL_NZ as
``npu_format_cast`` writes it, row-major ``[K, N]``, or an nn.Linear ``[N, K]`` tensor passed transposed.
"""
from __future__ import annotations

import math
import os
import sys

import torch

_PKG = os.path.join(os.getcwd(), "ascend-python_amd")
if _PKG not in sys.path:
    sys.path.insert(1, _PKG)

import op_plugin_amd as q  # noqa: E402
from op_plugin_amd.mlp import quant_mlp  # noqa: E402

_DT = {"fp16": torch.float16, "bf16": torch.bfloat16}
_EPS = 1e-6

# [in, out] of the linear layers: the configurations' (4096 x 4096, 8192 x 28672, 4096 x 11008, 8192 x 8192,
# 4096 x 28672, 14336 x 4096) and their ways back, the tests' and the sweep's (5120 x 13696, 5120 x 1536,
# 2048 x 3072, 4096 x 1000, 4160 x 4096), a vocabulary head, and tensor-parallel halves and eighths.
_SHAPES = [
    (4096, 4096), (8192, 8192), (4096, 11008), (11008, 4096), (8192, 28672), (28672, 8192), (4096, 28672),
    (14336, 4096), (5120, 13696), (13696, 5120), (5120, 1536), (2048, 3072), (4096, 1000), (4160, 4096),
    (4096, 32000), (4096, 5504), (5504, 4096), (8192, 3584), (3584, 8192),
]
_MLP_SHAPES = [(4096, 14336), (4096, 11008), (5120, 13696), (2048, 5504)]  # hidden, intermediate
_ROW_WIDTHS = [1536, 2048, 4096, 5120, 8192, 11008, 13696, 14336, 28672]

# No drawn pass is longer than the longest listed ones of its kind: M * N * K of the 4096-row W8A8 prefill, of
# the 2048-row W4A16 prefill and of the 512-token MLP block.
_MOST = {"w8a8": 4096 * 8192 * 8192, "w4a16": 2048 * 4096 * 11008, "w8a16": 2048 * 4096 * 11008,
         "mlp": 512 * 3 * 4096 * 14336}


def listed():
    return [
        # One token of a decode step: the norm in front of a layer.  The smallest call, launch latency alone.
        dict(name="rms_quant_decode", kind="rows", op="rms", M=1, K=4096, dtype="bf16"),
        # The activations of a 4096-token prefill at width 8192 (with outlier channels), a pure memory stream.
        dict(name="dynamic_quant_prefill", kind="rows", op="dynamic", M=4096, K=8192, dtype="fp16"),
        # Four sequences in decode, the wide projection of a large model: a stream of 235 MB of weights.
        dict(name="w8a8_decode", kind="w8a8", M=4, K=8192, N=28672, layout="nz", bias=False, dtype="fp16"),
        # A batch of 128 sequences in decode on a square layer, the weight as it came from the checkpoint.
        dict(name="w8a8_batch", kind="w8a8", M=128, K=4096, N=4096, layout="kn", bias=True, dtype="fp16"),
        # The compute-bound prefill, weight cast at load time.
        dict(name="w8a8_prefill", kind="w8a8", M=4096, K=8192, N=8192, layout="nz", bias=True, dtype="fp16"),
        # A prompt of an odd length on an nn.Linear weight whose width is no multiple of a tile.
        dict(name="w8a8_prompt_ragged", kind="w8a8", M=997, K=5120, N=13696, layout="nk", bias=False, dtype="bf16"),
        # Weight-only int4 decode, 16 sequences, up projection.
        dict(name="w4a16_decode", kind="w4a16", M=16, K=4096, N=11008, layout="nz", group=128, offset=True,
             bias=False, dtype="bf16"),
        # Interactive decode, one token, the way back of the same block (down projection).
        dict(name="w4a16_decode_down", kind="w4a16", M=1, K=11008, N=4096, layout="nz", group=128, offset=True,
             bias=False, dtype="bf16"),
        # A short prompt or a large decode batch of an odd size, fp16, symmetric int4 rows as packed.
        dict(name="w4a16_batch_ragged", kind="w4a16", M=77, K=5120, N=13696, layout="kn", group=128, offset=False,
             bias=False, dtype="fp16"),
        # Weight-only int4 prefill on the row-major weight.
        dict(name="w4a16_prefill", kind="w4a16", M=2048, K=4096, N=11008, layout="kn", group=128, offset=True,
             bias=False, dtype="bf16"),
        # Weight-only int8 nn.Linear with one scale per channel and a bias, a small odd batch.
        dict(name="w8a16_linear", kind="w8a16", M=23, K=4096, N=11008, layout="nk", group=0, offset=False,
             bias=True, dtype="bf16"),
        # The whole quantized MLP block over a 512-token chunk.
        dict(name="mlp_block", kind="mlp", M=512, K=4096, N=14336, layout="nz", dtype="bf16"),
    ]


def _tokens(rng, most):
    """A token count, spread over its logarithm from 1 to `most`; every other one is odd."""
    m = int(round(math.exp(rng.uniform(0.0, math.log(max(1, most))))))
    if rng.random() < 0.5:
        m |= 1
    return max(1, min(m, most))


def draw(rng):
    kind = rng.choice(["rows", "w8a8", "w8a8", "w4a16", "w4a16", "w8a16", "mlp"])
    dtype = rng.choice(["fp16", "bf16"])
    if kind == "rows":
        op = rng.choice(["dynamic", "rms", "swiglu"])
        K = rng.choice(_ROW_WIDTHS)
        most = 4096 * 8192 // (K * (2 if op == "swiglu" else 1))
        return dict(kind=kind, op=op, M=_tokens(rng, min(4096, most)), K=K, dtype=dtype)
    if kind == "mlp":
        H, I = rng.choice(_MLP_SHAPES)
        return dict(kind=kind, M=_tokens(rng, min(2048, _MOST[kind] // (3 * H * I))), K=H, N=I,
                    layout=rng.choice(["nz", "nz", "kn", "nk"]), dtype=dtype)
    K, N = rng.choice(_SHAPES)
    M = _tokens(rng, min(4096, _MOST[kind] // (K * N)))
    block = 128 if kind == "w4a16" else 64
    layouts = ["kn"] if kind == "w4a16" else ["kn", "nk"]
    if K % block == 0 and N % 16 == 0:  # what npu_format_cast takes; a loaded weight is mostly cast
        layouts += ["nz"] * len(layouts)
    case = dict(kind=kind, M=M, K=K, N=N, layout=rng.choice(layouts), bias=rng.random() < 0.4, dtype=dtype)
    if kind != "w8a8":
        groups = [128, 128, 64, 0] if kind == "w4a16" else [0, 0, 128]
        case.update(group=rng.choice([g for g in groups if g == 0 or K % g == 0]), offset=rng.random() < 0.5)
    return case


# ---------------------------------------------------------------- inputs


def _uniform(g, shape, lo, hi):
    return lo + (hi - lo) * torch.rand(shape, generator=g, device="cuda")


def _activations(g, M, K, dtype):
    """N(0, 1) with 1 % of the channels 20 times as large, as activations in front of a quantizer are."""
    x = torch.randn((M, K), generator=g, device="cuda")
    x[:, torch.randperm(K, generator=g, device="cuda")[: max(1, K // 100)]] *= 20.0
    return x.to(dtype)


def _int8_weight(g, rows, cols):
    return torch.randint(-127, 128, (rows, cols), generator=g, device="cuda", dtype=torch.int8)


def _raw(case, seed):
    """The case's inputs as numbers, before any layout: weights are int8 values [in, out]."""
    g = torch.Generator(device="cuda").manual_seed(int(seed))
    kind, M, K, dtype = case["kind"], case["M"], case["K"], _DT[case["dtype"]]
    r = {}
    if kind == "rows":
        r["x"] = _activations(g, M, K * (2 if case["op"] == "swiglu" else 1), dtype)
        if case["op"] == "rms":
            r["gamma"] = (1.0 + 0.02 * torch.randn(K, generator=g, device="cuda")).to(dtype)
        return r
    N = case["N"]
    if kind == "mlp":
        r["x"] = torch.randn((M, K), generator=g, device="cuda").to(dtype)
        r["gamma"] = (1.0 + 0.02 * torch.randn(K, generator=g, device="cuda")).to(dtype)
        r["w_gu"], r["s_gu"] = _int8_weight(g, K, 2 * N), _uniform(g, 2 * N, 1e-3, 1e-2)
        r["w_d"], r["s_d"] = _int8_weight(g, N, K), _uniform(g, K, 1e-3, 1e-2)
        return r
    if kind == "w8a8":
        r["x"], r["w"] = _activations(g, M, K, dtype), _int8_weight(g, K, N)
        r["scale"] = _uniform(g, N, 1e-3, 1e-2)
    else:
        r["x"] = torch.randn((M, K), generator=g, device="cuda").to(dtype)
        rows = (K // case["group"], N) if case["group"] else (N,)
        if kind == "w4a16":
            r["w"] = torch.randint(-8, 8, (K, N), generator=g, device="cuda", dtype=torch.int8)
            r["scale"] = _uniform(g, rows, 5e-3, 2e-2).half()
        else:
            r["w"] = _int8_weight(g, K, N)
            r["scale"] = _uniform(g, rows, 3e-4, 1.2e-3).half()
        r["offset"] = _uniform(g, rows, -1.0, 1.0).half() if case["offset"] else None
    r["bias"] = (0.1 * torch.randn(N, generator=g, device="cuda")).to(torch.bfloat16 if kind == "w8a8" else dtype) \
        if case["bias"] else None
    return r


def _lay_out(w, layout, int4):
    """An int8 [in, out] weight as a program keeps it after loading."""
    if layout == "nk":
        return w.t().contiguous().t()
    if int4:
        w = q.npu_convert_weight_to_int4pack(w)
    return q.npu_format_cast(w, q.ACL_FORMAT_FRACTAL_NZ) if layout == "nz" else w


def prepare(case, seed):
    r = _raw(case, seed)
    kind = case["kind"]
    state = dict(r, case=case)
    if kind == "mlp":
        state["w_gu"] = _lay_out(r["w_gu"], case["layout"], False)
        state["w_d"] = _lay_out(r["w_d"], case["layout"], False)
    elif kind != "rows":
        state["w"] = _lay_out(r["w"], case["layout"], kind == "w4a16")
    return state


def run(state):
    s, case = state, state["case"]
    kind = case["kind"]
    if kind == "rows":
        if case["op"] == "dynamic":
            return q.npu_dynamic_quant(s["x"])
        if case["op"] == "rms":
            return q.npu_rms_norm_dynamic_quant(s["x"], s["gamma"], _EPS)
        return q.npu_swiglu_dynamic_quant(s["x"])
    if kind == "mlp":
        return quant_mlp(s["x"], s["gamma"], s["w_gu"], s["s_gu"], s["w_d"], s["s_d"], _EPS)
    if kind == "w8a8":
        xq, xs = q.npu_dynamic_quant(s["x"])
        return xq, xs, q.npu_quant_matmul(xq, s["w"], s["scale"], pertoken_scale=xs, bias=s["bias"],
                                          output_dtype=torch.bfloat16)
    return q.npu_weight_quant_batchmatmul(s["x"], s["w"], s["scale"], s["offset"], bias=s["bias"],
                                          antiquant_group_size=case["group"])


# ---------------------------------------------------------------- what a pass cannot do without


def work(case):
    kind, M, K = case["kind"], case["M"], case["K"]
    if kind == "rows":
        wide = 2 if case["op"] == "swiglu" else 1
        per_row = 4 + (4 if case["op"] == "rms" else 0)
        return dict(bytes=M * (2 * K * wide + K + per_row) + (2 * K if case["op"] == "rms" else 0), flops=0)
    N = case["N"]
    if kind == "mlp":
        return dict(bytes=M * 2 * K + 2 * K + 3 * K * N + 4 * (2 * N + K) + M * 2 * K, flops=2 * M * 3 * K * N)
    b = M * 2 * K + M * 2 * N + (2 * N if case["bias"] else 0)
    if kind == "w8a8":
        b += M * (K + 4) + K * N + 4 * N
    else:
        rows = K // case["group"] if case["group"] else 1
        b += K * N // (2 if kind == "w4a16" else 1) + rows * N * 2 * (2 if case["offset"] else 1)
    return dict(bytes=b, flops=2 * M * N * K)


# ---------------------------------------------------------------- correctness


def tolerance(case):
    kind = case["kind"]
    if kind == "rows" and case["op"] == "dynamic":
        return "exact"  # a maximum, a division and a rounding to whole numbers: nothing is left open
    if kind == "rows":
        # a 16-bit value on a rounding edge may fall either way before it is quantized
        return dict(rel=2e-3 if case["dtype"] == "bf16" else 3e-4, max=8e-3, differ=1e-3)
    if kind == "w8a8":
        # int8 rows and int32 sums are exact; the scaling may round a bf16 value the other way now and then
        return dict(rel=5e-4, max=8e-3, differ=0.0)
    if kind == "mlp":
        return dict(rel=1e-2 if case["dtype"] == "bf16" else 5e-3, max=0.2)
    # one 16-bit rounding of a 32-bit sum, four times what the path is off its 64-bit value
    return dict(rel=7e-3, max=4e-2) if case["dtype"] == "bf16" else dict(rel=1e-3, max=1e-2)


def _quantized(y):
    """Per-token int8 of y as the quantizer's contract has it (32-bit scale and quotient), with its 32-bit scale."""
    y = y.float()
    s = y.abs().amax(-1, keepdim=True) / 127.0
    return torch.where(s > 0, torch.round(y / s), torch.zeros_like(y)), s


def _columns(a, w, columns=4096):
    """a @ w in 64 bits, `columns` of the weight at a time; w(lo, hi) gives them as float64."""
    n = w(None, None)
    return torch.cat([a @ w(lo, min(n, lo + columns)) for lo in range(0, n, columns)], dim=1)


def _weight(w, scale=None, offset=None, group=0):
    """The columns of a weight, dequantized in 64 bits, for _columns."""
    def take(lo, hi):
        if lo is None:
            return w.shape[1]
        d = w[:, lo:hi].double()
        if scale is None:
            return d
        s = scale[..., lo:hi].double()
        o = offset[..., lo:hi].double() if offset is not None else None
        if group:
            s = s.repeat_interleave(group, 0)
            o = o.repeat_interleave(group, 0) if o is not None else None
        return (d + o if o is not None else d) * s
    return take


def exact(case, seed):
    r = _raw(case, seed)
    kind = case["kind"]
    if kind == "rows":
        x = r["x"].double()
        if case["op"] == "dynamic":
            return None, x.abs().amax(-1) / 127.0
        if case["op"] == "swiglu":
            a, b = x.chunk(2, dim=-1)
            return None, (a * torch.sigmoid(a) * b).abs().amax(-1) / 127.0
        rstd = torch.rsqrt(x.square().mean(-1, keepdim=True) + _EPS)
        return None, (x * rstd * r["gamma"].double()).abs().amax(-1) / 127.0, rstd
    if kind == "w8a8":
        xq, xs = _quantized(r["x"])
        out = _columns(xq.double(), _weight(r["w"])) * xs.double() * r["scale"].double()
        return None, xs.double().squeeze(-1), out if r["bias"] is None else out + r["bias"].double()
    if kind == "mlp":
        x, dtype = r["x"].double(), torch.bfloat16
        y = (x * torch.rsqrt(x.square().mean(-1, keepdim=True) + _EPS) * r["gamma"].double()).to(r["x"].dtype)
        y1, s1 = _quantized(y)
        gu = (_columns(y1.double(), _weight(r["w_gu"])) * s1.double() * r["s_gu"].double()).to(dtype).double()
        a, b = gu.chunk(2, dim=-1)
        y2, s2 = _quantized((a * torch.sigmoid(a) * b).to(dtype))
        return _columns(y2.double(), _weight(r["w_d"])) * s2.double() * r["s_d"].double()
    out = _columns(r["x"].double(), _weight(r["w"], r["scale"], r["offset"], case["group"]))
    return out if r["bias"] is None else out + r["bias"].double()
