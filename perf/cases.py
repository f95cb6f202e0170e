"""The work that programs built on this package give it, for timing: whole passes through its public entry points.

The sizes are the five benchmark configurations of ``segquant_amd.workloads`` and generic ones of the same ranges:
one conditioning vector to 9216 tokens, whole and ragged sizes, every activation / weight format pair, static and
dynamic scales, DualScale, the three float types, the chained and the fused forms of the layers, the reference-named
operators, and the encoding of weights.  A case is a dict of plain values:

    kind "linear"    one SegmentLinear on (M, K) -> (M, N), its outputs in `segments` equal runs
         "block"     the three linears of a transformer block: qkv, mlp_up and mlp_down of width `dim`
         "mlp"       fc1 -> GELU(tanh) -> fc2 (DualScale) through forward_into
         "geglu"     proj -> x * gelu(gate) -> ff_out, int4 weights with one scale per 128 input channels
         "parts"     a linear on the concatenation of an attention output and a GELU'd MLP state (forward_parts)
         "operator"  the reference-named operators of ext_dict on (S, M, K) tensors
         "svd"       a smoothed linear with a 16-bit low-rank branch
         "weights"   weights -> codes, and for e4m3 the float -> e4m3 -> float round trip as well
"""
from __future__ import annotations

import math

import torch

from segquant_amd import ops
from segquant_amd.layers import ext_dict
from segquant_amd.layers.SegmentLinear import SegmentLinear
from segquant_amd.optimum.smooth import SmoothOptimizer
from segquant_amd.utils.extension import load_fake_quant_fp8_ext, load_real_quant_fp8_ext, load_real_quant_int4_ext, load_real_quant_int8_ext

_DEV = "cuda"
_DT = {"fp32": torch.float32, "fp16": torch.float16, "bf16": torch.bfloat16}
_SIZE = {"fp32": 4, "fp16": 2, "bf16": 2}
_CODE_BYTES = {"int8": 1.0, "fpe4m3": 1.0, "int4": 0.5}


def listed():
    return [
        # the modulation linear of a block on the conditioning vectors of a batch of two: launches and latency
        dict(name="modulation_2", kind="linear", M=2, K=1536, N=9216, segments=6, act="int8", weight="int8", dtype="fp16",
             dynamic=False, per_channel=False, group=0),
        # configuration 1: six output segments, fp32 in and out
        dict(name="adaln_256", kind="linear", M=256, K=1536, N=9216, segments=6, act="int8", weight="int8", dtype="fp32",
             dynamic=False, per_channel=False, group=0),
        # a batch of text tokens through an adapter: no dimension is a multiple of a tile
        dict(name="ragged_333", kind="linear", M=333, K=1168, N=1000, segments=1, act="int8", weight="int8", dtype="bf16",
             dynamic=False, per_channel=True, group=0),
        # int4 weights on two prompts of 77 tokens: reading the weights is what such a call is made for
        dict(name="int4_154", kind="linear", M=154, K=1280, N=5120, segments=1, act="int8", weight="int4", dtype="bf16",
             dynamic=True, per_channel=True, group=0),
        # configuration 3: the headline workload, dynamic scale per token
        dict(name="block_4608", kind="block", M=4608, dim=3072, act="int8", dtype="bf16"),
        # configuration 2: two chained linears in e4m3, the second DualScale
        dict(name="mlp_4096", kind="mlp", M=4096, K=1536, H=6144, act="fpe4m3", dtype="bf16"),
        # configuration 4: a gated feed-forward, int4 weights, a scale per 128 input channels
        dict(name="geglu_8192", kind="geglu", M=8192, K=1280, H=5120, dtype="bf16"),
        # configuration 5 at its largest and (e4m3) at its smallest: two input segments, the second GELU'd and DualScale
        dict(name="parts_int8_9216", kind="parts", M=9216, K0=3072, K1=12288, N=3072, act="int8", dtype="bf16"),
        dict(name="parts_e4m3_1024", kind="parts", M=1024, K0=3072, K1=12288, N=3072, act="fpe4m3", dtype="bf16"),
        # the reference's own operator, two segments, DualScale: how a program that kept its layers calls this package
        dict(name="operator_dual", kind="operator", S=2, M=2048, K=3072, N=1536, dual=True, act="int8", weight="int8", dtype="fp16"),
        # SmoothQuant division and a rank-32 branch around the largest linear of configuration 3
        dict(name="svd_4608", kind="svd", M=4608, K=3072, N=12288, rank=32, dtype="bf16"),
        # a layer's weights at load time: codes, and the fake-quantised weights a quality check compares with
        dict(name="weights_e4m3", kind="weights", N=9216, K=3072, fmt="fpe4m3", group=0, dtype="bf16"),
    ]


def _log(rng, lo, hi, step=1):
    """A multiple of `step` in [lo, hi], spread over the logarithm."""
    v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return min(hi, max(step, lo, round(v / step) * step))


def draw(rng):
    kind = rng.choice(["few", "few", "ragged", "ragged", "int4", "block", "mlp", "geglu", "parts", "operator", "svd", "weights"])
    fmt = rng.choice(["int8", "fpe4m3"])
    dtype = rng.choice(["bf16", "bf16", "fp16", "fp32"])
    d16 = rng.choice(["bf16", "fp16"])
    if kind == "few":  # conditioning vectors and few tokens
        seg = rng.choice([1, 2, 3, 6])
        return dict(kind="linear", M=_log(rng, 1, 320), K=_log(rng, 256, 6144, 128), N=seg * _log(rng, 512, 3072, 64), segments=seg,
                    act=fmt, weight=fmt, dtype=dtype, dynamic=rng.random() < 0.5, per_channel=rng.random() < 0.5, group=0)
    if kind == "ragged":  # any size the layers take: K in sixteens, anything else at all
        return dict(kind="linear", M=_log(rng, 9, 5000), K=_log(rng, 144, 5000, 16), N=_log(rng, 96, 6000), segments=1, act=fmt,
                    weight=fmt, dtype=dtype, dynamic=rng.random() < 0.5, per_channel=rng.random() < 0.5, group=0)
    if kind == "int4":
        group = rng.choice([0, 0, 128])
        return dict(kind="linear", M=_log(rng, 1, 4096), K=_log(rng, 512, 5120, 128 if group else 32), N=_log(rng, 640, 10240, 64), segments=1,
                    act="int8", weight="int4", dtype=d16, dynamic=True, per_channel=True, group=group)
    if kind == "block":
        return dict(kind="block", M=_log(rng, 200, 4608), dim=rng.choice([1152, 1536, 2048, 2432, 3072]), act=fmt, dtype=d16)
    if kind == "mlp":
        k = rng.choice([1152, 1280, 1536, 2048, 3072])
        return dict(kind="mlp", M=_log(rng, 100, 4608), K=k, H=4 * k, act=fmt, dtype=d16)
    if kind == "geglu":
        k = rng.choice([640, 1280, 1536])
        return dict(kind="geglu", M=_log(rng, 77, 8192), K=k, H=4 * k, dtype=d16)
    if kind == "parts":
        k = rng.choice([1536, 2048, 3072])
        return dict(kind="parts", M=_log(rng, 256, 9216), K0=k, K1=4 * k, N=k, act=fmt, dtype=d16)
    if kind == "operator":
        wf = rng.choice([fmt, fmt, "int4"])
        return dict(kind="operator", S=rng.choice([1, 2, 3]), M=_log(rng, 16, 3000), K=_log(rng, 256, 4096, 64), N=_log(rng, 256, 3072, 8),
                    dual=rng.random() < 0.5, act="int8" if wf == "int4" else fmt, weight=wf, dtype=dtype)
    if kind == "svd":
        return dict(kind="svd", M=_log(rng, 256, 4608), K=_log(rng, 1024, 3072, 128), N=_log(rng, 1024, 12288, 128), rank=rng.choice([32, 64]), dtype=d16)
    wf = rng.choice(["int8", "fpe4m3", "int4", "int4"])
    return dict(kind="weights", N=_log(rng, 500, 6144, 2), K=_log(rng, 512, 6144, 128), fmt=wf,
                group=128 if wf == "int4" and rng.random() < 0.5 else 0, dtype=dtype)


# ---- inputs and layers ------------------------------------------------------------------------------------------------

def _activations(gen, rows, cols, gelu=False):
    """N(0, 1) with one channel in a hundred twenty times as large, as ``workloads.make_input``; on request behind a GELU."""
    x = torch.randn(rows, cols, generator=gen, device=_DEV)
    x[:, torch.randperm(cols, generator=gen, device=_DEV)[:math.ceil(0.01 * cols)]] *= 20.0
    return torch.nn.functional.gelu(x, approximate="tanh") if gelu else x


def _layer(gen, k, n, x, act, weight, *, seg_mode="weight", chunksizes=None, dynamic=False, dual=False, per_channel=False, group=0,
           opt_type="default", dtype=torch.bfloat16):
    """A layer calibrated on x, its weights ~ N(0, 0.02^2) and biases ~ N(0, 0.01^2) as ``workloads`` draws them."""
    args = {"real_quant": True, "dual_scale": dual, "axis": -1 if dynamic else None, "dynamic": dynamic}
    wargs = {"real_quant": True, "axis": 1 if per_channel or group else None, **({"group_size": group} if group else {})}
    layer = SegmentLinear(k, n, bias=True, seg_mode=seg_mode, chunks=len(chunksizes) if chunksizes else 1, chunksizes=chunksizes,
                          custom_weight_tensor=torch.randn(n, k, generator=gen, device=_DEV) * 0.02,
                          custom_bias_tensor=(torch.randn(n, generator=gen, device=_DEV) * 0.01).to(dtype),
                          input_quant_type=act, weight_quant_type=weight, input_quant_args=args, weight_quant_args=wargs,
                          opt_type=opt_type, opt_kwargs={"low_rank": 32} if opt_type == "svd" else None, device=_DEV)
    if opt_type == "default":
        layer.calibrate(x)
        layer.finish_calibrate()
    return layer


def prepare(case, seed):
    gen = torch.Generator(device=_DEV).manual_seed(int(seed))
    c, kind, dt = case, case["kind"], _DT[case["dtype"]]
    if kind == "linear":
        x = _activations(gen, c["M"], c["K"])
        chunks = [c["N"] // c["segments"]] * c["segments"] if c["segments"] > 1 else None
        layer = _layer(gen, c["K"], c["N"], x, c["act"], c["weight"], chunksizes=chunks, dynamic=c["dynamic"],
                       per_channel=c["per_channel"], group=c["group"], dtype=dt)
        return dict(kind=kind, x=x.to(dt), layer=layer)
    if kind == "block":
        m, d = c["M"], c["dim"]
        kw = dict(dynamic=True, dtype=dt)
        xs = [_activations(gen, m, d), _activations(gen, m, d), _activations(gen, m, 4 * d)]
        layers = [_layer(gen, d, 3 * d, xs[0], c["act"], c["act"], chunksizes=[d] * 3, **kw),
                  _layer(gen, d, 4 * d, xs[1], c["act"], c["act"], per_channel=True, **kw),
                  _layer(gen, 4 * d, d, xs[2], c["act"], c["act"], per_channel=True, **kw)]
        return dict(kind=kind, xs=[x.to(dt) for x in xs], layers=layers)
    if kind == "mlp":
        x = _activations(gen, c["M"], c["K"])
        fc1 = _layer(gen, c["K"], c["H"], x, c["act"], c["act"], dtype=dt)
        hidden = torch.nn.functional.gelu(fc1(x.to(dt)), approximate="tanh").float()
        fc2 = _layer(gen, c["H"], c["K"], hidden, c["act"], c["act"], dual=True, dtype=dt)
        return dict(kind=kind, x=x.to(dt), fc1=fc1, fc2=fc2)
    if kind == "geglu":
        x = _activations(gen, c["M"], c["K"])
        proj = _layer(gen, c["K"], 2 * c["H"], x, "int8", "int4", chunksizes=[c["H"]] * 2, dynamic=True, group=128, dtype=dt)
        ff = _layer(gen, c["H"], c["K"], _activations(gen, 64, c["H"]), "int8", "int4", dynamic=True, group=128, dtype=dt)
        return dict(kind=kind, x=x.to(dt), proj=proj, ff=ff)
    if kind == "parts":
        parts = [_activations(gen, c["M"], c["K0"]), _activations(gen, c["M"], c["K1"])]
        seen = torch.cat([parts[0], torch.nn.functional.gelu(parts[1], approximate="tanh")], dim=-1)
        layer = _layer(gen, c["K0"] + c["K1"], c["N"], seen, c["act"], c["act"], seg_mode="input", chunksizes=[c["K0"], c["K1"]],
                       dual=[False, True], dtype=dt)
        return dict(kind=kind, parts=[p.to(dt) for p in parts], layer=layer)
    if kind == "operator":
        s, m, k, n = c["S"], c["M"], c["K"], c["N"]
        x = _activations(gen, s * m, k, gelu=c["dual"])
        limit = {"int8": 127.0, "fpe4m3": 448.0, "int4": 7.0}
        w = torch.randn(s, n, k, generator=gen, device=_DEV) * 0.02
        ext = {"int8": load_real_quant_int8_ext, "fpe4m3": load_real_quant_fp8_ext, "int4": load_real_quant_int4_ext}[c["weight"]](required=True)[0]
        sw, codes = [], []
        for i in range(s):
            sw.append(limit[c["weight"]] / w[i].abs().max().item())
            code = ext.create_quantized_weights(w[i])
            ext.real_quantized_quantize_weights(w[i], code, sw[-1])
            codes.append(code)
        xs = x.view(s, -1)
        scales = [limit[c["act"]] / xs.amax(dim=1), (128.0 if c["act"] == "int8" else 448.0) / (-xs).amax(dim=1)] if c["dual"] else \
            [limit[c["act"]] / xs.abs().amax(dim=1)]
        fns = ext_dict[f"W{c['weight']}A{c['act']}"]
        return dict(kind=kind, fn=fns["gemm_dual_scaled_fn" if c["dual"] else "gemm_scaled_fn"],
                    args=[x.view(s, m, k).to(dt), torch.stack(codes), *[t.float().contiguous() for t in scales],
                          torch.tensor(sw, dtype=torch.float32, device=_DEV)])
    if kind == "svd":
        x = _activations(gen, c["M"], c["K"])
        layer = _layer(gen, c["K"], c["N"], x, "int8", "int8", dynamic=True, per_channel=True, opt_type="svd", dtype=dt)
        opt = layer.optimizer
        layer.trace(x)
        # a decomposed checkpoint: the residual's weights and the two factors, no SVD here
        SmoothOptimizer.smooth(opt)
        opt.low_rank = c["rank"]
        opt.l1s = torch.randn(1, c["K"], c["rank"], generator=gen, device=_DEV) * 0.05
        opt.l2s = torch.randn(1, c["rank"], c["N"], generator=gen, device=_DEV) * 0.05
        opt.has_svd = True
        layer.calibrate(x)
        layer.finish_calibrate()
        return dict(kind="linear", x=x.to(dt), layer=layer)
    w = (torch.randn(c["N"], c["K"], generator=gen, device=_DEV) * 0.02).to(dt)
    state = dict(kind=kind, w=w, fmt=c["fmt"], group=c["group"])
    if c["group"]:
        state["scale"] = (7.0 / w.float().view(c["N"], -1, c["group"]).abs().amax(dim=-1)).t().contiguous()
        state["ext"] = load_real_quant_int4_ext(required=True)[0]
    else:
        limit = {"int8": 127.0, "fpe4m3": 448.0, "int4": 7.0}[c["fmt"]]
        state["scale"] = (limit / w.float().abs().amax(dim=1)).contiguous()
        state["ext"] = {"int8": load_real_quant_int8_ext, "fpe4m3": load_real_quant_fp8_ext,
                        "int4": load_real_quant_int4_ext}[c["fmt"]](required=True)[0]
        if c["fmt"] == "fpe4m3":
            state["fake"], state["scaled"] = load_fake_quant_fp8_ext(required=True), (w.float() * state["scale"][:, None]).to(dt)
    return state


def run(state):
    kind = state["kind"]
    if kind == "linear":
        return state["layer"](state["x"])
    if kind == "block":
        return [layer(x) for layer, x in zip(state["layers"], state["xs"])]
    if kind == "mlp":
        return state["fc1"].forward_into(state["fc2"], state["x"], pre_op="gelu_tanh")
    if kind == "geglu":
        value, gate = state["proj"](state["x"]).chunk(2, dim=-1)
        return state["ff"](value, pre_op="gelu", gate=gate)
    if kind == "parts":
        return state["layer"].forward_parts(state["parts"], pre_ops=[None, "gelu_tanh"])
    if kind == "operator":
        return state["fn"](*state["args"])
    w, ext = state["w"], state["ext"]
    if state["group"]:
        return ext.quantize_weights_groups(w, state["scale"], state["group"])
    codes = ext.create_quantized_weights(w)
    ext.real_quantized_quantize_weights(w, codes, state["scale"])
    if state["fmt"] == "fpe4m3":
        return codes, state["fake"].fake_e4m3fy(state["scaled"])
    return codes


# ---- what a pass cannot do without --------------------------------------------------------------------------------------

def _linear_work(m, k, n, weight, esz, x_bytes=None):
    """Input read, weight codes read, output written, each once; one multiply-add per product (DualScale counted once)."""
    return (m * k * esz if x_bytes is None else x_bytes) + n * k * _CODE_BYTES[weight] + n * esz + m * n * esz, 2.0 * m * n * k


def work(case):
    c, e = case, _SIZE[case["dtype"]]
    kind = c["kind"]
    if kind == "linear":
        jobs = [_linear_work(c["M"], c["K"], c["N"], c["weight"], e)]
        if c["group"]:
            jobs.append((4.0 * c["N"] * c["K"] / c["group"], 0.0))
    elif kind == "block":
        m, d = c["M"], c["dim"]
        jobs = [_linear_work(m, d, 3 * d, c["act"], e), _linear_work(m, d, 4 * d, c["act"], e), _linear_work(m, 4 * d, d, c["act"], e)]
    elif kind == "mlp":  # the hidden tensor is not an output
        jobs = [(c["M"] * c["K"] * e + 2 * c["K"] * c["H"] + (c["K"] + c["H"]) * e + c["M"] * c["K"] * e, 4.0 * c["M"] * c["K"] * c["H"])]
    elif kind == "geglu":
        k, h = c["K"], c["H"]
        jobs = [(2 * c["M"] * k * e + 3 * k * h * (0.5 + 4.0 / 128) + (2 * h + k) * e, 6.0 * c["M"] * k * h)]
    elif kind == "parts":
        jobs = [_linear_work(c["M"], c["K0"] + c["K1"], c["N"], c["act"], e)]
    elif kind == "operator":
        jobs = [_linear_work(c["M"], c["K"], c["N"], c["weight"], e)] * c["S"]
    elif kind == "svd":
        b, f = _linear_work(c["M"], c["K"], c["N"], "int8", e)
        jobs = [(b + (c["K"] + c["N"]) * c["rank"] * e, f + 2.0 * c["rank"] * c["M"] * (c["K"] + c["N"]))]
    else:
        n = c["N"] * c["K"]
        jobs = [(n * (e + _CODE_BYTES[c["fmt"]]) + 4.0 * (n / c["group"] if c["group"] else c["N"]), 0.0)]
        if c["fmt"] == "fpe4m3":
            jobs.append((2.0 * n * e, 0.0))
    return {"bytes": float(sum(b for b, _ in jobs)), "flops": float(sum(f for _, f in jobs))}


def tolerance(case):
    """About four times the distance from the same codes multiplied and scaled in 64 bits: the output's one rounding (1.7e-3 in
    bf16, 2.1e-4 in fp16) or, with fp32 outputs, the fp32 scaling (8e-8) and the matrix cores' e4m3 sums (4.5e-5).  Behind an
    activation function single codes fall to the other side of a step as well (e4m3: an eighth of the value; 2.3e-3 in all)."""
    kind, dtype = case["kind"], case["dtype"]
    if kind == "weights":
        return "exact"
    if dtype == "fp32":
        return {"rel": 3e-7, "max": 1.5e-6} if case["act"] == "int8" else {"rel": 1.8e-4, "max": 3e-3}
    if kind == "mlp" and case["act"] == "fpe4m3":
        return {"rel": 9e-3, "max": 0.08}
    most = 1.2e-2 if kind in ("mlp", "geglu", "parts") else 3.5e-3
    return {"rel": 7e-3, "max": 1.7e-2} if dtype == "bf16" else {"rel": 9e-4, "max": most}
