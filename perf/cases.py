"""Performance cases of the MI355X execution path: what its users run, over the sizes they run it at.

A case is one kind of work and its sizes:

    mlp, resnet_cifar, resnet_224, decoder   a model compiled once (`compile_workload`: pass pipeline, plan,
                                             one hipGraph) and fed one batch per pass, as a serving loop does
    linear, linear_fp8, linear_fp4           one Linear layer through the C ABI on preallocated buffers
    attention, conv                          one attention / convolution layer, likewise

`prepare` makes inputs and weights from the seed and compiles the plan, `run` is one pass, `exact` the same
result in float64 by plain torch.
"""

import json
import math

import numpy as np
import torch
import torch.nn.functional as F

from hackathon_amd import _lib, models
from hackathon_amd.device import DeviceArray, init
from hackathon_amd.workloads import compile_workload

MODELS = ("mlp", "resnet_cifar", "resnet_224", "decoder")
CODE = {"fp32": _lib.F32, "fp16": _lib.F16, "bf16": _lib.BF16}
TYPE = {"fp32": torch.float32, "fp16": torch.float16, "bf16": torch.bfloat16}
HEAD = 64  # the attention layer's head size (every decoder of this framework)


# ---------------------------------------------------------------- the cases
def listed():
    return [
        # The fp32 classifier on its benchmark batch: three small GEMMs, bound by launches and latency.
        {"name": "mlp_256", "kind": "mlp", "batch": 256},
        # CIFAR ResNet-18 in fp32 (the default policy), benchmark batch: implicit-GEMM convolutions on fp32 MFMA.
        {"name": "resnet_cifar_fp32_256", "kind": "resnet_cifar", "batch": 256},
        # ImageNet-size ResNet-18 in bf16, benchmark batch: the throughput workload.
        {"name": "resnet_224_bf16_256", "kind": "resnet_224", "batch": 256, "policy": "bf16"},
        # Decoder layers at the fp16 benchmark's sizes (prefill of 64 sequences) with the logits and their argmax.
        {"name": "decoder_fp16_64x256", "kind": "decoder", "policy": "fp16", "batch": 64, "seq": 256, "d": 512,
         "heads": 8, "ffn": 2048, "layers": 2, "vocab": 8192},
        # The whole fp16 decoder on one ragged sequence: what a single request waits for.
        {"name": "decoder_fp16_1x200", "kind": "decoder", "policy": "fp16", "batch": 1, "seq": 200, "d": 512,
         "heads": 8, "ffn": 2048, "layers": 6, "vocab": 8192},
        # The same layers under the deploy CLI's default policy, fp32.
        {"name": "decoder_fp32_8x256", "kind": "decoder", "policy": "fp32", "batch": 8, "seq": 256, "d": 512,
         "heads": 8, "ffn": 2048, "layers": 2, "vocab": 8192},
        # W8A8 decoder layers at the int8 benchmark's batch and width: quantized Linears, 1024-token attention.
        {"name": "decoder_w8a8_16x1024", "kind": "decoder", "policy": "w8a8", "batch": 16, "seq": 1024, "d": 768,
         "heads": 12, "ffn": 3072, "layers": 2, "vocab": 8192},
        # One Linear of a small request (FFN2 with its residual): few rows, a deep K.
        {"name": "linear_fp16_333", "kind": "linear", "type": "fp16", "out": "fp16", "m": 333, "k": 2048, "n": 512,
         "act": "none", "residual": True},
        # One E4M3 Linear at the decoder's prefill size: row quantization of the activation and the fp8 GEMM.
        {"name": "linear_fp8_16384", "kind": "linear_fp8", "m": 16384, "k": 512, "n": 2048, "act": "gelu"},
        # One MXFP4-weight Linear on an ordinary ragged token count.
        {"name": "linear_fp4_3000", "kind": "linear_fp4", "m": 3000, "k": 2048, "n": 512, "act": "none"},
        # Causal attention of one W8A8 decoder layer.
        {"name": "attention_bf16_16x1024", "kind": "attention", "type": "bf16", "batch": 16, "heads": 12,
         "seq": 1024, "causal": True},
        # One residual 3x3 convolution of ResNet-18's second stage on an odd batch.
        {"name": "conv_bf16_37x28", "kind": "conv", "type": "bf16", "batch": 37, "hw": 28, "cin": 128, "cout": 128,
         "ksize": 3, "stride": 1, "residual": True},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case: a kind, then its sizes over the range served (log-uniform where it is wide)."""
    kind = rng.choice(["mlp", "resnet_cifar", "resnet_224", "decoder", "decoder_w8a8", "decoder_fp32", "linear",
                       "linear", "linear_fp8", "linear_fp4", "attention", "conv"])
    if kind == "mlp":
        return {"kind": kind, "batch": _log_int(rng, 1, 8192)}
    if kind == "resnet_cifar":
        return {"kind": kind, "batch": _log_int(rng, 1, 255)}
    if kind == "resnet_224":
        return {"kind": kind, "batch": _log_int(rng, 1, 255), "policy": rng.choice(["bf16", "fp16"])}
    if kind == "decoder":
        seq = _log_int(rng, 16, 1024)
        return {"kind": kind, "policy": rng.choice(["fp16", "fp16", "bf16", "fp8", "fp4"]), "batch": _log_int(rng, 1, max(2, 16384 // seq)),
                "seq": seq, "d": 512, "heads": 8, "ffn": 2048, "layers": rng.choice([1, 2, 4]), "vocab": 8192}
    if kind == "decoder_w8a8":
        seq = _log_int(rng, 64, 1024)
        return {"kind": "decoder", "policy": "w8a8", "batch": _log_int(rng, 1, 16384 // seq), "seq": seq, "d": 768,
                "heads": 12, "ffn": 3072, "layers": 1, "vocab": rng.choice([1000, 8192])}
    if kind == "decoder_fp32":
        seq = _log_int(rng, 16, 512)
        d = rng.choice([128, 512])
        return {"kind": "decoder", "policy": "fp32", "batch": _log_int(rng, 1, max(2, 2048 // seq)), "seq": seq,
                "d": d, "heads": d // HEAD, "ffn": 4 * d, "layers": rng.choice([1, 2]), "vocab": rng.choice([14, 1000, 8192])}
    if kind in ("linear", "linear_fp8", "linear_fp4"):
        d = rng.choice([512, 768])
        k, n = rng.choice([(d, 3 * d), (d, d), (d, 4 * d), (4 * d, d), (512, 1000)])
        c = {"kind": kind, "m": _log_int(rng, 1, 16384), "k": k, "n": n, "act": rng.choice(["none", "relu", "gelu"])}
        if kind == "linear":
            c["type"] = rng.choice(["fp16", "bf16", "fp32"])
            c["out"] = "fp32" if c["type"] == "fp32" or rng.random() < 0.2 else c["type"]
            c["residual"] = rng.random() < 0.5
            if c["type"] == "fp32":
                c["m"] = _log_int(rng, 1, 4096)
        return c
    if kind == "attention":
        seq = _log_int(rng, 16, 2048)
        return {"kind": kind, "type": rng.choice(["fp16", "bf16"]), "batch": _log_int(rng, 1, max(2, 8192 // seq)),
                "heads": rng.choice([8, 12]), "seq": seq, "causal": rng.random() < 0.8}
    cin, cout, hw, k, stride = rng.choice([(64, 64, 56, 3, 1), (64, 128, 56, 3, 2), (64, 128, 56, 1, 2),
                                           (128, 128, 28, 3, 1), (128, 256, 28, 3, 2), (256, 256, 14, 3, 1),
                                           (256, 512, 14, 3, 2), (256, 512, 14, 1, 2), (512, 512, 7, 3, 1)])
    dt = rng.choice(["bf16", "fp16", "fp32"])
    return {"kind": "conv", "type": dt, "batch": _log_int(rng, 1, 64 if dt == "fp32" else 256), "hw": hw, "cin": cin,
            "cout": cout, "ksize": k, "stride": stride, "residual": stride == 1 and rng.random() < 0.5}


# ---------------------------------------------------------------- models
def _scales(model):
    """Activation scales of a W8A8 model from the committed calibration (same width, other layer counts)."""
    known = json.loads(models.calibration_path("decoder_w8a8").read_text())["scales"]
    return {n: known[n] for n in model}


def _model(case, seed):
    """The case's graph and host weights, built for one sample: the batch is a property of the plan."""
    kind = case["kind"]
    if kind == "mlp":
        m = models.build("mlp", batch=1, seed=seed)
    elif kind == "resnet_cifar":
        m = models.build("resnet18_cifar", batch=1, seed=seed)
    elif kind == "resnet_224":
        m = models.build("resnet18_224", batch=1, precision=case["policy"], seed=seed)
    else:
        quantized = case["policy"] == "w8a8"
        kw = dict(batch=1, seq=case["seq"], d_model=case["d"], heads=case["heads"], ffn=case["ffn"],
                  layers=case["layers"], vocab=case["vocab"], seed=seed)
        if quantized:
            names = ["layer%d.%s" % (i, p) for i in range(case["layers"]) for p in ("qkv", "out", "ffn1", "ffn2")]
            kw["act_scales"] = _scales(["%s.%s_scale" % (p, s) for p in names + ["lm_head"] for s in ("act", "out")])
        m = models.build_decoder(precision="fp16" if quantized else case["policy"], quantized=quantized,
                                 name="decoder", **kw)
    return m


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _model_input(case, seed):
    g, b = _gen(seed), case["batch"]
    if case["kind"] == "mlp":
        return torch.rand(b, 784, device="cuda", generator=g)
    if case["kind"] == "resnet_cifar":
        return torch.randn(b, 3, 32, 32, device="cuda", generator=g)
    if case["kind"] == "resnet_224":
        return torch.randn(b, 3, 224, 224, device="cuda", generator=g)
    return torch.randint(0, case["vocab"], (b, case["seq"]), device="cuda", generator=g)


class _Memory:
    """A device array of the framework as torch can see it (no copy)."""

    def __init__(self, arr, owner):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": arr.shape, "typestr": arr.dtype.str, "data": (arr.ptr, False),
                                         "strides": None, "version": 2}


def _prepare_model(case, seed):
    init(0)
    m = _model(case, seed)
    name = next(iter(m.inputs))
    x = _model_input(case, seed)
    m.inputs = {name: np.broadcast_to(m.inputs[name][:1], tuple(x.shape))}  # the plan takes the batch from here
    _, _, prog = compile_workload(m.name, model=m)
    feed = {name: DeviceArray(x.data_ptr(), tuple(x.shape), m.inputs[name].dtype, owner=x)}
    out = {k: torch.as_tensor(_Memory(v, prog), device="cuda") for k, v in prog.output_arrays.items()}
    return {"prog": prog, "feed": feed, "out": out}


# ---------------------------------------------------------------- single layers
GELU = (math.sqrt(2.0), 1.0, 0.5)  # the constants of the exported Div / Erf / Add / Mul / Mul chain


def _epilogue(e, bias, residual, act):
    e.alpha = e.beta = 1.0
    e.bias, e.bias_mode = bias.data_ptr(), 2
    e.residual = residual.data_ptr() if residual is not None else None
    e.act = {"none": 0, "relu": 1, "gelu": 2}[act]
    if act == "gelu":
        e.n_imm = 3
        e.imm[0], e.imm[1], e.imm[2] = GELU


def _linear_data(case, seed):
    """(x, weight [n][k], bias, residual): LayerNorm-like activations, the initialisation's weight spread."""
    g = _gen(seed)
    dt, out = TYPE[case.get("type", "fp16")], TYPE[case.get("out", "fp16")]
    x = torch.randn(case["m"], case["k"], device="cuda", generator=g).to(dt)
    w = torch.randn(case["n"], case["k"], device="cuda", generator=g) / math.sqrt(case["k"])
    bias = torch.randn(case["n"], device="cuda", generator=g) * 0.1
    res = torch.randn(case["m"], case["n"], device="cuda", generator=g).to(out) if case.get("residual") else None
    return x, w, bias, res


def _prepare_linear(case, seed):
    x, w, bias, res = _linear_data(case, seed)
    w = w.to(x.dtype)
    out = torch.empty(case["m"], case["n"], device="cuda", dtype=TYPE[case["out"]])
    a = _lib.GemmArgs()
    a.a, a.b, a.out = x.data_ptr(), w.data_ptr(), out.data_ptr()
    a.m, a.n, a.k, a.lda, a.ldb, a.ldo, a.batch = case["m"], case["n"], case["k"], case["k"], case["k"], case["n"], 1
    a.trans_b, a.in_dtype, a.out_dtype = 1, CODE[case["type"]], CODE[case["out"]]
    _epilogue(a.epi, bias, res, case["act"])
    return {"calls": [a], "out": out, "keep": (x, w, bias, res)}


def _prepare_linear_fp8(case, seed):
    x, w, bias, _ = _linear_data(case, seed)
    m, n, k = case["m"], case["n"], case["k"]

    def quantizer(src, codes, scale, code):
        q = _lib.Fp8QuantArgs()
        q.x, q.out, q.scale = src.data_ptr(), codes.data_ptr(), scale.data_ptr()
        q.rows, q.cols, q.ldx, q.ldo, q.x_dtype = src.shape[0], k, k, k, code
        return q

    qx, sx = torch.empty(m, k, device="cuda", dtype=torch.uint8), torch.empty(m, device="cuda")
    qw, sw = torch.empty(n, k, device="cuda", dtype=torch.uint8), torch.empty(n, device="cuda")
    _lib.launch(quantizer(w, qw, sw, _lib.F32))  # the weight is quantized once
    out = torch.empty(m, n, device="cuda", dtype=torch.float16)
    a = _lib.Fp8GemmArgs()
    a.a, a.b, a.a_scale, a.b_scale, a.out = (t.data_ptr() for t in (qx, qw, sx, sw, out))
    a.m, a.n, a.k, a.lda, a.ldb, a.ldo, a.out_dtype = m, n, k, k, k, n, _lib.F16
    _epilogue(a.epi, bias, None, case["act"])
    return {"calls": [quantizer(x, qx, sx, _lib.F16), a], "out": out, "keep": (x, w, bias, qx, sx, qw, sw)}


def _prepare_linear_fp4(case, seed):
    x, w, bias, _ = _linear_data(case, seed)
    m, n, k = case["m"], case["n"], case["k"]
    codes = torch.empty(n, k // 2, device="cuda", dtype=torch.uint8)
    scales = torch.empty(n, k // 32, device="cuda", dtype=torch.uint8)
    q = _lib.Mxfp4QuantArgs()
    q.x, q.codes, q.scales = w.data_ptr(), codes.data_ptr(), scales.data_ptr()
    q.rows, q.cols, q.ldx, q.ldc, q.lds, q.x_dtype = n, k, k, k // 2, k // 32, _lib.F32
    _lib.launch(q)
    out = torch.empty(m, n, device="cuda", dtype=torch.float16)
    a = _lib.W4A16GemmArgs()
    a.a, a.b_codes, a.b_scales, a.out = (t.data_ptr() for t in (x, codes, scales, out))
    a.m, a.n, a.k, a.lda, a.ldb, a.ldbs, a.ldo, a.out_dtype = m, n, k, k, k // 2, k // 32, n, _lib.F16
    _epilogue(a.epi, bias, None, case["act"])
    return {"calls": [a], "out": out, "keep": (x, w, bias, codes, scales)}


def _qkv(case, seed):
    """Packed [B, S, 3 H 64] projection, as the decoder's QKV Linear leaves it."""
    g = _gen(seed)
    return torch.randn(case["batch"], case["seq"], 3 * case["heads"] * HEAD, device="cuda", generator=g).to(TYPE[case["type"]])


def _prepare_attention(case, seed):
    qkv = _qkv(case, seed)
    b, s, h = case["batch"], case["seq"], case["heads"]
    w = h * HEAD
    out = torch.empty(b, s, h, HEAD, device="cuda", dtype=qkv.dtype)
    a = _lib.FlashArgs()
    p = qkv.data_ptr()
    a.q, a.k, a.v, a.out = p, p + 2 * w, p + 4 * w, out.data_ptr()
    a.batch, a.heads, a.seq_q, a.seq_k, a.head_dim, a.dtype = b, h, s, s, HEAD, CODE[case["type"]]
    for t in "qkv":
        setattr(a, t + "_sb", s * 3 * w), setattr(a, t + "_sh", HEAD), setattr(a, t + "_ss", 3 * w)
    a.o_sb, a.o_sh, a.o_ss = s * w, HEAD, w
    a.scale, a.mask_kind = 1.0 / math.sqrt(HEAD), 1 if case["causal"] else 0
    return {"calls": [a], "out": out, "keep": (qkv,)}


def _conv_geometry(case):
    pad = case["ksize"] // 2
    return pad, (case["hw"] + 2 * pad - case["ksize"]) // case["stride"] + 1


def _conv_data(case, seed):
    """(x NHWC, weight [o][kh][kw][c], bias, residual NHWC): post-ReLU activations, He-initialised weights."""
    g, dt = _gen(seed), TYPE[case["type"]]
    _, ho = _conv_geometry(case)
    k, cin, cout = case["ksize"], case["cin"], case["cout"]
    x = torch.randn(case["batch"], case["hw"], case["hw"], cin, device="cuda", generator=g).relu_().to(dt)
    w = (torch.randn(cout, k, k, cin, device="cuda", generator=g) * math.sqrt(2.0 / (cin * k * k))).to(dt)
    bias = torch.randn(cout, device="cuda", generator=g) * 0.1
    res = torch.randn(case["batch"], ho, ho, cout, device="cuda", generator=g).to(dt) if case["residual"] else None
    return x, w, bias, res


def _prepare_conv(case, seed):
    x, w, bias, res = _conv_data(case, seed)
    pad, ho = _conv_geometry(case)
    out = torch.empty(case["batch"], ho, ho, case["cout"], device="cuda", dtype=x.dtype)
    a = _lib.ConvArgs()
    a.x, a.w, a.out = x.data_ptr(), w.data_ptr(), out.data_ptr()
    a.n, a.c, a.h, a.w_, a.c_stride, a.c_pack, a.o = (case["batch"], case["cin"], case["hw"], case["hw"], case["cin"],
                                                      case["cin"], case["cout"])
    a.kh = a.kw = case["ksize"]
    a.sh = a.sw = case["stride"]
    a.pad_top = a.pad_left = pad
    a.dh = a.dw = 1
    a.ho = a.wo = ho
    a.out_layout, a.in_dtype, a.out_dtype = 1, CODE[case["type"]], CODE[case["type"]]
    _epilogue(a.epi, bias, res, "relu")
    return {"calls": [a], "out": out, "keep": (x, w, bias, res)}


_LAYERS = {"linear": _prepare_linear, "linear_fp8": _prepare_linear_fp8, "linear_fp4": _prepare_linear_fp4,
           "attention": _prepare_attention, "conv": _prepare_conv}


def prepare(case, seed):
    if case["kind"] in MODELS:
        return _prepare_model(case, seed)
    init(0)
    return _LAYERS[case["kind"]](case, seed)


def run(state):
    if "prog" in state:
        state["prog"].run(state["feed"])
        return state["out"]
    for args in state["calls"]:
        _lib.launch(args)
    return state["out"]


# ---------------------------------------------------------------- what a pass cannot do without
def _resnet_work(case):
    """(flops per image, weights) of ResNet-18's convolutions and classifier."""
    imagenet = case["kind"] == "resnet_224"
    hw, classes = (56, 1000) if imagenet else (32, 10)
    flops, weights = (2 * 112 * 112 * 64 * 147, 64 * 147) if imagenet else (2 * 32 * 32 * 64 * 27, 64 * 27)
    cin = 64
    for stage, c in enumerate((64, 128, 256, 512)):
        hw = hw // 2 if stage else hw
        taps = [9 * cin, 9 * c, 9 * c, 9 * c] + ([cin] if cin != c else [])
        flops += sum(2 * hw * hw * c * t for t in taps)
        weights += sum(c * t for t in taps)
        cin = c
    return flops + 2 * 512 * classes, weights + 512 * classes


def work(case):
    kind = case["kind"]
    if kind == "mlp":
        params = 784 * 512 + 512 * 256 + 256 * 10
        return {"bytes": 4 * (params + case["batch"] * 794), "flops": 2 * case["batch"] * params}
    if kind in ("resnet_cifar", "resnet_224"):
        flops, weights = _resnet_work(case)
        image, classes, size = (3 * 32 * 32, 10, 4) if kind == "resnet_cifar" else (3 * 224 * 224, 1000, 2)
        return {"bytes": size * weights + 4 * case["batch"] * (image + classes), "flops": flops * case["batch"]}
    if kind == "decoder":
        d, f, v, t = case["d"], case["ffn"], case["vocab"], case["batch"] * case["seq"]
        size = {"fp32": 4.0, "fp16": 2.0, "bf16": 2.0, "w8a8": 1.0, "fp8": 1.0, "fp4": 17 / 32}[case["policy"]]
        params = case["layers"] * (4 * d * d + 2 * d * f) + d * v
        pairs = case["batch"] * case["heads"] * case["seq"] * (case["seq"] + 1) // 2
        return {"bytes": size * params + min(t, v) * d * 2 + t * (16 + 4 * v),
                "flops": 2 * t * params + case["layers"] * 4 * HEAD * pairs}
    if kind.startswith("linear"):
        m, n, k = case["m"], case["n"], case["k"]
        si, so = torch.empty(0, dtype=TYPE[case.get("type", "fp16")]).element_size(), \
            torch.empty(0, dtype=TYPE[case.get("out", "fp16")]).element_size()
        wb = {"linear": si, "linear_fp8": 1, "linear_fp4": 17 / 32}[kind]
        return {"bytes": m * k * si + n * k * wb + 4 * n + m * n * so * (2 if case.get("residual") else 1),
                "flops": 2 * m * n * k}
    if kind == "attention":
        b, h, s = case["batch"], case["heads"], case["seq"]
        pairs = b * h * (s * (s + 1) // 2 if case["causal"] else s * s)
        return {"bytes": 4 * b * h * s * HEAD * 2, "flops": 4 * HEAD * pairs}
    _, ho = _conv_geometry(case)
    size = 4 if case["type"] == "fp32" else 2
    outs, taps = case["batch"] * ho * ho * case["cout"], case["cin"] * case["ksize"] ** 2
    return {"bytes": size * (case["batch"] * case["hw"] ** 2 * case["cin"] + case["cout"] * taps
                             + outs * (2 if case["residual"] else 1)), "flops": 2 * outs * taps}


def tolerance(case):
    """About four times the difference from float64 that each type shows.

    A W8A8 decoder rounds to int8 before and after every Linear: a value beside a code boundary takes the other
    code after any change of bf16 rounding before it, and the layers after see a whole step of difference (the
    out projection's step is a third of its output's spread: 0.11 from the float64 run of the same graph)."""
    kind = case["kind"]
    if kind in ("mlp", "resnet_cifar") or case.get("type") == "fp32":
        return {"rel": 5e-6}
    if kind == "resnet_224":
        return {"rel": 1.5e-2 if case["policy"] == "bf16" else 2e-3}
    if kind == "decoder":
        rel = {"fp32": 5e-6, "fp16": 4e-3, "bf16": 3e-2, "w8a8": 1.5e-1, "fp8": 3e-2, "fp4": 4e-3}[case["policy"]]
        return {"rel": rel, "differ": {"fp32": 0.001, "w8a8": 0.3}.get(case["policy"], 0.05)}
    if kind == "attention":
        return {"rel": 8e-3 if case["type"] == "bf16" else 1e-3}
    if kind == "linear_fp8":
        return {"rel": 4e-3}
    out = case.get("out", case.get("type", "fp16"))
    return {"rel": {"fp32": 5e-6, "fp16": 1e-3, "bf16": 7e-3}[out]}


# ---------------------------------------------------------------- float64 results
def _d(x):
    return torch.as_tensor(np.ascontiguousarray(x)).cuda().double()


def _exact_mlp(case, seed):
    w, h = _model(case, seed).weights, _model_input(case, seed).double()
    for i in (1, 2, 3):
        h = h @ _d(w["fc%d.weight" % i]).t() + _d(w["fc%d.bias" % i])
        h = h.relu() if i < 3 else h
    return {"logits": h}


def _conv64(x, w, stride, pad):
    """NCHW convolution in float64 as unfold + matmul, a few images at a time."""
    o, k = w.shape[0], w.shape[2]
    ho = (x.shape[2] + 2 * pad - k) // stride + 1
    step = max(1, int(2 ** 27 // (w[0].numel() * ho * ho)))
    parts = [torch.matmul(w.reshape(o, -1), F.unfold(x[i:i + step], k, padding=pad, stride=stride))
             for i in range(0, x.shape[0], step)]
    return torch.cat(parts).reshape(x.shape[0], o, ho, ho)


def _exact_resnet(case, seed):
    p = _model(case, seed).weights
    x = _model_input(case, seed).double()

    def conv_bn(h, name, stride, pad):
        y = _conv64(h, _d(p[name + ".conv.weight"]), stride, pad)
        g, b, mean, var = (_d(p["%s.bn.%s" % (name, s)]) for s in ("weight", "bias", "running_mean", "running_var"))
        f = g / torch.sqrt(var + 1e-5)
        return y * f[:, None, None] + (b - mean * f)[:, None, None]

    imagenet = case["kind"] == "resnet_224"
    h = conv_bn(x, "stem", 2 if imagenet else 1, 3 if imagenet else 1).relu_()
    if imagenet:
        h = F.max_pool2d(h, 3, 2, 1)
    for stage in range(4):
        for blk in range(2):
            name, stride = "layer%d.%d" % (stage + 1, blk), 2 if stage and not blk else 1
            y = conv_bn(conv_bn(h, name + ".a", stride, 1).relu_(), name + ".b", 1, 1)
            h = (y + (conv_bn(h, name + ".down", stride, 0) if stride == 2 else h)).relu_()
    return {"logits": h.mean((2, 3)) @ _d(p["fc.weight"]).t() + _d(p["fc.bias"])}


def _exact_decoder(case, seed):
    p, ids = _model(case, seed).weights, _model_input(case, seed)
    heads = case["heads"]

    def linear(h, name):
        return h @ _d(p[name + ".weight"]) + _d(p[name + ".bias"])

    def norm(h, name):
        return F.layer_norm(h, h.shape[-1:], _d(p[name + ".weight"]), _d(p[name + ".bias"]), 1e-5)

    x = _d(p["embed.tok"])[ids] + _d(p["embed.pos"])
    b, s, d = x.shape
    causal = torch.full((s, s), -math.inf, device="cuda", dtype=torch.float64).triu(1)
    for i in range(case["layers"]):
        name = "layer%d" % i
        q, k, v = (t.reshape(b, s, heads, HEAD).transpose(1, 2) for t in
                   linear(norm(x, name + ".ln1"), name + ".qkv").split(d, -1))
        ctx = torch.empty_like(x)
        for j in range(b):  # a sequence at a time: the scores of all of them need not fit
            pr = torch.softmax(q[j] @ k[j].transpose(1, 2).contiguous() / math.sqrt(HEAD) + causal, -1)
            ctx[j] = (pr @ v[j].contiguous()).transpose(0, 1).reshape(s, d)
        x = x + linear(ctx, name + ".out")
        x = x + linear(F.gelu(linear(norm(x, name + ".ln2"), name + ".ffn1")), name + ".ffn2")
    return {"logits": linear(norm(x, "final.ln"), "lm_head"), "argmax": None}


def _act64(v, act):
    return F.gelu(v) if act == "gelu" else v.relu() if act == "relu" else v


def _fp8_rows(x):
    """Row-wise E4M3 quantization: codes of x * (448 / max |x|) and the scale max |x| / 448, as values."""
    amax = x.float().abs().amax(1, keepdim=True)
    return (x.float() * (448.0 / amax)).to(torch.float8_e4m3fn).double() * (amax.double() / 448.0)


def _mxfp4(w):
    """MXFP4 blocks of 32 along k: E2M1 elements (ties to even) times a power of two, as values."""
    n, k = w.shape
    v = w.double().reshape(n, k // 32, 32)
    amax = v.abs().amax(2, keepdim=True)
    scale = torch.exp2((torch.floor(torch.log2(amax)) - 2).clamp(-13, 13))
    y = v.abs() / scale
    code = torch.zeros_like(y, dtype=torch.long)
    for i, mid in enumerate((0.25, 0.75, 1.25, 1.75, 2.5, 3.5, 5.0)):
        code += ((y > mid) | ((y == mid) & (i % 2 == 1))).long()
    grid = torch.tensor([0, 0.5, 1, 1.5, 2, 3, 4, 6], device="cuda", dtype=torch.float64)
    return (grid[code] * torch.sign(v) * scale).reshape(n, k)


def exact(case, seed):
    kind = case["kind"]
    if kind == "mlp":
        return _exact_mlp(case, seed)
    if kind in ("resnet_cifar", "resnet_224"):
        return _exact_resnet(case, seed)
    if kind == "decoder":
        # the int8, E4M3 and MXFP4 policies round codes along the way: float64 has no such value
        return _exact_decoder(case, seed) if case["policy"] in CODE else None
    if kind.startswith("linear"):
        x, w, bias, res = _linear_data(case, seed)
        a = _fp8_rows(x) if kind == "linear_fp8" else x.double()
        b = _fp8_rows(w) if kind == "linear_fp8" else _mxfp4(w) if kind == "linear_fp4" else w.to(x.dtype).double()
        v = a @ b.t() + bias.double()
        return _act64(v + res.double() if res is not None else v, case["act"])
    if kind == "attention":
        qkv = _qkv(case, seed)
        b, s, h = case["batch"], case["seq"], case["heads"]
        out = torch.empty(b, s, h, HEAD, device="cuda", dtype=torch.float64)
        for j in range(b):
            q, k, v = (t.reshape(s, h, HEAD).transpose(0, 1).contiguous().double() for t in qkv[j].split(h * HEAD, -1))
            sc = q @ k.transpose(1, 2).contiguous() / math.sqrt(HEAD)
            if case["causal"]:
                sc += torch.full((s, s), -math.inf, device="cuda", dtype=torch.float64).triu(1)
            out[j] = (torch.softmax(sc, -1) @ v).transpose(0, 1)
        return out
    x, w, bias, res = _conv_data(case, seed)
    pad, _ = _conv_geometry(case)
    y = _conv64(x.permute(0, 3, 1, 2).double(), w.permute(0, 3, 1, 2).contiguous().double(), case["stride"], pad)
    y = y.permute(0, 2, 3, 1) + bias.double()
    return (y + res.double() if res is not None else y).relu()
