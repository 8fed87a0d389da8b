"""The calls whose speed this framework is judged by, as data.

listed() names twelve of them, draw() gives further ones of the same ranges;
prepare() makes what a program holds before the call (operands, layer,
output buffer), run() is one pass through the public entry points, exact()
the same result in 64-bit torch arithmetic.

Kinds:
  gemm    hipgemm_amd.fp8_gemm_bf16: e4m3 x e4m3 -> bf16, per-tensor scales,
          into a buffer the caller owns.
  linear  torch_ops.Fp8Linear: bf16 activations quantised per token, e4m3
          weights with per-channel scales, bias and activation fused.
  grad    hipgemm_amd.gemm: e5m2 gradients x e4m3 operands -> fp32 (weight
          gradient) or bf16 (input gradient).
  chain   hipgemm_amd.gemm: e4m3 -> e4m3 with static scales, bias and
          activation, for a following e4m3 layer.
  mx      hipgemm_amd.mx_pack_scales of the activations' block scales, then
          hipgemm_amd.gemm with MX block scales (fp4 or e4m3 elements).
"""
import math

import torch

import hipgemm_amd as hg
from hipgemm_amd.torch_ops import Fp8Linear

E4M3, E5M2 = torch.float8_e4m3fn, torch.float8_e5m2
#: Magnitudes of the eight non-negative E2M1 codes and the midpoints between.
FP4 = (0.0, 0.5, 1.0, 1.5, 2.0, 3.0, 4.0, 6.0)
FP4_MID = (0.25, 0.75, 1.25, 1.75, 2.5, 3.5, 5.0)
ACTS = ("none", "relu", "silu", "gelu_tanh")
MAX_FLOPS = 2.0 * 8192 * 28672 * 8192


def listed():
    return [
        # The smallest call: what one launch costs a caller.
        dict(name="gemm 512", kind="gemm", M=512, N=512, K=512),
        # Decode of 16 sequences through one square projection: a pass over
        # the weights.
        dict(name="decode 16", kind="gemm", M=16, N=8192, K=8192),
        # Decode of 32 sequences through an up projection, as a layer.
        dict(name="decode layer", kind="linear", M=32, N=14336, K=4096,
             act="silu", bias=False),
        # A large decode batch, between memory- and compute-bound.
        dict(name="decode 128", kind="gemm", M=128, N=8192, K=8192),
        # A prefill chunk through a square projection: fewer tiles than CUs
        # on large tiles.
        dict(name="prefill gemm", kind="gemm", M=2048, N=4096, K=4096),
        # A prefill chunk through an up projection with bias, as a layer.
        dict(name="prefill layer", kind="linear", M=2048, N=14336, K=4096,
             act="gelu_tanh", bias=True),
        # Tile edges on every side and a short last round of tiles.
        dict(name="ragged gemm", kind="gemm", M=4000, N=5000, K=3584),
        # A statically quantised MLP's first half, e4m3 for the second.
        dict(name="static e4m3", kind="chain", M=4096, N=4096, K=4096,
             act="gelu_tanh"),
        # A weight gradient over 8192 tokens, accumulated in fp32 outside.
        dict(name="weight gradient", kind="grad", M=4096, N=4096, K=8192,
             out="float32"),
        # Microscaled fp4 activations and weights, the scales of the
        # activations packed on every call.
        dict(name="mxfp4", kind="mx", M=4096, N=8192, K=8192, fmt="fp4"),
        # The compute-bound square and the largest projection.
        dict(name="gemm 8192", kind="gemm", M=8192, N=8192, K=8192),
        dict(name="gemm largest", kind="gemm", M=8192, N=28672, K=8192),
    ]


def _log(rng, lo, hi, step):
    """A multiple of step, log-uniform between lo and hi."""
    v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return max(step, int(round(v / step)) * step)


def draw(rng):
    kind = rng.choice(("gemm", "gemm", "gemm", "linear", "linear", "grad",
                       "chain", "mx"))
    while True:
        # One size in four is odd where the path takes odd ones.
        ragged = rng.random() < 0.25
        if kind == "gemm":
            c = dict(kind=kind, M=_log(rng, 1, 8192, 1),
                     N=_log(rng, 512, 28672, 1 if ragged else 128),
                     K=_log(rng, 512, 28672, 16 if ragged else 128))
            if c["M"] > 256 and not ragged:
                c["M"] = _log(rng, 256, 8192, 64)
        elif kind == "linear":
            c = dict(kind=kind, M=_log(rng, 1, 4096, 1),
                     N=_log(rng, 1024, 28672, 8 if ragged else 128),
                     K=_log(rng, 1024, 8192, 16 if ragged else 128),
                     act=rng.choice(ACTS), bias=rng.random() < 0.5)
        elif kind == "grad":
            c = dict(kind=kind, M=_log(rng, 1024, 8192, 8 if ragged else 128),
                     N=_log(rng, 1024, 8192, 8 if ragged else 128),
                     K=_log(rng, 1024, 16384, 16 if ragged else 128),
                     out=rng.choice(("float32", "bfloat16")))
        elif kind == "chain":
            c = dict(kind=kind, M=_log(rng, 128, 8192, 1 if ragged else 64),
                     N=_log(rng, 1024, 14336, 16 if ragged else 128),
                     K=_log(rng, 1024, 8192, 16 if ragged else 128),
                     act=rng.choice(ACTS))
        else:
            c = dict(kind=kind, M=_log(rng, 128, 8192, 1 if ragged else 64),
                     N=_log(rng, 1024, 8192, 8 if ragged else 128),
                     K=_log(rng, 1024, 8192, 32 if ragged else 128),
                     fmt=rng.choice(("fp4", "e4m3")))
        if 2.0 * c["M"] * c["N"] * c["K"] <= MAX_FLOPS:
            return c


# ---- inputs ---------------------------------------------------------------

def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed) & 0x7FFFFFFF)


def _normal(g, rows, cols, std=1.0, dtype=torch.float32):
    return torch.randn((rows, cols), generator=g, device="cuda").mul_(std).to(dtype)


def _scalar(g):
    return torch.rand(1, generator=g, device="cuda") * 1.5 + 0.5


def _mx_quantise(x, fmt):
    """x (rows x K fp32) as MX blocks of 32: element bytes and E8M0 scales,
    the scale the largest power of two that keeps the block's maximum in the
    element format's top binade."""
    rows, K = x.shape
    b = x.view(rows, K // 32, 32)
    top = 2 if fmt == "fp4" else 8
    e = torch.floor(torch.log2(b.abs().amax(2).clamp_min(2.0 ** -100))) - top
    scales = (e + 127).clamp(0, 254).to(torch.uint8)
    q = (b * torch.exp2(-e)[:, :, None]).view(rows, K)
    if fmt == "e4m3":
        return q.clamp(-448, 448).to(E4M3), scales
    mid = torch.tensor(FP4_MID, device=x.device)
    code = torch.bucketize(q.abs(), mid).to(torch.uint8) | ((q < 0).to(torch.uint8) << 3)
    code = code.view(rows, K // 2, 2)
    return code[:, :, 0] | (code[:, :, 1] << 4), scales


def _operands(case, seed):
    """The random values of a case: everything exact() needs."""
    g = _gen(seed)
    M, N, K, kind = case["M"], case["N"], case["K"], case["kind"]
    if kind == "gemm":
        return dict(a=_normal(g, M, K).to(E4M3), b=_normal(g, N, K).to(E4M3),
                    sa=_scalar(g), sb=_scalar(g))
    if kind == "linear":
        d = dict(x=_normal(g, M, K, dtype=torch.bfloat16),
                 w=_normal(g, N, K, K ** -0.5))
        d["bias"] = _normal(g, 1, N, 0.1)[0] if case["bias"] else None
        return d
    if kind == "grad":
        return dict(a=_normal(g, M, K).to(E5M2), b=_normal(g, N, K).to(E4M3),
                    sa=_scalar(g) * 2.0 ** -10, sb=_scalar(g))
    if kind == "chain":
        # Scales that leave the product near unit variance, as calibration
        # does, and an output scale that fits it into e4m3.
        return dict(a=_normal(g, M, K).to(E4M3), b=_normal(g, N, K).to(E4M3),
                    sa=_scalar(g), sb=_scalar(g) * K ** -0.5,
                    bias=_normal(g, 1, N, 0.1)[0],
                    so=torch.full((1,), 32.0, device="cuda"))
    aq, ascale = _mx_quantise(_normal(g, M, K), case["fmt"])
    bq, bscale = _mx_quantise(_normal(g, N, K, K ** -0.5), case["fmt"])
    return dict(a=aq, ascale=ascale, b=bq, bscale=bscale)


def prepare(case, seed):
    s = _operands(case, seed)
    M, N, K, kind = case["M"], case["N"], case["K"], case["kind"]
    s["kind"] = kind
    if kind == "linear":
        lin = torch.nn.Linear(K, N, bias=case["bias"], device="meta")
        lin.weight = torch.nn.Parameter(s.pop("w"), requires_grad=False)
        if case["bias"]:
            lin.bias = torch.nn.Parameter(s["bias"], requires_grad=False)
        s["layer"] = Fp8Linear.from_linear(
            lin, activation=None if case["act"] == "none" else case["act"])
        return s
    dtype = {"grad": getattr(torch, case.get("out", "bfloat16")), "chain": E4M3}.get(
        kind, torch.bfloat16)
    s["out"] = torch.empty((M, N), dtype=dtype, device="cuda")
    if kind == "chain":
        s["act"] = None if case["act"] == "none" else case["act"]
    if kind == "mx":
        s["K"] = K
        s["fmt"] = hg.FMT_FP4_E2M1 if case["fmt"] == "fp4" else hg.FMT_E4M3
        s["bpacked"] = hg.mx_pack_scales(s["bscale"], K)  # weights: packed once
    return s


def run(s):
    kind = s["kind"]
    if kind == "gemm":
        return hg.fp8_gemm_bf16(s["a"], s["b"], s["sa"], s["sb"], out=s["out"])
    if kind == "linear":
        return s["layer"](s["x"])
    if kind == "grad":
        return hg.gemm(s["a"], s["b"], scale_a=s["sa"], scale_b=s["sb"],
                       out=s["out"])
    if kind == "chain":
        return hg.gemm(s["a"], s["b"], scale_a=s["sa"], scale_b=s["sb"],
                       bias=s["bias"], activation=s["act"], out=s["out"],
                       scale_out=s["so"])
    packed = hg.mx_pack_scales(s["ascale"], s["K"])
    return hg.gemm(s["a"], s["b"], a_format=s["fmt"], b_format=s["fmt"],
                   mx_scale_a=packed, mx_scale_b=s["bpacked"], out=s["out"])


# ---- what a pass cannot do without ---------------------------------------

def work(case):
    M, N, K, kind = case["M"], case["N"], case["K"], case["kind"]
    in_a, in_b, out = 1.0, 1.0, 2.0  # bytes per element
    extra = 0.0
    if kind == "linear":
        in_a = 2.0  # bf16 activations
        extra = 4.0 * N * (2 if case["bias"] else 1)
    elif kind == "grad":
        out = 4.0 if case["out"] == "float32" else 2.0
    elif kind == "chain":
        out, extra = 1.0, 4.0 * N
    elif kind == "mx":
        e = 0.5 if case["fmt"] == "fp4" else 1.0
        in_a = in_b = e + 1.0 / 32  # one scale byte per 32 elements
    return {"bytes": in_a * M * K + in_b * N * K + out * M * N + extra,
            "flops": 2.0 * M * N * K}


def tolerance(case):
    kind = case["kind"]
    if kind == "chain":
        # Another order of the fp32 sums moves a value across an e4m3
        # rounding boundary now and then: one step, an eighth of the value.
        return {"rel": 1e-2, "max": 0.14}
    if kind == "grad" and case["out"] == "float32":
        # fp32 sums in another order, in the matrix unit's own rounding (1.1e-5
        # from the exact sums over 8192 terms).
        return {"rel": 4.5e-5, "max": 5e-4}
    # bf16 outputs (1.7e-3 from the exact values): a rounding the other way is
    # 2^-7 of a value at most.
    return {"rel": 6e-3, "max": 1.6e-2}


# ---- the same in 64 bits --------------------------------------------------

def _act64(v, act):
    if act == "relu":
        return v.clamp_min_(0)
    if act == "silu":
        return v.mul_(torch.sigmoid(v))
    if act == "gelu_tanh":
        return torch.nn.functional.gelu(v, approximate="tanh")
    return v


def _quant64(x):
    """Per-row e4m3 values and scales of x."""
    x = x.double()
    amax = x.abs().amax(1)
    s = torch.where(amax > 0, amax / 448.0, torch.ones_like(amax))
    q = (x / s[:, None]).clamp_(-448.0, 448.0).to(E4M3)
    return q.double(), s


def _mx64(q, scales, fmt):
    if fmt == "fp4":
        table = torch.tensor([*FP4, *(-v for v in FP4)], dtype=torch.float64,
                             device=q.device)
        v = table[torch.stack((q & 15, q >> 4), 2).view(q.shape[0], -1).int()]
    else:
        v = q.double()
    s = torch.exp2(scales.double() - 127)
    return (v.view(q.shape[0], -1, 32) * s[:, :, None]).view(q.shape[0], -1)


def exact(case, seed):
    s = _operands(case, seed)
    kind = case["kind"]
    if kind == "linear":
        q, sx = _quant64(s["x"])
        w, sw = _quant64(s["w"])
        v = (q @ w.t()).mul_(sx[:, None]).mul_(sw[None, :])
        if s["bias"] is not None:
            v += s["bias"].double()
        return _act64(v, case["act"])
    if kind == "mx":
        return _mx64(s["a"], s["ascale"], case["fmt"]) @ _mx64(
            s["b"], s["bscale"], case["fmt"]).t()
    v = (s["a"].double() @ s["b"].double().t()).mul_(s["sa"].double() * s["sb"].double())
    if kind == "chain":
        v = _act64(v.add_(s["bias"].double()), case["act"])
        v = (v * s["so"].double()).clamp_(-448.0, 448.0)
    return v
