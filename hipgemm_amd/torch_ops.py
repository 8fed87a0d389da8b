"""PyTorch custom operators over the hipgemm C ABI, and an FP8 linear layer.

Importing this module registers, in the ``hipgemm`` namespace:

  torch.ops.hipgemm.fp8_gemm(a, b_t, scale_a=None, scale_b=None, variant=0)
      bf16 (M x N) = scale_a * scale_b * a (M x K e4m3) . b_t (N x K e4m3)^T,
      per-tensor scales (1-element float32 device tensors) -- the C ABI's
      hipgemm_fp8_gemm_bf16_ws.
  torch.ops.hipgemm.fp8_gemm_rowcol(a, b_t, scale_rows=None, scale_cols=None,
                                    variant=0)
      the same with per-row (M) / per-column (N) float32 scale vectors --
      hipgemm_fp8_gemm_bf16_rowcol.
  torch.ops.hipgemm.gemm(a, b_t, scale_a=None, scale_b=None, scale_rows=None,
                         scale_cols=None, bias=None, activation="none",
                         out_f16=False, variant=0, out_dtype=None,
                         scale_out=None, mx_scale_a=None, mx_scale_b=None)
      the general entry point (hipgemm_gemm): a / b_t float8_e4m3fn or
      float8_e5m2 (uint8 bytes: e4m3), or both float4_e2m1fn_x2 (K / 2
      bytes per row); fused bias and activation ("none", "relu", "silu",
      "gelu_tanh"); output bf16, fp16 (out_f16 or out_dtype), fp32 or
      float8_e4m3fn (out_dtype; saturating, after multiplying by the
      1-element scale_out); MX block scales packed by
      hipgemm_amd.mx_pack_scales (mx_scale_a / mx_scale_b, uint8).

All have fake (meta) implementations, so they trace under torch.compile,
torch.export and FakeTensorMode without running, and they run inside CUDA
graph capture (the split-K workspace is allocated on first use per stream,
before capture if the caller warms up).  The device implementation is
libhipgemm.so; CPU tensors raise HipGemmError -- there is no CPU path.

Fp8Linear is a drop-in for torch.nn.Linear in LLM projections (the reference
has no layer; its LLM shapes are benchmark configurations): e4m3 weights with
one fp32 scale per output channel, activations quantised per token (row) on
the fly, the product through hipgemm::gemm with the bias and activation
fused into its epilogue.
"""
from __future__ import annotations

from typing import Optional

import torch

from . import ACTIVATIONS, HipGemmError, fp8_gemm_bf16, fp8_gemm_bf16_rowcol
from . import _check, lib
from . import gemm as _gemm

__all__ = ["fp8_gemm", "fp8_gemm_rowcol", "gemm", "Fp8Linear",
           "quantize_rows"]

E4M3_MAX = 448.0


@torch.library.custom_op("hipgemm::fp8_gemm", mutates_args=())
def fp8_gemm(a: torch.Tensor, b_t: torch.Tensor,
             scale_a: Optional[torch.Tensor] = None,
             scale_b: Optional[torch.Tensor] = None,
             variant: int = 0) -> torch.Tensor:
    return fp8_gemm_bf16(a, b_t, scale_a, scale_b, variant=variant)


@fp8_gemm.register_fake
def _fp8_gemm_fake(a, b_t, scale_a=None, scale_b=None, variant=0):
    _check_shapes(a, b_t)
    return a.new_empty((a.shape[0], b_t.shape[0]), dtype=torch.bfloat16)


@torch.library.custom_op("hipgemm::fp8_gemm_rowcol", mutates_args=())
def fp8_gemm_rowcol(a: torch.Tensor, b_t: torch.Tensor,
                    scale_rows: Optional[torch.Tensor] = None,
                    scale_cols: Optional[torch.Tensor] = None,
                    variant: int = 0) -> torch.Tensor:
    return fp8_gemm_bf16_rowcol(a, b_t, scale_rows, scale_cols,
                                variant=variant)


@fp8_gemm_rowcol.register_fake
def _fp8_gemm_rowcol_fake(a, b_t, scale_rows=None, scale_cols=None,
                          variant=0):
    _check_shapes(a, b_t)
    if scale_rows is not None and tuple(scale_rows.shape) != (a.shape[0],):
        raise HipGemmError("scale_rows must have M elements")
    if scale_cols is not None and tuple(scale_cols.shape) != (b_t.shape[0],):
        raise HipGemmError("scale_cols must have N elements")
    return a.new_empty((a.shape[0], b_t.shape[0]), dtype=torch.bfloat16)


@torch.library.custom_op("hipgemm::gemm", mutates_args=())
def gemm(a: torch.Tensor, b_t: torch.Tensor,
         scale_a: Optional[torch.Tensor] = None,
         scale_b: Optional[torch.Tensor] = None,
         scale_rows: Optional[torch.Tensor] = None,
         scale_cols: Optional[torch.Tensor] = None,
         bias: Optional[torch.Tensor] = None, activation: str = "none",
         out_f16: bool = False, variant: int = 0,
         out_dtype: Optional[torch.dtype] = None,
         scale_out: Optional[torch.Tensor] = None,
         mx_scale_a: Optional[torch.Tensor] = None,
         mx_scale_b: Optional[torch.Tensor] = None) -> torch.Tensor:
    return _gemm(a, b_t, out_dtype=_out_dtype(out_f16, out_dtype),
                 scale_a=scale_a, scale_b=scale_b, scale_rows=scale_rows,
                 scale_cols=scale_cols, bias=bias, activation=activation,
                 variant=variant, scale_out=scale_out, mx_scale_a=mx_scale_a,
                 mx_scale_b=mx_scale_b)


def _out_dtype(out_f16, out_dtype):
    if out_dtype is not None:
        if out_dtype not in (torch.bfloat16, torch.float16, torch.float32,
                             torch.float8_e4m3fn):
            raise HipGemmError(f"unsupported out_dtype {out_dtype}")
        return out_dtype
    return torch.float16 if out_f16 else torch.bfloat16


@gemm.register_fake
def _gemm_fake(a, b_t, scale_a=None, scale_b=None, scale_rows=None,
               scale_cols=None, bias=None, activation="none", out_f16=False,
               variant=0, out_dtype=None, scale_out=None, mx_scale_a=None,
               mx_scale_b=None):
    _check_shapes(a, b_t)
    if activation not in ACTIVATIONS:
        raise HipGemmError(f"unknown activation {activation!r}")
    for v, n, name in ((scale_rows, a.shape[0], "scale_rows"),
                       (scale_cols, b_t.shape[0], "scale_cols"),
                       (bias, b_t.shape[0], "bias")):
        if v is not None and tuple(v.shape) != (n,):
            raise HipGemmError(f"{name} must have {n} elements")
    return a.new_empty((a.shape[0], b_t.shape[0]),
                       dtype=_out_dtype(out_f16, out_dtype))


def _check_shapes(a, b_t):
    if a.dim() != 2 or b_t.dim() != 2 or a.shape[1] != b_t.shape[1]:
        raise HipGemmError(f"expected a (M, K) and b_t (N, K), got "
                           f"{tuple(a.shape)} and {tuple(b_t.shape)}")


# Input types of hipgemm_quantize_rows_e4m3.
_QUANT_TYPES = {torch.float32: 0, torch.bfloat16: 1, torch.float16: 2}


def _plain_eager(x: torch.Tensor) -> bool:
    """x is an ordinary tensor on the current GPU and nothing watches the
    operations on it: no autograd graph to record (reverse or forward), no
    transform, trace, compilation or dispatch mode.  Everything else takes the
    tensor operations, which all of those see."""
    return (type(x) in (torch.Tensor, torch.nn.Parameter) and x.is_cuda
            and x.layout is torch.strided and not x.is_neg()
            and not (x.requires_grad and torch.is_grad_enabled())
            and not torch.compiler.is_compiling()
            and torch._C._get_tracing_state() is None
            and torch._C._len_torch_dispatch_stack() == 0
            and torch._C._len_torch_function_stack() == 0
            and not torch._C._are_functorch_transforms_active()
            and torch.autograd.forward_ad._current_level < 0
            and x.device.index == torch.cuda.current_device())


def _kernel_ahead(M: int, K: int, ld: int, size: int, ptr: int) -> bool:
    """The kernel is faster than the tensor operations on M rows of K elements
    of `size` bytes.  It gives each row a workgroup, so that it falls behind on
    many rows of a few elements, where a workgroup has little to do, and on a
    few very long rows, which leave CUs idle.  Measured against the operations
    in a graph, which is where they are cheapest (us, kernel / operations):
    bf16 65536x16 110 / 40, 65536x256 111 / 130, 16384x16 28 / 32; fp32
    262144x64 207 / 164, x192 209 / 292; bf16 1x131072 30 / 35, 1x262144 60 /
    36, 16x1048576 318 / 266, 256x1048576 604 / 1919; rows without 16-byte
    loads: 262144x33 120 / 105, 1x16385 22 / 30, 1x65537 81 / 39, 256x65537 150
    / 121, 1024x65537 172 / 464.  (At 256 to 20480 elements always.)"""
    if (ptr | ld * size | K * size) % 16 == 0:
        short, few, long, many = 512 // size, 8192 * size, (256 << 10) // size, 256
    else:
        short, few, long, many = 65, 65536, 20480, 1024
    return (K >= short or M <= few) and (K <= long or M >= many)


def quantize_rows(x: torch.Tensor):
    """Per-row e4m3 quantisation: returns (q, s) with q = x / s rounded to
    e4m3 (saturated to +-448) and s = amax(|row|) / 448 (float32, one per
    row; rows of zeros get s = 1).  x ~= q * s[:, None].

    Rows of float32, bfloat16 or float16 on the GPU go through one kernel
    (hipgemm_quantize_rows_e4m3) where that is faster (_kernel_ahead), with the
    same results bit for bit; under autograd, a transform or a trace, on the CPU
    and for other layouts these are tensor operations."""
    return _quantize_rows(x, _plain_eager(x))


def _quantize_rows(x: torch.Tensor, plain: bool):
    """quantize_rows, with _plain_eager(x) known."""
    kind = _QUANT_TYPES.get(x.dtype)
    if plain and kind is not None and x.dim() == 2:
        (M, K), (ld, unit) = x.shape, x.stride()
        if (0 < M < 2 ** 31 and 0 < K < 2 ** 31 and unit == 1 and ld >= K
                and (256 <= K <= 20480
                     or _kernel_ahead(M, K, ld, x.element_size(), x.data_ptr()))):
            dev = x.device
            q = torch.empty((M, K), dtype=torch.float8_e4m3fn, device=dev)
            s = torch.empty(M, dtype=torch.float32, device=dev)
            _check(lib().hipgemm_quantize_rows_e4m3(
                x.data_ptr(), kind, M, K, ld, q.data_ptr(), s.data_ptr(),
                torch._C._cuda_getCurrentRawStream(dev.index)),
                "hipgemm_quantize_rows_e4m3")
            return q, s
    return _quantize_rows_ops(x)


def _quantize_rows_ops(x: torch.Tensor):
    """quantize_rows as tensor operations."""
    xf = x.float()
    amax = xf.abs().amax(dim=1)
    s = torch.where(amax > 0, amax / E4M3_MAX, torch.ones_like(amax))
    q = (xf / s[:, None]).clamp_(-E4M3_MAX, E4M3_MAX).to(torch.float8_e4m3fn)
    return q, s


class Fp8Linear(torch.nn.Module):
    """y = act(x W^T + b) with W (out x in) held as e4m3 rows and one
    float32 scale per output feature; x is quantised per token (row) to e4m3
    with its own scale, and the product runs through hipgemm's general
    entry point with the scales, the bias and the activation fused:
    y[t, o] = bf16(act(fma(acc[t, o], sx[t] * sw[o], b[o]))).
    in_features must be a multiple of 16.  activation: None, "relu", "silu"
    or "gelu_tanh"."""

    def __init__(self, weight_e4m3: torch.Tensor, weight_scale: torch.Tensor,
                 bias: Optional[torch.Tensor] = None, variant: int = 0,
                 activation: Optional[str] = None):
        super().__init__()
        if weight_e4m3.dtype != torch.float8_e4m3fn or weight_e4m3.dim() != 2:
            raise HipGemmError("weight must be a 2-D float8_e4m3fn tensor")
        if weight_e4m3.shape[1] % 16 != 0:
            raise HipGemmError("in_features must be a multiple of 16")
        if tuple(weight_scale.shape) != (weight_e4m3.shape[0],):
            raise HipGemmError("weight_scale must have out_features elements")
        self.register_buffer("weight", weight_e4m3.contiguous())
        self.register_buffer("weight_scale",
                             weight_scale.to(torch.float32).contiguous())
        self.register_buffer("bias", None if bias is None else
                             bias.to(torch.float32).contiguous())
        if activation not in ACTIVATIONS:
            raise HipGemmError(f"unknown activation {activation!r}")
        self.activation = activation or "none"
        self.variant = variant

    @property
    def in_features(self) -> int:
        return self.weight.shape[1]

    @property
    def out_features(self) -> int:
        return self.weight.shape[0]

    @classmethod
    def from_linear(cls, linear: torch.nn.Linear, variant: int = 0,
                    activation: Optional[str] = None):
        """Quantise a Linear's weight per output channel (amax / 448)."""
        w, s = quantize_rows(linear.weight.detach())
        return cls(w, s, linear.bias.detach() if linear.bias is not None
                   else None, variant, activation)

    def forward(self, x: torch.Tensor) -> torch.Tensor:
        lead = x.shape[:-1]
        x2 = x.reshape(-1, self.in_features)
        plain = _plain_eager(x2)
        q, s = _quantize_rows(x2, plain)
        # Where nothing watches the operations (as for quantize_rows), the
        # call itself instead of the operator around it: the dispatcher and the
        # operator's wrappers take about 20 us of host time.
        w, sw, bias = self.weight, self.weight_scale, self.bias
        gemm = _gemm if plain and _plain_buffers(w, sw, bias) else torch.ops.hipgemm.gemm
        y = gemm(q, w, scale_rows=s, scale_cols=sw, bias=bias,
                 activation=self.activation, variant=self.variant)
        return y if x.dim() == 2 else y.reshape(*lead, self.out_features)


def _plain_buffers(*tensors) -> bool:
    grad = torch.is_grad_enabled()
    return all(t is None or (type(t) in (torch.Tensor, torch.nn.Parameter)
                             and not (grad and t.requires_grad))
               for t in tensors)
