"""UnquantizedLinearMethod.apply(layer, x, bias) = F.linear
(python/sglang/srt/layers/quantization/unquant.py:110-122).

Decode-sized inputs (M <= 64 rows) and every fp32 input go to the hand-written kernels behind
mi355_linear (weight-streaming MFMA / exact-fp32 tiled).  Large-M bf16/f16 GEMMs (prefill) run on the
hand-written 256 x 256-tile matrix-core kernel behind mi355_linear_tiled, which can apply SiLU-and-mul in
its epilogue, and few rows (to 256) on the smaller tiles behind mi355_linear_few, whose call also costs the host less than the
library's (8 us for 20).  PREFILL_GEMM (env MI355_PREFILL_GEMM) picks: "tiled" (default) = that kernel for every
shape it serves (at least TILED_MIN_TILES output tiles; smaller problems, but for few rows and for long reductions, and shapes it
does not take fall back to the library GEMM, torch.nn.functional.linear -> hipBLASLt); "auto" = the faster of the two
per projection as measured on MI355X (the hand-written kernel for gate_up with the fused activation,
1.02x the library pair; the library for the plain projections, where it is 4-6 % faster); "library" =
hipBLASLt everywhere."""
import os
from typing import Optional

import torch
import torch.nn.functional as F

from ...ops import FEW_MAX_M
from ...ops_backend import get_ops

SKINNY_MAX_M = 64
# Deferred split-K reduction / fused decode step (bit-identical to the unfused kernels but for the norm inside a projection of one or two
# rows, ops.norm_linear_packed, which adds the squares in another order; the switch exists so that tests and profiles can run both).
DECODE_FUSION = True
# "tiled" | "auto" | "library" for 16-bit GEMMs with more than SKINNY_MAX_M rows (see the module docstring)
PREFILL_GEMM = os.environ.get("MI355_PREFILL_GEMM", "tiled")
# below this many 256 x 256 output tiles the kernel leaves too many CUs idle (us, library | tiled: 6144 x 4096 with 1300 rows, 144 tiles, 70 | 82,
# 1700, 168, 74 | 81, 1962, 192, 83 | 83, 2300, 216, 86 | 86; 4096 x 4096 with 2300, 144, 67 | 75, 2800, 176, 76 | 79, 3100, 208, 81 | 82; 8192 x
# 2048 with 1300, 192, 42 | 45, 1700, 224, 49 | 48)
TILED_MIN_TILES = 192
# ... unless the tiles share long reductions: with K split over the idle CUs the kernel is ahead of the library from K = 8192 on, but
# for the few rows whose sums cost as much as the product (us, library | split: 4096 x 14336 with 126 rows 41 | 35, 330 65 | 53, 646
# 88 | 78, 1134 130 | 114; 4096 x 11264 with 80 rows 32 | 30, 128 47 | 31, 700 73 | 68; 2048 x 8192 with 128 rows 20 | 22, 200
# 28 | 24, 1000 48 | 47, 1353 53 | 56, 2100 73 | 73; 2048 x 5632 with 400 rows 22 | 27, 1000 36 | 39, 1500 40 | 48).  Products of less
# than 2.1 billion multiply-adds are launches and sums more than anything else (library / split: 512 x 8192 with 300 rows 0.83, 128 x 16384 with
# 256 0.64, 1024 x 14336 with 128 0.97, 150 1.23; 1280 x 8192 with 200 1.03), and columns of 16384 leave at most four workgroups a
# tile (x 8192 with 150 to 300 rows 0.77 to 1.01, x 16384 0.85 to 1.25; 8192 x 8192 0.88 to 1.36, x 14336 1.01 to 1.77)
SPLIT_MIN_K = 8192
SPLIT_MIN_MK = 1200000
SPLIT_MIN_MACS = 2.1e9
SPLIT_MAX_N = 8192


def _use_tiled(m: int, n_out_tiles_cols: int, n: int, k: int, dtype, silu_mul: bool) -> bool:
    if PREFILL_GEMM == "library" or (PREFILL_GEMM == "auto" and not silu_mul):
        return False
    tiles = ((m + 255) // 256) * ((n_out_tiles_cols + 255) // 256)
    ops = get_ops()
    return ((tiles >= TILED_MIN_TILES or (k >= SPLIT_MIN_K and m * k >= SPLIT_MIN_MK and m * n * k >= SPLIT_MIN_MACS and n <= SPLIT_MAX_N
                                          and ops.tiled_tail_splits(m, n, k, False, silu_mul) > 1))
            and ops.linear_tiled_supported(m, n, k, dtype, silu_mul))


def pack_for_decode(layer) -> None:
    """Keep a second copy of a 16-bit weight in the decode GEMM's streaming order (MFMA-fragment
    blocks, ops.pack_weight).  The row-major copy stays: prefill GEMMs, the embedding gather and
    checkpoint loading use it.  2x weight bytes is the price of reading decode weights as whole
    contiguous lines; at 288 GB of HBM per GPU it is not the binding constraint.  (Output heads at 64 rows, plain / packed:
    32768 x 4096 63 / 46 us, 32768 x 2048 34 / 25.)"""
    w = layer.weight
    layer.weight_packed = None
    if w.is_cuda and w.dtype in (torch.bfloat16, torch.float16) and w.shape[1] % 32 == 0:
        layer.weight_packed = get_ops().pack_weight(w.data)


def decode_linear(layer, x2: torch.Tensor, bias: Optional[torch.Tensor], out_dtype=None, scale: Optional[float] = None) -> torch.Tensor:
    """M <= 64 rows (or fp32): the hand-written kernels, on the packed copy when there is one.  scale: of an fp32 result, applied to the
    widened values."""
    ops = get_ops()
    wp = getattr(layer, "weight_packed", None)
    if wp is not None and x2.shape[0] <= SKINNY_MAX_M and x2.stride(0) % 8 == 0:
        return ops.linear_packed(x2, wp, layer.weight.shape[0], bias, out_dtype=out_dtype, scale=1.0 if scale is None else scale)
    y = ops.linear(x2, layer.weight, bias, out_dtype=out_dtype)
    return y if scale is None else y.mul_(scale)


def pack_gate_up_for_decode(layer) -> None:
    """gate_up_proj: the decode copy interleaves gate and up rows (8 + 8 per MFMA tile) so that the
    GEMM epilogue can apply SiLU-and-mul in registers (ops.linear_packed_silu_mul).  It replaces
    the plain packed copy: the unfused GEMM + activation remains the path for large M."""
    w = layer.weight
    layer.weight_packed = None
    layer.weight_packed_gate_up = None
    if (w.is_cuda and w.dtype in (torch.bfloat16, torch.float16) and w.shape[1] % 256 == 0
            and w.shape[0] % 16 == 0 and w.shape[0] < 65536):
        layer.weight_packed_gate_up = get_ops().pack_weight_gate_up(w.data)
    else:
        pack_for_decode(layer)


def gate_up_silu_mul(layer, act_fn, x: torch.Tensor) -> torch.Tensor:
    """act_fn(gate_up_proj(x)) (models/llama.py:94-98), fused for decode-sized inputs."""
    x2 = x.view(-1, x.shape[-1])
    wp = getattr(layer, "weight_packed_gate_up", None)
    if wp is not None and x2.shape[0] <= SKINNY_MAX_M and x2.stride(0) % 8 == 0:
        y = get_ops().linear_packed_silu_mul(x2, wp, layer.weight.shape[0])
        return y.view(*x.shape[:-1], y.shape[-1])
    w = layer.weight
    plain = x2.is_cuda and isinstance(layer.quant_method, UnquantizedLinearMethod) and getattr(layer, "bias", None) is None
    if plain and SKINNY_MAX_M < x2.shape[0] <= FEW_MAX_M and PREFILL_GEMM != "library":
        y = get_ops().linear_few(x2, w, None, silu_mul=True)
        if y is not None:
            return y.view(*x.shape[:-1], y.shape[-1])
    if (plain and x2.stride(1) == 1 and x2.stride(0) % 8 == 0
            and _use_tiled(x2.shape[0], w.shape[0], w.shape[0], w.shape[1], x2.dtype, True)):
        y = get_ops().linear_tiled(x2, w, None, silu_mul=True, split_tail=True)
        return y.view(*x.shape[:-1], y.shape[-1])
    gate_up, _ = layer(x)
    return act_fn(gate_up)


class SplitKPartials:
    """Output of a decode GEMM whose split-K partials ([splits, M, N] fp32) are still to be summed
    -- by the kernel that consumes it (the fused add + RMSNorm, or the fused decode attention).
    x_scale / w_scale: the fp8 GEMM's per-token and per-channel scales (None for a 16-bit GEMM)."""

    def __init__(self, part: torch.Tensor, x_scale=None, w_scale=None):
        self.part = part
        self.x_scale = x_scale
        self.w_scale = w_scale
        self.shape = part.shape[1:]


class QuantizedAct:
    """A decode activation that already went through per-token fp8 quantisation inside the kernel
    that produced it (row norm, SiLU-mul): xq [M, K] e4m3fn, x_scale [M, 1]; `dense` is the 16-bit
    tensor when the producer also wrote it (None otherwise)."""

    def __init__(self, xq: torch.Tensor, x_scale: torch.Tensor, dtype: torch.dtype,
                 dense: Optional[torch.Tensor] = None):
        self.xq = xq
        self.x_scale = x_scale
        self.dtype = dtype      # the activation dtype of the model (output dtype of the GEMM that follows)
        self.dense = dense
        self.shape = xq.shape


class PendingAllReduce:
    """This rank's partial sums of a row-parallel projection whose sum over the TP group has been
    left to the consumer: the RMSNorm behind it does all-reduce + residual add + norm in one launch
    (the reference defers the same all-reduce through LayerCommunicator, layers/communicator.py)."""

    def __init__(self, partial: torch.Tensor):
        self.partial = partial

    @property
    def shape(self):
        return self.partial.shape

    @property
    def dtype(self):
        return self.partial.dtype


def linear_for_norm(layer, x: torch.Tensor):
    """layer(x) for a post-norm that sums a decode product's splits itself (SplitKPartials), the tensor where there are none."""
    y = decode_linear_deferred(layer, x) if x.shape[0] <= SKINNY_MAX_M and layer.weight.shape[0] % 8 == 0 and layer.weight.shape[0] <= 8192 else None
    return layer(x)[0] if y is None else y


def decode_linear_deferred(layer, x, needs_all_reduce: bool = True):
    """layer(x) on the decode path, leaving the split-K reduction to the kernel that consumes it; None
    when the layer, the shape or the ops backend does not support it.  A row-parallel layer
    (needs_all_reduce) qualifies only at TP=1: its output would have to cross ranks first.  x is a
    [M, K] tensor or, for an fp8 layer, a QuantizedAct."""
    if not DECODE_FUSION or len(x.shape) != 2 or not 1 <= x.shape[0] <= SKINNY_MAX_M:     # (first: prompts ask twice a layer, 2 us less each)
        return None
    from .w8a8_fp8 import W8A8Fp8LinearMethod

    ops = get_ops()
    wp = getattr(layer, "weight_packed", None)
    if wp is None or (needs_all_reduce and getattr(layer, "tp_size", 1) != 1):
        return None
    n = layer.weight.shape[0]
    if isinstance(layer.quant_method, W8A8Fp8LinearMethod):
        if isinstance(x, QuantizedAct):
            xq, xs = x.xq, x.x_scale
        else:
            if layer.k_padded == x.shape[1] and (fused := ops.fp8_quant_packed_partials(x, wp, n)) is not None:
                return SplitKPartials(fused[0], fused[1], layer.weight_scale.data)
            xq, xs = ops.per_token_quant_fp8(x, pad_to=layer.k_padded)
        if xq.shape[1] != layer.k_padded:
            return None
        part = ops.fp8_packed_partials(xq, wp, n)
        return None if part is None else SplitKPartials(part, xs, layer.weight_scale.data)
    if (isinstance(x, QuantizedAct) or not isinstance(layer.quant_method, UnquantizedLinearMethod)
            or x.stride(0) % 8 != 0):
        return None
    part = ops.linear_packed_partials(x, wp, n)
    return None if part is None else SplitKPartials(part)


def takes_norm_in_front(layer, packed, hidden, norm, silu_mul: bool = False) -> bool:
    """Whether `layer` (16-bit, its packed weight given) forms the rows of the norm in front of it by itself (ops.norm_linear_packed): few rows of
    a decode step whose projection has left its sum to that norm."""
    return (DECODE_FUSION and isinstance(hidden, SplitKPartials) and hidden.x_scale is None and packed is not None and packed.is_cuda
            and isinstance(layer.quant_method, UnquantizedLinearMethod) and packed.dtype == norm.weight.dtype and getattr(layer, "bias", None) is None
            and hidden.part.shape[0] <= 8 and get_ops().norm_linear_packed_splits(hidden.shape[0], layer.weight.shape[0], hidden.shape[1], silu_mul) > 0)


def prefill_linear_act(layer, x: torch.Tensor, act: str) -> Optional[torch.Tensor]:
    """The unit act ("gelu_erf", or "gelu_tanh_mul" over [gate; up]) of layer(x) for 2-d rows and a layer without a bias, in the product's epilogue;
    None where the 256 x 256 tiles do not serve the product."""
    w = layer.weight
    if not (x.shape[0] > FEW_MAX_M and x.is_cuda and _use_tiled(x.shape[0], w.shape[0], w.shape[0], w.shape[1], x.dtype, act == "gelu_tanh_mul")
            and isinstance(layer.quant_method, UnquantizedLinearMethod) and getattr(layer, "bias", None) is None
            and x.stride(1) == 1 and x.stride(0) % 8 == 0 and w.is_contiguous()):
        return None
    return get_ops().linear_tiled(x, w, None, split_tail=True, act=act)


def prefill_linear(x2: torch.Tensor, weight: torch.Tensor, bias: Optional[torch.Tensor] = None) -> torch.Tensor:
    """16-bit rows [M, K] (M > SKINNY_MAX_M) against a plain weight [N, K]."""
    if x2.shape[0] <= FEW_MAX_M and x2.is_cuda and PREFILL_GEMM == "tiled":
        y = get_ops().linear_few(x2, weight, bias)
        if y is not None:
            return y
    if (x2.stride(1) == 1 and x2.stride(0) % 8 == 0 and weight.is_contiguous()
            and _use_tiled(x2.shape[0], weight.shape[0], weight.shape[0], weight.shape[1], x2.dtype, False)):
        return get_ops().linear_tiled(x2, weight, bias, split_tail=True)
    return F.linear(x2, weight, bias)


class UnquantizedLinearMethod:
    def process_weights_after_loading(self, layer) -> None:
        pack_for_decode(layer)

    def apply(self, layer, x: torch.Tensor, bias: Optional[torch.Tensor] = None) -> torch.Tensor:
        x2 = x.view(-1, x.shape[-1])
        if x2.shape[0] <= SKINNY_MAX_M or x2.dtype == torch.float32 or not x2.is_cuda:
            y = decode_linear(layer, x2, bias)
        else:
            y = prefill_linear(x2, layer.weight, bias)
        return y.view(*x.shape[:-1], y.shape[-1])
