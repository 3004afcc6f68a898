"""Prefill-sized fp8 projections on rows that the norm or the SiLU-mul in front has quantised: the bits of quantising them afterwards.
(bf16 alone: the library product that small shapes take refuses fp16 results.)"""
import types

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("m,n,k", [(65, 512, 1024), (129, 1024, 4096), (700, 6144, 4096), (2500, 4096, 2304)])
def test_projection_of_quantised_rows(m, n, k):
    from sglang_custom_amd.layers.layernorm import RMSNorm
    from sglang_custom_amd.layers.quantization.unquant import QuantizedAct
    from sglang_custom_amd.layers.quantization.w8a8_fp8 import W8A8Fp8LinearMethod, prefill_takes_quantised_rows
    from sglang_custom_amd import ops

    dtype = torch.bfloat16
    g = torch.Generator().manual_seed(m)
    method = W8A8Fp8LinearMethod()
    layer = types.SimpleNamespace(weight=(torch.randn(n, k, generator=g) * k ** -0.5).to(DEV, dtype), quant_method=method)
    method.process_weights_after_loading(layer)
    norm = RMSNorm(k).to(DEV, dtype)
    norm.weight.data.copy_(1 + 0.1 * torch.randn(k, generator=g))
    x = (torch.randn(m, k, generator=g) * torch.rand(m, 1, generator=g) * 3).to(DEV, dtype)
    r = torch.randn(m, k, generator=g).to(DEV, dtype)
    assert prefill_takes_quantised_rows(layer, m, dtype) and not prefill_takes_quantised_rows(layer, 64, dtype)
    for residual in (None, r):
        a, b = (None if residual is None else residual.clone() for _ in range(2))
        want, got = norm(x.clone(), a), norm(x.clone(), b, quant_fp8=True, dense=False)
        if residual is not None:
            (want, a), (got, b) = want, got
            assert torch.equal(a, b)
        assert isinstance(got, QuantizedAct) and got.dense is None and got.dtype == dtype and got.shape == x.shape
        assert torch.equal(method.apply(layer, got), method.apply(layer, want))
    gate_up = torch.randn(m, 2 * k, generator=g).to(DEV, dtype)
    assert torch.equal(method.apply(layer, QuantizedAct(*ops.silu_and_mul_quant_fp8(gate_up), dtype)), method.apply(layer, ops.silu_and_mul(gate_up)))
