"""Which prefill products take the tiled kernel: enough tiles, or long reductions whose tiles share K where that is ahead of the library."""
from types import SimpleNamespace

import pytest
import torch

from sglang_custom_amd import ops_backend
from sglang_custom_amd.layers.quantization import unquant, w8a8_fp8


@pytest.mark.parametrize("m,n,k,splits,bf16,fp8", [
    (12 * 256, 4096, 4096, 0, True, True), (12 * 256 - 256, 4096, 4096, 0, False, True), (9 * 256, 4096, 4096, 0, False, True), (8 * 256, 4096, 4096, 0, False, False),
    (300, 4096, 14336, 5, True, True), (300, 4096, 14336, 0, False, False), (300, 4096, 8128, 5, False, False), (90, 4096, 14336, 16, True, False),   # long, split, not
    (83, 4096, 14336, 16, False, False), (142, 4096, 14336, 16, True, False), (143, 4096, 14336, 16, True, True),
    (300, 512, 8192, 32, False, False), (520, 512, 8192, 32, True, False), (256, 128, 16384, 64, False, False), (1100, 2048, 8192, 6, True, True),   # few columns
    (1073, 2048, 8192, 6, True, True), (800, 2048, 8192, 8, True, False),
    (150, 16384, 16384, 4, False, False), (127, 8192, 16384, 8, True, False), (128, 8192, 16384, 8, True, True),                                      # many, few rows
])
def test_tiles_and_long_reductions(monkeypatch, m, n, k, splits, bf16, fp8):
    monkeypatch.setattr(ops_backend, "_backend", SimpleNamespace(tiled_tail_splits=lambda *a: splits, linear_tiled_supported=lambda *a: True,
                                                                 fp8_scaled_mm_tiled_supported=lambda *a: True))
    monkeypatch.setattr(unquant, "PREFILL_GEMM", "tiled")
    assert unquant._use_tiled(m, n, n, k, torch.bfloat16, False) == bf16
    assert w8a8_fp8._tiled_ok(m, n, k, torch.bfloat16, False) == fp8
