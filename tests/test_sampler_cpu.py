"""The sampler's host path without a GPU: a batch that does not decode greedily, through the CPU checker backend."""
import os
import sys
from types import SimpleNamespace

import pytest
import torch

sys.path.insert(0, os.path.dirname(os.path.abspath(__file__)))
import cpu_ops  # noqa: E402

from sglang_custom_amd import ops_backend  # noqa: E402
from sglang_custom_amd.layers.sampler import Sampler  # noqa: E402
from sglang_custom_amd.sampling.sampling_batch_info import SamplingBatchInfo  # noqa: E402
from sglang_custom_amd.sampling.sampling_params import SamplingParams  # noqa: E402


@pytest.mark.parametrize("return_logprob", [False, True])
@pytest.mark.parametrize("min_p", [0.0, 0.2])
def test_draw_of_a_mixed_batch(monkeypatch, return_logprob, min_p):
    monkeypatch.setattr(ops_backend, "_backend", cpu_ops)
    g = torch.Generator().manual_seed(7)
    logits = torch.randn(5, 200, generator=g) * 3
    params = [SamplingParams(temperature=t, top_k=k, top_p=p, min_p=min_p) for t, k, p in ((0.7, 20, 0.9), (1.3, 50, 1.0), (1.0, 1, 1.0), (2.0, 200, 0.5), (0.5, 3, 0.99))]
    info = SamplingBatchInfo.from_reqs([SimpleNamespace(sampling_params=p) for p in params], 200, "cpu")
    assert not info.is_all_greedy
    out = SimpleNamespace(next_token_logits=logits.clone(), next_token_logprobs=None)
    ids = Sampler(torch.Generator().manual_seed(3))(out, info, return_logprob=return_logprob)
    # in place: the probabilities; every id is of the set that top-k, top-p and min-p keep
    probs = torch.softmax(logits / info.temperatures, -1)
    assert torch.allclose(out.next_token_logits, probs, atol=1e-6)
    kept = cpu_ops.ops_ref.kept_distribution(probs, info.top_ks, info.top_ps, info.min_ps if min_p else None)
    assert ids.dtype == torch.int32 and (kept[torch.arange(5), ids.long()] > 0).all()
    assert ids[2] == logits[2].argmax()
    if return_logprob:
        assert torch.allclose(out.next_token_logprobs, probs.log()[torch.arange(5), ids.long()], atol=1e-5)
