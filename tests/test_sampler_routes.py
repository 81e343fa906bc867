"""Which batches of an odd number of softmax ranges the sampler hands to the one call."""
import types

import pytest
import torch


@pytest.mark.parametrize("dtype,vocab,top_k,taken", [
    (torch.bfloat16, 4096, True, True), (torch.bfloat16, 4096, False, False), (torch.bfloat16, 16383, False, False), (torch.bfloat16, 16384, False, True),
    (torch.float32, 4096, True, False), (torch.float32, 16384, True, True), (torch.float32, 128256, False, False),
])
def test_any_ranges(monkeypatch, dtype, vocab, top_k, taken):
    from sglang_amd import kernels
    from sglang_amd.layers.sampler import LogitsProcessorOutput, Sampler, SamplingBatchInfo

    seen = []
    monkeypatch.setattr(kernels, "sample_from_logits", lambda *a, any_ranges: seen.append(any_ranges) or torch.zeros(3, dtype=torch.int32))
    info = SamplingBatchInfo(torch.ones((3, 1)), torch.full((3,), 0.9), torch.full((3,), 50 if top_k else 1 << 30, dtype=torch.int32), torch.zeros(3),
                             is_all_greedy=False, need_top_p_sampling=True, need_top_k_sampling=top_k, need_min_p_sampling=False)
    Sampler()(LogitsProcessorOutput(next_token_logits=torch.zeros((3, vocab), dtype=dtype)), info)
    assert seen == [taken]
