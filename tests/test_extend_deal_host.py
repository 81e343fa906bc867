"""Which extends are dealt to workgroups that stay."""
import pytest

from sglang_amd import native


@pytest.mark.parametrize("lens,pre,hq,hkv,d,stays", [
    ([128] * 60, [896] * 60, 32, 8, 128, False),                        # all contexts alike
    ([128] * 60, [50 + 97 * i for i in range(60)], 32, 8, 128, True),
    ([1100, 3100, 2000, 1500, 2700, 2200], [0] * 6, 64, 8, 128, True),
    ([1100, 3100, 2000, 1500, 2700, 2200], [0] * 6, 14, 2, 64, False),   # head dim 64: four waves
    ([20, 300, 100], [0] * 3, 32, 8, 128, False),                        # fewer tiles than CUs
    ([150 + i for i in range(513)], [7 * i for i in range(513)], 32, 8, 128, False),
    ([40000, 100], [0, 0], 32, 8, 128, True),
    ([300000, 100], [0, 0], 32, 8, 128, False),                          # more tiles of 64 tokens than levels
    ([262144, 100], [0, 0], 32, 8, 128, True),
    ([262145, 100], [0, 0], 32, 8, 128, False),
    ([150 + i % 40 for i in range(512)], [7 * i for i in range(512)], 32, 8, 128, True),
    # one request that stands out does not put a batch of short walks into the queue, a long prefix that would be dealt last does
    ([200] * 30 + [700], [300] * 30 + [0], 32, 8, 128, False),
    ([200] * 12 + [700], [200] * 12 + [0], 32, 8, 128, False),
    ([200] * 31, [300] * 30 + [1500], 32, 8, 128, True),
    ([237] * 40 + [200], [0] * 40 + [1500], 32, 8, 128, True),
    ([700, 910, 500, 800, 600, 900, 490, 700], [0] * 8, 32, 32, 128, False),      # a query head to a kv head
    ([150] * 16, [100] * 15 + [3000], 32, 32, 128, True),
])
def test_rule(lens, pre, hq, hkv, d, stays):
    total = [p + n for p, n in zip(pre, lens)]
    shape = (max(lens), max(total), hq, hkv, d)
    parts = native.lib().sgl_amd_extend_attention_store_parts(len(lens), sum(lens), sum(total), *shape)
    assert (parts == 0) == stays
    general = native.lib().sgl_amd_extend_attention_parts(len(lens), sum(lens), *shape)
    assert general >= 1 and (stays or parts == general)
    assert native.lib().sgl_amd_extend_attention_store_parts(len(lens), sum(lens), 0, *shape) == general      # the sum is not known
