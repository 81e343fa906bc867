"""Large extends by workgroups that stay and take their query tiles from a queue: every query tile is computed as a launched workgroup computes it, so
the results of the two launches are the same bits."""
import pytest
import torch

from sglang_amd import kernels, native

pytestmark = pytest.mark.gpu
BF, FP8 = torch.bfloat16, torch.float8_e4m3fn


def _ragged(n, lo, hi):
    return [lo + (i * 7919 + 13) % (hi - lo + 1) for i in range(n)]


# (extend lengths, prefixes, query heads, kv heads): tiles of 64, 32, 51 (group 5) and 256 tokens; few and many key tiles (what is read ahead starts at nine);
# batches beyond a wave of requests; prefixes of one length and of many; requests without new tokens; one request alone
SHAPES = {
    "shared": ([128] * 60, [896] * 60, 32, 8),
    "cold ragged": ([1500, 37, 700, 2900, 0, 64, 1], [0] * 7, 64, 8),
    "mixed prefixes": (_ragged(40, 5, 300), _ragged(40, 0, 2500), 32, 8),
    "many requests": (_ragged(150, 30, 120), _ragged(150, 0, 70), 64, 8),
    "one": ([4097], [11], 32, 8),
    "group 5": (_ragged(30, 100, 333), _ragged(30, 0, 400), 40, 8),
    "group 1": (_ragged(9, 600, 900), _ragged(9, 3, 900), 32, 32),
    "two kv heads": (_ragged(20, 500, 700), [130] * 20, 32, 2),
}


@pytest.mark.parametrize("kv_fp8", [False, True])
@pytest.mark.parametrize("name", list(SHAPES))
def test_walked_extends_give_the_same_bits(name, kv_fp8, monkeypatch):
    _walked_and_launched(name, *SHAPES[name], kv_fp8, monkeypatch)


# Requests that have new tokens and no keys (their rows are zeros): the first tile that every workgroup takes (the longest prefixes stand first), tiles in the
# middle of the list, behind one another and between others, and all of them.
@pytest.mark.parametrize("kv_fp8", [False, True])
@pytest.mark.parametrize("name,without", [("first", lambda i: i >= 44), ("middle", lambda i: 9 < i < 14), ("every other", lambda i: i % 2 == 0), ("all", lambda i: True)])
def test_requests_without_keys(name, without, kv_fp8, monkeypatch):
    _walked_and_launched(name, [100 + i for i in range(64)], [40 * i for i in range(64)], 32, 8, kv_fp8, monkeypatch, [i for i in range(64) if without(i)])


def _walked_and_launched(name, lens, pre, hq, hkv, kv_fp8, monkeypatch, no_keys=()):
    d, b, t = 128, len(lens), sum(lens)
    g = torch.Generator(device="cuda")
    g.manual_seed(len(name))
    total = [p + n for p, n in zip(pre, lens)]
    monkeypatch.setattr(native.lib(), "sgl_amd_extend_attention_store_parts", lambda *a: 0)      # (also where it does not pay)
    slots = sum(total) + 8
    at = torch.randperm(slots - 1, device="cuda", generator=g).to(torch.int32) + 1
    table = torch.zeros((b + 3, max(total) + 5), dtype=torch.int32, device="cuda")
    rows = torch.randperm(b + 3, device="cuda", generator=g)[:b]
    loc, o = [], 0
    for i, n in enumerate(total):
        table[rows[i], :n] = at[o:o + n]
        loc.append(at[o + pre[i]:o + n])
        o += n
    loc = torch.cat(loc).to(torch.int64)
    qkv = torch.randn((t, (hq + 2 * hkv) * d), device="cuda", generator=g).to(BF)
    q, k, v = (x.reshape(t, -1, d) for x in qkv.split([hq * d, hkv * d, hkv * d], dim=-1))
    pool = [torch.randn((slots, hkv, d), device="cuda", generator=g).to(FP8 if kv_fp8 else BF) for _ in range(2)]
    seq, prefix = (torch.tensor(x, dtype=torch.int32, device="cuda") for x in ([0 if i in no_keys else n for i, n in enumerate(total)], pre))
    indptr = torch.tensor([0] + lens, dtype=torch.int32, device="cuda").cumsum(0, dtype=torch.int32)
    for causal in (True, False):
        outs, pools = [], []
        for walked in (True, False):
            kc, vc = (x.view(torch.uint8).clone() if kv_fp8 else x.clone() for x in pool)
            out = torch.full((t, hq, d), 7.0, dtype=BF, device="cuda")
            args = (q, out, kc, vc, table, rows, seq, prefix, indptr, max(lens), d ** -0.5, causal, kv_fp8)
            if walked:
                for _ in range(2):                                     # (the counters are zeroed by every call)
                    kernels.extend_attention(*args, max_kv_len=max(total), new_rows=(k, v, loc))
            else:
                kernels.store_kv_cache(k, v, kc, vc, loc, **(dict(num_kv_heads=hkv, head_dim=d, kv_fp8=True) if kv_fp8 else {}))
                native.call("sgl_amd_debug_extend_attention_shape", 82, 0)
                try:
                    kernels.extend_attention(*args)
                finally:
                    native.call("sgl_amd_debug_extend_attention_shape", 0, 0)
            outs.append(out)
            pools.append((kc, vc))
        assert torch.equal(outs[0], outs[1]), (name, causal, (outs[0] != outs[1]).any(-1).any(-1).nonzero().flatten()[:8].tolist())
        assert all(torch.equal(a, c) for a, c in zip(*pools))
        for i in no_keys:
            assert not outs[0][sum(lens[:i]):sum(lens[:i + 1])].any()
