"""A decode step's new K / V rows are in the pool before any request of the batch attends: a row of the batch may read a slot that another row writes in
the same step (two rows that end in one slot; consecutive tokens of one request as rows of their own; a slot in the middle of another context)."""
import types

import pytest
import torch

BF, FP8 = torch.bfloat16, torch.float8_e4m3fn


def _backend(dev, rows, width, slots, hq, hkv, d, fp8=False, page=1, hnd=False):
    from sglang_amd.layers.attention.hip_backend import HipAttnBackend
    from sglang_amd.layers.radix_attention import RadixAttention
    from sglang_amd.mem_cache.memory_pool import MHATokenToKVPool, ReqToTokenPool

    req_pool, pool = ReqToTokenPool(rows, width, dev), MHATokenToKVPool(slots, page, FP8 if fp8 else BF, hkv, d, 1, dev, use_hnd=hnd)
    backend = HipAttnBackend(types.SimpleNamespace(device=dev, req_to_token_pool=req_pool, token_to_kv_pool=pool, num_attention_heads_per_rank=hq,
                                                   num_kv_heads_per_rank=hkv, head_dim=d))
    return backend, req_pool, pool, RadixAttention(hq, d, d ** -0.5, hkv, 0)


def _step(backend, req_pool, pool, rows, lens, loc):
    from sglang_amd.model_executor.forward_batch_info import ForwardBatch, ForwardMode

    dev = req_pool.req_to_token.device
    seq = torch.tensor(lens)
    return ForwardBatch.init_new(forward_mode=ForwardMode.DECODE, input_ids=torch.zeros(len(lens), dtype=torch.int64, device=dev),
                                 req_pool_indices=torch.tensor(rows, device=dev), seq_lens=seq.int().to(dev), out_cache_loc=loc.to(dev), seq_lens_cpu=seq,
                                 req_to_token_pool=req_pool, token_to_kv_pool=pool, attn_backend=backend)


@pytest.mark.parametrize("fp8", [False, True])
def test_the_rows_are_stored_in_front_of_the_attention(monkeypatch, fp8):
    from sglang_amd import kernels

    backend, req_pool, pool, layer = _backend(torch.device("cpu"), 4, 64, 256, 8, 2, 128, fp8)
    fb = types.SimpleNamespace(batch_size=2, req_pool_indices=torch.tensor([1, 2]), out_cache_loc=torch.tensor([7, 8]))
    backend.forward_metadata = types.SimpleNamespace(cascade=object(), seq_lens_i32=torch.tensor([5, 9], dtype=torch.int32))
    done = []
    monkeypatch.setattr(kernels, "store_kv_cache", lambda k, v, kc, vc, loc, **kw: done.append(("store", loc.tolist())))
    monkeypatch.setattr(kernels, "cascade_decode_attention", lambda *a, **kw: done.append(("attend", sorted(kw))))
    k, v = torch.zeros((2, 2, 128), dtype=BF), torch.zeros((2, 2, 128), dtype=BF)
    backend.forward_decode(torch.zeros((2, 8 * 128), dtype=BF), k, v, layer, fb)
    assert done[0] == ("store", [7, 8]) and [x[0] for x in done] == ["store", "attend"] and "new_rows" not in done[1][1]


EDGES = [1, 2, 15, 16, 17, 32, 33, 63, 64, 65, 127, 128, 129, 145, 161, 256, 257]
LONG = [1500 + 67 * i for i in range(12)]
SHAPES = [
    # Hq, Hkv, D, e4m3, page, hnd, table width, lengths
    (32, 8, 128, 0, 1, 0, 16384, EDGES),                # items in the looping form
    (32, 8, 128, 0, 1, 0, 16384, EDGES + LONG),         # spans
    (32, 8, 128, 0, 1, 0, 512, EDGES),                  # one workgroup a unit
    (32, 8, 128, 1, 1, 0, 16384, EDGES + LONG),
    (32, 32, 128, 0, 1, 0, 8192, EDGES),
    (14, 2, 64, 0, 1, 0, 512, EDGES),
    (16, 4, 64, 1, 1, 0, 16384, EDGES + LONG),
    (32, 8, 128, 0, 16, 1, 16384, EDGES + LONG),        # head-major pages
]


@pytest.mark.gpu
@pytest.mark.parametrize("Hq,Hkv,D,fp8,page,hnd,width,lens", SHAPES, ids=[f"{s[0]}-{s[1]}-{s[2]}-fp8{s[3]}-hnd{s[5]}-w{s[6]}-{len(s[7])}" for s in SHAPES])
def test_rows_that_read_what_others_write(device, Hq, Hkv, D, fp8, page, hnd, width, lens):
    """Before the call the written slots hold NaN in a bf16 pool and 416 in one of e4m3 rows: a row read as the pool held it shows.  New keys lie along the
    queries, so that they carry weight.  Against float64 attention over the rows as the pool keeps them."""
    g = torch.Generator().manual_seed(Hq + D + len(lens) + fp8)
    lens = list(lens)
    B = len(lens)
    backend, req_pool, pool, layer = _backend(device, B + 4, width, (sum(lens) // page + B + 4) * page, Hq, Hkv, D, bool(fp8), page, bool(hnd))
    pages = [-(-n // page) for n in lens]
    perm = torch.randperm(sum(pages), generator=g).int() + 1
    table = torch.zeros(req_pool.req_to_token.shape, dtype=torch.int32)
    at = 0
    for b, n in enumerate(lens):
        table[b + 1, :n] = (perm[at:at + pages[b]][:, None] * page + torch.arange(page, dtype=torch.int32)).flatten()[:n]
        at += pages[b]
    rows = list(range(1, B + 1))
    loc = torch.stack([table[b + 1, n - 1] for b, n in enumerate(lens)]).long()
    spare = (sum(pages) + 1) * page                              # a slot of no request
    # the last row ends in the slot that row 3 writes, and its own row goes elsewhere
    table[B, lens[-1] - 1], loc[-1] = int(loc[3]), spare
    # row 4's new slot stands in the middle of row 10's context, row 5's at its front
    table[11, 40], table[11, 0] = int(loc[4]), int(loc[5])
    # rows 12 and 13 are consecutive tokens of one request (row 13's length is one more)
    rows[13], lens[13] = rows[12], lens[12] + 1
    table[13, lens[13] - 1] = int(loc[13])
    assert loc.unique().numel() == B
    req_pool.req_to_token.copy_(table)
    for buf in (pool.get_key_buffer(0), pool.get_value_buffer(0)):
        x = torch.randn(buf.shape, generator=g) * 0.5
        rows_of = x.transpose(1, 2).reshape(-1, Hkv, D) if hnd else x
        rows_of[loc] = 416.0 if fp8 else float("nan")
        x = rows_of.view(-1, page, Hkv, D).transpose(1, 2) if hnd else rows_of
        buf.copy_(x.to(FP8).view(torch.uint8) if fp8 else x.to(BF))
    qkv = (torch.randn((B, (Hq + 2 * Hkv) * D), generator=g) * 0.7).to(BF).to(device)
    q, k, v = (x.view(B, -1, D) for x in qkv.split([Hq * D, Hkv * D, Hkv * D], dim=-1))
    k.copy_(q.view(B, Hkv, Hq // Hkv, D).float().mean(2) * (Hq // Hkv) ** 0.5 * (128 / D) ** 0.5)
    fb = _step(backend, req_pool, pool, rows, lens, loc)
    backend.init_forward_metadata(fb)
    out = layer(q.reshape(B, -1), k, v, fb).view(B, Hq, D)

    def kept(buf):
        x = buf.view(FP8).double() if fp8 else buf.double()
        return (x.transpose(1, 2).reshape(-1, Hkv, D) if hnd else x).cpu()

    kc, vc = kept(pool.get_key_buffer(0)), kept(pool.get_value_buffer(0))
    new_k, new_v = (x.cpu().to(FP8).double() if fp8 else x.cpu().double() for x in (k.contiguous(), v.contiguous()))
    assert torch.equal(kc[loc], new_k) and torch.equal(vc[loc], new_v)
    for b in range(B):
        s = table[rows[b], :lens[b]].long()
        kk, vv = (x[s].repeat_interleave(Hq // Hkv, 1) for x in (kc, vc))
        p = torch.softmax(torch.einsum("hd,nhd->hn", q[b].cpu().double(), kk) * D ** -0.5, -1)
        want = torch.einsum("hn,nhd->hd", p, vv)
        # a probability and the output are rounded to bf16: 2^-9 each of the largest value that is summed
        assert float((out[b].cpu().double() - want).abs().max()) <= 2.0 ** -8 * float(vv.abs().max()), (b, lens[b])
