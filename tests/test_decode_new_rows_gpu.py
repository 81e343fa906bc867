"""A decode step's rows stored by the attention's own launch (cascade_decode_attention's new_rows): the bits of store_kv_cache and the attention one after the
other, for pools of every format, both forms of the launch, and tables and slots that the plan has and has not looked at."""
import re

import pytest
import torch

from test_no_spills import HIPCC, Path, _resource_usage

BF, FP8 = torch.bfloat16, torch.float8_e4m3fn
# Hq, Hkv, D, e4m3, page, hnd, table width, lengths
EDGES = [1, 2, 15, 16, 17, 63, 64, 65, 127, 128, 129, 193, 257]
SHAPES = [
    (32, 8, 128, 0, 1, 0, 16384, EDGES * 2),                                  # items of 128 tokens, looping form
    (32, 8, 128, 0, 1, 0, 16384, EDGES + [1500 + 67 * i for i in range(12)]), # spans
    (32, 8, 128, 0, 1, 0, 512, EDGES),                                        # one workgroup a unit
    (32, 8, 128, 1, 1, 0, 16384, EDGES + [1500 + 67 * i for i in range(12)]),
    (32, 8, 128, 1, 1, 0, 512, EDGES),
    (14, 2, 64, 0, 1, 0, 512, EDGES * 10),                                    # more than 64 requests
    (16, 4, 64, 1, 1, 0, 512, EDGES),
    (16, 4, 64, 1, 1, 0, 16384, EDGES * 6),
    (16, 4, 64, 0, 16, 1, 2048, EDGES),                                       # head-major pages
    (32, 2, 128, 0, 1, 0, 512, [1, 2]),
    (64, 4, 128, 0, 1, 0, 8192, [3, 130, 700]),                               # 16 query rows a kv head
]


@pytest.mark.gpu
@pytest.mark.parametrize("slots_are", ["new", "read_elsewhere", "twice", "unplanned", "others_planned", "without_tokens"])
@pytest.mark.parametrize("Hq,Hkv,D,fp8,page,hnd,width,lens", SHAPES, ids=[f"{s[0]}-{s[1]}-{s[2]}-fp8{s[3]}-hnd{s[5]}-w{s[6]}-{len(s[7])}" for s in SHAPES])
def test_the_bits_of_both_calls(device, Hq, Hkv, D, fp8, page, hnd, width, lens, slots_are):
    from sglang_amd import kernels

    g = torch.Generator().manual_seed(Hq + D + len(lens) + fp8 + len(slots_are))
    B, lens = len(lens), list(lens)
    pages = [-(-n // page) for n in lens]
    slots = (sum(pages) + B + 2) * page
    perm = torch.randperm(sum(pages), generator=g).int() + 1
    table, at = torch.zeros((B + 2, width), dtype=torch.int32), 0
    for b, n in enumerate(lens):
        table[b + 1, :n] = (perm[at:at + pages[b]][:, None] * page + torch.arange(page, dtype=torch.int32)).flatten()[:n]
        at += pages[b]
    loc = torch.tensor([int(table[b + 1, n - 1]) for b, n in enumerate(lens)])
    spare = (sum(pages) + 1) * page
    if slots_are == "read_elsewhere":                                # a slot of one row at the front of another's context; a row that ends in another's slot
        long = max(range(B), key=lambda b: lens[b])
        table[long + 1, 0] = int(loc[(long + 1) % B])
        if B > 3:
            table[2, lens[1] - 1], loc[1] = int(loc[0]), spare
    if slots_are == "twice":                                         # two rows to one slot, which both read; two to the sink
        table[B, lens[B - 1] - 1] = loc[B - 1] = int(loc[0])
        if B > 4:
            loc[2] = loc[3] = 0
    if slots_are == "without_tokens":
        lens[0] = 0
    fmt = dict(kv_fp8=bool(fp8), page_size=page, hnd=bool(hnd), **(dict(k_scale=0.75, v_scale=1.25) if fp8 else {}))
    shape = (slots // page, Hkv, page, D) if hnd else (slots, Hkv, D)
    pools = [(torch.randn(shape, generator=g) * 0.5).to(FP8 if fp8 else BF) for _ in range(2)]
    pools = [(x.view(torch.uint8) if fp8 else x).to(device) for x in pools]
    q, k, v = (x.to(device) for x in (torch.randn((B, (Hq + 2 * Hkv) * D), generator=g) * 0.7).to(BF).split([Hq * D, Hkv * D, Hkv * D], dim=-1))
    q, k, v = q.view(B, Hq, D), k.view(B, Hkv, D), v.view(B, Hkv, D)
    table, loc, seq, rows = table.to(device), loc.to(device), torch.tensor(lens, dtype=torch.int32, device=device), torch.arange(1, B + 1, device=device)
    ws = kernels.CascadeWorkspace(B, Hq, D, width, device)
    planned = None if slots_are == "unplanned" else loc.roll(1) if slots_are == "others_planned" else loc
    got = []
    for riding in (False, True):
        kc, vc = (x.clone() for x in pools)
        out = torch.zeros((B, Hq, D), dtype=BF, device=device)
        kernels.cascade_plan(ws, table, rows, seq, Hq, Hkv, new_loc=planned)
        if not riding:
            kernels.store_kv_cache(k, v, kc, vc, loc, **(dict(num_kv_heads=Hkv, head_dim=D, **fmt) if fp8 or hnd else {}))
        kernels.cascade_decode_attention(ws, q, kc, vc, out, table, rows, seq, D ** -0.5, **fmt, **(dict(new_rows=(k, v, loc)) if riding else {}))
        got.append((out, kc, vc))
    (o0, k0, v0), (o1, k1, v1) = got
    if slots_are == "twice":
        # which of two rows a launch of both leaves is not said; the attention's own keeps the later one, and any in the sink
        flat = [x.transpose(1, 2).reshape(-1, Hkv, D) if hnd else x for x in (k0, v0, k1, v1)]
        keep = torch.ones(flat[0].shape[0], dtype=torch.bool, device=device)
        keep[loc[0]] = keep[0] = False
        assert torch.equal(flat[0][keep], flat[2][keep]) and torch.equal(flat[1][keep], flat[3][keep])
        if not (fp8 or hnd):
            assert torch.equal(flat[2][loc[0]], k[B - 1]) and torch.equal(flat[3][loc[0]], v[B - 1])
            sink = [b for b in range(B) if int(loc[b]) == 0]
            assert not sink or any(torch.equal(flat[2][0], k[b]) for b in sink)
        readers = [b for b in range(B) if b not in (0, B - 1) and (int(loc[0]) not in table[b + 1, :lens[b]].tolist())]
        assert torch.equal(o0[readers], o1[readers])
        return
    assert torch.equal(k0, k1) and torch.equal(v0, v1) and torch.equal(o0, o1)


@pytest.mark.gpu
@pytest.mark.parametrize("without", ["every_third", "all", "the_last_two_of_one_slot", "one_whose_slot_is_read"])
@pytest.mark.parametrize("Hq,Hkv,D,fp8,width,B", [(32, 8, 128, 0, 16384, 26), (32, 8, 128, 0, 512, 26), (14, 2, 64, 0, 512, 130), (32, 8, 128, 1, 16384, 70), (16, 4, 64, 1, 512, 5)])
def test_requests_without_tokens(device, Hq, Hkv, D, fp8, width, B, without):
    """Their rows are stored though no unit reads them, and the plan says no more of them than that: other rows are then not stored by every wave."""
    from sglang_amd import kernels

    g = torch.Generator().manual_seed(B + Hq)
    lens = [EDGES[b % len(EDGES)] + (b > 20) * 200 for b in range(B)]
    slots = sum(lens) + 1
    table, at, perm = torch.zeros((B + 1, width), dtype=torch.int32), 0, torch.randperm(slots - 1, generator=g).int() + 1
    for b, n in enumerate(lens):
        table[b + 1, :n] = perm[at:at + n]
        at += n
    loc = torch.tensor([int(table[b + 1, n - 1]) for b, n in enumerate(lens)])
    empty = {"every_third": range(0, B, 3), "all": range(B), "the_last_two_of_one_slot": [B - 2, B - 1], "one_whose_slot_is_read": [1]}[without]
    for b in empty:
        lens[b] = 0
    found = 2                                                        # kPlanUnread
    if without == "the_last_two_of_one_slot":
        loc[B - 2], found = loc[B - 1], 3                            # and kPlanMeet
    if without == "one_whose_slot_is_read":
        table[3, 4], found = loc[1], 3
    pools = [(torch.randn((slots, Hkv, D), generator=g) * 0.5).to(FP8 if fp8 else BF) for _ in range(2)]
    pools = [(x.view(torch.uint8) if fp8 else x).to(device) for x in pools]
    q, k, v = ((torch.randn((B, h, D), generator=g) * 0.7).to(BF).to(device) for h in (Hq, Hkv, Hkv))
    table, loc, seq, rows = table.to(device), loc.to(device), torch.tensor(lens, dtype=torch.int32, device=device), torch.arange(1, B + 1, device=device)
    fmt = dict(kv_fp8=True, k_scale=0.75, v_scale=1.25) if fp8 else {}
    ws, got = kernels.CascadeWorkspace(B, Hq, D, width, device), []
    for riding in (False, True):
        kc, vc = (x.clone() for x in pools)
        out = torch.zeros((B, Hq, D), dtype=BF, device=device)
        kernels.cascade_plan(ws, table, rows, seq, Hq, Hkv, new_loc=loc)
        if not riding:
            # (of two rows with one slot a launch of both may leave either; the attention's own keeps the later one)
            keep = slice(0, B) if without != "the_last_two_of_one_slot" else [b for b in range(B) if b != B - 2]
            kernels.store_kv_cache(k[keep].contiguous(), v[keep].contiguous(), kc, vc, loc[keep].contiguous(), **(dict(num_kv_heads=Hkv, head_dim=D, **fmt) if fp8 else {}))
        kernels.cascade_decode_attention(ws, q, kc, vc, out, table, rows, seq, D ** -0.5, **fmt, **(dict(new_rows=(k, v, loc)) if riding else {}))
        got += [out, kc, vc]
    assert all(torch.equal(a, b) for a, b in zip(got[:3], got[3:]))
    words = 9 + 9 * B + 8 * ws.max_items + 769                        # cascade_plan_view (cascade_plan.hpp): ints in front of the pieces ...
    words = (words + 3) // 4 * 4 + 8 * (B + 768) + B                 # ... and of what was found
    bits = 0
    for x in ws.plan[words:words + 64].tolist():
        bits |= x
    assert bits == found


@pytest.mark.gpu
def test_replays_with_other_slots(device):
    """A captured step whose slots, lengths and tables change between replays, among them to ones that meet and back."""
    from sglang_amd import kernels

    B, Hq, Hkv, D, width = 6, 8, 2, 128, 16384
    g = torch.Generator().manual_seed(5)
    pool = [(torch.randn((4096, Hkv, D), generator=g) * 0.5).to(BF).to(device) for _ in range(2)]
    q, k, v = ((torch.randn((B, h, D), generator=g) * 0.7).to(BF).to(device) for h in (Hq, Hkv, Hkv))
    table, rows = torch.zeros((B + 1, width), dtype=torch.int32, device=device), torch.arange(1, B + 1, device=device)
    seq, loc = torch.ones(B, dtype=torch.int32, device=device), torch.zeros(B, dtype=torch.int64, device=device)
    ws, out = kernels.CascadeWorkspace(B, Hq, D, width, device), torch.zeros((B, Hq, D), dtype=BF, device=device)
    kc, vc = (x.clone() for x in pool)

    def step():
        kernels.cascade_plan(ws, table, rows, seq, Hq, Hkv, new_loc=loc)
        kernels.cascade_decode_attention(ws, q, kc, vc, out, table, rows, seq, D ** -0.5, new_rows=(k, v, loc))

    stream = torch.cuda.Stream()
    with torch.cuda.stream(stream):
        step()
        stream.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=stream):
            step()
    torch.cuda.synchronize()
    for n, meet in ((1, False), (70, False), (70, True), (300, False), (300, True), (301, False)):
        lens = [n + 3 * b for b in range(B)]
        t = torch.randperm(4095, generator=g)[: sum(lens)].int() + 1
        for b, x in enumerate(t.split(lens)):
            table[b + 1, : lens[b]] = x.to(device)
        loc.copy_(torch.stack([table[b + 1, m - 1] for b, m in enumerate(lens)]))
        if meet:
            table[1, 5] = int(loc[4])
        seq.copy_(torch.tensor(lens))
        for to, x in zip((kc, vc), pool):
            to.copy_(x)
        graph.replay()
        want, (k1, v1) = torch.zeros_like(out), (x.clone() for x in pool)
        kernels.store_kv_cache(k, v, k1, v1, loc)
        other = kernels.CascadeWorkspace(B, Hq, D, width, device)
        kernels.cascade_plan(other, table, rows, seq, Hq, Hkv)
        kernels.cascade_decode_attention(other, q, k1, v1, want, table, rows, seq, D ** -0.5)
        torch.cuda.synchronize()
        assert torch.equal(out, want) and torch.equal(kc, k1) and torch.equal(vc, v1), (n, meet)


def _planned_slots(monkeypatch, pool, fb, requests=3, **attrs):
    """new_loc of the plan that a decode step of `fb` makes over `pool`."""
    from types import SimpleNamespace

    from sglang_amd.layers.attention import hip_backend as H

    b, got = H.HipAttnBackend.__new__(H.HipAttnBackend), []
    vars(b).update(token_to_kv_pool=pool, req_to_token_pool=SimpleNamespace(req_to_token=None), num_q_heads=8, num_kv_heads=2, _seq_src=None,
                   forward_metadata=H._Meta(torch.ones(requests, dtype=torch.int32), cascade=object()), **attrs)
    monkeypatch.setattr(H.kernels, "cascade_plan", lambda *a, new_loc=None, **k: got.append(new_loc))
    b.init_forward_metadata_in_graph(fb)
    assert b.forward_metadata.slots_planned == (got[0] is not None)
    return got[0]


@pytest.mark.parametrize("what", ["no_slots", "slots_none", "slots_on_the_host", "pool_takes_no_rows"])
def test_steps_whose_rows_are_in_the_pool_need_no_slots(monkeypatch, what):
    """A model that stores its rows itself plans a step whatever its batch says of slots, over pools that take no rows."""
    from types import SimpleNamespace

    from sglang_amd.mem_cache.memory_pool import MHATokenToKVPool
    from sglang_amd.model_executor.forward_batch_info import ForwardMode

    fb = SimpleNamespace(forward_mode=ForwardMode.DECODE, req_pool_indices=torch.zeros(3, dtype=torch.int64), out_cache_loc=torch.zeros(3, dtype=torch.int64))
    pool = MHATokenToKVPool.__new__(MHATokenToKVPool)
    if what == "no_slots":
        del fb.out_cache_loc
    elif what == "slots_none":
        fb.out_cache_loc = None
    elif what == "pool_takes_no_rows":
        pool = SimpleNamespace()
    assert _planned_slots(monkeypatch, pool, fb) is None


@pytest.mark.parametrize("fp8,hnd,page,streams,looks", [(False, False, 1, True, False), (False, False, 1, False, False), (True, False, 1, True, False), (True, False, 1, False, True),
                                                        (False, True, 16, False, False), (True, True, 16, False, False)])
def test_the_plan_looks_only_where_a_layer_stores_with_it(monkeypatch, fp8, hnd, page, streams, looks):
    """The package's own model stores its rows itself over bf16 pools and where the projection streams; over head-major pages the store keeps its launch."""
    from types import SimpleNamespace

    from sglang_amd.harness import models
    from sglang_amd.layers.attention.hip_backend import HipAttnBackend
    from sglang_amd.mem_cache.memory_pool import MHATokenToKVPool
    from sglang_amd.model_executor.forward_batch_info import ForwardMode

    pool, loc = MHATokenToKVPool.__new__(MHATokenToKVPool), torch.zeros(3, dtype=torch.int64)
    vars(pool).update(dtype=FP8 if fp8 else BF, is_fp8=fp8, use_hnd=hnd, page_size=page)
    monkeypatch.setattr(HipAttnBackend, "_new_slots", lambda *a: loc)
    monkeypatch.setattr(models.kernels, "wstream_preferred", lambda *a: streams)
    attn = SimpleNamespace(rotary_emb=SimpleNamespace(is_neox_style=True), qkv_proj=SimpleNamespace(weight=torch.zeros(1, 1)))
    model = SimpleNamespace(layers=[SimpleNamespace(self_attn=attn)])
    fb = SimpleNamespace(forward_mode=ForwardMode.DECODE, req_pool_indices=loc)
    got = _planned_slots(monkeypatch, pool, fb, _brings_rows=lambda *a: models.CausalLM.brings_rows(model, *a))
    assert (got is loc) == looks
    assert (_planned_slots(monkeypatch, pool, fb) is loc) == (not hnd)      # a backend that is not told
    assert (_planned_slots(monkeypatch, pool, fb, 512) is loc) == (not hnd) and _planned_slots(monkeypatch, pool, fb, 513) is None


@pytest.mark.skipif(not Path(HIPCC).exists(), reason="hipcc not installed")
def test_registers(tmp_path):
    usage = _resource_usage("cascade_attention.hip", tmp_path)
    loop = {k: v for k, v in usage.items() if "cascade_store_loop_kernel" in k}
    one = {k: v for k, v in usage.items() if re.search("cascade_store_kernel", k)}
    assert len(loop) == 4 and len(one) == 4, sorted(usage)
    for name, u in loop.items():
        assert u["vgpr_spill_count"] <= (8 if "ILi128ELb1E" in name else 0) and u["sgpr_spill_count"] == 0 and u["vgpr_count"] <= 128, (name, u)
    for name, u in one.items():                                       # 96 registers: five workgroups a CU
        assert u["vgpr_spill_count"] <= (16 if "ELb1E" in name else 5) and u["sgpr_spill_count"] == 0 and u["vgpr_count"] <= 96, (name, u)
