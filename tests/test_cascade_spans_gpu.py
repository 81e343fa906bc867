"""GPU tests of the shared-prefix decode plan's spans: behind large request tables the private tokens of a batch are cut into equal parts
whose ends fall anywhere in a request.  The output is checked against the CPU oracle (oracle/ops.py decode_attention), the slot counts against
the cut restated here."""
import pytest
import torch

from oracle import ops as oo

pytestmark = pytest.mark.gpu
BF = torch.bfloat16
SPAN_UNITS, MIN_TILES, ONE_ROUND, TILE, CHUNK = 768, 3, 1024, 64, 128


def _spans(lens, shared, n_shared_items, Hkv):
    """(tiles of a span or 0, partial slots of every request)"""
    tiles = [(n - s + TILE - 1) // TILE for n, s in zip(lens, shared)]
    per_head = SPAN_UNITS // Hkv
    want = max(per_head - n_shared_items, per_head // 2, 1)
    span = (sum(tiles) + want - 1) // want
    items = n_shared_items + sum(-(-(n - s) // CHUNK) for n, s in zip(lens, shared))
    if span < MIN_TILES or items * Hkv <= ONE_ROUND:
        return 0, [-(-s // CHUNK) + -(-(n - s) // CHUNK) for n, s in zip(lens, shared)]
    slots, at = [], 0
    for t, s in zip(tiles, shared):
        slots.append(-(-s // CHUNK) + ((at + t - 1) // span - at // span + 1 if t else 0))
        at += t
    return span, slots


LONG = [2000 + 37 * i for i in range(10)]
SHAPES = [
    # Hq, Hkv, D, e4m3, page, hnd, lengths, shared prefix of the first three requests
    (32, 8, 128, 0, 1, 0, [1, 15, 16, 17, 63, 64, 65, 127, 128, 129, 191, 193] + LONG, 0),    # spans of several requests, pieces of one token
    (32, 8, 128, 0, 1, 0, LONG + [5003, 1, 640], 1500),                                       # shared items ahead of the spans
    (32, 8, 128, 1, 1, 0, LONG + [5003, 130, 1], 0),
    (32, 8, 128, 1, 16, 1, [600] * 6 + LONG, 700),
    (16, 2, 64, 0, 16, 1, [33 + 211 * i for i in range(60)], 0),                              # 8 rows a kv head
    (16, 2, 64, 1, 1, 0, [33 + 211 * i for i in range(60)], 300),
    (8, 8, 64, 0, 1, 0, LONG + [4100, 2], 0),                                                 # one row a kv head
    (6, 2, 128, 1, 1, 0, [977 + 130 * i for i in range(50)], 0),                              # three
    (32, 2, 128, 0, 1, 0, [3000 + 64 * i for i in range(40)], 0),                             # 16 rows a kv head: items, no spans
    (32, 8, 128, 1, 1, 0, [70, 128, 1, 200, 129, 64, 300, 17], 0),                            # too few tokens for spans: e4m3 items
]


@pytest.mark.parametrize("Hq,Hkv,D,fp8,page,hnd,lens,shared", SHAPES, ids=[f"{s[0]}-{s[1]}-{s[2]}-fp8{s[3]}-hnd{s[5]}-{len(s[6])}" for s in SHAPES])
def test_spans_match_oracle(device, Hq, Hkv, D, fp8, page, hnd, lens, shared):
    from sglang_amd import kernels as K

    g = torch.Generator().manual_seed(Hq + D + len(lens))
    B, width = len(lens), 16384
    # pages in any order: request b's token t sits in slot page_id * page + t % page
    pages = [-(-n // page) for n in lens]
    perm = torch.randperm(sum(pages), generator=g).int() + 1
    slots = (sum(pages) + 1) * page
    r2t = torch.zeros((B + 1, width), dtype=torch.int32)
    at = 0
    for b, n in enumerate(lens):
        rows = (perm[at:at + pages[b]][:, None] * page + torch.arange(page, dtype=torch.int32)).flatten()[:n]
        r2t[b + 1, :n] = rows
        at += pages[b]
    for b in (1, 2):
        n = min(shared, lens[b] - 1) // page * page
        r2t[b + 1, :n] = r2t[1, :n]
    kc = torch.randn((slots, Hkv, D), generator=g) * 0.5
    vc = torch.randn((slots, Hkv, D), generator=g) * 0.5
    q = (torch.randn((B, Hq, D), generator=g) * 0.5).to(BF)
    hot = r2t[B, lens[-1] // 2].long()
    kc[hot] *= 12.0                              # one key whose score may end every running maximum before it
    ks, vs = (0.5, 0.25) if fp8 else (1.0, 1.0)
    if fp8:
        kc8, vc8 = (kc / ks).to(torch.float8_e4m3fn), (vc / vs).to(torch.float8_e4m3fn)
        kc, vc = kc8.float() * ks, vc8.float() * vs
        kd, vd = kc8.view(torch.uint8), vc8.view(torch.uint8)
    else:
        kd, vd = kc.to(BF), vc.to(BF)
        kc, vc = kd.float(), vd.float()
    if hnd:
        kd, vd = (x.view(-1, page, Hkv, D).transpose(1, 2).contiguous() for x in (kd, vd))
    kd, vd = kd.to(device), vd.to(device)
    pool, seq = torch.arange(1, B + 1), torch.tensor(lens, dtype=torch.int32)
    ws = K.CascadeWorkspace(B, Hq, D, width, device)
    ws.ws_acc.fill_(float("nan"))                # a slot that nobody writes shows
    ws.ws_ml.fill_(float("nan"))
    r2t_d, pool_d, seq_d = r2t.to(device), pool.to(device), seq.to(device)
    K.cascade_plan(ws, r2t_d, pool_d, seq_d, Hq, Hkv)
    out = torch.empty((B, Hq, D), dtype=BF, device=device)
    K.cascade_decode_attention(ws, q.to(device), kd, vd, out, r2t_d, pool_d, seq_d, D ** -0.5, bool(fp8), ks, vs, page, bool(hnd))
    plan = K.cascade_plan_summary(ws, B)
    header = ws.plan[:8].cpu().tolist()
    span, slot_counts = _spans(lens, plan["req_shared"], plan["n_shared_items"], Hkv) if Hq // Hkv <= 8 else (0, None)
    loop = B * (width // CHUNK + 1) * Hkv > (2048 if Hq // Hkv <= 8 else 10240)
    assert loop and header[4] == span
    if slot_counts is not None:
        off = 8 + 4 * B + B + 1 + 8 * ws.max_items + B + 2 * B
        assert ws.plan[off:off + B].cpu().tolist() == slot_counts
        assert max(slot_counts) <= ws.slots
    ref = oo.decode_attention(q, kc, vc, r2t, pool, seq.long(), D ** -0.5, compute_dtype=torch.float32).float()
    err = (out.cpu().float() - ref).abs()
    # probabilities are rounded to bf16 (relative 2^-9 each, the sum in fp32) and so is the output: 2^-8 of the largest value a row can take
    assert float(err.max()) <= 2.0 ** -8 * float(vc.abs().max()) , float(err.max())
    # a second step over the same buffers gives the same bits (partial slots of the first one do not leak)
    out2 = torch.empty_like(out)
    K.cascade_plan(ws, r2t_d, pool_d, seq_d, Hq, Hkv)
    K.cascade_decode_attention(ws, q.to(device), kd, vd, out2, r2t_d, pool_d, seq_d, D ** -0.5, bool(fp8), ks, vs, page, bool(hnd))
    assert torch.equal(out, out2)


@pytest.mark.parametrize("fp8", [0, 1])
@pytest.mark.parametrize("lens,plan_heads,Hq,Hkv,D", [([5000 + 37 * i for i in range(8)], (16, 4), 16, 4, 128),      # spans; one workgroup a unit when asked for
                                                     ([5000 + 37 * i for i in range(8)], (16, 4), 8, 2, 128),       # ... and by itself, for fewer heads than the plan's
                                                     ([5000 + 37 * i for i in range(8)], (16, 4), 16, 4, 64),       # bf16 rows of 64 elements stay with the items
                                                     ([130, 700, 64, 1, 1000, 333, 512, 95], (32, 8), 32, 8, 128)])  # too few tokens for spans
def test_every_launch_form_reads_the_plan_it_gets(device, lens, plan_heads, Hq, Hkv, D, fp8):
    """Both launch forms over one plan, whether or not it holds spans, at every line of the switch: the oracle's bar each, and where no
    spans are walked the same bits from bf16 rows (e4m3 items of few rows are cut into other tiles)."""
    from sglang_amd import kernels as K, native

    B, width = len(lens), 8192
    g = torch.Generator().manual_seed(Hq + B)
    r2t = torch.zeros((B + 1, width), dtype=torch.int32)
    perm, at = (torch.randperm(sum(lens), generator=g) + 1).int(), 0
    for b, n in enumerate(lens):
        r2t[b + 1, :n], at = perm[at:at + n], at + n
    r2t[2, :min(384, lens[1] - 1)] = r2t[5, :min(384, lens[1] - 1)]                 # a shared prefix too
    kc, vc = (torch.randn((sum(lens) + 1, Hkv, D), generator=g) * 0.5 for _ in range(2))
    q = (torch.randn((B, Hq, D), generator=g) * 0.5).to(BF)
    if fp8:
        kd, vd = kc.to(torch.float8_e4m3fn), vc.to(torch.float8_e4m3fn)
        kc, vc, kd, vd = kd.float(), vd.float(), kd.view(torch.uint8), vd.view(torch.uint8)
    else:
        kd, vd = kc.to(BF), vc.to(BF)
        kc, vc = kd.float(), vd.float()
    pool, seq = torch.arange(1, B + 1), torch.tensor(lens, dtype=torch.int32)
    ref = oo.decode_attention(q, kc, vc, r2t, pool, seq.long(), D ** -0.5, compute_dtype=torch.float32).float()
    bar = 2.0 ** -8 * float(vc.abs().max())                                         # as above
    ws = K.CascadeWorkspace(B, plan_heads[0], D, width, device)
    r2t_d, pool_d, seq_d, q_d, kd, vd = (x.to(device) for x in (r2t, pool, seq, q, kd, vd))
    K.cascade_plan(ws, r2t_d, pool_d, seq_d, *plan_heads)
    spans = int(ws.plan[4]) > 0
    assert spans == (lens[0] == 5000) and K.cascade_plan_summary(ws, B)["n_shared_items"] > 0
    outs = []
    try:
        for line in (0, 1, 16384):
            native.call("sgl_amd_debug_cascade_launch_form", line, 0)
            out = torch.empty((B, Hq, D), dtype=BF, device=device)
            ws.ws_acc.fill_(float("nan"))
            ws.ws_ml.fill_(float("nan"))
            K.cascade_decode_attention(ws, q_d, kd, vd, out, r2t_d, pool_d, seq_d, D ** -0.5, bool(fp8))
            outs.append(out)
            err = float((out.cpu().float() - ref).abs().max())
            assert err <= bar, (line, err, bar)
    finally:
        native.call("sgl_amd_debug_cascade_launch_form", 0, 0)
    if (not spans or D == 64) and not fp8:
        assert torch.equal(outs[0], outs[1]) and torch.equal(outs[0], outs[2])


@pytest.mark.parametrize("own,prefix,groups,want", [(100, 2000, 1, False), (130, 1000, 16, False), (190, 1100, 1, False), (300, 1000, 6, True), (100, 500, 1, True)])
def test_no_spans_beside_shared_items_that_fill_the_chip(device, own, prefix, groups, want):
    """96 requests, 8 kv heads: more than 48 shared items (384 units) leave the private tokens in items.  Either way the oracle's result."""
    from sglang_amd import kernels as K

    Hq, Hkv, D, B, width = 32, 8, 128, 96, 8192
    g = torch.Generator().manual_seed(own + prefix)
    perm = (torch.randperm(groups * prefix + B * own, generator=g) + 1).int()
    r2t = torch.zeros((B + 1, width), dtype=torch.int32)
    for b in range(B):
        s = b * groups // B * prefix
        r2t[b + 1, :prefix] = perm[s:s + prefix]
        r2t[b + 1, prefix:prefix + own] = perm[groups * prefix + b * own:groups * prefix + (b + 1) * own]
    kc, vc = ((torch.randn((perm.numel() + 1, Hkv, D), generator=g) * 0.5).to(BF) for _ in range(2))
    q = (torch.randn((B, Hq, D), generator=g) * 0.5).to(BF)
    pool, seq = torch.arange(1, B + 1), torch.full((B,), prefix + own, dtype=torch.int32)
    ws = K.CascadeWorkspace(B, Hq, D, width, device)
    r2t_d, pool_d, seq_d = r2t.to(device), pool.to(device), seq.to(device)
    K.cascade_plan(ws, r2t_d, pool_d, seq_d, Hq, Hkv)
    plan = K.cascade_plan_summary(ws, B)
    assert (int(ws.plan[4]) > 0) == want and (plan["n_shared_items"] * Hkv <= SPAN_UNITS // 2) == want
    out = torch.empty((B, Hq, D), dtype=BF, device=device)
    K.cascade_decode_attention(ws, q.to(device), kc.to(device), vc.to(device), out, r2t_d, pool_d, seq_d, D ** -0.5)
    ref = oo.decode_attention(q, kc, vc, r2t, pool, seq.long(), D ** -0.5, compute_dtype=torch.float32).float()
    assert float((out.cpu().float() - ref).abs().max()) <= 2.0 ** -8 * float(vc.float().abs().max())      # as above
