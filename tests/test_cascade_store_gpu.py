"""GPU tests of the decode attention that stores the step's own K / V rows (cascade_decode_attention's new_rows): it leaves the pool and gives the
output of store_kv_cache followed by the plain call, wherever the newest token falls in a unit.  Before the call the newest slots hold NaN: a row
read from the pool in the place of the new one, or a stale one multiplied by a probability of zero, shows.  The new keys lie along the queries, so
that the newest token has a tenth of the weight and more: another row in its place shows too."""
import pytest
import torch

pytestmark = pytest.mark.gpu
BF = torch.bfloat16
EDGES = [1, 2, 15, 16, 17, 32, 33, 63, 64, 65, 127, 128, 129, 145, 161, 256, 257]
LONG = [1500 + 67 * i for i in range(12)]
SHAPES = [
    # Hq, Hkv, D, e4m3, page, hnd, table width, lengths, prefix shared by the first three
    (32, 8, 128, 0, 1, 0, 16384, EDGES, 0),             # items in the looping form
    (32, 8, 128, 0, 1, 0, 16384, EDGES + LONG, 0),      # spans
    (32, 8, 128, 0, 1, 0, 16384, LONG + EDGES, 640),    # shared items ahead of spans
    (32, 8, 128, 0, 1, 0, 512, EDGES, 0),               # one workgroup a unit: the rows are stored by a launch of their own
    (32, 8, 128, 1, 1, 0, 16384, EDGES, 0),
    (32, 8, 128, 1, 1, 0, 16384, LONG + EDGES, 640),
    (32, 2, 128, 1, 1, 0, 16384, EDGES * 3, 0),         # 16 query rows a kv head
    (32, 32, 128, 0, 1, 0, 8192, EDGES, 0),
    (14, 2, 64, 0, 1, 0, 512, EDGES, 0),                # one workgroup a unit, head dim 64
    (14, 2, 64, 1, 1, 0, 512, EDGES, 0),
    (14, 2, 64, 0, 1, 0, 16384, LONG + EDGES * 3, 640),
    (16, 4, 64, 1, 1, 0, 16384, EDGES + LONG, 0),
    (32, 8, 128, 0, 16, 1, 16384, EDGES + LONG, 0),     # head-major pages
    (16, 2, 64, 1, 16, 1, 512, EDGES, 0),
]


@pytest.mark.parametrize("Hq,Hkv,D,fp8,page,hnd,width,lens,shared", SHAPES, ids=[f"{s[0]}-{s[1]}-{s[2]}-fp8{s[3]}-hnd{s[5]}-w{s[6]}-{len(s[7])}" for s in SHAPES])
def test_new_rows_equal_store_then_attend(device, Hq, Hkv, D, fp8, page, hnd, width, lens, shared):
    from sglang_amd import kernels as K

    g = torch.Generator().manual_seed(Hq + D + len(lens) + fp8)
    B = len(lens)
    pages = [-(-n // page) for n in lens]
    perm = torch.randperm(sum(pages), generator=g).int() + 1
    slots = (sum(pages) + 2) * page
    r2t = torch.zeros((B + 1, width), dtype=torch.int32)
    at = 0
    for b, n in enumerate(lens):
        r2t[b + 1, :n] = (perm[at:at + pages[b]][:, None] * page + torch.arange(page, dtype=torch.int32)).flatten()[:n]
        at += pages[b]
    for b in (1, 2):
        n = min(shared, lens[b] - 1) // page * page
        r2t[b + 1, :n] = r2t[1, :n]
    loc = torch.stack([r2t[b + 1, n - 1] for b, n in enumerate(lens)]).long()
    loc[-1] = slots - 1                                     # a row that goes elsewhere than its request's last slot: that slot is read as it stands
    ks, vs = (0.5, 0.25) if fp8 else (1.0, 1.0)
    pools = []
    for _ in range(2):
        x = torch.randn((slots, Hkv, D), generator=g) * 0.5
        x[loc] = float("nan")
        x = x.to(torch.float8_e4m3fn).view(torch.uint8) if fp8 else x.to(BF)
        pools.append((x.view(-1, page, Hkv, D).transpose(1, 2).contiguous() if hnd else x).to(device))
    qkv = (torch.randn((B, (Hq + 2 * Hkv) * D), generator=g) * 0.7).to(BF).to(device)
    q, k, v = (x.view(B, -1, D) for x in qkv.split([Hq * D, Hkv * D, Hkv * D], dim=-1))
    k.copy_(q.view(B, Hkv, Hq // Hkv, D).float().mean(2) * (Hq // Hkv) ** 0.5 * (128 / D) ** 0.5)
    pool, seq, loc = torch.arange(1, B + 1).to(device), torch.tensor(lens, dtype=torch.int32).to(device), loc.to(device)
    r2t = r2t.to(device)
    ws = K.CascadeWorkspace(B, Hq, D, width, device)
    outs = []
    for ride in (False, True):
        kd, vd = (x.clone() for x in pools)
        out = torch.full((B, Hq, D), float("nan"), dtype=BF, device=device)
        K.cascade_plan(ws, r2t, pool, seq, Hq, Hkv)
        if not ride:
            fmt = dict(num_kv_heads=Hkv, head_dim=D, kv_fp8=bool(fp8), k_scale=ks, v_scale=vs, page_size=page, hnd=bool(hnd)) if fp8 or hnd else {}
            K.store_kv_cache(k, v, kd, vd, loc, **fmt)
        K.cascade_decode_attention(ws, q, kd, vd, out, r2t, pool, seq, D ** -0.5, bool(fp8), ks, vs, page, bool(hnd), new_rows=(k, v, loc) if ride else None)
        outs.append((out, kd, vd))
    (a, ka, va), (b, kb, vb) = outs
    assert bool(torch.isfinite(b).all())
    # a probability is rounded to bf16 in one call and kept in fp32 in the other, and both outputs are rounded: 2^-8 of the largest value each way
    top = max(float(v.abs().max()), 3.0)
    assert float((a.float() - b.float()).abs().max()) <= 2.0 ** -7 * top
    assert torch.equal(ka.view(torch.uint8), kb.view(torch.uint8)) and torch.equal(va.view(torch.uint8), vb.view(torch.uint8))
