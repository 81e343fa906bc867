"""Experts whose weights bound their products (moe_weight_bound_kernel, moe_sum_parts): tiles of 240 rows with three stages of weights, K of the down projection in
parts, against float64."""
import pytest
import torch

from sglang_amd import kernels as K

BF = torch.bfloat16


def test_where_these_tiles_are_taken():
    for rows, experts, up, down, most in ((39, 8, 14336, 4096, 320), (40, 8, 14336, 4096, 240), (39, 8, 7168, 4096, 320), (40, 8, 7168, 4096, 240), (330, 8, 14336, 4096, 240),
                                          (331, 8, 14336, 4096, 320), (256, 32, 7168, 4096, 240), (257, 32, 7168, 4096, 320), (130, 4, 1024, 1024, 320), (400, 32, 2048, 2048, 240),
                                          (254, 128, 768, 2048, 240), (258, 128, 768, 2048, 320)):
        assert K.moe_weight_bound(rows * experts, experts, up, down)[0] == most, (rows, experts)
    assert K.moe_weight_bound(8 * 130, 8, 14336, 4096) == (240, 4) and K.moe_weight_bound(64 * 130, 64, 1408, 2048) == (240, 2)
    assert K.moe_weight_bound(6000, 8, 14336, 4096) == (320, 2)
    for pairs, experts, up, down in ((8 * 479, 8, 14336, 4096), (8 * 1281, 8, 14336, 4096), (8 * 750, 8, 7168, 4096)):
        assert K.moe_weight_bound(pairs, experts, up, down) == (320, 0)


def test_from_how_many_rows_on():
    """Few column tiles of few experts, and a short K of the down projection, from 50 rows an expert on; others from 40."""
    for experts, up, down, least in ((8, 4096, 6144, 50), (8, 3584, 4096, 50), (96, 384, 4096, 50), (16, 2048, 7168, 40), (16, 2048, 2048, 40), (4, 14336, 4096, 40), (60, 1408, 2048, 40)):
        assert K.moe_weight_bound((least - 1) * experts, experts, up, down)[1] == 0 and K.moe_weight_bound(least * experts, experts, up, down)[0] == 240


def test_copies_of_the_rows_are_bounded():
    """fp32 copies that the parts of the down projection take: 256 MiB with tiles of 240 rows, 320 with tiles of 320; one copy, as the other tiles have, without a bound."""
    seen = set()
    for experts in (4, 8, 16, 32, 64, 100, 128, 200):
        for up in (384, 768, 1408, 2048, 4096, 7168, 8192, 14336, 20480):
            for down in (1024, 2048, 4096, 6144, 8192):
                for rows in (40, 56, 130, 240, 241, 330, 400, 480, 481, 640, 960, 1280):
                    most, parts = K.moe_weight_bound(rows * experts, experts, up, down)
                    if parts > 1:
                        seen.add((most, parts))
                        assert parts * rows * experts * down * 4 <= (256 if most == 240 else 320) << 20, (experts, up, down, rows)
    assert {(240, 2), (240, 4), (320, 2)} <= seen


def test_no_more_parts_than_steps():
    """A part of K has a step of 64 at least (sgl_amd_moe_rows_gemm refuses others): intermediate sizes of few steps over all that the rule takes."""
    taken = 0
    for experts in (64, 112, 128, 160, 192, 220):
        for up in (64, 128, 192, 256, 320):
            for down in (64, 256, 512, 1024, 2048):
                for rows in (40, 56, 90, 130, 250):
                    most, parts = K.moe_weight_bound(rows * experts, experts, up, down)
                    taken += parts > 0
                    assert parts <= up // 64, (experts, up, down, rows)
    assert taken > 20


@pytest.mark.gpu
def test_a_layer_of_three_steps():
    """128 experts of 192 / 512 with 56 rows: four parts would suit its tiles, its K has three steps."""
    g = torch.Generator().manual_seed(11)
    M, E, N, H, top = 896, 128, 192, 512, 8
    x = torch.randn((M, H), generator=g).to(BF).cuda()
    w13, w2 = (torch.randn((E, 2 * N, H), generator=g) * 0.05).to(BF).cuda(), (torch.randn((E, H, N), generator=g) * 0.05).to(BF).cuda()
    tw, ids = torch.randn((M, E), generator=g).softmax(-1).topk(top)
    tw, ids = tw.float().contiguous().cuda(), ids.int().contiguous().cuda()
    assert K.moe_weight_bound(M * top, E, N, H)[1] > 0
    got, want = K.fused_experts(x, w13, w2, tw, ids), torch.zeros((M, H), dtype=torch.float64, device="cuda")
    for i in range(E):
        tok, k = (ids == i).nonzero(as_tuple=True)
        gu = x[tok].double() @ w13[i].double().T.contiguous()
        want.index_add_(0, tok, (torch.nn.functional.silu(gu[:, :N]) * gu[:, N:]) @ w2[i].double().T.contiguous() * tw[tok, k].double()[:, None])
    # bf16 roundings of gate and activation, of their product, of a pair's row and of the result, 2^-9 each
    assert float((got.double() - want).norm() / want.norm()) < 5 * 2.0 ** -9


def _pairs(loads, topk, g):
    """Pairs of every expert in no order, `topk` a token."""
    ids = torch.repeat_interleave(torch.arange(len(loads)), torch.tensor(loads))
    return ids[torch.randperm(ids.numel(), generator=g)].to(torch.int32).view(-1, topk).cuda()


def _estimate(loads, N, Kd, most, max_parts, gated):
    """(parts of K, tiles of a part) that the kernel chooses for a product: the number of units of 16 rows and of parts whose rounds of tiles over 256 compute units take least."""
    best, nk, cols = None, Kd // 64, -(-N // (128 if gated else 256))
    units = [-(-n // 16) for n in loads if n]
    for m in range(most // 16, most // 32 - 1, -1):
        tiles = [-(-u // m) for u in units]
        fullest = max(-(-u // t) for u, t in zip(units, tiles))
        step = max(12 + fullest * 3 // 4 if most == 240 else 24, fullest + 9)
        for n in range(1, max(1, max_parts) + 1):
            rounds = -(-sum(tiles) * cols * n // 256)
            cost = rounds * -(-nk // n) * step + (n - 1) * int(3e-5 * sum(loads) * N) if max_parts else rounds * step
            if best is None or cost < best[0]:
                best = cost, n, sum(tiles) * cols
    return best[1:]


@pytest.mark.gpu
@pytest.mark.parametrize("most", [240, 320])
@pytest.mark.parametrize("loads,N,Kd", [((1, 16, 17, 0), 64, 64), ((239, 240, 241, 2), 320, 128), ((15, 241, 480, 481), 288, 192), ((225, 224, 0, 33), 576, 512),
                                        ((320, 321, 640, 7), 256, 832)])
def test_products_of_few_rows(most, loads, N, Kd):
    g = torch.Generator().manual_seed(sum(loads) + N)
    E, numel = len(loads), sum(loads)
    ids = _pairs(loads, 2 if numel % 2 == 0 else 1, g)
    M, topk = ids.shape
    flat = ids.flatten().long()
    s, e, post = K.moe_align_block_size(ids, 256, E)
    x = torch.randn((M, Kd), generator=g).to(BF).cuda()
    rows = x[torch.arange(numel, device="cuda") // topk]
    # gated up projection: the activation's argument is one fp32 sum, its value rounded to bf16 twice (2^-8 of it each) and once more with `up`
    w13 = (torch.randn((E, 2 * N, Kd), generator=g) * 0.05).to(BF).cuda()
    up = torch.empty((numel, N), dtype=BF, device="cuda")
    K.moe_rows_gemm(x, w13, up, s, e, post, topk, numel, most, act=K.SILU)
    want = torch.empty((numel, 2 * N), dtype=torch.float64, device="cuda")
    for i in range(E):
        want[flat == i] = rows[flat == i].double() @ w13[i].double().T.contiguous()
    want = torch.nn.functional.silu(want[:, :N]) * want[:, N:]
    assert bool(((up.double() - want).abs() <= 2.0 ** -6 * want.abs() + 1e-3).all())
    # parts of K: fp32 sums of Kd products in any order
    w2 = (torch.randn((E, N, Kd), generator=g) * 0.05).to(BF).cuda()
    want, bound = torch.empty((numel, N), dtype=torch.float64, device="cuda"), torch.empty((numel, N), dtype=torch.float64, device="cuda")
    for i in range(E):
        want[flat == i] = rows[flat == i].double() @ w2[i].double().T.contiguous()
        bound[flat == i] = rows[flat == i].double().abs() @ w2[i].double().abs().T.contiguous() * (Kd + 4) * 2.0 ** -24
    tw = torch.rand((M, topk), generator=g).cuda()
    for most_parts in {1, min(4, Kd // 64)}:
        parts = torch.full((most_parts, numel, N), float("nan"), device="cuda")
        splits = torch.zeros(1, dtype=torch.int32, device="cuda")
        K.moe_rows_gemm(x, w2, parts, s, e, post, topk, numel, most, splits=splits)
        n = int(splits)
        assert n == _estimate(loads, N, Kd, most, most_parts, False)[0] and (n > 1 or most_parts == 1)
        assert bool(((parts[:n].double().sum(0) - want).abs() <= bound).all())
        out = torch.empty((M, N), dtype=BF, device="cuda")
        K.moe_sum_parts(parts, splits, tw, out, 0.5)
        total = parts[0].clone()
        for i in range(1, n):
            total += parts[i]
        acc = torch.zeros((M, N), device="cuda")
        for k in range(topk):
            acc += total.to(BF).float().view(M, topk, N)[:, k] * tw[:, k:k + 1]
        assert torch.equal(out, (acc * 0.5).to(BF))


@pytest.mark.gpu
@pytest.mark.parametrize("most", [240, 320])
@pytest.mark.parametrize("loads,N,Kd,cut", [((500, 3, 239, 241, 0, 322, 97, 16), 9024, 64, False), ((500, 3, 239, 241, 0, 322, 97, 16), 9024, 128, False),
                                            ((130, 641, 33, 0, 240, 480, 15, 320), 9024, 192, False), ((700, 650, 0, 5, 720), 9220, 448, False),
                                            ((30, 17, 0, 48, 16, 5), 7684, 4160, True), ((100, 17, 260, 0, 48, 5), 6404, 4160, True)])
def test_workgroups_that_take_several_tiles(most, loads, N, Kd, cut):
    """More tiles than compute units, of uneven experts and of output columns that fill no tile: the next tile's stages behind steps of one, two and three and of odd counts, and from a
    part of K to the next, which is not as long."""
    g = torch.Generator(device="cuda").manual_seed(sum(loads) + N + Kd)
    E, numel = len(loads), sum(loads)
    ids = _pairs(loads, 1, torch.Generator().manual_seed(numel))
    flat = ids.flatten().long()
    s, e, post = K.moe_align_block_size(ids, 256, E)
    x = torch.randn((numel, Kd), generator=g, device="cuda").to(BF)
    if N % 32 == 0:
        parts, tiles = _estimate(loads, N, Kd, most, 0, True)
        assert tiles > 256
        w13 = (torch.randn((E, 2 * N, Kd), generator=g, device="cuda") * 0.05).to(BF)
        up = torch.empty((numel, N), dtype=BF, device="cuda")
        K.moe_rows_gemm(x, w13, up, s, e, post, 1, numel, most, act=K.SILU)
        for i in range(E):
            gu = x[flat == i].double() @ w13[i].double().T.contiguous()
            want = torch.nn.functional.silu(gu[:, :N]) * gu[:, N:]
            assert bool(((up[flat == i].double() - want).abs() <= 2.0 ** -6 * want.abs() + 1e-3).all()), i
        del w13
    w2 = (torch.randn((E, N, Kd), generator=g, device="cuda") * 0.05).to(BF)
    most_parts = min(4, Kd // 64)
    out = torch.full((most_parts, numel, N), float("nan"), device="cuda")
    splits = torch.zeros(1, dtype=torch.int32, device="cuda")
    K.moe_rows_gemm(x, w2, out, s, e, post, 1, numel, most, splits=splits)
    n = int(splits)
    want_n, tiles = _estimate(loads, N, Kd, most, most_parts, False)
    assert n == want_n and tiles * n > 256 and (n > 1) == cut, (n, want_n, tiles)
    got = out[:n].double().sum(0)
    for i in range(E):
        a, w = x[flat == i].double(), w2[i].double().T.contiguous()
        assert bool(((got[flat == i] - a @ w).abs() <= a.abs() @ w.abs() * (Kd + 4) * 2.0 ** -24).all()), i


@pytest.mark.gpu
@pytest.mark.parametrize("M,E,N,H,plan", [(520, 8, 7168, 1024, (240, 4)), (2003, 8, 10240, 512, (320, 2)), (1530, 16, 2048, 768, (240, 4))])
def test_layers_that_take_these_tiles(M, E, N, H, plan):
    """fused_experts by its own rule, against 64 bits."""
    g = torch.Generator(device="cuda").manual_seed(M)
    x = torch.randn((M, H), generator=g, device="cuda").to(BF)
    w13, w2 = (torch.randn((E, 2 * N, H), generator=g, device="cuda") * 0.03).to(BF), (torch.randn((E, H, N), generator=g, device="cuda") * 0.03).to(BF)
    tw, ids = (torch.randn((M, E), generator=g, device="cuda") + torch.randn((1, E), generator=g, device="cuda") * 0.5).softmax(-1).topk(2)
    tw, ids = tw.float().contiguous(), ids.int().contiguous()
    assert K.moe_weight_bound(2 * M, E, N, H) == plan
    got, want = K.fused_experts(x, w13, w2, tw, ids, 0.5), torch.zeros((M, H), dtype=torch.float64, device="cuda")
    for i in range(E):
        tok, k = (ids == i).nonzero(as_tuple=True)
        gu = x[tok].double() @ w13[i].double().T.contiguous()
        want.index_add_(0, tok, (torch.nn.functional.silu(gu[:, :N]) * gu[:, N:]) @ w2[i].double().T.contiguous() * tw[tok, k].double()[:, None] * 0.5)
    # bf16 roundings of gate and activation, of their product, of a pair's row and of the result, 2^-9 each
    assert float((got.double() - want).norm() / want.norm()) < 5 * 2.0 ** -9
    assert torch.equal(got, K.fused_experts(x, w13, w2, tw, ids, 0.5))


@pytest.mark.gpu
@pytest.mark.parametrize("form", ["rows_of_out", "columns_of_out", "rows_of_ids", "stride_of_out"])
def test_what_the_other_tiles_take_or_refuse(form):
    """Outputs, ids and weights with more rows than there are tokens, as padded buffers have, and an output whose rows are not 16 bytes apart."""
    g = torch.Generator().manual_seed(12)
    M, E, N, H, top = 250, 8, 3584, 256, 2
    x = torch.randn((M, H), generator=g).to(BF).cuda()
    w13, w2 = (torch.randn((E, 2 * N, H), generator=g) * 0.05).to(BF).cuda(), (torch.randn((E, H, N), generator=g) * 0.05).to(BF).cuda()
    tw, ids = torch.randn((M + 9, E), generator=g).softmax(-1).topk(top)
    tw, ids = tw.float().contiguous().cuda(), ids.int().contiguous().cuda()
    assert K.moe_weight_bound(M * top, E, N, H)[1] > 0
    want = K.fused_experts(x, w13, w2, tw[:M].contiguous(), ids[:M].contiguous()).float()
    if form == "stride_of_out":
        with pytest.raises(RuntimeError, match="multiples of 8"):
            K.fused_experts(x, w13, w2, tw[:M].contiguous(), ids[:M].contiguous(), out=torch.empty((M, H + 4), dtype=BF, device="cuda")[:, :H])
        return
    if form == "rows_of_ids":
        got = K.fused_experts(x, w13, w2, tw, ids)
    else:
        out = torch.full((M + (5 if form == "rows_of_out" else 0), H + (8 if form == "columns_of_out" else 0)), 7.0, dtype=BF, device="cuda")
        got = K.fused_experts(x, w13, w2, tw[:M].contiguous(), ids[:M].contiguous(), out=out)
        assert got is out and bool((out[M:] == 7).all()) and bool((out[:, H:] == 7).all())
        got = got[:M, :H]
    d = (got.float() - want).abs()                     # (other tiles: an ulp where one of three roundings falls the other way)
    assert float((d > 2.0 ** -7 * want.abs() + 1e-3).float().mean()) < 1e-3


@pytest.mark.gpu
@pytest.mark.parametrize("override", [(240, 4), (320, 2)])
def test_the_layer_agrees_with_the_other_tiles(monkeypatch, override):
    """Same products, other order of their fp32 sums: bf16 results differ by an ulp where one of three roundings falls the other way."""
    g = torch.Generator().manual_seed(3)
    M, E, N, H = 500, 8, 768, 1024
    x = torch.randn((M, H), generator=g).to(BF).cuda()
    w13, w2 = (torch.randn((E, 2 * N, H), generator=g) * 0.03).to(BF).cuda(), (torch.randn((E, H, N), generator=g) * 0.03).to(BF).cuda()
    tw, ids = torch.randn((M, E), generator=g).softmax(-1).topk(2)
    tw, ids = tw.float().contiguous().cuda(), ids.int().contiguous().cuda()
    monkeypatch.setattr(K, "MOE_TILE_OVERRIDE", (128, 128, 128))
    base = K.fused_experts(x, w13, w2, tw, ids).float()
    monkeypatch.setattr(K, "MOE_PARTS_OVERRIDE", override)
    d = (K.fused_experts(x, w13, w2, tw, ids).float() - base).abs()
    assert float((d > 2.0 ** -7 * base.abs() + 1e-3).float().mean()) < 1e-3
