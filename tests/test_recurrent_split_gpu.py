"""The chunked recurrences of 16-bit activations on the bf16 matrix cores (three-piece operands): edges of chunks, tiles and columns,
states that must stay as exact as fp32, and agreement with the general kernels, which rows at odd addresses take."""
import math

import pytest
import torch

from oracle import hybrid as oh
from sglang_amd import kernels, native
from test_hybrid_kernels_gpu import _err, _segments

pytestmark = pytest.mark.gpu
BF = torch.bfloat16
LENS = [1, 15, 16, 31, 32, 33, 63, 64, 65, 97, 128, 130, 200]


def _state_want(rule, S, seq, A_log, bias, heads, groups, K, V):
    """The state behind one segment in 64 bits, token by token."""
    S = S.double()
    for act, gates in zip(*(t.double() for t in seq)):
        if rule == "mamba2":
            x, B = act[:heads * V].view(heads, V), act[heads * V:heads * V + groups * K].view(groups, K).repeat_interleave(heads // groups, 0)
            dt = oh.softplus(gates[:heads] + bias.double())
            S = S * torch.exp(-torch.exp(A_log.double()) * dt)[:, None, None] + (dt[:, None] * B)[:, :, None] * x[:, None, :]
        else:
            k = oh.unit(act[groups * K:2 * groups * K].view(groups, K)).repeat_interleave(heads // groups, 0)
            v, beta = act[2 * groups * K:].view(heads, V), torch.sigmoid(gates[:heads])
            S = S * torch.exp(-torch.exp(A_log.double()) * oh.softplus(gates[heads:] + bias.double()))[:, None, None]
            S = S + k[:, :, None] * (beta[:, None] * (v - (k[:, None, :] @ S)[:, 0]))[:, None, :]
    return S


@pytest.mark.parametrize("rule", ["mamba2", "delta"])
@pytest.mark.parametrize("heads,groups,K,V,decay", [(2, 1, 128, 128, 0.0), (4, 2, 64, 64, 0.0), (2, 2, 32, 16, 0.0), (3, 3, 40, 24, -1.0), (2, 1, 72, 136, -2.0),
                                                    (4, 2, 8, 8, 0.5), (2, 1, 104, 72, 4.0)])
def test_split_recurrence(device, rule, heads, groups, K, V, decay):
    """decay 4: sixteen tokens fall by far more than e^60 (exponentials taken one by one).  Odd segments repeat their keys; every second
    one continues a state.  Outputs: one 16-bit rounding, as the general forms' bar.  States: fp32 sums of up to 200 terms, 4e-6 of the
    largest (2^-24 sqrt(200) per element, times the few operations of a term)."""
    g = torch.Generator().manual_seed(heads * K + V)
    T = sum(LENS)
    width = heads * V + 2 * groups * K
    act, gates = torch.randn(T, width, generator=g).to(BF), torch.randn(T, 2 * heads, generator=g).to(BF)
    keys = slice(heads * V, heads * V + groups * K) if rule == "mamba2" else slice(groups * K, 2 * groups * K)
    at, spans, pos = 0, [], []
    for i, n in enumerate(LENS):
        if i % 2:
            act[at:at + n, keys] = act[at, keys]
        spans.append((at, at + n))
        pos.append(torch.arange(n) + (7 if i % 2 == 0 else 0))
        at += n
    A_log, bias, D = torch.randn(heads, generator=g) * 0.5 + decay, torch.randn(heads, generator=g) * 0.5 - 1.0, torch.randn(heads, generator=g)
    state0 = torch.randn(len(LENS) + 1, heads, K, V, generator=g) * 0.3
    slots = torch.randperm(len(LENS), generator=g) + 1
    seg, pos = _segments(LENS, device), torch.cat(pos).to(device)
    dev = [t.to(device) for t in (A_log, bias, D)]

    def run(rows, gate):
        state = state0.to(device)
        if rule == "mamba2":
            y = kernels.mamba2_scan(rows, gate[:, :heads], *dev, state, slots.to(device), pos, seg, groups, form="chunk")
        else:
            y = kernels.gated_delta_scan(rows, gate[:, :heads], gate[:, heads:], *dev[:2], state, slots.to(device), pos, seg, groups, K ** -0.5, form="chunk")
        return y, state

    y, state = run(act.to(device), gates.to(device))
    odd = torch.zeros(T, width + 9, dtype=BF, device=device)
    odd[:, 1:1 + width] = act.to(device)
    y0, general = run(odd[:, 1:1 + width], gates.to(device))             # rows at odd addresses: the general kernel
    assert _err(y, y0.cpu()) < 1.2e-2 and torch.equal(state[0].cpu(), state0[0])
    for i, (lo, hi) in enumerate(spans):
        start = state0[slots[i]] if i % 2 == 0 else torch.zeros(heads, K, V)
        want = _state_want(rule, start, (act[lo:hi], gates[lo:hi]), A_log, bias, heads, groups, K, V)
        scale = want.abs().max()
        off = (state[slots[i]].double().cpu() - want).abs().max() / scale
        assert off < 4e-6, (i, float(off), float((general[slots[i]].double().cpu() - want).abs().max() / scale))


def _one_term(device, n, fall, seed):
    """(split kernel's, general kernel's) relative errors of products (inverse) x (right-hand side) alone.  Only token n - 2 has a value, so U of
    token n - 1 is one such product; its key reaches into the upper half of the head dim, where no other token's does, and the state there
    holds that product times the (exact) key.  The keys' lengths are powers of two: what is left is the gates' and the product's."""
    g = torch.Generator().manual_seed(seed)
    B, heads, groups, K, V = 64, 8, 8, 64, 64
    act = torch.randn(B, n, 2 * groups * K + heads * V, generator=g)
    k = act[:, :, groups * K:2 * groups * K].view(B, n, groups, K)
    k.zero_()
    k[:, :n - 1, :, :16] = 256.0
    k[:, n - 1, :, 8:16] = 256.0
    k[:, n - 1, :, 32:40] = torch.randint(0, 2, (B, groups, 8), generator=g) * 512.0 - 256.0
    act[:, torch.arange(n) != n - 2, 2 * groups * K:] = 0.0
    gates = torch.randn(B, n, 2 * heads, generator=g)
    gates[:, :, heads:] = fall
    gates[:, n - 2:, heads:] = torch.randn(B, min(n, 2), heads, generator=g) - 6.0   # the last two tokens fall by little
    act, gates = act.to(BF), gates.to(BF)
    A_log, bias = torch.zeros(heads), torch.zeros(heads)
    want = torch.stack([_state_want("delta", torch.zeros(heads, K, V), (act[b], gates[b]), A_log, bias, heads, groups, K, V) for b in range(B)])[:, :, 32:40]
    pos, rows = torch.arange(n).repeat(B).to(device), torch.zeros(B * n, act.shape[-1] + 9, dtype=BF, device=device)
    out = []
    for odd in (0, 1):                                                               # (rows at odd addresses: the general kernel)
        x = rows[:, odd:odd + act.shape[-1]]
        x.copy_(act.flatten(0, 1))
        x = x if odd else x.contiguous()
        state, gt = torch.zeros(B, heads, K, V, device=device), gates.flatten(0, 1).to(device)
        kernels.gated_delta_scan(x, gt[:, :heads], gt[:, heads:], A_log.to(device), bias.to(device), state, torch.arange(B, device=device), pos,
                                 _segments([n] * B, device), groups, K ** -0.5, form="chunk")
        err = (state[:, :, 32:40].cpu().double() - want) / want
        out.append((float(err.mean()) * 2.0 ** 24, float(err.abs().max()) * 2.0 ** 24))
    return out


def test_products_of_pieces_do_not_shrink(device):
    """Mean relative error over 512 independent products, in units of 2^-24: that of the general kernel, whose products are fp32 (roundings of
    gates and products are a few units each, their means agree to 0.1).  Terms left out of a product of truncated pieces all have its sign:
    0.7 on average without m l and l m."""
    (mean, big), (mean0, big0) = _one_term(device, 2, 0.0, 1)
    assert abs(mean - mean0) < 0.15 and big < big0 + 2.0, (mean, mean0, big, big0)


@pytest.mark.parametrize("n,fall", [(16, 3.9), (16, 2.0), (16, 0.5), (32, 3.9)])
def test_decays_between_neighbours_behind_a_steep_fall(device, n, fall):
    """The decay between the last two tokens, e^-0.003, is a product of two exponentials whose exponents are the whole tile's fall (up to e^56).
    Largest relative error in units of 2^-24: that of the general kernel, which takes one exponential, and two for the other factor and the
    product's rounding, plus what products of pieces leave out (7)."""
    (_, big), (_, big0) = _one_term(device, n, fall, 1)
    assert big < big0 + 9.0, (big, big0)


@pytest.mark.parametrize("rule", ["mamba2", "delta"])
def test_gates_whose_falls_leave_the_floats(device, rule):
    """A fall of 3e38 a token: everything in front is forgotten, the sums of the falls lie beyond the largest float, nothing becomes NaN."""
    g = torch.Generator().manual_seed(3)
    heads, groups, K, V, T = 2, 1, 64, 64, 150
    act, gates = torch.randn(T, heads * V + 2 * groups * K, generator=g).to(BF), torch.randn(T, 2 * heads, generator=g).to(BF)
    gates[20:T:7] = 3.0e38
    A_log, bias, D = torch.zeros(heads), torch.zeros(heads), torch.zeros(heads)
    if rule == "mamba2":                                        # (its values are scaled by the same gates)
        act[:, :heads * V] *= 1e-20
        act[:, heads * V:] *= 1e-15
    ref = None
    for odd in (1, 0):
        rows = torch.zeros(T, act.shape[1] + 9, dtype=BF, device=device)[:, odd:odd + act.shape[1]]
        rows.copy_(act)
        rows = rows if odd else rows.contiguous()
        state, gt, seg, pos = torch.zeros(1, heads, K, V, device=device), gates.to(device), _segments([T], device), torch.arange(T, device=device)
        par = [t.to(device) for t in (A_log, bias, D)]
        if rule == "mamba2":
            y = kernels.mamba2_scan(rows, gt[:, :heads], *par, state, torch.zeros(1, dtype=torch.int64, device=device), pos, seg, groups, form="chunk")
        else:
            y = kernels.gated_delta_scan(rows, gt[:, :heads], gt[:, heads:], *par[:2], state, torch.zeros(1, dtype=torch.int64, device=device), pos, seg, groups,
                                         K ** -0.5, form="chunk")
        assert bool(y.isfinite().all()) and bool(state.isfinite().all()), odd
        if odd:
            ref = y.cpu()
    if rule == "delta":                                         # (Mamba-2: chunks of 64 here and 32 there, and small falls behind 1e38 are lost in a chunk's sum)
        assert _err(y, ref) < 1.2e-2                            # one 16-bit rounding, as the other outputs here


def _one_token_states(device, B, x, gate, dim):
    """Mamba-2 states behind one token each, from the split kernel and from the general one (rows at odd addresses)."""
    n, heads, V = x.shape
    act, out = torch.cat([x.flatten(1), B.flatten(1), torch.zeros(n, dim).to(BF)], 1), []
    zero, pos = torch.zeros(heads, device=device), torch.zeros(n, dtype=torch.int64, device=device)
    for odd in (0, 1):
        rows = torch.zeros(n, act.shape[1] + 9, dtype=BF, device=device)[:, odd:odd + act.shape[1]]
        rows.copy_(act)
        state = torch.zeros(n, heads, dim, V, device=device)
        kernels.mamba2_scan(rows if odd else rows.contiguous(), gate.to(device), zero, zero, zero, state, torch.arange(n, device=device), pos,
                            _segments([1] * n, device), 1, form="chunk")
        out.append(state.cpu())
    return out


def test_pieces_of_a_product_add_up_to_it(device):
    """The state behind one token is B (dt x): for B of powers of two the pieces of dt x leave exactly the float that the general kernel has."""
    g = torch.Generator().manual_seed(2)
    n, heads, K, V = 40, 4, 64, 64
    B = torch.exp2(torch.randint(-3, 4, (n, 1, K), generator=g).float()).to(BF)
    x, gate = torch.randn(n, heads, V, generator=g).to(BF), torch.randn(n, heads, generator=g).to(BF)
    split, general = _one_token_states(device, B, x, gate, K)
    assert torch.equal(split, general)


@pytest.mark.parametrize("rule", ["mamba2", "delta"])
def test_long_memory_of_one_sign(device, rule):
    """2500 tokens of positive values that are hardly forgotten: what every chunk's addition loses is lost with the state's sign and adds up.
    The relative error of the state (2-norm) is no larger than the general kernel's, whose sums are fp32 products one after the other."""
    g = torch.Generator().manual_seed(8)
    heads, groups, K, V, T = 4, 1, 128, 64, 2500
    act = (torch.randn(T, heads * V + 2 * groups * K, generator=g).abs() + 0.05).to(BF)
    gates = torch.randn(T, 2 * heads, generator=g).to(BF)
    A_log, bias, D = torch.full((heads,), -6.0), torch.full((heads,), -3.0), torch.zeros(heads)
    want = _state_want(rule, torch.zeros(heads, K, V), (act, gates), A_log, bias, heads, groups, K, V)
    errs = []
    for odd in (0, 1):
        rows = torch.zeros(T, act.shape[1] + 9, dtype=BF, device=device)[:, odd:odd + act.shape[1]]
        rows.copy_(act)
        rows, state, gt = rows if odd else rows.contiguous(), torch.zeros(1, heads, K, V, device=device), gates.to(device)
        slot, pos, seg, par = torch.zeros(1, dtype=torch.int64, device=device), torch.arange(T, device=device), _segments([T], device), [t.to(device) for t in (A_log, bias, D)]
        if rule == "mamba2":
            kernels.mamba2_scan(rows, gt[:, :heads], *par, state, slot, pos, seg, groups, form="chunk")
        else:
            kernels.gated_delta_scan(rows, gt[:, :heads], gt[:, heads:], *par[:2], state, slot, pos, seg, groups, K ** -0.5, form="chunk")
        errs.append(float((state[0].cpu().double() - want).norm() / want.norm()))
    assert errs[0] <= errs[1], errs


@pytest.mark.parametrize("rule", ["mamba2", "delta"])
@pytest.mark.parametrize("bad", [float("nan"), float("inf"), float("-inf")])
def test_values_that_are_no_numbers_reach_no_further(device, rule, bad):
    """One NaN or infinity in a row of one segment, in any input, at places around the borders of tiles and chunks: the outputs and states that
    are not finite are the general kernel's (its tile of 16 tokens, what follows, the state), and the rest is what it is without it."""
    g = torch.Generator().manual_seed(6)
    heads, groups, K, V, n = 2, 1, 64, 32, 150
    places = [0, 3, 15, 16, 30, 31, 32, 47, 50, 63, 64, 100, 149]
    inputs = ["value", "key", "query", "gate"] + ["beta"] * (rule == "delta")
    T = n * len(places) * len(inputs)
    act, gates = torch.randn(T, heads * V + 2 * groups * K, generator=g).to(BF), torch.randn(T, 2 * heads, generator=g).to(BF)
    spoilt, sgates, at = act.clone(), gates.clone(), 0
    cols = dict(value=5, key=heads * V + 9, query=heads * V + groups * K + 9) if rule == "mamba2" else dict(value=2 * groups * K + 5, key=groups * K + 9, query=9)
    for what in inputs:
        for p in places:
            if what in cols:
                spoilt[at + p, cols[what]] = bad
            else:
                sgates[at + p, heads if (what == "gate") == (rule == "delta") else 0] = bad
            at += n
    segs = len(places) * len(inputs)
    A_log, bias, D = torch.zeros(heads), torch.zeros(heads), torch.ones(heads)
    slots, pos, seg, par = torch.arange(segs, device=device), torch.arange(n).repeat(segs).to(device), _segments([n] * segs, device), [t.to(device) for t in (A_log, bias, D)]

    def run(a, gt, odd):
        rows = torch.zeros(T, a.shape[1] + 9, dtype=BF, device=device)[:, odd:odd + a.shape[1]]
        rows.copy_(a)
        rows, state, gt = rows if odd else rows.contiguous(), torch.zeros(segs, heads, K, V, device=device), gt.to(device)
        if rule == "mamba2":
            y = kernels.mamba2_scan(rows, gt[:, :heads], *par, state, slots, pos, seg, groups, form="chunk")
        else:
            y = kernels.gated_delta_scan(rows, gt[:, :heads], gt[:, heads:], *par[:2], state, slots, pos, seg, groups, K ** -0.5, form="chunk")
        return y.view(segs, n, -1).cpu(), state.cpu()

    (y, state), (y0, state0), (clean, clean_state) = run(spoilt, sgates, 0), run(spoilt, sgates, 1), run(act, gates, 0)
    for i in range(segs):
        where = (inputs[i // len(places)], places[i % len(places)])
        assert torch.equal(y[i].isfinite(), y0[i].isfinite()), where
        assert torch.equal(state[i].isfinite(), state0[i].isfinite()), where
        ok, sok = y[i].isfinite(), state[i].isfinite()
        assert torch.equal(y[i][ok & (torch.arange(n)[:, None] < where[1])], clean[i][ok & (torch.arange(n)[:, None] < where[1])]), where
        assert _err(y[i][ok], y0[i][ok]) < 1.2e-2 if ok.any() else True, where
        assert _err(state[i][sok], state0[i][sok]) < 1e-4 if sok.any() else True, where


def test_rows_longer_than_the_floats(device):
    """A key or query of finite elements whose squared length is infinite counts as zero (1 / sqrt(inf)), as in the general kernel."""
    g = torch.Generator().manual_seed(7)
    heads, groups, K, V, T = 2, 1, 64, 32, 150
    act, gates = torch.randn(T, 2 * groups * K + heads * V, generator=g).to(BF), torch.randn(T, 2 * heads, generator=g).to(BF)
    act[[5, 100], :K] = 3.0e19                                  # queries (not in one chunk with such a key in front: their product is infinite)
    act[[20, 64, 130], K:2 * K] = -4.0e19                       # keys
    A_log, bias, out = torch.zeros(heads, device=device), torch.zeros(heads, device=device), []
    for odd in (0, 1):
        rows = torch.zeros(T, act.shape[1] + 9, dtype=BF, device=device)[:, odd:odd + act.shape[1]]
        rows.copy_(act)
        state, gt = torch.zeros(1, heads, K, V, device=device), gates.to(device)
        y = kernels.gated_delta_scan(rows if odd else rows.contiguous(), gt[:, :heads], gt[:, heads:], A_log, bias, state, torch.zeros(1, dtype=torch.int64, device=device),
                                     torch.arange(T, device=device), _segments([T], device), groups, K ** -0.5, form="chunk")
        assert bool(y.isfinite().all()) and bool(state.isfinite().all()), odd
        out.append((y.cpu(), state.cpu()))
    assert _err(out[0][0], out[1][0]) < 1.2e-2 and _err(out[0][1], out[1][1]) < 1e-4


@pytest.mark.parametrize("dt,fall", [(1e15, 3.7), (1e12, 3.9), (1e30, 0.5), (1e11, 3.7)])
def test_steps_so_long_that_a_factor_leaves_the_floats(device, dt, fall):
    """dt is part of the second factor of a decay on the diagonal, which may be e^60 already: sixteen falls of 3.7 at dt = 1e15 are 8e38."""
    g = torch.Generator().manual_seed(9)
    heads, groups, K, V, T = 2, 1, 64, 32, 150
    act, gates = torch.randn(T, heads * V + 2 * groups * K, generator=g).to(BF), torch.full((T, heads), dt).to(BF)
    A_log, zero, out = torch.full((heads,), math.log(fall / dt), device=device), torch.zeros(heads, device=device), []
    for odd in (0, 1):
        rows = torch.zeros(T, act.shape[1] + 9, dtype=BF, device=device)[:, odd:odd + act.shape[1]]
        rows.copy_(act)
        state = torch.zeros(1, heads, K, V, device=device)
        y = kernels.mamba2_scan(rows if odd else rows.contiguous(), gates.to(device), A_log, zero, zero, state, torch.zeros(1, dtype=torch.int64, device=device),
                                torch.arange(T, device=device), _segments([T], device), groups, form="chunk")
        assert bool(y.isfinite().all()) and bool(state.isfinite().all()), odd
        out.append((y.cpu(), state.cpu()))
    assert _err(out[0][0], out[1][0]) < 1.2e-2 and _err(out[0][1], out[1][1]) < 1e-4


def test_rule_of_two_launches():
    """Where the first launch pays: from so many chunks of the longest segment on, fewer where workgroups stand behind each other."""
    size = native.lib().sgl_amd_delta_chunk_workspace
    assert size(1500, 1, 1500, 32, 128, 128) == (1500 // 32 + 1) * 32 * 10240
    for args, two in (((288, 1, 288, 32, 128, 128), True), ((256, 1, 256, 32, 128, 128), False), ((8 * 33, 8, 33, 32, 128, 128), True), ((4 * 33, 4, 33, 32, 128, 128), False),
                      ((512, 16, 32, 32, 128, 128), True), ((256, 8, 32, 32, 128, 128), False), ((1500, 1, 1500, 32, 136, 128), False), ((0, 1, 1500, 32, 128, 128), False),
                      ((200000, 4, 50000, 32, 128, 128), False)):
        assert (size(*args) > 0) == two, args


@pytest.mark.parametrize("heads,groups,K,V,decay,copies", [(2, 1, 128, 128, 0.0, 1), (4, 2, 64, 64, 0.0, 1), (2, 2, 32, 16, 0.0, 1), (3, 3, 40, 24, -1.0, 1),
                                                           (2, 1, 72, 136, -2.0, 1), (4, 2, 8, 8, 0.5, 1), (2, 1, 104, 72, 4.0, 1), (7, 7, 128, 64, 0.0, 3), (8, 4, 56, 72, 4.0, 2)])
def test_delta_rule_in_two_launches(device, heads, groups, K, V, decay, copies):
    """The same bars as the one launch (test_split_recurrence), at the edges of chunks, tiles and columns; several copies: more workgroups than compute units.
    A workspace full of NaN: nothing is read that the first launch does not write.  Empty segments change nothing."""
    g = torch.Generator().manual_seed(heads * K + V)
    lens = ([0] + LENS + [0, 300]) * copies
    T, width = sum(lens), heads * V + 2 * groups * K
    act, gates = torch.randn(T, width, generator=g).to(BF), torch.randn(T, 2 * heads, generator=g).to(BF)
    A_log, bias = torch.randn(heads, generator=g) * 0.5 + decay, torch.randn(heads, generator=g) * 0.5 - 1.0
    state0 = torch.randn(len(lens) + 1, heads, K, V, generator=g) * 0.3
    slots = torch.randperm(len(lens), generator=g) + 1
    spans, pos, at = [], [], 0
    for i, n in enumerate(lens):
        if i % 2 and n:
            act[at:at + n, groups * K:2 * groups * K] = act[at, groups * K:2 * groups * K].clone()
        spans.append((at, at + n))
        pos.append(torch.arange(n) + (7 if i % 2 == 0 else 0))
        at += n
    start = torch.tensor([min(lo, T - 1) for lo, _ in spans], dtype=torch.int32, device=device)
    length, pos = torch.tensor(lens, dtype=torch.int32, device=device), torch.cat(pos).to(device)
    dev = [t.to(device) for t in (A_log, bias, slots)]
    gt, stream = gates.to(device), torch.cuda.current_stream().cuda_stream
    units = (T // 32 + len(lens)) * heads * 10240

    def run(rows, two):
        state, o = state0.to(device), torch.full((T, heads * V), 7.0, dtype=BF, device=device)
        a = gt[:, heads:]
        args = (0, rows.data_ptr(), rows.stride(0), gt.data_ptr(), a.data_ptr(), gt.stride(0), dev[0].data_ptr(), dev[1].data_ptr(), state.data_ptr(), dev[2].data_ptr(),
                pos.data_ptr(), start.data_ptr(), length.data_ptr(), o.data_ptr(), o.stride(0), len(lens), heads, groups, K, V, K ** -0.5)
        if two:
            ws = torch.full((units // 2,), float("nan"), dtype=BF, device=device)
            native.call("sgl_amd_delta_chunk_ws", *args, T, max(lens), ws.data_ptr(), units, stream)
        else:
            native.call("sgl_amd_delta_chunk", *args, stream)
        return o, state

    y, state = run(act.to(device), True)
    odd = torch.zeros(T, width + 9, dtype=BF, device=device)
    odd[:, 1:1 + width] = act.to(device)
    y0, general = run(odd[:, 1:1 + width], False)                        # rows at odd addresses: the general kernel
    assert _err(y, y0.cpu()) < 1.2e-2 and torch.equal(state[0].cpu(), state0[0])
    for i, (lo, hi) in enumerate(spans):
        if lo == hi:
            assert torch.equal(state[slots[i]].cpu(), state0[slots[i]])
            continue
        if i >= len(LENS) + 3:                                           # (copies: against the general kernel alone)
            off = (state[slots[i]] - general[slots[i]]).abs().max() / general[slots[i]].abs().max()
            assert off < 8e-6, (i, float(off))
            continue
        begin = state0[slots[i]] if i % 2 == 0 else torch.zeros(heads, K, V)
        want = _state_want("delta", begin, (act[lo:hi], gates[lo:hi]), A_log, bias, heads, groups, K, V)
        off = (state[slots[i]].double().cpu() - want).abs().max() / want.abs().max()
        assert off < 4e-6, (i, float(off), float((general[slots[i]].double().cpu() - want).abs().max() / want.abs().max()))
    # the same bits every time
    again, state2 = run(act.to(device), True)
    assert torch.equal(again, y) and torch.equal(state2, state)


@pytest.mark.parametrize("V,copies", [(128, 1), (72, 1), (128, 70)])
def test_segments_that_the_callers_tokens_leave_no_room_for(device, V, copies):
    """More tokens in the segments than the call says: what has room is computed as ever, the rest has no numbers for outputs (and never the buffer's old ones) and
    keeps its state; by the fetching wave's form and by the one of more workgroups than compute units."""
    heads, K, lens = 2, 64, [64] * copies + [320, 5]
    g = torch.Generator().manual_seed(V + copies)
    T = sum(lens)
    qkv = torch.randn(T, 2 * heads * K + heads * V, generator=g).to(BF).to(device)
    gt = torch.randn(T, 2 * heads, generator=g).to(BF).to(device)
    A_log, bias = (torch.randn(heads, generator=g).to(device) for _ in range(2))
    state0 = torch.randn(len(lens), heads, K, V, generator=g).to(device)
    slots = torch.arange(len(lens), device=device)
    length = torch.tensor(lens, dtype=torch.int32, device=device)
    start = (length.cumsum(0) - length).to(torch.int32)
    pos = torch.cat([torch.arange(n) + 1 for n in lens]).to(device)
    outs = []
    for tokens in (T, 32 * (2 * copies + 3 - len(lens))):                 # (room for all; for three chunks more than the copies have)
        state, o = state0.clone(), torch.full((T, heads * V), 7.0, dtype=BF, device=device)
        units = (tokens // 32 + len(lens)) * heads * 10240
        ws = torch.empty(units, dtype=torch.uint8, device=device)
        native.call("sgl_amd_delta_chunk_ws", 0, qkv.data_ptr(), qkv.stride(0), gt.data_ptr(), gt[:, heads:].data_ptr(), gt.stride(0), A_log.data_ptr(), bias.data_ptr(),
                    state.data_ptr(), slots.data_ptr(), pos.data_ptr(), start.data_ptr(), length.data_ptr(), o.data_ptr(), o.stride(0), len(lens), heads, heads, K, V,
                    K ** -0.5, tokens, max(lens), ws.data_ptr(), units, torch.cuda.current_stream().cuda_stream)
        outs.append((o, state))
    (o, state), (o2, state2) = outs
    assert bool(o.isfinite().all())
    room, at, cut = tokens // 32 + len(lens), 0, []
    for n in lens:
        at += -(-n // 32)
        cut.append(at > room)
    assert any(cut) and not cut[0]
    for i, (lo, n) in enumerate(zip(start.tolist(), lens)):
        if cut[i]:
            assert bool(o2[lo:lo + n].isnan().all()) and torch.equal(state2[i], state0[i]), i
        else:
            assert torch.equal(o2[lo:lo + n], o[lo:lo + n]) and torch.equal(state2[i], state[i]), i
