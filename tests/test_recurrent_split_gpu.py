"""The chunked recurrences of 16-bit activations on the bf16 matrix cores (three-piece operands): edges of chunks, tiles and columns,
states that must stay as exact as fp32, and agreement with the general kernels, which rows at odd addresses take."""
import pytest
import torch

from oracle import hybrid as oh
from sglang_amd import kernels
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
