"""GPU tests of the branches inside the one-call sampler: the division by the temperature through one reciprocal, the single- and the
two-level cut of the candidate lists, one to four softmax ranges a workgroup.  Ids and kept counts must equal those of the two calls
(softmax over the row, then sample from the probabilities) on every row, bit for bit."""
import pytest
import torch

pytestmark = pytest.mark.gpu


# (rows, columns): 4, 2 and 1 ranges a workgroup in 16 groups; ranges joined further for short rows; tails of 1, 2 and 3 columns
@pytest.mark.parametrize("B,V", [(32, 128256), (64, 151936), (128, 128256), (128, 32000), (64, 65537), (128, 40002), (16, 33003), (2, 50257)])
@pytest.mark.parametrize("fp32", [False, True])
def test_one_call_equals_softmax_then_sample(device, B, V, fp32):
    from sglang_amd import kernels as K

    Vp = V + (-V) % 4                                   # (rows start 8- or 16-byte aligned)
    g = torch.Generator(device=device).manual_seed(V + B)
    rn = lambda *s: torch.randn(s, generator=g, device=device)
    lg = rn(B, Vp) * 2.5
    temps = torch.rand((B, 1), generator=g, device=device) + 0.4
    temps[0] = 1.0
    temps[1] = 1.0e-7                                   # below the reciprocal's range
    if B >= 16:
        temps[2] = 3.0e6                                # above it: a flat row
        lg[3] -= 9.0                                    # the cut far (in keys) below the largest: the two-level select, across zero
        lg[4] = -lg[4].abs() * 0.01 - 1e-4              # negative rows
        lg[5, torch.randperm(Vp, generator=torch.Generator().manual_seed(1))[: Vp - 90].to(device)] = -float("inf")   # a masked vocabulary
        lg[6, 1:] = -float("inf")                       # one token left
        lg[7] *= 1e30                                   # quotients near the largest float
        lg[8] = 0.0
        lg[9] = lg[9].abs() * -0.0                      # -0 beside +0
        lg[9, ::3] = 0.0
        lg[10, 17] = float("nan")
        lg[11, 19] = float("inf")
        lg[12] = rn(Vp) * 1e-39                         # denormals
    padded = lg if fp32 else lg.to(torch.bfloat16)
    lg = padded[:, :V]
    top_k = torch.tensor(([50, 1, 64, 40, 1 << 30, 7, 20, 60] * 16)[:B], dtype=torch.int32, device=device)
    top_p = torch.tensor(([0.9, 1.0, 1.0, 0.95, 0.6, 0.999] * 22)[:B], device=device)
    seeds, pos = torch.arange(B, device=device) * 977 + 5, torch.arange(B, device=device)
    for min_p in (None, torch.full((B,), 0.02, device=device)):
        probs = K.softmax_temperature_(padded.clone()[:, :V], temps) if fp32 else K.softmax_temperature_from_bf16(lg, temps)
        want, want_n = K.top_k_top_p_min_p_sample(probs, top_k, top_p, min_p, seeds, pos, return_n_keep=True)
        out = K.sample_from_logits(lg, temps, top_k, top_p, min_p, seeds, pos, return_n_keep=True, return_fallback=True)
        assert out is not None
        got, got_n, redone = out
        same = (got == want) & (got_n == want_n)
        bad = same.logical_not().nonzero().flatten().tolist()
        assert not bad, [(r, int(got[r]), int(want[r]), int(got_n[r]), int(want_n[r]), int(redone[r])) for r in bad]
        usual = [r for r in range(13, B) if int(top_k[r]) <= 64]
        assert not any(redone.tolist()[r] for r in usual)          # gaussian rows are decided by their candidates


@pytest.mark.parametrize("fp32", [False, True])
@pytest.mark.parametrize("V", [101, 41, 130, 203, 515, 959])
@pytest.mark.parametrize("B,splits", [(64, 16), (128, 16), (40, 32), (8, 48), (3, 64)])
def test_short_rows_whose_last_ranges_are_empty(device, B, splits, V, fp32):
    """Ranges are rounded up to four columns, so a short row's last columns may lie in any range of a workgroup.  (The Python entry leaves rows
    below 512 columns a range to the two calls; the native one takes them.)  The largest logit sits in the last column of every second row."""
    from sglang_amd import kernels as K, native

    g = torch.Generator(device=device).manual_seed(V + B)
    Vp = V + (-V) % 4
    padded = torch.randn((B, Vp), generator=g, device=device) * 2.5
    padded[::2, V - 1] = 30.0
    padded = padded if fp32 else padded.to(torch.bfloat16)
    lg = padded[:, :V]
    temps = torch.rand((B, 1), generator=g, device=device) + 0.4
    top_k, top_p = torch.full((B,), 20, dtype=torch.int32, device=device), torch.full((B,), 0.95, device=device)
    seeds, pos = torch.arange(B, device=device) * 977 + 5, torch.arange(B, device=device)
    probs = torch.empty((B, Vp), device=device)
    probs[:, :V] = torch.softmax(lg.float() / temps, dim=-1)
    want, want_n = K.top_k_top_p_min_p_sample(probs[:, :V], top_k, top_p, None, seeds, pos, return_n_keep=True)
    got, got_n = torch.full((B,), -1, dtype=torch.int32, device=device), torch.full((B,), -1, dtype=torch.int32, device=device)
    ws = torch.zeros(native.lib().sgl_amd_sample_from_logits_workspace_bytes(B, splits) // 8 + 2, dtype=torch.int64, device=device)
    scratch = torch.empty((B, Vp), device=device)
    native.call("sgl_amd_top_k_top_p_min_p_sample_from_logits", lg.data_ptr(), int(not fp32), lg.stride(0), temps.data_ptr(), scratch.data_ptr(),
                scratch.stride(0), B, V, top_k.data_ptr(), top_p.data_ptr(), None, seeds.data_ptr(), pos.data_ptr(), got.data_ptr(), None, None,
                got_n.data_ptr(), splits, ws.data_ptr(), torch.cuda.current_stream().cuda_stream)
    assert (got[::2] == V - 1).all() and (got_n[::2] == 1).all()
    # (the softmax sums differ in the last bits: a row's cut may fall one column further at most, the rest is equal)
    assert ((got_n - want_n).abs() <= 1).all() and (got == want)[got_n == want_n].all()


def test_rows_that_keep_some_hundred_columns_are_decided_from_the_lists(device):
    """32000 columns in 16 lists of their ranges' 64 largest: rows that keep 400 columns need no second look at the probabilities."""
    from sglang_amd import kernels as K

    B, V = 128, 32000
    g = torch.Generator(device=device).manual_seed(5)
    lg = (torch.randn((B, V), generator=g, device=device) * 2.5).to(torch.bfloat16)
    top_k, seeds, pos = torch.full((B,), 400, dtype=torch.int32, device=device), torch.arange(B, device=device), torch.arange(B, device=device)
    out = K.sample_from_logits(lg, torch.ones((B, 1), device=device), top_k, None, None, seeds, pos, return_n_keep=True, return_fallback=True)
    assert bool((out[1] == 400).all()) and not bool(out[2].any())


def _rows(device, B, V, seed):
    """bf16 logits [B, V] of several kinds, with temperatures, seeds and positions."""
    Vp = V + (-V) % 4
    g = torch.Generator(device=device).manual_seed(seed)
    rn = lambda *s: torch.randn(s, generator=g, device=device)
    lg = rn(B, Vp) * 2.5
    temps = torch.rand((B, 1), generator=g, device=device) * 0.6 + 0.6
    temps[0] = 1.0
    if B >= 12:
        lg[1] = (rn(Vp) * 8).round() / 8                            # few keys, hundreds of columns each
        lg[2] = rn(Vp) * 0.3                                        # flat: the nucleus crosses zero
        lg[3] = -(rn(Vp).abs() * 3 + 1)                             # no positive column
        lg[4] = rn(Vp) * 1e-6                                       # distinct logits, equal probabilities
        lg[4, 5] = 3.0
        lg[5, torch.randperm(Vp, generator=torch.Generator().manual_seed(1))[: Vp - 90].to(device)] = -float("inf")
        lg[6] = rn(Vp) * 8                                          # peaked
        lg[7] -= 20.0
        lg[8] = 0.0
        lg[9, 3] = float("nan")
        temps[10] = 4.0
        temps[11] = 0.05
    return lg.to(torch.bfloat16)[:, :V], temps, torch.arange(B, device=device) * 7919 + 3, torch.arange(B, device=device) + 11


@pytest.mark.parametrize("B,V", [(1, 128256), (12, 128256), (40, 128256), (45, 50257), (100, 151936), (120, 40002), (90, 65537)])
@pytest.mark.parametrize("top_k,top_p,min_p", [(200, 1.0, 0.0), (200, 0.7, 0.0), (65, 0.999, 0.02), (1000, 0.9, 0.0), (1 << 30, 0.9, 0.0),
                                               (1 << 30, 0.5, 0.01), (1 << 30, 1.0, 0.05), (40, 0.9, 0.0)])
def test_rows_decided_by_their_keys_equal_softmax_then_sample(device, B, V, top_k, top_p, min_p):
    """Nuclei beyond one wave are decided from the counts of their 16-bit keys, from the candidate lists or from the row; any number of ranges."""
    from sglang_amd import kernels as K

    lg, temps, seeds, pos = _rows(device, B, V, V + B + top_k % 1000)
    ks = torch.full((B,), top_k, dtype=torch.int32, device=device)
    ps, ms = torch.full((B,), top_p, device=device), torch.full((B,), min_p, device=device) if min_p else None
    probs = K.softmax_temperature_from_bf16(lg, temps)
    assert probs is not None
    want, want_n = K.top_k_top_p_min_p_sample(probs, ks, ps, ms, seeds, pos, return_n_keep=True)
    got, got_n = K.sample_from_logits(lg, temps, ks, ps, ms, seeds, pos, return_n_keep=True, any_ranges=True)
    bad = ((got == want) & (got_n == want_n)).logical_not().nonzero().flatten().tolist()
    assert not bad, [(r, int(got[r]), int(want[r]), int(got_n[r]), int(want_n[r])) for r in bad]


@pytest.mark.parametrize("top_k", [100, 300, 700])
@pytest.mark.parametrize("V", [33000, 65536])
def test_kept_columns_of_one_probability_are_decided_from_their_counts(device, V, top_k):
    """Peaked rows that keep columns of many keys whose probabilities are all zero: nothing is sorted in memory."""
    from sglang_amd import kernels as K

    B, g = 32, torch.Generator(device=device).manual_seed(V + top_k)
    lg = (torch.randn((B, V), generator=g, device=device) * 6.0).to(torch.bfloat16)
    temps, pos = torch.linspace(0.03, 0.12, B, device=device)[:, None], torch.arange(B, device=device)
    args = (torch.full((B,), top_k, dtype=torch.int32, device=device), None, None, pos * 31, pos)
    probs = K.softmax_temperature_from_bf16(lg, temps)
    assert bool(((probs > 0).sum(-1) < top_k).any())
    want, want_n = K.top_k_top_p_min_p_sample(probs, *args, return_n_keep=True)
    K.sample_from_logits(lg, temps, *args)
    scratch = K._SAMPLE_WS["from_logits", B, V, 64, str(lg.device)][1]               # rows that go the long way are written here as probabilities
    scratch.fill_(-1.0)
    got, got_n = K.sample_from_logits(lg, temps, *args, return_n_keep=True)
    assert torch.equal(got, want) and torch.equal(got_n, want_n)
    assert bool((scratch == -1.0).all()), (scratch != -1.0).any(-1).nonzero().flatten().tolist()


@pytest.mark.parametrize("B,V", [(1, 128256), (12, 32000), (33, 50257), (100, 151936), (128, 40002), (700, 33000), (3, 1025)])
@pytest.mark.parametrize("fp32", [False, True])
def test_unfiltered_from_logits_equals_softmax_then_sample(device, B, V, fp32):
    from sglang_amd import kernels as K

    lg, temps, seeds, pos = _rows(device, B, V, V + B)
    lg = torch.nn.functional.pad(lg, (0, (-V) % 4))
    lg = lg.float() if fp32 else lg
    splits = min(64, 2048 // B, V // 512)
    probs = torch.empty((B, lg.shape[1]), device=device)
    ws = torch.empty(B * splits * 2, device=device)
    from sglang_amd import native
    if fp32:
        probs.copy_(lg)
        native.call("sgl_amd_softmax_temperature_split", probs.data_ptr(), temps.data_ptr(), B, V, probs.stride(0), splits, ws.data_ptr(), K._stream())
    else:
        native.call("sgl_amd_softmax_temperature_split_bf16", lg.data_ptr(), probs.data_ptr(), temps.data_ptr(), B, V, lg.stride(0), probs.stride(0), splits,
                    ws.data_ptr(), K._stream())
    want = K.top_k_top_p_min_p_sample(probs[:, :V], None, None, None, seeds, pos, filtered=False)
    before = lg.clone()
    got = K.sample_unfiltered_from_logits(lg[:, :V], temps, seeds, pos)
    assert torch.equal(lg.nan_to_num(7.0), before.nan_to_num(7.0))
    bad = (got != want).nonzero().flatten().tolist()
    assert not bad, [(r, int(got[r]), int(want[r])) for r in bad]


def _seed_with_hash(col, want=0):
    """The seed (its upper half and the position 0) whose hash of column `col` is `want`: every step of the hash can be undone."""
    M = 0xffffffff
    inv = lambda x: pow(x, -1, 1 << 32)
    rotr = lambda x, r: (x >> r) | (x << (32 - r)) & M

    def unshift(h, r):
        x = h
        for _ in range(32 // r + 1):
            x = h ^ (x >> r)
        return x

    def scramble(k):
        k = k * 0xCC9E2D51 & M
        return ((k << 15 | k >> 17) & M) * 0x1B873593 & M

    def unmix(h, k):                                              # h in front of mm_mix(h, k)
        return rotr((h - 0xE6546B64) * inv(5) & M, 13) ^ scramble(k)

    h = unshift(want, 16) * inv(0xC2B2AE35) & M
    h = unshift(h, 13) * inv(0x85EBCA6B) & M
    h = unmix(unmix(unmix(unshift(h, 16) ^ 16, col), 0), 0)       # column, position, upper half
    k = rotr((h - 0xE6546B64) * inv(5) & M, 13)                    # scramble(lower half) ^ 0
    return rotr(k * inv(0x1B873593) & M, 15) * inv(0xCC9E2D51) & M


@pytest.mark.parametrize("fp32", [False, True])
@pytest.mark.parametrize("below", [85, 97, 103, 120])
def test_unfiltered_rows_whose_largest_probability_has_hash_0(device, fp32, below):
    """Its noise is -709.8, so that a column of the far tail wins: probabilities below the least normal float, whole binades apart or zero."""
    from sglang_amd import kernels as K

    B, V = 48, 32000
    g = torch.Generator().manual_seed(below)
    lg = 30.0 - below + torch.randn((B, V), generator=g) * 2.0
    top = torch.randint(0, V, (B,), generator=g)
    lg[torch.arange(B), top] = 30.0
    lg = lg.to(torch.bfloat16).to(device)
    lg = lg.float() if fp32 else lg
    seeds = torch.tensor([_seed_with_hash(int(c)) for c in top], device=device)
    temps, pos = torch.ones((B, 1), device=device), torch.zeros(B, dtype=torch.int64, device=device)
    probs = torch.empty((B, V), device=device)
    ws = torch.empty(B * 64 * 2, device=device)
    from sglang_amd import native
    splits = min(64, 2048 // B, V // 512)
    if fp32:
        probs.copy_(lg)
        native.call("sgl_amd_softmax_temperature_split", probs.data_ptr(), temps.data_ptr(), B, V, V, splits, ws.data_ptr(), K._stream())
    else:
        native.call("sgl_amd_softmax_temperature_split_bf16", lg.data_ptr(), probs.data_ptr(), temps.data_ptr(), B, V, V, V, splits, ws.data_ptr(), K._stream())
    want = K.top_k_top_p_min_p_sample(probs, None, None, None, seeds, pos, filtered=False)
    if below < 120:                                               # (of 120 all others are zero and the largest wins)
        assert not bool((want.cpu() == top).any())
    got = K.sample_unfiltered_from_logits(lg, temps, seeds, pos)
    bad = (got != want).nonzero().flatten().tolist()
    assert not bad, [(r, int(got[r]), int(want[r])) for r in bad]
