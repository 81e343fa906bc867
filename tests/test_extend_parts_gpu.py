"""Extend attention with the keys of a request dealt over workgroups, and the four-wave form of one part."""
import pytest
import torch

import oracle.ops as oo
from sglang_amd import kernels, native
from test_kernels_gpu import BF, _random_case


def test_rule_splits_few_rows_behind_long_contexts_only():
    parts = native.lib().sgl_amd_extend_attention_parts
    assert parts(1, 203, 203, 4003, 32, 8, 128) > 1 and parts(3, 66, 22, 4571, 32, 32, 128) > 1 and parts(1, 500, 500, 4500, 14, 2, 64) > 1
    for one in ((60, 128, 1024, 32, 8, 128), (6, 3107, 3107, 64, 8, 128), (1, 37, 37, 14, 2, 64), (1, 512, 512, 32, 8, 128), (1, 203, 0, 32, 8, 128),
                (0, 5, 500, 32, 8, 128), (1, 5, 500, 32, 8, 96), (1, 5, 5000, 256, 1, 128)):
        assert parts(one[0], one[0] * one[1], *one[1:]) == 1, one


@pytest.mark.gpu
@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("Hq,Hkv,D,causal", [(32, 8, 128, True), (14, 2, 64, True), (4, 4, 128, True), (64, 1, 64, True), (16, 4, 128, False)])
def test_parts_against_the_oracle(device, Hq, Hkv, D, causal, fp8):
    """Walks of no tile, one and many, tile-straddling extends, more parts than a request has tiles, a key that dominates inside one
    part; rows behind the requests' tokens are left alone.  Bars of the other extend tests; e4m3 rows are compared on their
    dequantised values."""
    prefix = [0, 896, 5, 0, 63, 64, 200, 1000] if causal else [0, 0, 0, 0]
    extend = [130, 128, 1, 333, 65, 64, 7, 70] if causal else [50, 64, 129, 300]
    c = _random_case(len(prefix), Hq, Hkv, D, prefix, extend, seed=Hq + D + 7, spike=True)
    c["q"][-3] = (c["k_cache"][c["req_to_token"][c["req_pool_indices"][-1], 3].long(), 0] * 30).to(BF)
    kc, vc = (x.to(torch.float8_e4m3fn) if fp8 else x for x in (c["k_cache"], c["v_cache"]))
    ref = oo.extend_attention(c["q"], kc.to(BF), vc.to(BF), c["req_to_token"], c["req_pool_indices"], c["seq_lens"], c["extend_prefix_lens"],
                              c["extend_seq_lens"], c["scaling"], causal=causal, compute_dtype=torch.float32)
    T, spare = c["q"].shape[0], 5
    q = torch.cat([c["q"], torch.zeros(spare, Hq, D, dtype=BF)]).to(device)
    qo = torch.zeros(len(prefix) + 1, dtype=torch.int32)
    qo[1:] = torch.cumsum(torch.tensor(extend), 0)
    kc, vc = ((x.view(torch.uint8) if fp8 else x).to(device) for x in (kc, vc))
    r2t, pool, seq, pre, qo = (c["req_to_token"].to(device), c["req_pool_indices"].to(device), c["seq_lens"].to(torch.int32).to(device),
                               torch.tensor(prefix, dtype=torch.int32, device=device), qo.to(device))
    for parts in (1, 2, 5, 16):
        out = torch.full_like(q, 7.0)
        n = (T + spare) * Hq
        acc, ml = torch.full((parts, n, D), float("nan"), device=device), torch.full((parts, n, 2), float("nan"), device=device)
        native.call("sgl_amd_extend_attention_kv", q.data_ptr(), out.data_ptr(), kc.data_ptr(), vc.data_ptr(), r2t.data_ptr(), r2t.stride(0), pool.data_ptr(),
                    seq.data_ptr(), pre.data_ptr(), qo.data_ptr(), len(prefix), T + spare, max(extend), int(seq.max()), Hq, Hkv, D, q.stride(0), out.stride(0),
                    Hkv * D, c["scaling"], int(causal), int(fp8), 1.0, 1.0, parts, acc.data_ptr(), ml.data_ptr(), torch.cuda.current_stream().cuda_stream)
        torch.testing.assert_close(out[:T].float().cpu(), ref.float(), atol=4e-3, rtol=1e-2, msg=lambda m: f"{parts} parts: {m}")
        assert bool((out[T:] == 7.0).all()), parts


@pytest.mark.gpu
@pytest.mark.parametrize("shape", [0, 82])
@pytest.mark.parametrize("Hq,Hkv,D,fp8", [(32, 8, 128, False), (14, 2, 64, True)])
def test_request_without_keys_gives_zero_rows(device, Hq, Hkv, D, fp8, shape):
    """Query rows of a request whose context is empty (seq_lens 0) are zeros in one part, in several and in the eight-wave form; nothing is
    read or written for it anywhere else (one part has no partial rows), and its neighbours' rows are what they are without it."""
    c = _random_case(3, Hq, Hkv, D, [0, 300, 70], [40, 130, 65], seed=Hq + 3)
    kc, vc = ((x.to(torch.float8_e4m3fn).view(torch.uint8) if fp8 else x).to(device) for x in (c["k_cache"], c["v_cache"]))
    q, r2t, pool = c["q"].to(device), c["req_to_token"].to(device), c["req_pool_indices"].to(device)
    pre, qo = torch.tensor([0, 300, 70], dtype=torch.int32, device=device), torch.tensor([0, 40, 170, 235], dtype=torch.int32, device=device)

    def run(lens, parts):
        out = torch.full_like(q, 7.0)
        n = q.shape[0] * Hq
        acc, ml = torch.full((parts, n, D), float("nan"), device=device), torch.full((parts, n, 2), float("nan"), device=device)
        ws = (acc.data_ptr(), ml.data_ptr()) if parts > 1 else (None, None)
        seq = torch.tensor(lens, dtype=torch.int32, device=device)
        native.call("sgl_amd_extend_attention_kv", q.data_ptr(), out.data_ptr(), kc.data_ptr(), vc.data_ptr(), r2t.data_ptr(), r2t.stride(0), pool.data_ptr(),
                    seq.data_ptr(), pre.data_ptr(), qo.data_ptr(), 3, q.shape[0], 130, 430, Hq, Hkv, D, q.stride(0), out.stride(0), Hkv * D, D ** -0.5, 1,
                    int(fp8), 1.0, 1.0, parts, *ws, torch.cuda.current_stream().cuda_stream)
        return out

    native.call("sgl_amd_debug_extend_attention_shape", shape, 0)
    try:
        for parts in (1, 2) if shape == 0 else (1,):
            want = run([40, 430, 135], parts)
            for empty, rows in ((0, slice(0, 40)), (1, slice(40, 170)), (2, slice(170, 235))):
                lens = [40, 430, 135]
                lens[empty] = 0
                got, ref = run(lens, parts), want.clone()
                ref[rows] = 0.0
                assert torch.equal(got, ref), (parts, empty)
    finally:
        native.call("sgl_amd_debug_extend_attention_shape", 0, 0)


@pytest.mark.gpu
@pytest.mark.parametrize("bad", [float("nan"), float("inf")])
def test_a_key_that_is_no_number_makes_its_rows_nan_in_any_number_of_parts(device, bad):
    """Softmax over a NaN or infinite score is NaN: rows that see the key are NaN however the keys are dealt, the rest are what they are
    without it."""
    Hq, Hkv, D, prefix, extend = 8, 2, 128, [700, 300], [40, 30]
    c = _random_case(2, Hq, Hkv, D, prefix, extend, seed=11)
    qo = torch.tensor([0, 40, 70], dtype=torch.int32, device=device)
    q, r2t, pool, seq, pre = (c["q"].to(device), c["req_to_token"].to(device), c["req_pool_indices"].to(device), c["seq_lens"].to(torch.int32).to(device),
                              torch.tensor(prefix, dtype=torch.int32, device=device))
    spoilt = c["k_cache"].clone()
    spoilt[c["req_to_token"][c["req_pool_indices"][0], 710].long(), 1] = bad             # seen by tokens 10 and on of request 0, by kv head 1's rows
    vc = c["v_cache"].to(device)
    for parts in (1, 2, 5, 16):
        outs = []
        for kc in (c["k_cache"].to(device), spoilt.to(device)):
            out, n = torch.empty_like(q), q.shape[0] * Hq
            acc, ml = torch.empty((parts, n, D), device=device), torch.empty((parts, n, 2), device=device)
            native.call("sgl_amd_extend_attention_kv", q.data_ptr(), out.data_ptr(), kc.data_ptr(), vc.data_ptr(), r2t.data_ptr(), r2t.stride(0), pool.data_ptr(),
                        seq.data_ptr(), pre.data_ptr(), qo.data_ptr(), 2, 70, 40, 740, Hq, Hkv, D, q.stride(0), out.stride(0), Hkv * D, D ** -0.5, 1, 0, 1.0, 1.0,
                        parts, acc.data_ptr(), ml.data_ptr(), torch.cuda.current_stream().cuda_stream)
            outs.append(out)
        nan = torch.zeros(70, Hq, dtype=torch.bool, device=device)
        nan[10:40, 4:] = True
        assert bool(outs[1][nan].isnan().all()), parts
        assert torch.equal(outs[1][~nan], outs[0][~nan]), parts


@pytest.mark.gpu
@pytest.mark.parametrize("Hq,Hkv,D,extend,max_kv", [(32, 8, 128, [130, 7], 0), (14, 2, 64, [300, 65], 365), (64, 8, 128, [700, 900], 1000)])
def test_pool_that_does_not_begin_at_a_16_byte_piece(device, Hq, Hkv, D, extend, max_kv):
    """Rows go to LDS in whole 16-byte pieces only where the pool begins at one; other pools give the same result another way."""
    prefix = [0, 100]
    c = _random_case(2, Hq, Hkv, D, prefix, extend, seed=Hq + D)
    ref = oo.extend_attention(c["q"], c["k_cache"], c["v_cache"], c["req_to_token"], c["req_pool_indices"], c["seq_lens"], c["extend_prefix_lens"],
                              c["extend_seq_lens"], c["scaling"], causal=True, compute_dtype=torch.float32)

    def shifted(x, by):
        flat = torch.empty(x.numel() + by, dtype=x.dtype, device=device)
        flat[by:] = x.reshape(-1).to(device)
        return flat[by:].view(x.shape)

    q = c["q"].to(device)
    qo = torch.tensor([0, extend[0], sum(extend)], dtype=torch.int32, device=device)
    args = (c["req_to_token"].to(device), c["req_pool_indices"].to(device), c["seq_lens"].to(torch.int32).to(device),
            torch.tensor(prefix, dtype=torch.int32, device=device), qo, max(extend), c["scaling"])
    for k_by, v_by in ((0, 0), (4, 0), (0, 4), (2, 4)):
        out = kernels.extend_attention(q, torch.empty_like(q), shifted(c["k_cache"], k_by), shifted(c["v_cache"], v_by), *args, max_kv_len=max_kv)
        torch.testing.assert_close(out.float().cpu(), ref.float(), atol=4e-3, rtol=1e-2, msg=lambda m: f"{k_by}, {v_by}: {m}")
