"""A prefill layer through kernels.extend_attention_layer, which looks at every argument once: the bits of the general wrappers, and everything that is not of the
plainest form left to them."""
import types

import pytest
import torch

BF, FP8 = torch.bfloat16, torch.float8_e4m3fn


def _layer(dev, lens, prefix, hq, hkv, d, fp8, seed=0):
    from sglang_amd.layers.attention.hip_backend import HipAttnBackend
    from sglang_amd.layers.radix_attention import RadixAttention
    from sglang_amd.mem_cache.memory_pool import MHATokenToKVPool, ReqToTokenPool
    from sglang_amd.model_executor.forward_batch_info import ForwardBatch, ForwardMode

    g = torch.Generator().manual_seed(seed)
    B, T, total = len(lens), sum(lens), sum(lens) + len(lens) * prefix
    req_pool, pool = ReqToTokenPool(B + 2, 2048, dev), MHATokenToKVPool(total + 8, 1, FP8 if fp8 else BF, hkv, d, 1, dev)
    for buf in (pool.get_key_buffer(0), pool.get_value_buffer(0)):
        x = (torch.randn(buf.shape, generator=g) * 0.5)
        buf.copy_((x.to(FP8).view(torch.uint8) if fp8 else x.to(BF)))
    slots, loc = torch.randperm(total, generator=g).int() + 1, []
    for b, n in enumerate(lens):
        s, slots = slots[: prefix + n], slots[prefix + n:]
        req_pool.req_to_token[b + 1, : prefix + n] = s.to(dev)
        loc.append(s[prefix:].long())
    backend = HipAttnBackend(types.SimpleNamespace(device=dev, req_to_token_pool=req_pool, token_to_kv_pool=pool, num_attention_heads_per_rank=hq,
                                                   num_kv_heads_per_rank=hkv, head_dim=d))
    seq = torch.tensor([prefix + n for n in lens])
    fb = ForwardBatch(ForwardMode.EXTEND, B, torch.zeros(T, dtype=torch.int64, device=dev), torch.arange(1, B + 1, device=dev), seq.int().to(dev), torch.cat(loc).to(dev),
                      seq_lens_cpu=seq, extend_seq_lens_cpu=lens, extend_prefix_lens_cpu=[prefix] * B, extend_prefix_lens=torch.full((B,), prefix, dtype=torch.int32, device=dev),
                      req_to_token_pool=req_pool, token_to_kv_pool=pool, attn_backend=backend)
    qkv = (torch.randn((T, (hq + 2 * hkv) * d), generator=g) * 0.7).to(BF).to(dev)
    return backend, fb, pool, RadixAttention(hq, d, d ** -0.5, hkv, 0), qkv.split([hq * d, hkv * d, hkv * d], dim=-1)


SHAPES = [(14, 2, 64, 0, [37], 0), (32, 8, 128, 0, [1, 64, 3], 0), (32, 8, 128, 1, [5, 20], 30), (32, 8, 128, 0, [203], 700), (64, 8, 128, 1, [120, 300, 700, 90], 0), (32, 32, 128, 0, [40, 80], 50)]


@pytest.mark.gpu
@pytest.mark.parametrize("hq,hkv,d,fp8,lens,prefix", SHAPES)
def test_the_general_wrappers_bits(device, monkeypatch, hq, hkv, d, fp8, lens, prefix):
    from sglang_amd import kernels

    got, plain = [], kernels.extend_attention_layer
    for general in (False, True):
        backend, fb, pool, layer, (q, k, v) = _layer(device, lens, prefix, hq, hkv, d, fp8)
        if fp8:
            layer.set_kv_scales(0.5, 2.0)
        took = []
        monkeypatch.setattr(kernels, "extend_attention_layer", lambda *a: None if general else took.append(plain(*a)) or took[-1])
        backend.init_forward_metadata(fb)
        got.append((layer(q, k, v, fb), pool.get_key_buffer(0), pool.get_value_buffer(0)))
        assert general or took[0] is not None
    assert all(torch.equal(a, b) for a, b in zip(*got))


@pytest.mark.gpu
def test_other_forms_are_left_to_the_general_wrappers(device, monkeypatch):
    from sglang_amd import kernels
    from sglang_amd.layers.radix_attention import AttentionType

    backend, fb, pool, layer, (q, k, v) = _layer(device, [17, 40], 0, 8, 2, 128, 0)
    seen, plain = [], kernels.extend_attention_layer
    monkeypatch.setattr(kernels, "extend_attention_layer", lambda *a: seen.append(plain(*a)) or seen[-1])
    backend.init_forward_metadata(fb)
    want, k3, v3 = layer(q, k, v, fb), k.view(-1, 2, 128), v.view(-1, 2, 128)
    assert seen.pop() is not None
    # queries of three dimensions: the general wrappers' answer
    assert torch.equal(backend.forward_extend(q.view(-1, 8, 128), k3, v3, layer, fb), want) and seen.pop() is None
    # slots of 32 bits: the general wrappers' answer
    loc, fb.out_cache_loc = fb.out_cache_loc, fb.out_cache_loc.int()
    assert torch.equal(backend.forward_extend(q, k3, v3, layer, fb), want) and seen.pop() is None
    fb.out_cache_loc = loc
    # what is refused: another type, another device, keys that are not 16-byte aligned
    odd = torch.empty(k3.numel() + 1, dtype=BF, device=device)[1:].view(k3.shape)
    odd.copy_(k3)
    for qq, kk in ((q.half(), k3), (q.cpu(), k3), (q, odd)):
        with pytest.raises((ValueError, RuntimeError)):
            backend.forward_extend(qq, kk, v3, layer, fb)
        assert seen.pop() is None
    # a layer's switches never get there
    for name, value in (("logit_cap", 30.0), ("sliding_window_size", 8)):
        before = getattr(layer, name)
        setattr(layer, name, value)
        assert not torch.equal(layer(q, k, v, fb), want) and not seen
        setattr(layer, name, before)
    layer.attn_type = AttentionType.ENCODER_ONLY
    assert not torch.equal(layer(q, k, v, fb), want) and seen.pop() is not None
    layer.attn_type = AttentionType.DECODER
    layer.is_cross_attention = True
    with pytest.raises(NotImplementedError):
        layer(q, k, v, fb)
