"""The work a user of this framework has it do, as measured cases.

Six kinds, each through the entry points a program calls:

  extend   one attention layer of a prefill pass: AttentionBackend.forward_extend, which stores the new keys and values and attends
  decode   the attention layers of one decode step, captured as a graph the way the decode graph runner captures them
  experts  a sparse feed-forward block: TopK and FusedMoE
  sample   Sampler.forward over a step's logits
  model    ModelRunner.forward: a decode step (graph replay) or a prefill pass of a whole model, or of its first layers
  scan     a recurrent layer of a hybrid decoder: Mamba-2 or the gated delta rule, whole prompts or one token a request

Sizes are those of the configurations in sglang_amd.harness (models.CONFIGS, genusun.CONFIGS) and of the repository's benchmark:
4 groups of 16 requests that share 896 prompt tokens, 128 of their own.
"""
import dataclasses
import math
import types

import torch

from sglang_amd import kernels
from sglang_amd.harness import genusun
from sglang_amd.harness.engine import ModelRunner
from sglang_amd.harness.models import CONFIGS
from sglang_amd.layers.attention.hip_backend import HipAttnBackend
from sglang_amd.layers.moe.fused_moe import FusedMoE
from sglang_amd.layers.moe.topk import TopK
from sglang_amd.layers.radix_attention import RadixAttention
from sglang_amd.layers.sampler import LogitsProcessorOutput, Sampler, SamplingBatchInfo
from sglang_amd.mem_cache.memory_pool import MHATokenToKVPool, ReqToTokenPool
from sglang_amd.model_executor.forward_batch_info import ForwardBatch, ForwardMode

BF, F32, F64, FP8 = torch.bfloat16, torch.float32, torch.float64, torch.float8_e4m3fn


def listed():
    return [
        # the first turn of a small model's user: one short prompt, nothing cached; launches and host time count
        dict(name="extend_first_turn", kind="extend", model="qwen2.5-0.5b", kv="bf16", requests=1, groups=1, prefix=0, tokens=37, spread=0.0),
        # a later turn of a conversation, or a chunk of a long prompt: few new tokens behind a long cached context
        dict(name="extend_later_turn", kind="extend", model="llama-3-8b", kv="bf16", requests=1, groups=1, prefix=3800, tokens=203, spread=0.0),
        # the benchmark's second pass: 60 requests whose 896-token prefixes are in the radix cache
        dict(name="extend_shared", kind="extend", model="llama-3-8b", kv="bf16", requests=60, groups=4, prefix=896, tokens=128, spread=0.0),
        # cold prompts of several lengths in one pass of a large model
        dict(name="extend_cold", kind="extend", model="llama-3-70b", kv="bf16", requests=6, groups=6, prefix=0, tokens=2100, spread=0.5),
        # the benchmark's decode step: shared prefixes, 64 tokens generated
        dict(name="decode_shared", kind="decode", model="llama-3-8b", kv="bf16", requests=64, groups=4, prefix=896, tokens=128, generated=64, spread=0.0, layers=8),
        # long conversations that share nothing, on an fp8 cache
        dict(name="decode_long_fp8", kind="decode", model="mixtral-8x7b", kv="fp8", requests=37, groups=37, prefix=0, tokens=3000, generated=200, spread=0.7, layers=4),
        # sparse feed-forward of a decode step
        dict(name="experts_decode", kind="experts", model="mixtral-8x7b", tokens=48),
        # sparse feed-forward of a prefill pass
        dict(name="experts_prefill", kind="experts", model="mixtral-8x7b", tokens=3000),
        # filtered sampling of a large vocabulary
        dict(name="sample_filtered", kind="sample", model="llama-3-8b", requests=128, top_k=50, top_p=0.9, min_p=0.0),
        # the benchmark's whole decode step, four of its 32 equal layers
        dict(name="model_decode", kind="model", model="llama-3-8b", mode="decode", layers=4, requests=64, groups=4, prefix=896, tokens=128, generated=64),
        # the two recurrences of a hybrid decoder over a prefill batch
        dict(name="scan_mamba2", kind="scan", model="genusun-1b", rule="mamba2", requests=4, tokens=2048, spread=0.2, start=0),
        dict(name="scan_delta", kind="scan", model="genusun-8b", rule="delta", requests=3, tokens=1500, spread=0.3, start=0),
    ]


# ------------------------------------------------------------------------------------------------ draws
def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["extend", "extend", "extend", "decode", "decode", "experts", "sample", "model", "scan", "scan"])
    while True:
        if kind == "extend":
            c = dict(kind=kind, model=rng.choice(["qwen2.5-0.5b", "llama-3-8b", "llama-3-70b", "mixtral-8x7b", "llava-1.6-7b"]),
                     kv=rng.choice(["bf16", "bf16", "fp8"]), requests=_log(rng, 1, 64), groups=1, prefix=0, tokens=_log(rng, 20, 4000), spread=rng.choice([0.0, 0.3, 0.6]))
            if rng.random() < 0.6:
                c["prefix"] = _log(rng, 64, 6000)
            c["groups"] = rng.choice([1, c["requests"], max(1, c["requests"] // 8)])
        elif kind == "decode":
            c = dict(kind=kind, model=rng.choice(["qwen2.5-0.5b", "llama-3-8b", "llama-3-70b", "mixtral-8x7b", "llava-1.6-7b"]),
                     kv=rng.choice(["bf16", "bf16", "fp8"]), requests=_log(rng, 1, 128), groups=1, prefix=rng.choice([0, _log(rng, 64, 4000)]),
                     tokens=_log(rng, 16, 4000), generated=_log(rng, 1, 500), spread=rng.choice([0.0, 0.4, 0.7]), layers=4)
            c["groups"] = rng.choice([1, c["requests"], max(1, c["requests"] // 8)])
        elif kind == "experts":
            c = dict(kind=kind, model="mixtral-8x7b", tokens=_log(rng, 1, 3000))
        elif kind == "sample":
            c = dict(kind=kind, model=rng.choice(["llama-3-8b", "qwen2.5-0.5b", "mixtral-8x7b"]), requests=_log(rng, 1, 128),
                     top_k=rng.choice([0, 20, 50, 200]), top_p=rng.choice([1.0, 0.9, 0.7]), min_p=rng.choice([0.0, 0.0, 0.05]))
        elif kind == "model":
            c = dict(kind=kind, model=rng.choice(["llama-3-8b", "qwen2.5-0.5b"]), mode=rng.choice(["decode", "decode", "prefill"]), layers=rng.choice([2, 3, 4]),
                     requests=_log(rng, 1, 64), groups=1, prefix=rng.choice([0, _log(rng, 64, 1500)]), tokens=_log(rng, 20, 600), generated=_log(rng, 1, 100))
            c["groups"] = rng.choice([1, c["requests"]])
        else:
            c = dict(kind=kind, model=rng.choice(["genusun-1b", "genusun-8b"]), rule=rng.choice(["mamba2", "delta"]), requests=_log(rng, 1, 16),
                     tokens=_log(rng, 16, 2048), spread=rng.choice([0.0, 0.2, 0.5]), start=rng.choice([0, 0, 2048]))
            if rng.random() < 0.25:
                c.update(requests=_log(rng, 1, 128), tokens=1, spread=0.0, start=1000)
        if _affordable(c):
            return c


def _affordable(c):
    """Within the listed cases' cost, the models' contexts and a few GiB of inputs."""
    w = work(c)
    if w["flops"] > 4.0e11 * (20 if c["kind"] == "experts" else 1) or w["bytes"] > 3.5e9:
        return False
    if c["kind"] in ("extend", "decode", "model"):
        prefix, lens, total = _lengths(c)
        return total <= 170_000 and sum(lens) <= 14_000 * (12 if c["kind"] == "decode" else 1) and max(lens) + prefix + c.get("generated", 0) <= 8000
    return c["kind"] != "scan" or c["requests"] * c["tokens"] <= 9000


# ------------------------------------------------------------------------------------------------ shapes
def _heads(c):
    m = CONFIGS[c["model"]]
    return m.num_attention_heads, m.num_key_value_heads, m.head_dim


def _ragged(n, tokens, spread):
    """n lengths around `tokens`, a fixed odd pattern: requests of one batch are not equally long."""
    return [max(1, int(round(tokens * (1.0 + spread * math.sin(1.0 + 2.4 * i))))) for i in range(n)]


def _lengths(c):
    """(shared prefix, own tokens of every request, slots in use)."""
    lens = _ragged(c["requests"], c["tokens"], c.get("spread", 0.0))
    return c["prefix"], lens, c["groups"] * c["prefix"] + sum(lens) + c["requests"] * c.get("generated", 0)


def _pairs(c):
    """Visible (query, key) pairs of an extend."""
    prefix, lens, _ = _lengths(c)
    return sum(n * prefix + n * (n + 1) // 2 for n in lens)


def work(case):
    c = case
    if c["kind"] == "extend":
        hq, hkv, d = _heads(c)
        prefix, lens, _ = _lengths(c)
        row, t = 2 * hkv * d, sum(lens)
        es = 1 if c["kv"] == "fp8" else 2
        return {"bytes": 2 * t * 2 * hq * d + t * row * (2 + es) + c["groups"] * prefix * row * es, "flops": 4 * hq * d * _pairs(c)}
    if c["kind"] == "decode":
        hq, hkv, d = _heads(c)
        prefix, lens, total = _lengths(c)
        row, b = 2 * hkv * d, c["requests"]
        es = 1 if c["kv"] == "fp8" else 2
        keys = b * prefix + total - c["groups"] * prefix
        return {"bytes": c["layers"] * (total * row * es + 2 * b * 2 * hq * d + b * row * 2), "flops": c["layers"] * 4 * hq * d * keys}
    if c["kind"] == "experts":
        m = CONFIGS[c["model"]]
        e, h, n, t = m.num_local_experts, m.hidden_size, m.intermediate_size, c["tokens"]
        used = e * (1.0 - (1.0 - m.num_experts_per_tok / e) ** t)
        return {"bytes": int(used * 3 * h * n * 2) + 2 * t * h * 2, "flops": t * m.num_experts_per_tok * 6 * h * n}
    if c["kind"] == "sample":
        v = CONFIGS[c["model"]].vocab_size
        return {"bytes": c["requests"] * v * 2, "flops": c["requests"] * v * 4}
    if c["kind"] == "model":
        m = CONFIGS[c["model"]]
        hq, hkv, d = _heads(c)
        prefix, lens, total = _lengths(c)
        layer = m.hidden_size * (hq + 2 * hkv) * d + hq * d * m.hidden_size + 3 * m.hidden_size * m.intermediate_size
        head, row, b, n = m.vocab_size * m.hidden_size, 2 * hkv * d, c["requests"], c["layers"]
        if c["mode"] == "decode":
            keys = b * prefix + total - c["groups"] * prefix
            return {"bytes": 2 * (n * layer + head) + n * total * row * 2 + b * m.vocab_size * 2, "flops": 2 * b * (n * layer + head) + n * 4 * hq * d * keys}
        t = sum(lens)
        return {"bytes": 2 * (n * layer + head) + n * (t + c["groups"] * prefix) * row * 2 + 2 * t * m.hidden_size * 2,
                "flops": 2 * t * n * layer + 2 * b * head + n * 4 * hq * d * _pairs(c)}
    s, t = _scan_sizes(c), sum(_ragged(c["requests"], c["tokens"], c["spread"]))
    if c["rule"] == "mamba2":
        cols = s["heads"] * s["v"] + 2 * s["groups"] * s["k"] + s["heads"]
        flops = t * s["heads"] * s["k"] * s["v"] * 4
    else:
        cols = 2 * s["groups"] * s["k"] + s["heads"] * s["v"] + 2 * s["heads"]
        flops = t * s["heads"] * s["k"] * s["v"] * 6
    state = c["requests"] * s["heads"] * s["k"] * s["v"] * 4
    return {"bytes": t * 2 * (cols + s["heads"] * s["v"]) + state * (2 if c["start"] else 1), "flops": flops}


def tolerance(case):
    """About four times the distance of today's results from 64 bits (exact() below): bf16 results of fp32 sums, a product of bf16 results
    (experts), layers of bf16 roundings (model).  Sampled ids are decided by seeded noise; only a near-tie may fall the other way."""
    return {"extend": {"rel": 9e-3}, "decode": {"rel": 9e-3}, "experts": {"rel": 1.6e-2}, "sample": {"rel": 0.0, "differ": 0.03}, "model": {"rel": 6e-2},
            "scan": {"rel": 7e-3}}[case["kind"]]


# ------------------------------------------------------------------------------------------------ states
def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _randn(g, *shape, dtype=BF, scale=1.0):
    return (torch.randn(shape, generator=g, device="cuda", dtype=F32) * scale).to(dtype)


def _layout(c, seed, rows, table):
    """Where the tokens of a batch lie in the pool, as a radix cache and a scheduler leave them: a group's prefix and a request's
    own tokens as runs, in no order, then one slot a request for every generated token.  Fills the request table; returns the
    rows, the slots of the requests' own tokens and of the last generated one."""
    prefix, lens, total = _lengths(c)
    b, groups, gen = c["requests"], c["groups"], c.get("generated", 0)
    host = torch.Generator()
    host.manual_seed(int(seed))
    runs = [prefix] * groups + lens
    starts, at = [0] * len(runs), 1
    for i in torch.randperm(len(runs), generator=host).tolist():
        starts[i], at = at, at + runs[i]
    idx = (torch.randperm(rows, generator=host)[:b] + 1).tolist()
    own = []
    for i in range(b):
        p = torch.arange(starts[i * groups // b], starts[i * groups // b] + prefix)
        o = torch.arange(starts[groups + i], starts[groups + i] + lens[i])
        own.append(o)
        g = at + i + b * torch.arange(gen)
        row = torch.cat([p, o, g]).to(torch.int32)
        table[idx[i], : row.numel()] = row.cuda()
    last = torch.tensor([at + i + b * (gen - 1) for i in range(b)]) if gen else None
    return idx, torch.cat(own), last


def _batch(c, seed, req_pool, kv_pool, backend, ids, decode):
    prefix, lens, _ = _lengths(c)
    idx, own, last = _layout(c, seed, req_pool.size, req_pool.req_to_token)
    seq = torch.tensor([prefix + n + c.get("generated", 0) if decode else prefix + n for n in lens], dtype=torch.int64)
    more = {} if decode else dict(extend_prefix_lens_cpu=[prefix] * len(lens), extend_seq_lens_cpu=lens)
    return ForwardBatch.init_new(forward_mode=ForwardMode.DECODE if decode else ForwardMode.EXTEND, input_ids=ids,
                                 req_pool_indices=torch.tensor(idx, device="cuda"), seq_lens=seq.to(torch.int32).cuda(),
                                 out_cache_loc=(last if decode else own).cuda(), seq_lens_cpu=seq, req_to_token_pool=req_pool,
                                 token_to_kv_pool=kv_pool, attn_backend=backend, **more)


def _attention(c, seed):
    g, decode = _gen(seed), c["kind"] == "decode"
    hq, hkv, d = _heads(c)
    prefix, lens, total = _lengths(c)
    n, t = c.get("layers", 1), c["requests"] if decode else sum(lens)
    req_pool = ReqToTokenPool(c["requests"], 8192, torch.device("cuda", 0))
    kv_pool = MHATokenToKVPool(total + 64, 1, FP8 if c["kv"] == "fp8" else BF, hkv, d, n, torch.device("cuda", 0))
    for i in range(n):
        for buf in (kv_pool.get_key_buffer(i), kv_pool.get_value_buffer(i)):
            x = _randn(g, *buf.shape)
            buf.copy_(x.to(FP8).view(torch.uint8) if c["kv"] == "fp8" else x)
    runner = types.SimpleNamespace(device=torch.device("cuda", 0), req_to_token_pool=req_pool, token_to_kv_pool=kv_pool, num_attention_heads_per_rank=hq,
                                   num_kv_heads_per_rank=hkv, head_dim=d)
    backend = HipAttnBackend(runner)
    fb = _batch(c, seed, req_pool, kv_pool, backend, torch.zeros(t, dtype=torch.int64, device="cuda"), decode)
    layers = [RadixAttention(hq, d, d ** -0.5, hkv, i) for i in range(n)]
    qkv = [_randn(g, t, (hq + 2 * hkv) * d) for _ in range(n)]
    return types.SimpleNamespace(backend=backend, fb=fb, layers=layers, qkv=[x.split([hq * d, hkv * d, hkv * d], dim=-1) for x in qkv], pool=kv_pool)


def _capture(s, step):
    """A decode step as the decode graph runner records one: two eager runs, then a graph."""
    stream = torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(stream):
        s.backend.init_cuda_graph_state(s.fb.batch_size, s.fb.batch_size)
        s.backend.init_forward_metadata_out_graph(s.fb, in_capture=True)
        step()
        step()
        stream.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=stream):
            s.out = step()
    torch.cuda.current_stream().wait_stream(stream)
    return graph


def prepare(case, seed):
    c, g = case, _gen(seed)
    if c["kind"] == "extend":
        s = _attention(c, seed)
        s.backend.init_forward_metadata(s.fb)
        s.kind = "extend"
        return s
    if c["kind"] == "decode":
        s = _attention(c, seed)

        def step():
            s.backend.init_forward_metadata_in_graph(s.fb)
            return [layer(q, k, v, s.fb) for layer, (q, k, v) in zip(s.layers, s.qkv)]

        s.graph = _capture(s, step)
        s.kind = "decode"
        return s
    if c["kind"] == "experts":
        m = CONFIGS[c["model"]]
        e, h, n = m.num_local_experts, m.hidden_size, m.intermediate_size
        w13, w2 = torch.empty((e, 2 * n, h), dtype=BF, device="cuda"), torch.empty((e, h, n), dtype=BF, device="cuda")
        for i in range(e):
            w13[i], w2[i] = _randn(g, 2 * n, h, scale=0.02), _randn(g, h, n, scale=0.02)
        x = _randn(g, c["tokens"], h)
        logits = _randn(g, c["tokens"], e, scale=1.5) + _randn(g, 1, e, scale=0.3)
        return types.SimpleNamespace(kind="experts", topk=TopK(m.num_experts_per_tok, renormalize=True), experts=FusedMoE(w13, w2, m.num_experts_per_tok), x=x, logits=logits)
    if c["kind"] == "sample":
        b, v = c["requests"], CONFIGS[c["model"]].vocab_size
        info = SamplingBatchInfo(torch.rand((b, 1), generator=g, device="cuda") * 0.6 + 0.6, torch.full((b,), c["top_p"], device="cuda"),
                                 torch.full((b,), c["top_k"] or 1 << 30, dtype=torch.int32, device="cuda"), torch.full((b,), c["min_p"], device="cuda"),
                                 is_all_greedy=False, need_top_p_sampling=c["top_p"] < 1.0, need_top_k_sampling=c["top_k"] > 0, need_min_p_sampling=c["min_p"] > 0.0,
                                 sampling_seed=torch.randint(0, 1 << 40, (b,), generator=g, device="cuda"))
        return types.SimpleNamespace(kind="sample", sampler=Sampler(), info=info, logits=_randn(g, b, v, scale=2.5),
                                     positions=torch.randint(1, 4000, (b,), generator=g, device="cuda"))
    if c["kind"] == "model":
        return _model(c, seed)
    return _scan(c, seed)


def _model(c, seed):
    g, decode = _gen(seed), c["mode"] == "decode"
    _, lens, total = _lengths(c)
    cfg = dataclasses.replace(CONFIGS[c["model"]], num_hidden_layers=c["layers"])
    r = ModelRunner(cfg, max_total_tokens=total + 64, max_running_requests=c["requests"], max_context_len=8192, use_graph=decode, graph_max_bs=c["requests"], strict_graph=True)
    for i in range(c["layers"]):
        for buf in (r.token_to_kv_pool.get_key_buffer(i), r.token_to_kv_pool.get_value_buffer(i)):
            buf.copy_(_randn(g, *buf.shape))
    ids = torch.randint(0, cfg.vocab_size, (c["requests"] if decode else sum(lens),), generator=g, device="cuda")
    fb = _batch(c, seed, r.req_to_token_pool, r.token_to_kv_pool, r.attn_backend, ids, decode)
    return types.SimpleNamespace(kind="model", runner=r, fb=fb, pool=r.token_to_kv_pool)


def _scan_sizes(c):
    kind = {"mamba2": "mamba2", "delta": "delta"}[c["rule"]]
    m = next(layer["mixer"] for layer in genusun.CONFIGS[c["model"]].layers if layer["type"] == kind)
    if kind == "mamba2":
        return dict(heads=m["heads"], groups=m["groups"], k=m["state"], v=m["vdim"])
    return dict(heads=m["heads"], groups=m["kv_heads"], k=m["dim"], v=m["vdim"])


def _scan(c, seed):
    g, s = _gen(seed), _scan_sizes(c)
    b, h, k, v = c["requests"], s["heads"], s["k"], s["v"]
    lens = _ragged(b, c["tokens"], c["spread"])
    t = sum(lens)
    act = torch.nn.functional.silu(_randn(g, t, (h * v + 2 * s["groups"] * k), dtype=F32)).to(BF)        # what the convolution in front leaves
    gates = _randn(g, t, 2 * h)
    a_log, bias = _randn(g, h, dtype=F32, scale=0.5), _randn(g, h, dtype=F32, scale=0.5) - 3.0
    state = _randn(g, b + 1, h, k, v, dtype=F32, scale=0.3)
    slots = torch.randperm(b, generator=g, device="cuda") + 1
    positions = torch.cat([torch.arange(c["start"], c["start"] + n) for n in lens]).cuda()
    if c["tokens"] == 1:
        seg = kernels.Segments()
    else:
        n = torch.tensor(lens)
        seg = kernels.Segments(torch.repeat_interleave(torch.arange(b, dtype=torch.int32), n).cuda(), (torch.cumsum(n, 0) - n).to(torch.int32).cuda(),
                               n.to(torch.int32).cuda(), max(lens))
    return types.SimpleNamespace(kind="scan", rule=c["rule"], act=act, gates=gates, a_log=a_log, bias=bias, skip=_randn(g, h, dtype=F32), state=state, slots=slots,
                                 positions=positions, seg=seg, sizes=s)


def run(state):
    s = state
    if s.kind == "extend":
        q, k, v = s.qkv[0]
        return {"out": s.layers[0](q, k, v, s.fb), "keys": s.pool.get_key_buffer(0), "values": s.pool.get_value_buffer(0)}
    if s.kind == "decode":
        s.graph.replay()
        n = len(s.layers)
        return {"out": s.out, "keys": [s.pool.get_key_buffer(i) for i in range(n)], "values": [s.pool.get_value_buffer(i) for i in range(n)]}
    if s.kind == "experts":
        return s.experts(s.x, s.topk(s.x, s.logits))
    if s.kind == "sample":
        return s.sampler(LogitsProcessorOutput(s.logits), s.info, positions=s.positions)
    if s.kind == "model":
        n = s.runner.config.num_hidden_layers
        logits = s.runner.forward(s.fb).next_token_logits
        return {"logits": logits, "keys": [s.pool.get_key_buffer(i) for i in range(n)], "values": [s.pool.get_value_buffer(i) for i in range(n)]}
    h = s.sizes["heads"]
    if s.rule == "mamba2":
        y = kernels.mamba2_scan(s.act, s.gates[:, :h], s.a_log, s.bias, s.skip, s.state, s.slots, s.positions, s.seg, s.sizes["groups"])
    else:
        y = kernels.gated_delta_scan(s.act, s.gates[:, :h], s.gates[:, h:], s.a_log, s.bias, s.state, s.slots, s.positions, s.seg, s.sizes["groups"],
                                     s.sizes["k"] ** -0.5)
    return {"out": y, "state": s.state}


# ------------------------------------------------------------------------------------------------ 64 bits
def _attend(q, k, v, scale, prefix):
    """q [n, Hq, D] at positions prefix .. prefix + n - 1 over k, v [m, Hkv, D], in 64 bits."""
    n, hq, d = q.shape
    m, hkv, _ = k.shape
    out = torch.empty((n, hq, d), dtype=F64, device=q.device)
    mask = torch.arange(m, device=q.device)[None, :] > prefix + torch.arange(n, device=q.device)[:, None]
    for j in range(hkv):
        qs = q[:, j * (hq // hkv):(j + 1) * (hq // hkv)].to(F64).transpose(0, 1).reshape(-1, d)
        p = (qs @ k[:, j].to(F64).T.contiguous() * scale).view(hq // hkv, n, m).masked_fill_(mask, float("-inf")).softmax(-1)
        out[:, j * (hq // hkv):(j + 1) * (hq // hkv)] = (p.view(-1, m) @ v[:, j].to(F64)).view(hq // hkv, n, d).transpose(0, 1)
    return out


def _rows(buf, fp8):
    return buf.view(FP8).to(F32) if fp8 else buf


def exact(case, seed):
    c = case
    if c["kind"] in ("extend", "decode"):
        s = _attention(c, seed)
        hq, hkv, d = _heads(c)
        fp8, decode, outs = c["kv"] == "fp8", c["kind"] == "decode", []
        table, lens = s.fb.req_to_token_pool.req_to_token, s.fb.seq_lens_cpu.tolist()
        new = [1] * len(lens) if decode else s.fb.extend_seq_lens_cpu
        kept = []
        for i, (q, k, v) in enumerate(s.qkv):
            kb, vb = s.pool.get_key_buffer(i), s.pool.get_value_buffer(i)
            kept.append((kb, vb))
            for buf, x in ((kb, k), (vb, v)):
                x = x.reshape(-1, hkv, d)
                buf[s.fb.out_cache_loc] = x.to(FP8).view(torch.uint8) if fp8 else x
            at, o = 0, []
            for b, n in enumerate(new):
                slots = table[s.fb.req_pool_indices[b], : lens[b]].long()
                o.append(_attend(q[at:at + n].reshape(n, hq, d), _rows(kb[slots], fp8), _rows(vb[slots], fp8), d ** -0.5, lens[b] - n))
                at += n
            outs.append(torch.cat(o).view(-1, hq * d))
        keys, values = ([None] * len(kept) if fp8 else [x[j].to(F64) for x in kept] for j in (0, 1))
        return {"out": outs, "keys": keys, "values": values} if decode else {"out": outs[0], "keys": keys[0], "values": values[0]}
    if c["kind"] == "experts":
        s = prepare(c, seed)
        w, ids = s.logits.to(F64).softmax(-1).sort(dim=-1, descending=True, stable=True)
        w, ids = w[:, : s.topk.top_k], ids[:, : s.topk.top_k]
        w = w / w.sum(-1, keepdim=True)
        y = torch.zeros(s.x.shape, dtype=F64, device="cuda")
        n = s.experts.w2_weight.shape[2]
        for e in range(s.experts.num_experts):
            tok, place = (ids == e).nonzero(as_tuple=True)
            u = s.x[tok].to(F64) @ s.experts.w13_weight[e].to(F64).T
            y.index_add_(0, tok, w[tok, place][:, None] * ((torch.nn.functional.silu(u[:, :n]) * u[:, n:]) @ s.experts.w2_weight[e].to(F64).T))
        return y
    if c["kind"] == "sample":
        return None
    if c["kind"] == "model":
        return _exact_model(c, seed)
    return _exact_scan(c, seed)


def _exact_model(c, seed):
    s = _model(c, seed)
    m, fb, model = s.runner.config, s.fb, s.runner.model
    hq, hkv, d = _heads(c)
    decode, lens, table = c["mode"] == "decode", s.fb.seq_lens_cpu.tolist(), s.fb.req_to_token_pool.req_to_token
    new = [1] * len(lens) if decode else fb.extend_seq_lens_cpu

    def norm(x, w):
        return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + m.rms_norm_eps) * w.weight.to(F64)

    def linear(x, layer):
        y = x @ layer.weight.to(F64).T
        return y if layer.bias is None else y + layer.bias.to(F64)

    ang = fb.positions.to(F64)[:, None] / m.rope_theta ** (torch.arange(0, d, 2, device="cuda", dtype=F64) / d)
    cos, sin = ang.cos()[:, None], ang.sin()[:, None]

    def turn(x):
        a, b = x[..., : d // 2], x[..., d // 2:]
        return torch.cat([a * cos - b * sin, b * cos + a * sin], -1)

    x, keys, values = model.embed_tokens[fb.input_ids].to(F64), [], []
    for i, layer in enumerate(model.layers):
        q, k, v = linear(norm(x, layer.input_layernorm), layer.self_attn.qkv_proj).split([hq * d, hkv * d, hkv * d], dim=-1)
        q, k, v = turn(q.view(-1, hq, d)), turn(k.reshape(-1, hkv, d)), v.reshape(-1, hkv, d)
        kb, vb = s.pool.get_key_buffer(i).to(F64), s.pool.get_value_buffer(i).to(F64)
        kb[fb.out_cache_loc], vb[fb.out_cache_loc] = k, v
        at, o = 0, []
        for b, n in enumerate(new):
            slots = table[fb.req_pool_indices[b], : lens[b]].long()
            o.append(_attend(q[at:at + n], kb[slots], vb[slots], d ** -0.5, lens[b] - n))
            at += n
        x = x + linear(torch.cat(o).view(-1, hq * d), layer.self_attn.o_proj)
        gate, up = linear(norm(x, layer.post_attention_layernorm), layer.mlp.gate_up_proj).chunk(2, dim=-1)
        x = x + linear(torch.nn.functional.silu(gate) * up, layer.mlp.down_proj)
        keys.append(kb)
        values.append(vb)
    x = norm(x, model.norm)
    if not decode:
        x = x[torch.cumsum(torch.tensor(new), 0).cuda() - 1]
    return {"logits": x @ model.lm_head.to(F64).T, "keys": keys, "values": values}


def _exact_scan(c, seed):
    s = _scan(c, seed)
    h, k, v, groups = s.sizes["heads"], s.sizes["k"], s.sizes["v"], s.sizes["groups"]
    lens = _ragged(c["requests"], c["tokens"], c["spread"])
    n, b = max(lens), len(lens)
    take = torch.zeros((b, n), dtype=torch.int64)
    live = torch.zeros((b, n), dtype=torch.bool)
    at = 0
    for i, m in enumerate(lens):
        take[i, :m], live[i, :m], at = torch.arange(at, at + m), True, at + m
    take, live = take.cuda(), live.cuda()
    act, gates = s.act[take].to(F64), s.gates[take].to(F64)
    decay, bias = -s.a_log.to(F64).exp(), s.bias.to(F64)
    softplus = lambda z: torch.logaddexp(z, torch.zeros_like(z))      # noqa: E731
    S = s.state[s.slots].to(F64) if c["start"] else torch.zeros((b, h, k, v), dtype=F64, device="cuda")
    out = torch.zeros((b, n, h, v), dtype=F64, device="cuda")
    wide = lambda x: x.repeat_interleave(h // groups, dim=2)          # noqa: E731
    if c["rule"] == "mamba2":
        x, B, C = act[..., : h * v].view(b, n, h, v), wide(act[..., h * v:h * v + groups * k].view(b, n, groups, k)), wide(act[..., h * v + groups * k:].view(b, n, groups, k))
        dt = softplus(gates[..., :h] + bias)
        for t in range(n):
            N = S * (decay * dt[:, t]).exp()[..., None, None] + (dt[:, t, :, None] * B[:, t])[..., None] * x[:, t, :, None, :]
            S = torch.where(live[:, t, None, None, None], N, S)
            out[:, t] = (C[:, t, :, None, :] @ S)[:, :, 0] + s.skip.to(F64)[:, None] * x[:, t]
    else:
        unit = lambda z: z / (z.square().sum(-1, keepdim=True) + 1e-6).sqrt()      # noqa: E731
        q, kk = wide(unit(act[..., : groups * k].view(b, n, groups, k))) * k ** -0.5, wide(unit(act[..., groups * k:2 * groups * k].view(b, n, groups, k)))
        x = act[..., 2 * groups * k:].view(b, n, h, v)
        beta, g = torch.sigmoid(gates[..., :h]), decay * softplus(gates[..., h:] + bias)
        for t in range(n):
            D = S * g[:, t].exp()[..., None, None]
            u = beta[:, t, :, None] * (x[:, t] - (kk[:, t, :, None, :] @ D)[:, :, 0])
            S = torch.where(live[:, t, None, None, None], D + kk[:, t, :, :, None] * u[:, :, None, :], S)
            out[:, t] = (q[:, t, :, None, :] @ S)[:, :, 0]
    state = s.state.to(F64)
    state[s.slots] = S
    return {"out": torch.cat([out[i, :m] for i, m in enumerate(lens)]).view(-1, h * v), "state": state}
