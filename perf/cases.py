"""Workloads of the framework's main paths with their inputs, their least work and their results in 64 bits.

Six kinds of case, each one pass through public entry points as a serving program makes it:

* ``step``     a captured decode step of the Qwen3-style decoder (``Qwen3ForCausalLM.forward`` over the paged cache)
* ``decode``   paged attention of one new token per sequence over long contexts, 16-bit or INT8 cache
* ``prefill``  the ``Attention`` layer over packed prompts or over cached prefixes, the cache store included
* ``memory``   the matrix memory of the recurrent design over prompts (``mlstm``)
* ``experts``  a mixture of experts with router, shared expert and the norm that sums it up (``SparseExperts``, ``stream_norm``)
* ``window``   prompts in sliding windows (``window_prefill``)

A case is a dict of plain values; lengths follow from its numbers alone, contents from the seed."""
from __future__ import annotations

import math
import random

import torch

DEVICE = "cuda"
EPS = 1e-6
DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}

# decoders: that of the engine benchmark, and those of about 1.7 and 8 billion parameters (some layers of them)
DECODERS = {"w1024": dict(width=1024, layers=8, heads=16, kv=8, ff=3072), "w2048": dict(width=2048, layers=8, heads=16, kv=8, ff=6144),
            "w4096": dict(width=4096, layers=4, heads=32, kv=8, ff=12288)}
# mixtures of experts of the same widths as the last two
MIXTURES = {"w2048": dict(width=2048, experts=64, top=6, ff=768, shared=1536), "w4096": dict(width=4096, experts=64, top=8, ff=1280, shared=2048)}
GROUPS, KEEP = 8, 4            # groups of experts, and how many of them a token may choose from
VOCAB = 32000
CAP_BYTES, CAP_FLOPS = 5.0e9, 6.0e11          # of drawn cases: below those of decode_long and experts_prompts


def listed():
    return [
        # one user waiting for the next token of a short conversation: the smallest call, launches and latency alone
        dict(name="step_one", kind="step", model="w1024", rows=1, low=300, high=300, block=256, most=512, lengths=1),
        # the engine benchmark's ordinary batch: 16 conversations, prompts of 32 to 96 tokens and up to 256 new ones
        dict(name="step_16", kind="step", model="w1024", rows=16, low=32, high=352, block=256, most=512, lengths=2),
        # a busier server on a decoder of 8 billion parameters' width, an odd number of requests
        dict(name="step_wide_61", kind="step", model="w4096", rows=61, low=64, high=1500, block=16, most=2048, lengths=3),
        # long contexts of very different lengths in one batch: memory bandwidth alone, the largest case
        dict(name="decode_long", kind="decode", batch=256, low=128, high=32768, heads=32, kv=8, dim=128, block=16, dtype="bf16", int8=False, lengths=4),
        # half the memory per token: the INT8 cache
        dict(name="decode_int8", kind="decode", batch=128, low=256, high=16384, heads=32, kv=8, dim=128, block=16, dtype="bf16", int8=True, lengths=6),
        # a ragged batch of new prompts
        dict(name="prefill_prompts", kind="prefill", prompts=16, low=64, high=2048, cached=0.0, heads=32, kv=8, dim=128, block=256, dtype="bf16", lengths=5),
        # follow-up turns: 90 % of what each conversation holds is cached, the smaller decoder's heads
        dict(name="prefill_turns", kind="prefill", prompts=7, low=500, high=6000, cached=0.9, heads=16, kv=8, dim=128, block=16, dtype="bf16", lengths=7),
        # a batch of prompts through a recurrent layer
        dict(name="memory_prompts", kind="memory", prompts=8, low=1024, high=1024, heads=16, dim=128, vdim=256, lengths=8),
        # the same prompts through a mixture of experts: the matrix unit alone
        dict(name="experts_prompts", kind="experts", model="w2048", rows=8192),
        # a short prompt, or a step that mixes one with decoded tokens: some rows for every expert
        dict(name="experts_mixed", kind="experts", model="w2048", rows=300),
        # a decode step of 32 requests through the wider mixture: most experts' weights for a row or two each
        dict(name="experts_decode", kind="experts", model="w4096", rows=32),
        # prompts through sliding-window attention, odd lengths
        dict(name="window_prompts", kind="window", prompts=5, low=700, high=4000, size=1024, heads=32, kv=8, dim=128, shared=False, lengths=9),
    ]


def _log_uniform(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    """One more case: every kind equally often, sizes over the whole range of the kind."""
    while True:
        kind = rng.choice(("step", "decode", "prefill", "memory", "experts", "window"))
        case = dict(kind=kind, lengths=rng.randrange(1 << 20))
        if kind == "step":
            high = _log_uniform(rng, 33, 2000)
            case.update(model=rng.choice(sorted(DECODERS)), rows=_log_uniform(rng, 1, 64), low=rng.randint(32, high), high=high,
                        block=rng.choice((16, 256)), most=2048)
        elif kind == "decode":
            high = _log_uniform(rng, 200, 32768)
            case.update(batch=_log_uniform(rng, 1, 256), low=rng.randint(16, high), high=high, kv=8, heads=rng.choice((16, 32)),
                        dim=rng.choice((64, 128, 128)), block=rng.choice((16, 256)), dtype=rng.choice(("bf16", "bf16", "fp16")),
                        int8=rng.random() < 0.3)
        elif kind == "prefill":
            high = _log_uniform(rng, 48, 8192)
            dtype = rng.choice(("bf16", "bf16", "bf16", "fp16", "fp32"))
            case.update(prompts=_log_uniform(rng, 1, 16), low=rng.randint(16, high), high=high, cached=rng.choice((0.0, 0.0, 0.5, 0.95)),
                        heads=rng.choice((16, 32)), kv=8, dim=64 if dtype == "fp32" else rng.choice((64, 128, 128)),
                        block=rng.choice((16, 256)), dtype=dtype)
        elif kind == "memory":
            high = _log_uniform(rng, 40, 8192)
            case.update(prompts=_log_uniform(rng, 1, 8), low=rng.randint(33, high), high=high, heads=rng.choice((8, 16)), dim=128, vdim=256)
        elif kind == "experts":
            del case["lengths"]
            case.update(model=rng.choice(sorted(MIXTURES)), rows=_log_uniform(rng, 1, 8192))
        else:
            high = _log_uniform(rng, 48, 8192)
            case.update(prompts=_log_uniform(rng, 1, 8), low=rng.randint(33, high), high=high, size=rng.choice((256, 512, 1024, 2048)),
                        heads=rng.choice((16, 32)), kv=8, dim=128, shared=rng.random() < 0.5)
        need = work(case)
        rows = sum(_lengths(case)) if kind in ("prefill", "memory", "window") else 0
        if need["bytes"] <= CAP_BYTES and need["flops"] <= CAP_FLOPS and rows <= 16384:
            return case


# ---- sizes and inputs ----

def _lengths(case):
    """Tokens of every sequence, cached ones included: spread over the logarithm of the range."""
    rng = random.Random(case["lengths"])
    return [_log_uniform(rng, case["low"], case["high"]) for _ in range(case.get("rows") or case.get("batch") or case["prompts"])]


def _new_lengths(case):
    """New tokens of every sequence of a prefill: what its cached prefix leaves, at least one."""
    return [max(n - int(n * case["cached"]), 1) for n in _lengths(case)]


def _random(seed):
    gen = torch.Generator(device=DEVICE).manual_seed(seed)

    def normal(*shape, std=1.0, mean=0.0, dtype=torch.bfloat16):
        return (torch.randn(shape, generator=gen, device=DEVICE) * std + mean).to(dtype)

    return gen, normal


def _tables(lengths, block, seed, width=0):
    """Block tables of sequences that took their blocks from a pool in use: int32 (sequences, width), and the pool's size."""
    need = [-(-n // block) for n in lengths]
    perm = torch.randperm(sum(need), generator=torch.Generator().manual_seed(seed)).to(torch.int32)
    tables = torch.full((len(need), max(width, max(need))), -1, dtype=torch.int32)
    at = 0
    for b, n in enumerate(need):
        tables[b, :n] = perm[at:at + n]
        at += n
    return tables, sum(need)


def _slots(tables, b, places, block):
    return tables[b].long()[places // block] * block + places % block


def _starts(lengths):
    return [0, *torch.tensor(lengths).cumsum(0).tolist()]


def _gather(cache, tables, b, n):
    """The first ``n`` rows of sequence ``b`` of a paged cache."""
    block = cache.shape[1]
    rows = cache[tables[b, :-(-n // block)].long().to(cache.device)]
    return rows.reshape(-1, *cache.shape[2:])[:n]


def _attend(q, k, v, scale, see=None, bias=None):
    """softmax(scale q k^T + bias) v of one kv head's query heads in 64 bits: q (rows, heads, dim), k and v (keys, dim)."""
    rows, heads, dim = q.shape
    s = (q.transpose(0, 1).reshape(heads * rows, dim) @ k.T).view(heads, rows, -1) * scale
    if bias is not None:
        s += bias
    if see is not None:
        s.masked_fill_(~see, float("-inf"))
    p = torch.softmax(s, -1).view(heads * rows, -1)
    return (p @ v).view(heads, rows, v.shape[-1]).transpose(0, 1)


# ---- a decode step of the Qwen3-style decoder ----

def _step_inputs(case, seed):
    z, lengths = DECODERS[case["model"]], _lengths(case)
    gen, normal = _random(seed)
    width, heads, kv, ff, dim = z["width"], z["heads"], z["kv"], z["ff"], 128
    weights = {"embedding_layer.weight": normal(VOCAB, width), "final_layernorm.weight": normal(width, std=0.1, mean=1.0)}
    for i in range(z["layers"]):
        p = f"layer_stack.{i}."
        weights.update({
            p + "input_layernorm.weight": normal(width, std=0.1, mean=1.0), p + "post_attention_layernorm.weight": normal(width, std=0.1, mean=1.0),
            p + "self_attn.rms_norm.weight": normal(dim, std=0.1, mean=1.0),
            p + "self_attn.qkv_projection.weight": normal((heads + 2 * kv) * dim, width, std=width ** -0.5),
            p + "self_attn.output_projection.weight": normal(width, heads * dim, std=(heads * dim) ** -0.5),
            p + "mlp.gate_up.weight": normal(2 * ff, width, std=width ** -0.5), p + "mlp.gate_down.weight": normal(width, ff, std=ff ** -0.5)})
    tables, blocks = _tables(lengths, case["block"], case["lengths"], -(-case["most"] // case["block"]))
    cache = normal(2, z["layers"], blocks, case["block"], kv, dim)
    ids = torch.randint(0, VOCAB, (len(lengths),), generator=gen, device=DEVICE)
    slots = torch.stack([_slots(tables, b, torch.tensor(n - 1), case["block"]) for b, n in enumerate(lengths)])
    return z, lengths, weights, tables, cache, ids, slots


def _prepare_step(case, seed):
    from minivllm_amd.layers.attention import decode_workspace_bytes
    from minivllm_amd.models.qwen3 import Qwen3ForCausalLM
    from minivllm_amd.utils.context import reset_context, set_context
    z, lengths, weights, tables, cache, ids, slots = _step_inputs(case, seed)
    with torch.device(DEVICE):
        model = Qwen3ForCausalLM(VOCAB, z["width"], z["heads"], 128, 1.0, z["kv"], EPS, base=1_000_000, max_position=case["most"],
                                 intermediate_size=z["ff"], ffn_bias=False, num_layers=z["layers"], block_size=case["block"], small_rows=64)
    model = model.to(torch.bfloat16).eval()
    model.load_state_dict(weights, strict=False)
    need = decode_workspace_bytes(len(lengths), z["heads"], 128, tables.shape[1], case["block"])
    workspace = torch.empty(max(need, 16), dtype=torch.uint8, device=DEVICE)
    for i, layer in enumerate(model.layer_stack):
        attention = layer.self_attn.attention
        attention.k_cache, attention.v_cache, attention.decode_workspace = cache[0, i], cache[1, i], workspace
    lens = torch.tensor(lengths, dtype=torch.int64, device=DEVICE)
    positions, slots, tables = lens - 1, slots.to(DEVICE), tables.to(DEVICE)
    # the step as a serving loop keeps it: one graph per batch size, replayed for every token
    with torch.no_grad():
        set_context(False, slot_mapping=slots, context_lens=lens, block_tables=tables)
        model(ids, positions)
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            hidden = model(ids, positions)
        reset_context()
    return dict(graph=graph, out=(hidden, cache), keep=(model, workspace, lens, positions, slots, tables, ids))


def _run_graph(state):
    state["graph"].replay()
    return state["out"]


def _exact_step(case, seed):
    z, lengths, weights, tables, cache, ids, slots = _step_inputs(case, seed)
    heads, kv, dim, rows = z["heads"], z["kv"], 128, len(lengths)
    w = lambda name: weights[name].double()
    rms = lambda t, g: t / torch.sqrt(t.pow(2).mean(-1, keepdim=True) + EPS) * g
    pos = torch.tensor(lengths, dtype=torch.float64, device=DEVICE) - 1
    angle = pos[:, None] * (1.0 / 1_000_000 ** (torch.arange(0, dim, 2, dtype=torch.float64, device=DEVICE) / dim))
    cos, sin = angle.cos()[:, None], angle.sin()[:, None]

    def turn(t):
        a, b = t.chunk(2, -1)
        return torch.cat([a * cos - b * sin, a * sin + b * cos], -1)

    x, cache = weights["embedding_layer.weight"][ids].double(), cache.double()
    slots = slots.to(DEVICE)
    for i in range(z["layers"]):
        p = f"layer_stack.{i}."
        qkv = rms(x, w(p + "input_layernorm.weight")) @ w(p + "self_attn.qkv_projection.weight").T
        q, k, v = qkv.split([heads * dim, kv * dim, kv * dim], -1)
        gamma = w(p + "self_attn.rms_norm.weight")
        q, k = turn(rms(q.view(rows, heads, dim), gamma)), turn(rms(k.view(rows, kv, dim), gamma))
        cache[0, i].view(-1, kv, dim)[slots] = k
        cache[1, i].view(-1, kv, dim)[slots] = v.reshape(rows, kv, dim)
        o = torch.empty_like(q)
        group = heads // kv
        for b, n in enumerate(lengths):
            keys, values = _gather(cache[0, i], tables, b, n), _gather(cache[1, i], tables, b, n)
            for h in range(kv):
                part = slice(h * group, (h + 1) * group)
                o[b:b + 1, part] = _attend(q[b:b + 1, part], keys[:, h], values[:, h], dim ** -0.5)
        x = x + o.reshape(rows, -1) @ w(p + "self_attn.output_projection.weight").T
        gate, up = (rms(x, w(p + "post_attention_layernorm.weight")) @ w(p + "mlp.gate_up.weight").T).chunk(2, -1)
        x = x + (gate * torch.sigmoid(gate) * up) @ w(p + "mlp.gate_down.weight").T
    return rms(x, w("final_layernorm.weight")), cache


def _work_step(case):
    z, lengths = DECODERS[case["model"]], _lengths(case)
    rows, dim = len(lengths), 128
    matrices = z["width"] * (2 * z["heads"] + 2 * z["kv"]) * dim + 3 * z["width"] * z["ff"]
    token = 2 * z["kv"] * dim * 2                                  # a token's key and value in one layer
    return {"bytes": z["layers"] * (2 * matrices + sum(lengths) * token + rows * token) + 2 * rows * z["width"] * 2,
            "flops": z["layers"] * (2 * rows * matrices + 4 * sum(lengths) * z["heads"] * dim)}


# ---- attention of one new token per sequence ----

def _decode_inputs(case, seed):
    lengths = _lengths(case)
    _, normal = _random(seed)
    dtype, kv, dim = DTYPES[case["dtype"]], case["kv"], case["dim"]
    tables, blocks = _tables(lengths, case["block"], case["lengths"])
    shape = (blocks, case["block"], kv, dim)
    q = normal(len(lengths), case["heads"], dim, dtype=dtype)
    caches, scales = [], []
    for _ in range(2):
        if not case["int8"]:
            cache = torch.empty(shape, dtype=dtype, device=DEVICE)
            for lo in range(0, blocks, 1 << 14):
                cache[lo:lo + (1 << 14)] = normal(*cache[lo:lo + (1 << 14)].shape, dtype=dtype)
        else:                                                      # codes up to 127 and scales as vectors of unit variance give them
            cache = torch.empty(shape, dtype=torch.int8, device=DEVICE)
            for lo in range(0, blocks, 1 << 14):
                part = cache[lo:lo + (1 << 14)]
                part.copy_((normal(*part.shape, dtype=torch.float32) * 45).clamp_(-127, 127).round_())
            scales.append(normal(*shape[:3], std=0.002, mean=0.022, dtype=torch.float32).clamp_(min=0.01))
        caches.append(cache)
    return lengths, q, tables, caches, scales


def _prepare_decode(case, seed):
    from minivllm_amd.layers.attention import paged_attention_decode, paged_attention_decode_int8
    lengths, q, tables, caches, scales = _decode_inputs(case, seed)
    tables, lens = tables.to(DEVICE), torch.tensor(lengths, dtype=torch.int64, device=DEVICE)
    call = paged_attention_decode_int8 if case["int8"] else paged_attention_decode
    return dict(call=call, args=(q, *caches, *scales, tables, lens, case["dim"] ** -0.5, case["heads"], case["kv"], case["dim"], case["block"]))


def _run_decode(state):
    return state["call"](*state["args"])


def _exact_decode(case, seed):
    lengths, q, tables, caches, scales = _decode_inputs(case, seed)
    group, out = case["heads"] // case["kv"], torch.empty(q.shape, dtype=torch.float64, device=DEVICE)
    for b, n in enumerate(lengths):
        k, v = (_gather(c, tables, b, n).double() for c in caches)
        if scales:
            k, v = (t * _gather(s, tables, b, n).double()[..., None] for t, s in zip((k, v), scales))
        for h in range(case["kv"]):
            part = slice(h * group, (h + 1) * group)
            out[b:b + 1, part] = _attend(q[b:b + 1, part].double(), k[:, h], v[:, h], case["dim"] ** -0.5)
    return out


def _work_decode(case):
    lengths = _lengths(case)
    vector = case["dim"] + 4 if case["int8"] else 2 * case["dim"]
    return {"bytes": 2 * sum(lengths) * case["kv"] * vector + 4 * len(lengths) * case["heads"] * case["dim"]
            + 4 * sum(-(-n // case["block"]) for n in lengths), "flops": 4 * sum(lengths) * case["heads"] * case["dim"]}


# ---- the attention layer over prompts ----

def _prefill_inputs(case, seed):
    lengths, new = _lengths(case), _new_lengths(case)
    _, normal = _random(seed)
    dtype, total = DTYPES[case["dtype"]], sum(new)
    q = normal(total, case["heads"], case["dim"], dtype=dtype)
    k, v = (normal(total, case["kv"], case["dim"], dtype=dtype) for _ in range(2))
    tables, blocks = _tables(lengths, case["block"], case["lengths"])
    cache = normal(2, blocks, case["block"], case["kv"], case["dim"], dtype=dtype)
    slots = torch.cat([_slots(tables, b, torch.arange(n - m, n), case["block"]) for b, (n, m) in enumerate(zip(lengths, new))])
    return lengths, new, q, k, v, tables, cache, slots


def _prepare_prefill(case, seed):
    from minivllm_amd.layers.attention import Attention
    lengths, new, q, k, v, tables, cache, slots = _prefill_inputs(case, seed)
    layer = Attention(case["heads"], case["dim"], 1.0, case["kv"], case["block"])
    layer.k_cache, layer.v_cache = cache[0], cache[1]
    cu_q, cu_k = (torch.tensor(_starts(n), dtype=torch.int32, device=DEVICE) for n in (new, lengths))
    context = (True, cu_q, cu_k, max(new), max(lengths), slots.to(DEVICE), None, tables.to(DEVICE) if case["cached"] else None)
    return dict(layer=layer, qkv=(q, k, v), cache=cache, context=context)


def _run_prefill(state):
    from minivllm_amd.utils.context import reset_context, set_context
    set_context(*state["context"])
    out = state["layer"](*state["qkv"])
    reset_context()
    return out, state["cache"]


def _exact_prefill(case, seed):
    lengths, new, q, k, v, tables, cache, slots = _prefill_inputs(case, seed)
    kv, dim, group = case["kv"], case["dim"], case["heads"] // case["kv"]
    cache, slots = cache.double(), slots.to(DEVICE)
    cache[0].view(-1, kv, dim)[slots] = k.double()
    cache[1].view(-1, kv, dim)[slots] = v.double()
    out, at = torch.empty(q.shape, dtype=torch.float64, device=DEVICE), 0
    for b, (n, m) in enumerate(zip(lengths, new)):
        keys, values = _gather(cache[0], tables, b, n), _gather(cache[1], tables, b, n)
        see = torch.arange(n, device=DEVICE)[None] <= torch.arange(n - m, n, device=DEVICE)[:, None]
        for h in range(kv):
            part = slice(h * group, (h + 1) * group)
            out[at:at + m, part] = _attend(q[at:at + m, part].double(), keys[:, h], values[:, h], dim ** -0.5, see)
        at += m
    return out.view(-1, case["heads"] * dim), cache


def _work_prefill(case):
    lengths, new = _lengths(case), _new_lengths(case)
    size, total = DTYPES[case["dtype"]].itemsize, sum(new)
    cached = sum(lengths) - total
    pairs = sum(m * (n - m) + m * (m + 1) // 2 for n, m in zip(lengths, new))
    return {"bytes": size * case["dim"] * (2 * total * case["heads"] + case["kv"] * (4 * total + 2 * cached)) + 8 * total,
            "flops": 4 * case["heads"] * case["dim"] * pairs}


# ---- the matrix memory over prompts ----

def _memory_inputs(case, seed):
    lengths = _lengths(case)
    _, normal = _random(seed)
    heads, dim, vdim, rows = case["heads"], case["dim"], case["vdim"], sum(_lengths(case))
    proj = normal(rows, heads * (2 * dim + 2 * vdim))
    gates = torch.cat([normal(rows, heads, dtype=torch.float32),
                       torch.nn.functional.logsigmoid(normal(rows, heads, mean=3.0, dtype=torch.float32))], 1).contiguous()
    return lengths, proj, gates, normal(heads * vdim, std=0.2, mean=1.0, dtype=torch.float32)


def _prepare_memory(case, seed):
    from minivllm_amd.engine.hybrid_cache import HybridCacheManager
    from minivllm_amd.engine.ragged import ragged_step
    from minivllm_amd.engine.sequence import Sequence
    from minivllm_amd.layers.recurrent import MlstmState
    lengths, proj, gates, weight = _memory_inputs(case, seed)
    heads, dim, vdim = case["heads"], case["dim"], case["vdim"]
    manager, seqs = HybridCacheManager([], 1, 16, len(lengths)), []
    for n in lengths:
        seq = Sequence([0] * n, block_size=16)
        manager.allocate(seq)
        seq.num_computed_tokens, seq.num_scheduled_tokens = 0, n
        seqs.append(seq)
    step = ragged_step(seqs, [], 16, torch.device(DEVICE, 0), heads * -(-vdim // 128))
    state = MlstmState.allocate(len(lengths), heads, dim, vdim, DEVICE)
    # prompts of 33 rows and more stay in the caller's order, and slots are given out in it
    return dict(step=step, args=(proj, gates, heads * (2 * dim + vdim), weight, state, EPS), state=state)


def _run_memory(state):
    from minivllm_amd.layers.recurrent import mlstm
    memory = state["state"]
    return mlstm(state["step"], *state["args"]), memory.s, memory.n, memory.m


def _exact_memory(case, seed):
    lengths, proj, gates, weight = _memory_inputs(case, seed)
    heads, dim, vdim = case["heads"], case["dim"], case["vdim"]
    starts, count, longest = _starts(lengths), len(lengths), max(lengths)

    def padded(t):                                                 # (longest, prompts, ...), zeros behind the shorter prompts
        rows = torch.zeros(count, longest, *t.shape[1:], dtype=torch.float64, device=DEVICE)
        for i, n in enumerate(lengths):
            rows[i, :n] = t[starts[i]:starts[i] + n].double()
        return rows.transpose(0, 1).contiguous()

    q, k, v, g = proj.split([heads * dim, heads * dim, heads * vdim, heads * vdim], -1)
    q, k, v = padded(q.unflatten(-1, (heads, dim))) * dim ** -0.5, padded(k.unflatten(-1, (heads, dim))), padded(v.unflatten(-1, (heads, vdim)))
    log_i, log_f = padded(gates[:, :heads]), padded(gates[:, heads:])
    s = torch.zeros(count, heads, dim, vdim, dtype=torch.float64, device=DEVICE)
    z, m = s.new_zeros(count, heads, dim), s.new_zeros(count, heads)
    lens = torch.tensor(lengths, device=DEVICE)
    outs = s.new_empty(longest, count, heads, vdim)
    for t in range(longest):
        live = (t < lens)[:, None]
        m_new = torch.where(live, torch.maximum(log_f[t] + m, log_i[t]), m)
        keep = torch.where(live, torch.exp(log_f[t] + m - m_new), torch.ones_like(m))
        add = torch.where(live, torch.exp(log_i[t] - m_new), torch.zeros_like(m))
        s.mul_(keep[..., None, None]).add_((add[..., None] * k[t])[..., None] * v[t][..., None, :])
        z, m = keep[..., None] * z + add[..., None] * k[t], m_new
        den = torch.maximum((z * q[t]).sum(-1).abs(), torch.exp(-m)) + 1e-6
        outs[t] = (s * q[t][..., None]).sum(-2) / den[..., None]
    rows = torch.cat([outs[:n, i] for i, n in enumerate(lengths)])
    rows = (rows / torch.sqrt(rows.pow(2).mean(-1, keepdim=True) + EPS)).reshape(-1, heads * vdim)
    return rows * weight.double() * torch.sigmoid(g.double()), s, z, m


def _work_memory(case):
    rows, heads, dim, vdim = sum(_lengths(case)), case["heads"], case["dim"], case["vdim"]
    return {"bytes": rows * heads * (2 * (2 * dim + 2 * vdim) + 2 * vdim + 8) + 4 * case["prompts"] * heads * (dim * (vdim + 1) + 1),
            # the state's update and its product with the query
            "flops": 4 * rows * heads * dim * vdim}


# ---- a mixture of experts ----

def _experts_inputs(case, seed):
    z = MIXTURES[case["model"]]
    _, normal = _random(seed)
    width, ff, shared, count = z["width"], z["ff"], z["shared"], z["experts"]
    linear = lambda *shape: normal(*shape, std=shape[-1] ** -0.5)
    weights = {"gate": linear(count, ff, width), "up": linear(count, ff, width), "down": linear(count, width, ff), "router": linear(count, width),
               "correction": normal(count, std=0.1, dtype=torch.float32), "shared.gate": linear(shared, width), "shared.up": linear(shared, width),
               "shared.down": linear(width, shared), "shared.sg": linear(1, width)}
    f32 = lambda *shape, std=0.1, mean=1.0: normal(*shape, std=std, mean=mean, dtype=torch.float32)
    frame = dict(x=normal(case["rows"], 2, width, dtype=torch.float32), out=f32(2), mix=f32(2, 2, std=0.05, mean=0.0) + torch.eye(2, device=DEVICE),
                 gain=f32(width), into=f32(2, mean=0.5), scale=f32(width, mean=0.7))
    return z, normal(case["rows"], width), weights, frame


def _prepare_experts(case, seed):
    from minivllm_amd.layers.experts import SparseExperts
    z, h, weights, frame = _experts_inputs(case, seed)
    layer = SparseExperts(z["width"], z["width"], z["experts"], z["top"], z["ff"], GROUPS, KEEP, z["shared"], small_rows=64)

    def get(name):
        if name[0] == "e" and name[1].isdigit():
            number, part = name[1:].split(".")
            return weights[part][int(number)]
        return weights[name]

    layer.load(get, lambda t: t.contiguous())
    state = dict(layer=layer.eval(), h=h, frame=frame)
    if case["rows"] <= 64:                                         # a decode step: captured, as a serving loop keeps it
        with torch.no_grad():
            _eager_experts(state)
            torch.cuda.synchronize()
            graph = torch.cuda.CUDAGraph()
            with torch.cuda.graph(graph):
                out = _eager_experts(state)
        state.update(graph=graph, out=out)
    return state


def _eager_experts(state):
    from minivllm_amd.layers.fused import stream_norm
    f = state["frame"]
    # the residual streams are kept as they are (as behind a model's last layer), so that a pass can be made again
    return stream_norm(f["x"], state["layer"](state["h"]), f["out"], f["mix"], f["gain"], EPS, f["into"], f["scale"], want_x=False)[0]


def _run_experts(state):
    if "graph" in state:
        return _run_graph(state)
    with torch.inference_mode():
        return _eager_experts(state)


def _exact_experts(case, seed):
    z, h, weights, f = _experts_inputs(case, seed)
    h, d = h.double(), lambda t: t.double()
    scores = torch.sigmoid(h @ d(weights["router"]).T)
    choice = scores + d(weights["correction"])
    groups = choice.view(len(h), GROUPS, -1)
    rank = groups.topk(2, -1).values.sum(-1)                       # a group counts with its two best
    kept = torch.zeros_like(rank, dtype=torch.bool).scatter_(1, rank.topk(KEEP, -1).indices, True)
    ids = groups.masked_fill(~kept[..., None], float("-inf")).view(len(h), -1).topk(z["top"], -1).indices
    weight = scores.gather(1, ids)
    weight = weight / weight.sum(-1, keepdim=True)
    unit = lambda t, gate, up, down: (torch.nn.functional.silu(t @ d(gate).T) * (t @ d(up).T)) @ d(down).T
    y = torch.sigmoid(h @ d(weights["shared.sg"]).T) * unit(h, weights["shared.gate"], weights["shared.up"], weights["shared.down"])
    for e in range(z["experts"]):
        rows, place = (ids == e).nonzero(as_tuple=True)
        if len(rows):
            y.index_add_(0, rows, weight[rows, place][:, None] * unit(h[rows], weights["gate"][e], weights["up"][e], weights["down"][e]))
    x = torch.einsum("st,nsw->ntw", d(f["mix"]), d(f["x"])) + d(f["out"])[None, :, None] * (d(f["scale"]) * y)[:, None]
    u = (d(f["into"])[None, :, None] * x).sum(1)
    return u / torch.sqrt(u.pow(2).mean(-1, keepdim=True) + EPS) * d(f["gain"])


def _work_experts(case):
    z, rows = MIXTURES[case["model"]], case["rows"]
    width, pairs = z["width"], rows * z["top"]
    used = z["experts"] * (1 - (1 - z["top"] / z["experts"]) ** rows)          # experts with a row, choices taken as even
    matrices = 3 * width * (used * z["ff"] + z["shared"]) + (z["experts"] + 1) * width
    return {"bytes": 2 * matrices + rows * width * (2 + 2 + 8), "flops": 6 * width * (pairs * z["ff"] + rows * z["shared"]) + 2 * rows * width * z["experts"]}


# ---- prompts in sliding windows ----

def _window_inputs(case, seed):
    lengths = _lengths(case)
    _, normal = _random(seed)
    rows, heads, kv, dim = sum(lengths), case["heads"], case["kv"], case["dim"]
    q, k = normal(rows, heads, dim), normal(rows, kv, dim)
    v = None if case["shared"] else normal(rows, kv, dim)
    gate = normal(rows, heads, dim) if case["shared"] else normal(rows, heads)          # of every channel, of every head
    slopes = torch.tensor([2.0 ** (-8.0 * (h + 1) / heads) for h in range(heads)], device=DEVICE) if case["shared"] else None
    return lengths, q, k, v, gate, slopes


def _prepare_window(case, seed):
    lengths, q, k, v, gate, slopes = _window_inputs(case, seed)
    cu = torch.tensor(_starts(lengths), dtype=torch.int32, device=DEVICE)
    options = dict(v=v, gate=gate)
    if case["shared"]:
        options.update(slopes=slopes, temperature=(0.1, 8192), positions=torch.cat([torch.arange(n, device=DEVICE) for n in lengths]))
    return dict(args=(q, k, cu, cu, case["dim"] ** -0.5, case["size"]), options=options)


def _run_window(state):
    from minivllm_amd.layers.window import window_prefill
    out = torch.empty_like(state["args"][0])
    window_prefill(out, *state["args"], **state["options"])
    return out


def _exact_window(case, seed):
    lengths, q, k, v, gate, slopes = _window_inputs(case, seed)
    group, out, at = case["heads"] // case["kv"], torch.empty(q.shape, dtype=torch.float64, device=DEVICE), 0
    for n in lengths:
        for lo in range(0, n, 2048):                               # rows in pieces, each with the keys its windows reach
            rows, first = torch.arange(lo, min(lo + 2048, n), device=DEVICE), max(lo - case["size"] + 1, 0)
            away = rows[:, None] - torch.arange(first, int(rows[-1]) + 1, device=DEVICE)[None]
            see = (away >= 0) & (away < case["size"])
            heat = 1 + 0.1 * torch.log(torch.floor((rows.double() + 1) / 8192) + 1) if case["shared"] else None
            for h in range(case["kv"]):
                part = slice(h * group, (h + 1) * group)
                queries = q[at + lo:at + int(rows[-1]) + 1, part].double()
                keys = k[at + first:at + int(rows[-1]) + 1, h].double()
                values = keys if v is None else v[at + first:at + int(rows[-1]) + 1, h].double()
                bias = None if slopes is None else -slopes[part].double()[:, None, None] * away
                if heat is not None:
                    queries = queries * heat[:, None, None]
                out[at + lo:at + int(rows[-1]) + 1, part] = _attend(queries, keys, values, case["dim"] ** -0.5, see, bias)
        at += n
    return out * torch.sigmoid(gate.double() if gate.dim() == 3 else gate.double()[..., None])


def _work_window(case):
    lengths, heads, kv, dim = _lengths(case), case["heads"], case["kv"], case["dim"]
    rows, size = sum(lengths), case["size"]
    pairs = sum(min(n, size) * (min(n, size) + 1) // 2 + max(n - size, 0) * size for n in lengths)
    gates = heads * dim if case["shared"] else heads
    return {"bytes": 2 * rows * (2 * heads * dim + (1 if case["shared"] else 2) * kv * dim + gates), "flops": 4 * heads * dim * pairs}


# ---- by kind ----

KINDS = {"step": (_prepare_step, _run_graph, _exact_step, _work_step), "decode": (_prepare_decode, _run_decode, _exact_decode, _work_decode),
         "prefill": (_prepare_prefill, _run_prefill, _exact_prefill, _work_prefill),
         "memory": (_prepare_memory, _run_memory, _exact_memory, _work_memory),
         "experts": (_prepare_experts, _run_experts, _exact_experts, _work_experts),
         "window": (_prepare_window, _run_window, _exact_window, _work_window)}


def prepare(case, seed):
    state = KINDS[case["kind"]][0](case, seed)
    state["run"] = KINDS[case["kind"]][1]
    return state


def run(state):
    return state["run"](state)


def work(case):
    need = KINDS[case["kind"]][3](case)
    return {"bytes": float(need["bytes"]), "flops": float(need["flops"])}


def tolerance(case):
    """About four times the distance from ``exact`` that the path shows: 16-bit roundings of a single operator are 2e-3 to 3e-3 of
    its result, those of four or eight layers on top of each other 0.8e-2 to 1.2e-2."""
    if case["kind"] == "step":
        return {"rel": 4e-2}
    return {"rel": 1e-5 if case.get("dtype") == "fp32" else 1e-2}


def exact(case, seed):
    return KINDS[case["kind"]][2](case, seed)
