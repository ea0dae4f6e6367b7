"""Niridra on the GPU: every mechanism against the plain oracle, and the model through its cache, batches and engine."""
import json
import math
import random

import numpy as np
import pytest
import torch

from minivllm_amd.engine import ragged
from minivllm_amd.engine.hybrid_runner import HybridModelRunner
from minivllm_amd.engine.ragged import ragged_step
from minivllm_amd.engine.sequence import Sequence
from minivllm_amd import _C
from minivllm_amd.layers.experts import ExpertOutput, SparseExperts, interleave_gate_up, moe_linear, moe_linear_tiles, moe_plan, moe_route
from minivllm_amd.layers.fused import stream_embed_norm, stream_norm
from minivllm_amd.layers.latent import head_linear, latent_decode, latent_norm_store, latent_width
from minivllm_amd.layers.mixers import DecayMemory, LatentAttention
from minivllm_amd.layers.recurrent import DecayMemoryState, decay_memory, gate_linear, gated_row_norm
from minivllm_amd.models.niridra import NiridraForCausalLM, engine_config
from minivllm_amd.sampling_parameters import SamplingParams
from niridra_cases import CONFIGS, config, latent_layer, lightning_layer, moe
from oracle import niridra_oracle as ref
from sokevik_cases import Driver, manager, tokens

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")
DTYPES = [torch.float32, torch.bfloat16]


def rel(got, want):
    """Root mean square error over the root mean square of the expected values."""
    got, want = got.detach().double().cpu(), want.double()
    assert got.shape == want.shape and bool(got.isfinite().all())
    return ((got - want).pow(2).mean().sqrt() / want.pow(2).mean().sqrt().clamp_min(1e-30)).item()


def row_rel(got, want):
    """The same of the worst row."""
    got, want = got.detach().double().cpu().flatten(1), want.double().flatten(1)
    assert got.shape == want.shape and bool(got.isfinite().all())
    return ((got - want).pow(2).mean(-1).sqrt() / want.pow(2).mean(-1).sqrt().clamp_min(1e-30)).max().item()


def tol(dtype, f32=2e-6, bf16=8e-3):
    return f32 if dtype == torch.float32 else bf16


def gen(seed):
    return torch.Generator().manual_seed(seed)


def make_step(lengths, before=None, slots=8, blocks=400, bs=16, units=1, m=None):
    """A step of sequences of which ``before[i]`` tokens are taken as computed already."""
    m = m or manager([0], blocks, bs, slots)
    seqs = []
    for i, n in enumerate(lengths):
        p0 = before[i] if before else 0
        s = Sequence([1] * (p0 + n), block_size=bs)
        m.allocate(s)
        s.num_computed_tokens, s.num_scheduled_tokens = p0, n
        seqs.append(s)
    return ragged_step(seqs, [0], bs, DEV, units, latent=True), seqs, m


# ---- residual streams, embedding ----
STREAM_SHAPES = [(1, 80), (2, 97), (3, 512), (4, 64), (5, 1028), (8, 320), (2, 4100), (6, 36), (7, 2050)]


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("streams,width", STREAM_SHAPES)
@pytest.mark.parametrize("rows", [1, 7, 600])
def test_stream_norm(dtype, streams, width, rows):
    g, eps, padded = gen(width), 1e-2, -(-width // 64) * 64
    r = lambda *s: torch.randn(*s, generator=g)
    x, y = r(rows, streams, width), r(rows, width).to(dtype)
    out_w, mix, in_w, gain, scale = r(streams), r(streams, streams), r(streams), r(width), r(width)
    on = lambda t: None if t is None else t.to(DEV)
    for use_in, use_scale, want_x in ((True, True, True), (False, False, False)):
        yy = y.double() * (scale.double() if use_scale else 1.0)
        want_streams = torch.einsum("st,nsw->ntw", mix.double(), x.double()) + out_w.double()[:, None] * yy[:, None]
        u = (want_streams * (in_w.double()[:, None] if use_in else 1.0)).sum(1)
        mine = on(x).clone()
        h, new = stream_norm(mine, on(y), on(out_w), on(mix), on(gain), eps, on(in_w) if use_in else None,
                             on(scale) if use_scale else None, padded, want_x)
        assert rel(h[:, :width], ref.rms(u, eps) * gain.double()) < tol(dtype, 4e-6, 4e-3) and not h[:, width:].any()
        if want_x:
            assert rel(new, want_streams) < 2e-6
        else:
            assert torch.equal(mine.cpu(), x)                          # nobody asked for the streams: they stay


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("width", [80, 97, 1028])
@pytest.mark.parametrize("top,shared,gated,sorted_rows", [(1, True, True, False), (3, False, False, True), (6, True, False, True), (4, True, True, True)])
def test_stream_norm_of_a_mixture(dtype, width, top, shared, gated, sorted_rows):
    """The weighted sum of the experts' rows wherever they lie, and the shared expert behind its gate."""
    g, rows, streams, eps = gen(width + top), 37, 2, 1e-3
    r = lambda *s: torch.randn(*s, generator=g)
    x, parts, weights, y = r(rows, streams, width), r(rows * top, width + 8).to(dtype), r(rows, top), r(rows, width).to(dtype)
    gates, out_w, mix, gain = r(rows, 5), r(streams), r(streams, streams), r(width)
    place = torch.randperm(rows * top, generator=g).int() if sorted_rows else None
    at = torch.arange(rows * top) if place is None else place.long()
    want = (weights.double()[..., None] * parts.double()[at][:, :width].view(rows, top, width)).sum(1)
    if shared:
        want = want + y.double() * (torch.sigmoid(gates[:, 3:4].double()) if gated else 1.0)
    streams_want = torch.einsum("st,nsw->ntw", mix.double(), x.double()) + out_w.double()[:, None] * want[:, None]
    out = ExpertOutput(parts.to(DEV), weights.to(DEV), None if place is None else place.to(DEV), y.to(DEV) if shared else None,
                       gates.to(DEV)[:, 3] if gated else None)
    h, new = stream_norm(x.to(DEV), out, out_w.to(DEV), mix.to(DEV), gain.to(DEV), eps)
    assert rel(new, streams_want) < 2e-6 and rel(h, ref.rms(streams_want.sum(1), eps) * gain.double()) < tol(dtype, 4e-6, 4e-3)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("streams,width", [(1, 80), (3, 97), (4, 1028)])
def test_stream_embedding_over_portions(dtype, streams, width):
    """Every cut gives the same rows: the token before a portion is state; slots come round with another sequence's token."""
    g, eps, hashing = gen(width), 1e-3, (37, 70001, 90007)
    embed, bigram = torch.randn(50, width, generator=g).to(dtype), torch.randn(38, width, generator=g).to(dtype)
    in_w, gain = torch.randn(streams, generator=g), torch.randn(width, generator=g)
    m = manager([0], 40, 16, 3)
    prev = torch.full((7,), 12345, dtype=torch.int64, device=DEV)
    cfg = {"scale": 3.5, "bigram": dict(zip(("buckets", "mul_prev", "mul_cur"), hashing))}
    for round_ in range(3):
        toks = {k: tokens(10 * round_ + k, n, 50) for k, n in enumerate((61, 9, 40))}
        want = {k: ref.embedding(t, {"embed": embed.double(), "bigram": bigram.double()}, cfg) for k, t in toks.items()}
        seqs, at, rng = {}, dict.fromkeys(toks, 0), random.Random(round_)
        while at:
            live = [k for k in at if rng.random() < 0.7] or [next(iter(at))]
            for k in live:
                if k not in seqs:
                    seqs[k] = Sequence(toks[k], block_size=16)
                    m.allocate(seqs[k])
                seqs[k].num_computed_tokens = at[k]
                seqs[k].num_scheduled_tokens = min(rng.choice([1, 1, 2, 3, 20]), len(toks[k]) - at[k])
            step = ragged_step([seqs[k] for k in live], [0], 16, DEV, latent=True)
            h, x = stream_embed_norm(step, step.input_ids, embed.to(DEV), 3.5, streams, gain.to(DEV), eps, in_w.to(DEV),
                                     bigram.to(DEV), hashing, prev, width + 3)
            for i, k in enumerate(live):
                n = seqs[k].num_scheduled_tokens
                rows, e = slice(step.starts[i], step.starts[i] + n), want[k][at[k]:at[k] + n]
                assert rel(x[rows], e[:, None].expand(-1, streams, -1)) < 1e-6
                assert rel(h[rows, :width], ref.rms(e * in_w.double().sum(), eps) * gain.double()) < tol(dtype, 4e-6, 4e-3)
                at[k] += n
                if at[k] == len(toks[k]):
                    m.deallocate(seqs.pop(k))
                    del at[k]


def test_stream_embedding_alone():
    embed, ids = torch.randn(30, 72, generator=gen(1)), torch.tensor([3, 29, 0, 3], device=DEV)
    step, _, _ = make_step([4])
    h, x = stream_embed_norm(step, ids, embed.to(DEV), 2.0, 2, torch.ones(72, device=DEV), 1e-5)
    assert torch.equal(x.cpu(), (embed[ids.cpu()] * 2)[:, None].expand(-1, 2, -1)) and rel(h, ref.rms(embed[ids.cpu()].double() * 4, 1e-5)) < 1e-6


# ---- matrix memory with constant decays ----
def memory_case(seed, rows, heads, dim, vdim, dtype, std=1.0):
    n = heads * (2 * dim + vdim)
    return (torch.randn(rows, -(-(n + heads * vdim) // 8) * 8, generator=gen(seed)) * std).to(dtype)


def memory_reference(proj, heads, dim, vdim, decay, silu=True):
    act = ref.silu if silu else (lambda z: z)
    p, rows = proj.double(), proj.shape[0]
    q, k = (act(p[:, i * heads * dim:(i + 1) * heads * dim]).view(rows, heads, dim) for i in range(2))
    v = act(p[:, 2 * heads * dim:heads * (2 * dim + vdim)]).view(rows, heads, vdim)
    return ref.decaying_memory(q, k, v, torch.tensor(decay, dtype=torch.float64)).reshape(rows, -1)


MEMORY_SHAPES = [(3, 24, 40), (2, 64, 64), (1, 128, 136), (2, 200, 72), (2, 20, 12), (1, 256, 264), (1, 300, 20), (2, 8, 130)]


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("heads,dim,vdim", MEMORY_SHAPES)
@pytest.mark.parametrize("cuts", [[300], [64, 64, 172], [1] * 12 + [31, 33, 2, 200, 1, 21], [190, 110]], ids=str)
def test_decay_memory_portions(dtype, heads, dim, vdim, cuts):
    """Any portions give the rows of the token-by-token recurrence: rows one by one, in blocks, across steps."""
    rows, decay = sum(cuts), [0.35 + 0.64 * i / heads for i in range(heads)]
    proj = memory_case(dim + vdim, rows, heads, dim, vdim, dtype)
    want = memory_reference(proj, heads, dim, vdim, decay)
    m = manager([], 1, 16, 2)
    s = Sequence([1] * rows, block_size=16)
    m.allocate(s)
    state = DecayMemoryState.allocate(2, decay, dim, vdim, DEV)
    state.s.fill_(float("nan"))                                       # what a slot held before must not matter
    at, got = 0, []
    for n in cuts:
        s.num_computed_tokens, s.num_scheduled_tokens = at, n
        got.append(decay_memory(ragged_step([s], [], 16, DEV, 1), proj[at:at + n].to(DEV), state).cpu())
        at += n
    got = torch.cat(got)
    assert rel(got, want) < tol(dtype, 2e-6, 5e-3) and row_rel(got, want) < tol(dtype, 2e-5, 3e-2)


@pytest.mark.parametrize("silu", [True, False])
@pytest.mark.parametrize("decay", [[0.0, 1.0], [1e-30, 0.9999], [0.01, 0.2]])
def test_decay_memory_extreme_decays(decay, silu):
    """Everything forgotten at once, nothing ever, and a first token that still counts hundreds of rows later."""
    heads, dim, vdim, rows = 2, 64, 72, 400
    proj = memory_case(1, rows, heads, dim, vdim, torch.bfloat16)
    proj[0] *= 8.0                                                    # one key and value stand out
    want = memory_reference(proj, heads, dim, vdim, decay, silu)
    for cut in (400, 97, 30):                                         # blocks; blocks with ends; row by row
        s, m = Sequence([1] * rows, block_size=16), manager([], 1, 16, 2)
        m.allocate(s)
        state, got = DecayMemoryState.allocate(2, decay, dim, vdim, DEV), []
        for at in range(0, rows, cut):
            s.num_computed_tokens, s.num_scheduled_tokens = at, min(cut, rows - at)
            got.append(decay_memory(ragged_step([s], [], 16, DEV, 1), proj[at:at + cut].to(DEV), state, silu).cpu())
        got = torch.cat(got)
        assert rel(got, want) < 6e-3 and rel(got[300:], want[300:]) < 6e-3, cut


@pytest.mark.parametrize("heads,dim,vdim", [(2, 64, 64), (1, 136, 200), (3, 24, 40)])
def test_decay_memory_segments_side_by_side(monkeypatch, heads, dim, vdim):
    """Long portions cut into segments (here of one block), several entries, a state to go on from: as in one piece."""
    monkeypatch.setattr(ragged, "MIN_SEGMENT_ROWS", 64)
    lengths, before, decay = [1, 333, 64, 20, 129, 700], [4, 0, 70, 0, 65, 3], [0.999 - 0.3 * i for i in range(heads)]
    m = manager([], 1, 16, 8)
    state = DecayMemoryState.allocate(8, decay, dim, vdim, DEV)
    cases, outs, seqs = [], {i: [] for i in range(len(lengths))}, []
    for i, (n, p) in enumerate(zip(lengths, before)):
        cases.append(memory_case(50 + i, n + p, heads, dim, vdim, torch.bfloat16))
        seqs.append(Sequence([1] * (n + p), block_size=16))
        m.allocate(seqs[-1])
    for phase in (0, 1):
        live = [i for i in range(len(lengths)) if phase == 1 or before[i]]
        for i in live:
            seqs[i].num_computed_tokens = before[i] if phase else 0
            seqs[i].num_scheduled_tokens = lengths[i] if phase else before[i]
        step = ragged_step([seqs[i] for i in live], [], 16, DEV, 1)
        if phase:
            assert step.split and step.segments.shape[0] > 10
        part = lambda i: slice(seqs[i].num_computed_tokens, seqs[i].num_computed_tokens + seqs[i].num_scheduled_tokens)
        out = decay_memory(step, torch.cat([cases[live[e]][part(live[e])] for e in step.order]).to(DEV), state).cpu()
        for j, i in enumerate(live):
            outs[i].append(out[step.starts[j]:step.starts[j] + seqs[i].num_scheduled_tokens])
    for i in range(len(lengths)):
        assert rel(torch.cat(outs[i]), memory_reference(cases[i], heads, dim, vdim, decay)) < 5e-3, i


@pytest.mark.parametrize("width", [8, 520, 2048, 2056, 8192, 8200])       # up to 8192 in chunks of eight, where rows are multiples of 16 bytes
@pytest.mark.parametrize("top", [1, 2, 3, 4, 7, 9])
@pytest.mark.parametrize("rows,odd", [(5, 0), (5, 4), (530, 0)])
def test_stream_norm_of_a_mixture_in_wide_chunks(width, top, rows, odd):
    """Two streams, a shared row behind a gate, choices that hand their input on (their places are -1); the streams are fp32 sums, so 4e-6, the output
    rounds to 16 bits, 4e-3."""
    g = gen(width + top)
    x, y, own = torch.randn(rows, 2, width, generator=g), torch.randn(rows, width, generator=g).bfloat16(), torch.randn(rows, width, generator=g).bfloat16()
    parts, weights = torch.randn(rows * top, width + odd, generator=g).bfloat16(), torch.rand(rows, top, generator=g)
    ids = torch.randint(-1, 3, (rows, top), generator=g).int()
    live = ids.view(-1) >= 0
    place = torch.full((rows * top,), -1)
    place[live] = torch.randperm(rows * top, generator=g)[:int(live.sum())]
    gate, out_w, mix, in_w, scale, gain = (torch.randn(n, generator=g) for n in (rows, 2, 4, 2, width, width))
    each = torch.where(live[:, None], parts[place.clamp(min=0), :width].double(), own.double().repeat_interleave(top, 0)).view(rows, top, width)
    total = torch.sigmoid(gate.double())[:, None] * y.double() + (weights.double()[..., None] * each).sum(1)
    new = torch.einsum("st,nsw->ntw", mix.view(2, 2).double(), x.double()) + out_w.double()[None, :, None] * (scale.double() * total)[:, None]
    u = (in_w.double()[None, :, None] * new).sum(1)
    on = lambda t: t.to(DEV)
    out = ExpertOutput(on(parts)[:, :width], on(weights), on(place.int()), on(y), on(gate), on(ids), on(own))
    h, mine = stream_norm(on(x), out, on(out_w), on(mix.view(2, 2)), on(gain), 1e-3, on(in_w), on(scale))
    assert rel(mine, new) < 4e-6 and rel(h, ref.rms(u, 1e-3) * gain.double()) < 4e-3


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("width", [36, 97, 640, 4096, 5000])
@pytest.mark.parametrize("rows", [3, 600])
def test_gated_row_norm(dtype, width, rows):
    g = gen(width)
    x, weight = torch.randn(rows, width, generator=g), torch.randn(width, generator=g)
    gate = torch.randn(rows, width + 12, generator=g).to(dtype)
    want = ref.rms(x.double(), 1e-2) * weight.double() * torch.sigmoid(gate[:, 4:4 + width].double())
    assert rel(gated_row_norm(x.to(DEV), weight.to(DEV), gate.to(DEV)[:, 4:4 + width], 1e-2), want) < tol(dtype, bf16=4e-3)


# ---- latents ----
@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("rank", [8, 40, 72, 96, 150, 512, 530, 1500, 2048])
def test_latent_norm_store(dtype, rank):
    g, rows, padded = gen(rank), 37, latent_width(rank)
    x = torch.randn(rows, padded + 8, generator=g).to(dtype)
    weight, slots = torch.randn(rank, generator=g), torch.randperm(64, generator=g)[:rows].clone()
    slots[::5] = -1
    cache = torch.full((4, 16, padded), 7.0, dtype=dtype, device=DEV)
    out = latent_norm_store(x.to(DEV)[:, :padded], weight.to(DEV), 1e-2, cache, slots.to(DEV)).cpu()
    assert rel(out[:, :rank], ref.rms(x[:, :rank].double(), 1e-2) * weight.double()) < tol(dtype, bf16=4e-3) and not out[:, rank:].any()
    flat = cache.cpu().view(64, padded)
    for t in range(rows):
        if slots[t] >= 0:
            assert torch.equal(flat[slots[t]], out[t])
    assert bool((flat[[i for i in range(64) if i not in slots.tolist()]] == 7.0).all())
    assert latent_norm_store(x.to(DEV)[:, :padded], weight.to(DEV), 1e-2, cache, slots.to(DEV), need_rows=False) is None


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("heads,n,k", [(1, 16, 8), (3, 48, 40), (5, 96, 64), (18, 192, 32), (2, 512, 128), (4, 128, 544)])
@pytest.mark.parametrize("rows", [1, 16, 45])
def test_head_linear(dtype, heads, n, k, rows):
    g = gen(n + k)
    x = torch.randn(rows, heads * k + 16, generator=g).to(dtype)
    w = (torch.randn(heads, n, k, generator=g) * k ** -0.5).to(dtype)
    want = torch.einsum("thk,hnk->thn", x[:, 8:8 + heads * k].double().view(rows, heads, k), w.double())
    view = x.to(DEV)[:, 8:8 + heads * k].unflatten(-1, (heads, k))
    assert rel(head_linear(view, w.to(DEV)), want) < tol(dtype, bf16=4e-3)
    out = torch.zeros(rows + 2, heads, n, dtype=dtype, device=DEV)
    head_linear(view, w.to(DEV), out=out[1:-1])
    assert rel(out[1:-1], want) < tol(dtype, bf16=4e-3) and not out[0].any() and not out[-1].any()


def latent_case(seed, lens, heads, padded, dtype, bs, entries=None):
    """Queries over cached latents; row i answers from entry ``entries[i]`` (its own by default)."""
    g = gen(seed)
    entries = list(range(len(lens))) if entries is None else entries
    need = [max(-(-max(n for n, e in zip(lens, entries) if e == i) // bs), 1) for i in range(max(entries) + 1)]
    order, width = torch.randperm(sum(need) + 3, generator=g), max(need) + 2
    tables, at = torch.full((len(need), width), -1, dtype=torch.int32), 0
    for i, n in enumerate(need):
        tables[i, :n] = order[at:at + n].int()
        at += n
    cache = torch.randn(sum(need) + 3, bs, padded, generator=g).to(dtype)
    q = torch.randn(len(lens), heads, padded, generator=g).to(dtype)
    rows = [cache[tables[e, :need[e]].long()].reshape(-1, padded)[:n].double() for n, e in zip(lens, entries)]
    return q, cache, tables, torch.tensor(entries, dtype=torch.int32), torch.tensor(lens), rows


def latent_reference(q, rows, scale):
    return torch.stack([torch.softmax(q[i].double() @ c.T * scale, -1) @ c if len(c) else torch.zeros_like(q[i]).double() for i, c in enumerate(rows)])


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("padded", [32, 64, 96, 128, 192, 256, 384, 512, 544, 1056, 2048])
@pytest.mark.parametrize("heads", [1, 5, 16, 18, 40])
def test_latent_decode(dtype, padded, heads):
    for bs, lens in ((16, [1, 2, 15, 16, 17, 63, 64, 65, 128, 129, 700]), (48, [300, 1])):
        q, cache, tables, entry, lengths, rows = latent_case(padded + heads, lens, heads, padded, dtype, bs)
        scale = 1.5 * padded ** -0.5
        got = latent_decode(q.to(DEV), cache.to(DEV), tables.to(DEV), entry.to(DEV), lengths.to(DEV), scale)
        want = latent_reference(q, rows, scale)
        assert rel(got, want) < tol(dtype, 2e-6, 6e-3) and row_rel(got, want) < tol(dtype, 1e-5, 1.5e-2), bs


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("padded", [32, 64, 96])
def test_latent_decode_joins_many_shares_of_narrow_rows(dtype, padded):
    """More shares than the pass that joins them has lanes with columns."""
    q, cache, tables, entry, lengths, rows = latent_case(padded, [5000, 3, 2049], 2, padded, dtype, 16)
    got = latent_decode(q.to(DEV), cache.to(DEV), tables.to(DEV), entry.to(DEV), lengths.to(DEV), 0.2)
    assert row_rel(got, latent_reference(q, rows, 0.2)) < tol(dtype, 1e-5, 1.5e-2)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("padded,heads", [(96, 4), (512, 32), (160, 3)])
def test_latent_decode_finds_single_keys(dtype, padded, heads):
    """One score stands out: first and last keys, both sides of page and tile borders, far back; one past the end never."""
    length = 2100
    q, cache, tables, entry, lengths, rows = latent_case(7, [length] * 2, heads, padded, dtype, 16)
    flat = lambda p: (int(tables[0, p // 16]), p % 16)
    for p in (0, 1, 15, 16, 63, 64, 65, 127, 128, 1000, 1023, 1024, 2047, 2048, 2098, 2099):
        target = rows[0][p].to(dtype)
        q[0] = target * (60.0 / float(target.double() @ target.double()))
        got = latent_decode(q.to(DEV), cache.to(DEV), tables.to(DEV), entry.to(DEV), lengths.to(DEV), 1.0)
        assert rel(got[0], target.double().expand(heads, -1)) < tol(dtype, 1e-3, 1e-2), p
        short = torch.tensor([max(p, 0), length])                      # the key is the first one not seen
        got = latent_decode(q.to(DEV), cache.to(DEV), tables.to(DEV), entry.to(DEV), short.to(DEV), 1.0)
        assert rel(got, latent_reference(q, [rows[0][:p], rows[1]], 1.0)) < tol(dtype, 2e-5, 2e-2), p
        assert flat(p) in [(int(b), o) for b in tables[0, :-2] for o in range(16)]


@pytest.mark.parametrize("dtype", DTYPES)
def test_latent_decode_rows_of_one_entry(dtype):
    """Several rows of an entry, each with a length of its own, beside another's; none at all gives zeros."""
    lens, entries = [33, 34, 35, 200, 0], [0, 0, 0, 1, 1]
    q, cache, tables, entry, lengths, rows = latent_case(3, lens, 6, 64, dtype, 16, entries)
    got = latent_decode(q.to(DEV), cache.to(DEV), tables.to(DEV), entry.to(DEV), lengths.to(DEV), 0.3)
    assert rel(got, latent_reference(q, rows, 0.3)) < tol(dtype, 2e-6, 6e-3) and not got[4].any()


# ---- latent attention as a layer ----
def latent_module(cfg, width, dtype, eps=1e-3, source=None, seed=0, weights=None):
    c = cfg["mixer"]
    w = weights or {k[len("l0.mix."):]: t for k, t in ref.random_weights(config([{**cfg, "mixer": {**c, "kv_from": None}}], width=width), seed).items()
                    if k.startswith("l0.mix.")}
    m = LatentAttention(width, c["heads"], c["dim"], c["vdim"], c["kv_rank"], c["scale"], 0, 16, dtype, eps, source, 64)
    m.load(lambda n: w[n], lambda t: t.to(DEV, dtype).contiguous(), width)
    return m, {k: t.double() for k, t in w.items()}


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("heads,dim,vdim,rank", [(5, 40, 24, 72), (2, 64, 64, 64), (18, 16, 48, 150), (1, 128, 8, 512), (3, 24, 136, 40), (4, 200, 100, 300)])
@pytest.mark.parametrize("cuts", [[200], [1] * 40 + [2] * 20, [31, 32, 33, 1, 2, 70, 31], [150, 50], [17, 183]], ids=str)
def test_latent_attention_portions(dtype, heads, dim, vdim, rank, cuts):
    """Peaked scores: absorbed rows, long portions behind cached ones and from the start all give the whole sequence's rows,
    the layer's own latents and, through other heads, a later layer's that reads them."""
    width, rows, eps = 96, sum(cuts), 1e-3
    cfg = latent_layer(heads, dim, vdim, rank, 2.0 * dim ** -0.5)
    own, w = latent_module(cfg, width, dtype)
    later_cfg = latent_layer(heads + 1, max(dim // 2 // 8 * 8, 8), vdim + 8, rank, -0.5)
    later, w2 = latent_module(later_cfg, width, dtype, source=own, seed=5)
    own.cache = torch.full((20, 16, own.latent_width), 3.0, dtype=dtype, device=DEV)
    h, h2 = (torch.randn(rows, width, generator=gen(i)).to(dtype) for i in (8, 9))
    c = ref.latent(h.double(), w, "", eps)
    want, want2 = ref.latent_attention(h.double(), c, w, "", cfg["mixer"]), ref.latent_attention(h2.double(), c, w2, "", later_cfg["mixer"])
    m = manager([0], 20, 16, 2)
    s = Sequence([1] * rows, block_size=16)
    m.allocate(s)
    got, got2, at = [], [], 0
    for n in cuts:
        s.num_computed_tokens, s.num_scheduled_tokens = at, n
        step = ragged_step([s], [0], 16, DEV, latent=True)
        got.append(own(h[at:at + n].to(DEV), step).cpu())
        got2.append(later(h2[at:at + n].to(DEV), step).cpu())
        at += n
    for g, x in ((torch.cat(got), want), (torch.cat(got2), want2)):
        assert rel(g, x) < tol(dtype, 5e-6, 2e-2) and row_rel(g, x) < tol(dtype, 1e-4, 0.15)


@pytest.mark.parametrize("dtype", DTYPES)
def test_latent_attention_single_keys_in_every_path(dtype):
    """Queries that pick one key each (the first, at page borders, their own, far back), in single rows, short and long
    portions; entries of one batch with shuffled blocks."""
    heads, dim, rank, n = 2, 48, 96, 330
    width, g = heads * dim + rank + 32, gen(2)
    eye = torch.eye(width)
    w = {"q": eye[:heads * dim].bfloat16(), "dkv": eye[heads * dim:heads * dim + rank].bfloat16(), "dkv.norm": torch.ones(rank).bfloat16(),
         "uk": (torch.randn(heads * dim, rank, generator=g) * rank ** -0.5).bfloat16(),
         "uv": (torch.randn(heads * dim, rank, generator=g) * rank ** -0.5).bfloat16(),
         "o": torch.nn.functional.pad(torch.eye(heads * dim), (0, 0, 0, width - heads * dim)).bfloat16()}
    cfg = latent_layer(heads, dim, dim, rank, 1.0)
    m, wd = latent_module(cfg, width, dtype, 1e-5, weights=w)
    h = torch.randn(2, n, width, generator=g)
    target = {}
    for b in range(2):
        c = ref.latent(h[b].double(), wd, "", 1e-5)
        k = (c @ wd["uk"].T).view(n, heads, dim)
        for i in range(n):
            j = [0, 15, 16, 31, 32, 63, 64, i, max(i - 1, 0), i - i % 16, i // 2, max(i - i % 16 - 1, 0)][i % 12]
            target[b, i] = j = min(j, i)
            h[b, i, :heads * dim] = (k[j] * 40 / k[j].pow(2).sum(-1, keepdim=True)).reshape(-1).float()
    h = h.to(dtype)
    want = [ref.latent_attention(x.double(), ref.latent(x.double(), wd, "", 1e-5), wd, "", cfg["mixer"]) for x in h]
    for cuts in ([n], [300] + [1] * 30, [20, 2, 3, 32, 1, 200, 31, 41], [64] * 5 + [10]):
        m.cache = torch.zeros(50, 16, m.latent_width, dtype=dtype, device=DEV)
        mgr = manager([0], 50, 16, 2)
        seqs = [Sequence([1] * n, block_size=16) for _ in range(2)]
        for q in range(0, n, 16):                                   # blocks handed out in turns
            for s in seqs:
                s.group_tables = s.group_tables or [[]]
                s.group_tables[0].append(mgr.pools[0].take_block())
        for i, s in enumerate(seqs):
            s.state_slot = i
        at, got = 0, [[], []]
        for c in cuts:
            for s in seqs:
                s.num_computed_tokens, s.num_scheduled_tokens = at, c
            step = ragged_step(seqs, [0], 16, DEV, latent=True)
            out = m(torch.cat([h[b, at:at + c] for b in step.order]).to(DEV), step).cpu()
            for b in range(2):
                got[b].append(out[step.starts[b]:step.starts[b] + c])
            at += c
        for b in range(2):
            assert row_rel(torch.cat(got[b])[:, :heads * dim], want[b][:, :heads * dim]) < tol(dtype, 1e-4, 0.1), cuts


# ---- mixture of experts ----
@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("rows", [5, 600])
@pytest.mark.parametrize("n,k", [(11, 128), (40, 64), (61, 192), (65, 1024), (81, 320), (200, 128)])
def test_router_logits(dtype, rows, n, k):
    """Any number of experts beside the shared expert's gate."""
    x, w = torch.randn(rows, k, generator=gen(n)).to(dtype), (torch.randn(n, k, generator=gen(k)) * k ** -0.5).to(dtype)
    assert row_rel(gate_linear(x.to(DEV), w.to(DEV), None, n, 0.0), x.double() @ w.double().T) < 1e-5


@pytest.mark.parametrize("rows", [1, 17, 512, 513, 4113])
@pytest.mark.parametrize("n,k", [(5, 576), (32, 1024), (33, 640), (64, 1088), (65, 2048), (90, 704)])
def test_router_logits_long_rows(rows, n, k):
    """Whole rows through LDS: every number of column tiles, 16 and 32 rows, parts of K of unequal length, strided rows."""
    x, w = torch.randn(rows, k + 40, generator=gen(n)).bfloat16()[:, 8:k + 8], (torch.randn(n, k, generator=gen(k)) * k ** -0.5).bfloat16()
    b = torch.randn(n, generator=gen(rows))
    x_gpu = x.to(DEV) if rows == 1 else torch.empty(rows, k + 40, dtype=x.dtype, device=DEV)[:, 8:k + 8].copy_(x)
    z = x.double() @ w.double().T + b.double()
    want = torch.cat([z[:, :n // 2], torch.nn.functional.logsigmoid(z[:, n // 2:])], dim=1)
    assert row_rel(gate_linear(x_gpu, w.to(DEV), b.to(DEV), n // 2, 0.0), want) < 1e-5


ROUTERS = [(10, 3, 2, 1), (12, 5, 3, 2), (5, 1, 1, 1), (64, 6, 8, 3), (128, 8, 16, 4), (200, 9, 4, 2), (1000, 12, 50, 7), (6, 6, 1, 1), (16, 2, 16, 3), (7, 4, 7, 5)]


@pytest.mark.parametrize("experts,top,groups,keep", ROUTERS)
@pytest.mark.parametrize("shift", [0.0, -3.0, 2.0])
def test_moe_route(experts, top, groups, keep, shift):
    """Choices and weights token by token; with a shift all choice scores are negative, and closed groups stay closed."""
    g, rows = gen(experts + top), 50
    z, correction = torch.randn(rows, experts + 3, generator=g) * 2, torch.randn(experts, generator=g) * 0.5 + shift
    ids, weights = moe_route(z.to(DEV), correction.to(DEV), experts, top, groups, keep)
    for t in range(rows):
        want, w = ref.route(z[t, :experts].double(), correction.double(), {"top": top, "groups": {"count": groups, "keep": keep}})
        assert ids[t].tolist() == want, t
        assert torch.allclose(weights[t].cpu().double(), w, atol=1e-6)
    ids, _ = moe_route(z.to(DEV), None, experts, top, groups, keep)
    want, _ = ref.route(z[0, :experts].double(), torch.zeros(experts).double(), {"top": top, "groups": {"count": groups, "keep": keep}})
    assert ids[0].tolist() == want


@pytest.mark.parametrize("rows,top,experts", [(1, 1, 1), (7, 3, 10), (700, 4, 12), (2500, 3, 300), (5000, 2, 1024)])
def test_moe_plan(rows, top, experts):
    ids = torch.randint(0, experts, (rows, top), generator=gen(rows)).int()
    if experts > 2:
        ids[ids == 1] = 0                                                 # an expert without rows
    place = moe_plan(ids.to(DEV), experts).place.cpu().long()
    assert sorted(place.tolist()) == list(range(rows * top))
    by_place = torch.empty(rows * top, dtype=torch.int32)
    by_place[place] = ids.view(-1)
    assert bool((by_place[1:] >= by_place[:-1]).all())


@pytest.mark.parametrize("rows,top,experts,n,k", [(1, 1, 1, 64, 64), (5, 3, 10, 80, 128), (64, 8, 16, 272, 1088), (170, 2, 3, 128, 320), (700, 3, 7, 336, 192),
                                                  (40, 6, 6, 1024, 64), (1500, 4, 30, 64, 576), (1300, 2, 4, 336, 192), (2100, 1, 3, 1040, 64),
                                                  (1100, 3, 5, 80, 704)])
@pytest.mark.parametrize("path", ["few", "many", "any"])
def test_moe_linear(rows, top, experts, n, k, path):
    """Both products of an expert over unsorted pairs and over a plan; rows of experts in any number, also none."""
    if path == "few" and rows * top > 512:
        pytest.skip("more pairs than the unsorted form takes")
    dtype, g = torch.float32 if path == "any" else torch.bfloat16, gen(n + k)
    f = -(-n // 64) * 64
    x, ids = torch.randn(rows, k + 8, generator=g).to(dtype), torch.randint(0, experts, (rows, top), generator=g).int()
    if experts > 3:
        ids[ids == 2] = 3
    gate, up = ((torch.randn(experts, f, k, generator=g) * k ** -0.5).to(dtype) for _ in range(2))
    down = (torch.randn(experts, -(-n // 16) * 16, f, generator=g) * f ** -0.5).to(dtype)
    both = torch.stack([interleave_gate_up(a, b) for a, b in zip(gate, up)])
    on = lambda t: t.to(DEV)
    plan = None if path == "few" else moe_plan(on(ids), experts)
    act = moe_linear(on(x)[:, :k], on(both), on(ids), plan, top, glu=True)
    place = torch.arange(rows * top) if plan is None else plan.place.cpu().long()
    e, xr = ids.view(-1).long(), x[:, :k].double().repeat_interleave(top, 0)
    want = torch.empty(rows * top, f, dtype=torch.float64)
    for i in range(experts):
        r = (e == i).nonzero()[:, 0]
        want[r] = ref.silu(xr[r] @ gate[i].double().T) * (xr[r] @ up[i].double().T)
    assert row_rel(act.cpu()[place], want) < tol(dtype, 1e-5, 1.5e-2)
    out = moe_linear(act, on(down), on(ids), plan).cpu()[place]
    mine, want = act.cpu()[place].double(), torch.empty(rows * top, down.shape[1], dtype=torch.float64)
    for i in range(experts):
        r = (e == i).nonzero()[:, 0]
        want[r] = mine[r] @ down[i].double().T
    assert row_rel(out, want) < tol(dtype, 1e-5, 1e-2)


@pytest.mark.parametrize("n,k", [(64, 64), (80, 128), (336, 192)])
@pytest.mark.parametrize("counts", [[63, 64, 65, 0, 1, 129, 2, 32, 33, 5], [256, 0, 257, 513, 320, 321, 640, 700, 1023, 449, 128, 2]], ids=["small", "large"])
def test_moe_linear_row_tile_edges(counts, n, k):
    """Few pairs per expert on average, so tiles of 64 rows, or many, so tiles of 256: experts one short of a tile, at it, past it and of
    several, and every number of 64-row parts of a last one; fewer steps along K than the ring has buffers."""
    g = gen(n + k)
    experts, pairs = len(counts), sum(counts)
    ids = torch.cat([torch.full((c,), i) for i, c in enumerate(counts)])[torch.randperm(pairs, generator=g)].int().view(-1, 1)
    x = torch.randn(pairs, k, generator=g).bfloat16()
    w = (torch.randn(experts, n, k, generator=g) * k ** -0.5).bfloat16()
    plan = moe_plan(ids.to(DEV), experts)
    place = plan.place.cpu().long()
    out = moe_linear(x.to(DEV), w.to(DEV), ids.to(DEV), plan, 1).cpu()[place]
    want = torch.einsum("pk,pnk->pn", x.double(), w.double()[ids.view(-1).long()])
    assert row_rel(out, want) < 1e-2


@pytest.mark.parametrize("n,k", [(336, 2048), (160, 4096), (272, 192)])
@pytest.mark.parametrize("glu", [False, True])
@pytest.mark.parametrize("counts", [[63, 65, 0, 1, 129, 2, 32, 5, 64], [128, 60, 129, 300, 0, 57, 100],
                                    [256, 257, 320, 321, 640, 700, 1023, 449, 2048, 1088, 1, 1600], [384, 400, 448, 500]], ids=["64", "128", "256", "256-few"])
def test_moe_linear_walks_and_shares(counts, n, k, glu):
    """Rows a multiple of 4 KB, where experts and weight tiles begin K at different steps, in every form; the shares of the XCDs with weight tiles that
    they do not divide, last tiles of up to 64 rows behind all others (from 8192 pairs on) and longer ones in order."""
    g = gen(n + k)
    experts, pairs = len(counts), sum(counts)
    ids = torch.cat([torch.full((c,), i) for i, c in enumerate(counts)])[torch.randperm(pairs, generator=g)].int().view(-1, 1)
    x = torch.randn(pairs, k, generator=g).bfloat16()
    w = (torch.randn(experts, n // 32 * 64 if glu else n, k, generator=g) * k ** -0.5).bfloat16()
    plan = moe_plan(ids.to(DEV), experts)
    out = moe_linear(x.to(DEV), w.to(DEV), ids.to(DEV), plan, 1, glu).cpu()[plan.place.cpu().long()]
    want = torch.empty(out.shape, dtype=torch.float64)
    for e in range(experts):
        rows = (ids.view(-1) == e).nonzero().view(-1)
        z = x[rows].double() @ w[e].double().T
        if glu:                                            # gate and up rows in turns of 32
            gate, up = z.view(len(rows), n // 32, 2, 32).unbind(2)
            z = torch.nn.functional.silu(gate) * up
        want[rows] = z.reshape(len(rows), out.shape[1])
    assert row_rel(out, want) < 1e-2


@pytest.mark.parametrize("counts,n,k,top", [
    ([1024] * 10, 2048, 64, 1),                                       # 320 tiles, 40 per XCD: one round, eight tiles of the second in halves
    ([1000] * 10 + [64, 1, 0, 300, 128, 640], 2048, 192, 3),          # the same with tiles that are not whole, halves without rows, few rows behind them
    ([300, 520, 20, 700] * 20, 1040, 128, 7),                         # last weight tile of 16 outputs; rows are pair / 7
    ([1024] * 10 + [20] * 20, 2048, 64, 1),                           # 40 tiles per XCD and 20 of few rows, which halves would push into a third round
    ([1024] * 10 + [20] * 30, 2048, 64, 1),                           # the same with 30, which need that round anyway
    ([4096] * 9 + [4000, 40], 1024, 4096, 1),                         # long K: a workgroup for every tile
])
@pytest.mark.parametrize("glu", [False, True])
def test_moe_linear_rounds_of_large_tiles(counts, n, k, top, glu):
    """More tiles of 256 rows than CUs, so that workgroups go from one to the next: every row against the product in float32, whose sums
    differ by less than a rounding to 16 bits (2^-9 of the value), the gated ones by those of its factors."""
    g = torch.Generator(device=DEV).manual_seed(n + k)
    pairs = sum(counts) // top * top
    ids = torch.cat([torch.full((c,), i, device=DEV) for i, c in enumerate(counts)])[torch.randperm(sum(counts), generator=g, device=DEV)]
    ids = ids[:pairs].int().view(-1, top).contiguous()
    x = torch.randn(pairs // top, k, generator=g, device=DEV).bfloat16()
    w = (torch.randn(len(counts), n // 64 * 64 if glu else n, k, generator=g, device=DEV) * k ** -0.5).bfloat16()
    plan = moe_plan(ids, len(counts))
    out = moe_linear(x, w, ids, plan, top, glu)[plan.place.long()].float()
    again = moe_linear(x, w, ids, plan, top, glu)[plan.place.long()].float()
    assert torch.equal(out, again)
    want = torch.empty_like(out)
    for e in range(len(counts)):
        rows = (ids.view(-1) == e).nonzero().view(-1)
        z = x[rows // top].float() @ w[e].float().T
        if glu:
            gate, up = z.view(len(rows), w.shape[1] // 64, 2, 32).unbind(2)
            z = (torch.nn.functional.silu(gate) * up).reshape(len(rows), w.shape[1] // 2)
        want[rows] = z
    worst = (out - want).abs().amax(1) / want.abs().amax(1)
    assert worst.max() < 2 ** -8, worst.max()


@pytest.mark.parametrize("rows,top,experts,n,k,sn,sk", [
    (3, 2, 5, 128, 128, 64, 64),                                          # tiles of 64 rows; one tile of the shared expert
    (130, 2, 6, 80, 192, 400, 320),                                       # ... three row tiles of it, its last weight tile of 16 outputs, more steps of K
    (257, 1, 3, 336, 128, 144, 64),                                       # tiles of 128 rows
    (300, 4, 16, 4096, 64, 720, 192),                                     # tiles of 256 rows of a plan with both, one for each workgroup
    (1100, 1, 2, 3072, 64, 6400, 192),                                    # tiles of 256 rows, several for a workgroup, the shared ones in place of three
    (2100, 1, 2, 3072, 192, 10304, 384),                                 # ... in whole rounds and a part of one
    (700, 3, 40, 4096, 4096, 272, 2048),                                  # long K: a workgroup for every tile
])
@pytest.mark.parametrize("glu", [False, True])
def test_moe_linear_shared(rows, top, experts, n, k, sn, sk, glu):
    """An expert that all rows go through beside the others, in every form of the tiles: the others' results are as without it, bit for bit, its own are the
    product in float32 to a rounding to 16 bits (2^-9 of the value; gated ones to those of its factors)."""
    g = torch.Generator(device=DEV).manual_seed(n + k + sn)
    normal = lambda *shape, std=1.0: (torch.randn(*shape, generator=g, device=DEV) * std).bfloat16()
    ids = torch.randint(0, experts, (rows, top), generator=g, device=DEV).int()
    x, xs, w, ws = normal(rows, k), normal(rows, sk + 8)[:, :sk], normal(experts, n // 64 * 64 if glu else n, k, std=k ** -0.5), normal(sn // 64 * 64 if glu else sn, sk, std=sk ** -0.5)
    plan = moe_plan(ids, experts)
    out, beside = moe_linear(x, w, ids, plan, top, glu, shared=(xs, ws))
    assert torch.equal(out, moe_linear(x, w, ids, plan, top, glu))
    want = xs.float() @ ws.float().T
    if glu:
        gate, up = want.chunk(2, 1)
        want = torch.nn.functional.silu(gate) * up
    worst = (beside.float() - want).abs().amax(1) / want.abs().amax(1)
    assert beside.shape == want.shape and worst.max() < 2 ** -8, worst.max()
    for bad in (dict(plan=None), dict(glu=(1.0, 7.0, 1.0)), dict(shared=(xs.float(), ws.float())), dict(shared=(xs[:, :-1], ws))):
        with pytest.raises((ValueError, RuntimeError)):
            moe_linear(x, w, ids, **{**dict(plan=plan, per_token=top, glu=glu, shared=(xs, ws)), **bad})


@pytest.mark.parametrize("rows,top,experts,n,k", [
    (1, 1, 1, 64, 768),                                                   # one tile
    (1, 6, 64, 1536, 2048), (5, 6, 64, 1536, 2048),                       # tiles of 32 rows, on both sides of the line's gap
    (16, 2, 8, 336, 1088),                                                # 32 pairs, the last weight tile of 16 rows, steps no multiple of the buffers
    (32, 1, 8, 192, 832),                                                 # experts of up to all 32 rows
    (33, 1, 9, 192, 832),                                                 # tiles of 64 rows
    (66, 1, 17, 1040, 768),                                               # ... and an expert of 65 rows: two tiles
    (40, 3, 30, 576, 4096), (40, 3, 30, 1152, 4096),                      # a turned K in 64 rows, on both sides of the gap
])
@pytest.mark.parametrize("glu,side", [(False, None), (True, None), ((1.5, 7.0, 1.0), None), (False, (64, 768)), (True, (64, 768)), (False, (208, 2112)), (True, (208, 2112))])
def test_moe_linear_few_workgroups(rows, top, experts, n, k, glu, side):
    """Weights in 64 rows per workgroup, most pairs one expert's: experts and, beside them, an expert of all rows against the products in float32, to a rounding
    to 16 bits (2^-9 of the value; gated ones to those of its factors)."""
    g = torch.Generator(device=DEV).manual_seed(rows + n + k)
    normal = lambda *shape, std=1.0: (torch.randn(*shape, generator=g, device=DEV) * std).bfloat16()
    n = n // 64 * 64 if glu else n
    assert moe_linear_tiles(rows * top, experts, n, k, None if side is None else (rows, *side)) == (32 if rows * top <= 32 else 64, 64)
    ids = torch.randint(0, experts, (rows, top), generator=g, device=DEV).int()
    ids[:, 0] = experts - 1                                               # (in the 66-row case one id more, of nobody)
    if rows == 66:
        ids[7, 0] = -1
    x, w = normal(rows, k + 8)[:, :k], normal(experts, n, k, std=k ** -0.5)
    plan, shared = moe_plan(ids, experts), None
    if side is not None:
        sn, sk = side
        shared = normal(rows, sk), normal(sn // 64 * 64 if glu else sn, sk, std=sk ** -0.5)
    out = moe_linear(x, w, ids, plan, top, glu, shared=shared)

    def gated(z, turns):
        if not glu:
            return z
        gate, up = z.unflatten(1, (-1, 2, 32)).permute(2, 0, 1, 3).flatten(2) if turns else z.chunk(2, 1)
        if glu is True:
            return torch.nn.functional.silu(gate) * up
        alpha, limit, shift = glu
        gate = gate.clamp(max=limit)
        return gate * torch.sigmoid(alpha * gate) * (up.clamp(-limit, limit) + shift)

    def close(got, want):
        assert got.shape == want.shape
        worst = (got.float() - want).abs().amax(1) / want.abs().amax(1)
        assert worst.max() < 2 ** -8, worst.max()

    if shared is not None:
        out, beside = out
        close(beside, gated(shared[0].float() @ shared[1].float().T, False))
    flat, place = ids.flatten().tolist(), plan.place.tolist()
    for p, e in enumerate(flat):
        if e >= 0:
            close(out[place[p]][None], gated(x[p // top][None].float() @ w[e].float().T, True))


def test_experts_call_a_shared_expert_that_is_not_as_built():
    """A hook on the shared expert or one of its parts is called, one that was replaced is used."""
    m = SparseExperts(128, 128, 4, 2, 64, shared_ff=64, small_rows=64)
    weights = dict(router=(4, 128), **{"shared.sg": (1, 128), "shared.gate": (64, 128), "shared.up": (64, 128), "shared.down": (128, 64)}, gate=(64, 128), up=(64, 128),
                   down=(128, 64))
    g = torch.Generator(device=DEV).manual_seed(0)
    m.load(lambda name: torch.zeros(4, device=DEV) if name == "correction" else
           (torch.randn(weights.get(name) or weights[name.split(".")[1]], generator=g, device=DEV) / 11).bfloat16(), lambda t: t.contiguous())
    h, calls = torch.randn(100, 128, generator=g, device=DEV).bfloat16(), []
    with torch.no_grad():
        plain = m(h).shared
        assert torch.allclose(plain.float(), m.shared(h).float(), atol=2 ** -6)
        for part in (m.shared, m.shared.gate_up, m.shared.activation, m.shared.gate_down):
            handle = part.register_forward_hook(lambda *a: calls.append(1))
            assert torch.allclose(plain.float(), m(h).shared.float(), atol=2 ** -6)
            handle.remove()
        assert len(calls) == 4
        m.shared = torch.nn.Identity()
        assert m(h).shared is h


@pytest.mark.parametrize("rows", [3, 100])
@pytest.mark.parametrize("which", ["gate_up", "gate_down"])
def test_experts_with_a_shared_expert_at_an_odd_address(which, rows):
    """A contiguous weight that begins two bytes into a buffer: what the module itself gives, as the launches do not take it."""
    g = torch.Generator(device=DEV).manual_seed(rows)
    weights = {"router": (4, 128), "correction": (4,), "gate": (64, 128), "up": (64, 128), "down": (128, 64), "shared.sg": (1, 128), "shared.gate": (64, 128),
               "shared.up": (64, 128), "shared.down": (128, 64)}
    m = SparseExperts(128, 128, 4, 2, 64, shared_ff=64)
    m.load(lambda name: (torch.randn(weights.get(name) or weights[name.split(".")[1]], generator=g, device=DEV) / 11).bfloat16(), lambda t: t.contiguous())
    h = torch.randn(rows, 128, generator=g, device=DEV).bfloat16()
    with torch.no_grad():
        beside = m(h).shared
        part = getattr(m.shared, which)
        flat = torch.empty(part.weight.numel() + 1, dtype=torch.bfloat16, device=DEV)
        flat[1:] = part.weight.flatten()
        part.weight = torch.nn.Parameter(flat[1:].view_as(part.weight), requires_grad=False)
        got = m(h).shared
        assert torch.equal(got, m.shared(h)) and torch.allclose(got.float(), beside.float(), atol=2 ** -6)


@pytest.mark.parametrize("width,ff,shared,sorted_pairs", [(704, 704, None, False), (768, 128, None, True), (128, 768, None, True), (128, 64, 64, True)])
def test_experts_of_one_row(width, ff, shared, sorted_pairs):
    """Few rows, on either side of the line from which their pairs are sorted too: as in a batch, whose products are those over sorted pairs."""
    m, g = SparseExperts(width, width, 8, 2, ff, shared_ff=shared or 0, small_rows=64), torch.Generator(device=DEV).manual_seed(width + ff)
    shape = {"router": (8, width), "correction": (8,), "gate": (ff, width), "up": (ff, width), "down": (width, ff), "shared.sg": (1, width)}
    if shared:
        shape.update({"shared.gate": (shared, width), "shared.up": (shared, width), "shared.down": (width, shared)})
    m.load(lambda name: torch.randn(shape.get(name) or shape[name.split(".")[1]], generator=g, device=DEV).mul_(width ** -0.5).bfloat16(), lambda t: t.contiguous())
    h = torch.randn(40, width, generator=g, device=DEV).bfloat16()
    batch = m(h)
    assert m(h[:0]).parts.shape[0] == 0
    for n in (1, 2, 8):
        out = m(h[:n])
        assert (out.part_row is not None) == sorted_pairs and torch.equal(out.weights, batch.weights[:n])
        place = out.part_row.long() if sorted_pairs else torch.arange(2 * n, device=DEV)
        assert row_rel(out.parts[place], batch.parts[batch.part_row.long()[:2 * n]].cpu()) < 1e-2


@pytest.mark.parametrize("n,k", [(2560, 128), (2304, 64), (768, 64)])      # products on tiles of 256 rows; those of 768 outputs (192 tiles), and those whose rows are no multiple of 16 bytes, on those of 128
@pytest.mark.parametrize("glu", [False, True])
@pytest.mark.parametrize("more", [0, 120])
def test_moe_linear_both_tilings_of_a_plan(n, k, glu, more):
    """Plans between small and large tiles have both: experts without rows, of every number of 64-row parts, past a large tile by a few rows (behind all
    others from 8192 pairs on) and by more; an output whose rows are no multiple of 16 bytes stays on the smaller ones."""
    counts = [0, 1, 63, 64, 65, 127, 128, 129, 192, 193, 255, 256, 257, 300, 320, 321] * 4
    counts = [c + (more if i % 5 == 0 else 0) - (c > 200 and more == 0 and 100) for i, c in enumerate(counts)]
    g, experts, pairs = gen(n + k), len(counts), sum(counts)
    assert 48 * experts < pairs < 384 * experts and (pairs >= 8192)
    ids = torch.cat([torch.full((c,), i) for i, c in enumerate(counts)])[torch.randperm(pairs, generator=g)].int().view(-1, 1)
    x = torch.randn(pairs, k, generator=g).bfloat16()
    w = (torch.randn(experts, n, k, generator=g) * k ** -0.5).bfloat16()
    xd, wd, idd = x.to(DEV), w.to(DEV), ids.to(DEV)
    plan = moe_plan(idd, experts)
    place = plan.place.cpu().long()
    out = moe_linear(xd, wd, idd, plan, 1, glu)
    want = torch.empty(out.shape, dtype=torch.float64)
    for e in range(experts):
        rows = (ids.view(-1) == e).nonzero().view(-1)
        z = x[rows].double() @ w[e].double().T
        if glu:
            gate, up = z.view(len(rows), n // 64, 2, 32).unbind(2)
            z = torch.nn.functional.silu(gate) * up
        want[rows] = z.reshape(len(rows), out.shape[1])
    assert row_rel(out.cpu()[place], want) < 1e-2
    stride = out.shape[1] + 4
    odd = torch.full((pairs, stride), float("nan"), dtype=torch.bfloat16, device=DEV)
    st = _C.load().mvllm_moe_linear(odd.data_ptr(), stride, xd.data_ptr(), k, wd.data_ptr(), idd.data_ptr(), plan.data.data_ptr(), pairs, experts, n, k, 1,
                                    int(glu), 1, _C.current_stream_ptr(odd.device))
    assert st == 0
    assert row_rel(odd[:, :out.shape[1]].cpu()[place], want) < 1e-2 and torch.isnan(odd[:, out.shape[1]:]).all()


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("cfg", [moe(), moe(experts=12, top=5, groups=(3, 2), ff=72, shared=100), moe(experts=5, top=1, groups=None, shared=None),
                                 moe(experts=40, top=8, groups=(8, 3), ff=64, shared=16)], ids=["a", "b", "c", "d"])
def test_experts(dtype, cfg):
    width, inputs = 80, 128
    w = {k[len("l0.mlp."):]: t for k, t in ref.random_weights(config([lightning_layer(mlp=cfg)]), 3).items() if k.startswith("l0.mlp.")}
    r, groups, shared = cfg["router"], cfg["router"]["groups"] or {"count": 1, "keep": 1}, cfg["shared"] or {"ff": 0}
    m = SparseExperts(width, inputs, r["experts"], r["top"], cfg["expert"]["ff"], groups["count"], groups["keep"], shared["ff"], small_rows=64)
    m.load(lambda n: w[n], lambda t: t.to(DEV, dtype).contiguous())
    wd = {k: t.double() for k, t in w.items()}
    h = torch.randn(600, width, generator=gen(4)).to(dtype)
    want = ref.experts(h.double(), wd, "", cfg)
    one = torch.ones(1, device=DEV)
    for lo, n in ((0, 600), (0, 1), (1, 5), (40, 64), (200, 150)):
        padded = torch.nn.functional.pad(h[lo:lo + n], (0, inputs - width)).to(DEV)
        _, x = stream_norm(torch.zeros(n, 1, width, device=DEV), m(padded), one, one[None], torch.ones(width, device=DEV), 1.0)
        err = (x[:, 0].cpu().double() - want[lo:lo + n]).pow(2).mean(-1).sqrt() / want.pow(2).mean().sqrt()
        assert err.max() < tol(dtype, 1e-5, 3e-2), (lo, n, int(err.argmax()))


# ---- the model ----
_runners: dict = {}


def make_runner(name, dtype, **extra):
    key = (name, dtype, tuple(sorted(extra.items())))
    if key not in _runners:
        cfg = CONFIGS[name]()
        full = engine_config({**cfg, "dtype": "fp32" if dtype == torch.float32 else "bf16", "block_size": 16, "max_cached_blocks": 64,
                              "max_num_sequences": 4, "max_position": 1024, **extra, "enforce_eager": True})
        runner = HybridModelRunner(full, NiridraForCausalLM)
        weights = ref.random_weights(cfg, seed=11)
        runner.model.load_weights(weights)
        if not extra.get("enforce_eager", True):
            runner.capture_decode_graphs()           # after the weights: a captured step holds their addresses
        _runners[key] = runner, cfg, weights
    return _runners[key]


_wanted: dict = {}


def oracle_logits(seed, n, cfg, weights):
    key = (json.dumps(cfg), seed, n)
    if key not in _wanted:
        _wanted[key] = ref.forward(tokens(seed, n, cfg["vocab"]), weights, cfg)
    return _wanted[key]


# a row's logits error over the logits' spread: all rows, the median.  bf16: a router's close call goes the other way in some
# rows of a random model, and from there into all later ones
MODEL_TOL = {torch.float32: (2e-4, 2e-5), torch.bfloat16: (1.0, 6e-2)}


def row_errors(got, want):
    d = got.double() - want
    return (d - d.mean(-1, keepdim=True)).pow(2).mean(-1).sqrt() / want.std()


def check_rows(got, want, dtype, *what):
    err = row_errors(got, want)
    assert err.max() < MODEL_TOL[dtype][0] and err.median() < MODEL_TOL[dtype][1], (*what, int(err.argmax()), float(err.max()), float(err.median()))


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("name", sorted(CONFIGS))
@pytest.mark.parametrize("sizes", [[170], [1], [2], [3, 5, 64, 1, 1, 33], [64], [150, 1]], ids=str)
def test_model_in_portions(dtype, name, sizes):
    runner, cfg, weights = make_runner(name, dtype)
    n = 170 if sizes != [1] or dtype == torch.float32 else 90
    want = oracle_logits(7, 170, cfg, weights)[:n]
    got = Driver(runner).run_alone("a", tokens(7, 170, cfg["vocab"])[:n], sizes)
    check_rows(got, want, dtype)


@pytest.mark.parametrize("name", sorted(CONFIGS))
def test_residual_streams_layer_by_layer(name):
    runner, cfg, weights = make_runner(name, torch.float32)
    toks, want, got = tokens(7, 60, cfg["vocab"]), [], []
    ref.forward(toks, weights, cfg, layer_outputs=want)
    s = Sequence(toks, block_size=16)
    runner.cache_manager.allocate(s)
    s.num_scheduled_tokens = 60
    runner.forward_step([s], got)
    runner.cache_manager.deallocate(s)
    assert len(got) == len(want) == len(cfg["layers"])
    for i, (a, b) in enumerate(zip(got, want)):
        assert rel(a, b) < 2e-5, i


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("name", sorted(CONFIGS))
def test_mixed_batches_and_reuse(dtype, name):
    """Portions beside decoded tokens, requests left out of steps, slots and pages given back and used again, in a pool
    that is just large enough: every request's logits are its own."""
    runner, cfg, weights = make_runner(name, dtype)
    lens = {"a": 170, "b": 61, "c": 7, "d": 130, "e": 96, "f": 33}
    toks = {k: tokens(20 + i, n, cfg["vocab"]) for i, (k, n) in enumerate(lens.items())}
    rng, drv, at, waiting, live = random.Random(4), Driver(runner), dict.fromkeys(lens, 0), list(lens), []
    while waiting or live:
        while waiting and len(live) < 4:
            live.append(waiting.pop(0))
        chosen = [k for k in live if rng.random() < 0.8] or live[:1]
        portions = {k: toks[k][at[k]:at[k] + rng.choice([1, 1, 1, 2, 3, 17, 40, 64])] for k in chosen}
        for k in chosen:
            at[k] += len(portions[k])
        ended = [k for k in chosen if at[k] == lens[k]]
        drv.step(portions, ended)
        live = [k for k in live if k not in ended]
    for i, k in enumerate(lens):
        check_rows(torch.cat(drv.logits[k]), oracle_logits(20 + i, lens[k], cfg, weights), dtype, k)
    assert len(runner.cache_manager.free_slots) == 4
    assert all(len(p.free_block_ids) == 64 for p in runner.cache_manager.pools)


def test_logits_do_not_depend_on_cuts_and_company():
    """bf16: the same tokens whole, in portions, token by token and beside others differ by rounding only (away from a
    router's close calls: in most rows)."""
    runner, cfg, _ = make_runner("mixed", torch.bfloat16)
    toks = tokens(3, 120, cfg["vocab"])
    base = Driver(runner).run_alone("a", toks, [120]).double()
    others = [Driver(runner).run_alone("a", toks, sizes) for sizes in ([1], [2], [33], [7, 60])]
    drv = Driver(runner)
    for at in range(0, 120, 40):
        drv.step({"x": tokens(50, 35, cfg["vocab"])[:35 - at // 4], "a": toks[at:at + 40], "y": tokens(51, 3, cfg["vocab"])[:1]}, ["x"])
    drv.step({"y": [1]}, ["y", "a"])
    for got in [*others, torch.cat(drv.logits["a"])]:
        assert row_errors(got, base).median() < 5e-2


def test_first_tokens_and_one_token_prompts():
    runner, cfg, weights = make_runner("mixed", torch.float32)
    want = oracle_logits(7, 170, cfg, weights)
    for n in (1, 2, 3, 4):
        check_rows(Driver(runner).run_alone("x", tokens(7, 170, cfg["vocab"])[:n], [n]), want[:n], torch.float32, n)


def test_long_decoding():
    """A few hundred decoded tokens, over many pages."""
    runner, cfg, weights = make_runner("other", torch.float32)
    got = Driver(runner).run_alone("x", tokens(31, 330, cfg["vocab"]), [5, 1])
    assert row_errors(got, oracle_logits(31, 330, cfg, weights)).max() < 2e-4


def greedy_reference(prompt, new, weights, cfg):
    """Greedy continuation by the oracle and the smallest lead of a chosen token over the next one."""
    toks, lead = list(prompt), math.inf
    for _ in range(new):
        logits = ref.forward(toks, weights, cfg)[-1]
        top = logits.topk(2)
        lead = min(lead, float(top.values[0] - top.values[1]) / float(logits.std()))
        toks.append(int(top.indices[0]))
    return toks[len(prompt):], lead


def generate(runner, prompts, new, budget=64, slots=4, **kw):
    from minivllm_amd.engine.llm_engine import LLMEngine
    runner.sample_calls = 0
    eng = LLMEngine(dict(runner.config, max_num_batched_tokens=budget, max_num_sequences=slots, **kw), model_runner=runner)
    return eng.generate(prompts, SamplingParams(greedy=True, max_tokens=new, ignore_eos=True))["token_ids"]


@pytest.mark.parametrize("name", ["mixed", "other"])
def test_greedy_generation_through_the_engine(name):
    """fp32: the engine's greedy ids are the oracle's; captured decode steps and small step budgets give the same ones."""
    runner, cfg, weights = make_runner(name, torch.float32)
    prompts = [tokens(60 + i, n, cfg["vocab"]) for i, n in enumerate([5, 40, 1, 23, 71, 2])]
    got = generate(runner, prompts, 12)
    for p, ids in zip(prompts, got):
        want, lead = greedy_reference(p, 12, weights, cfg)
        assert lead > 1e-3, "the case has a tie: choose other prompts"
        assert ids == want
    assert generate(runner, prompts, 12, budget=7) == got
    graphed, _, _ = make_runner(name, torch.float32, enforce_eager=False, max_model_length=256)
    for async_decode in (True, False):
        assert generate(graphed, prompts, 12, async_decode=async_decode) == got
    assert generate(graphed, prompts, 12, budget=9) == got


@pytest.mark.parametrize("name", ["mixed", "plain"])
def test_captured_decode(name):
    """bf16, decoding over several pages: replays of the captured step give the eager step's ids."""
    eager, cfg, _ = make_runner(name, torch.bfloat16)
    graphed, _, _ = make_runner(name, torch.bfloat16, enforce_eager=False, max_model_length=512)
    prompts = [tokens(80 + i, n, cfg["vocab"]) for i, n in enumerate([3, 18, 31, 64, 19])]
    want, got = generate(eager, prompts, 100), generate(graphed, prompts, 100)
    # greedy ids of a model with random weights part after a near-tie: the partings have to be rare
    same = sum(a == b for w, g in zip(want, got) for a, b in zip(w, g))
    assert same / 500 > 0.6 and all(w[:4] == g[:4] for w, g in zip(want, got))


def test_preempted_requests_start_over():
    """A pool too small for all of them: preempted requests are computed again and end with the same ids."""
    runner, cfg, _ = make_runner("other", torch.float32)
    prompts = [tokens(40 + i, n, cfg["vocab"]) for i, n in enumerate([30, 28, 45])]
    want = generate(runner, prompts, 40)
    small, _, _ = make_runner("other", torch.float32, max_cached_blocks=8)
    assert generate(small, prompts, 40) == want
    assert len(small.cache_manager.free_slots) == 4


def write_checkpoint(folder, cfg, weights):
    header, blobs, at = {}, [], 0
    for k, t in weights.items():
        raw = t.contiguous().view(torch.int16).numpy().tobytes()
        header[k] = {"dtype": "BF16", "shape": list(t.shape), "data_offsets": [at, at + len(raw)]}
        blobs.append(raw)
        at += len(raw)
    text = json.dumps(header).encode()
    (folder / "config.json").write_text(json.dumps(cfg))
    (folder / "model.safetensors").write_bytes(len(text).to_bytes(8, "little") + text + b"".join(blobs))


def test_trace_replay_and_command_line(tmp_path, capsys):
    """A checkpoint folder through the trace replay (files in the order of entries and places) and the generate command."""
    from minivllm_amd.__main__ import main
    from minivllm_amd.engine.replay import replay
    cfg = CONFIGS["mixed"]()
    weights = ref.random_weights(cfg, seed=3)
    write_checkpoint(tmp_path, cfg, weights)
    a, b = tokens(1, 50, cfg["vocab"]), tokens(2, 30, cfg["vocab"])
    steps = [{"step": 0, "entries": [{"id": "a", "tokens": a[:41], "want": [40, 3]}, {"id": "b", "tokens": b[:1], "want": [0]}], "end": []},
             {"step": 1, "entries": [{"id": "b", "tokens": b[1:30], "want": []}], "end": []},
             {"step": 2, "entries": [{"id": "a", "tokens": a[41:42], "want": [0]}], "end": ["b"]},
             {"step": 3, "entries": [{"id": "c", "tokens": b, "want": [29]}, {"id": "a", "tokens": a[42:], "want": [7]}], "end": ["a", "c"]}]
    said, out = [], tmp_path / "out"
    out.mkdir()
    replay(str(tmp_path), "float32", str(out), 128, [json.dumps(s) + "\n" for s in steps] + ["\n"], said.append)
    assert said == [f"done {i}" for i in range(4)] and sorted(p.name for p in out.iterdir()) == ["0.f32", "2.f32", "3.f32"]
    wa, wb = ref.forward(a, weights, cfg), ref.forward(b, weights, cfg)
    for n, rows in ((0, [wa[40], wa[3], wb[0]]), (2, [wa[41]]), (3, [wb[29], wa[49]])):
        got = torch.from_numpy(np.fromfile(out / f"{n}.f32", dtype="<f4")).view(len(rows), -1)
        check_rows(got, torch.stack(rows), torch.float32, n)
    capsys.readouterr()
    main(["generate", "--model", str(tmp_path), "--dtype", "float32", "--prompt", " ".join(map(str, b[:9])), "--max-tokens", "6", "--greedy"])
    ids = json.loads(capsys.readouterr().out.strip().splitlines()[-1])["token_ids"]
    want, lead = greedy_reference(b[:9], 6, weights, cfg)
    assert lead > 1e-3 and ids == [want]
