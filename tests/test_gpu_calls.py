"""The native way to the attention operators (csrc/calls.cpp): the same results, bit for bit, as the longer way, which everything else takes."""
import pytest
import torch
from torch.utils._python_dispatch import TorchDispatchMode

from minivllm_amd import _C
from minivllm_amd.layers import attention
from minivllm_amd.layers.window import window_prefill
from minivllm_amd.utils import reset_context, set_context

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


class Counted:
    """Passes calls on and counts those that were taken."""

    def __init__(self):
        self.calls, self.taken = _C.calls, 0

    def __getattr__(self, name):
        def call(*a):
            got = getattr(self.calls, name)(*a)
            self.taken += got is not None and got is not False
            return got
        return call


@pytest.fixture
def counted(monkeypatch):
    _C.load()
    assert _C.calls is not None
    counted = Counted()
    monkeypatch.setattr(_C, "calls", counted)
    return counted


def both(counted, monkeypatch, f, taken):
    """f() with the native way and without it; how many of its calls were taken."""
    counted.taken = 0
    a = f()
    assert counted.taken == taken
    with monkeypatch.context() as m:
        m.setattr(_C, "calls", None)
        b = f()
    assert a.dtype == b.dtype and a.shape == b.shape and a.stride() == b.stride()
    assert torch.equal(a, b)
    return a


def normal(*shape, dtype=torch.bfloat16):
    return torch.randn(*shape, device=DEV, generator=torch.Generator(DEV).manual_seed(sum(shape))).to(dtype)


def paged(lengths, block, kv, dim, dtype, int8=False):
    tables = torch.full((len(lengths), max(-(-n // block) for n in lengths) + 1), -1, dtype=torch.int32)
    at = 0
    for b, n in enumerate(lengths):
        need = -(-n // block)
        tables[b, :need] = torch.arange(at, at + need)
        at += need
    caches = [normal(at, block, kv, dim, dtype=torch.float32) for _ in range(2)]
    if int8:
        return tables.to(DEV), [(c * 40).round().clamp(-127, 127).to(torch.int8) for c in caches], [torch.rand(at, block, kv, device=DEV) + 0.01 for _ in range(2)]
    return tables.to(DEV), [c.to(dtype) for c in caches], []


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("lengths,block", [([5], 16), ([300, 1, 77], 16), ([2500, 3000], 256)])
def test_decode(counted, monkeypatch, dtype, lengths, block):
    tables, (k, v), _ = paged(lengths, block, 2, 64, dtype)
    q = normal(len(lengths), 8, 64, dtype=dtype)
    for lens in (torch.tensor(lengths, device=DEV), torch.tensor(lengths, dtype=torch.int32, device=DEV)):
        args = (q, k, v, tables, lens, 0.125, 8, 2, 64, block)
        both(counted, monkeypatch, lambda: attention.paged_attention_decode(*args), 1)
    need = attention.decode_workspace_bytes(len(lengths), 8, 64, tables.shape[1], block)
    own = torch.empty(need + 16, dtype=torch.uint8, device=DEV)
    both(counted, monkeypatch, lambda: attention.paged_attention_decode(*args, workspace=own), 1)
    # converted, or turned down
    wide = normal(len(lengths), 8, 128, dtype=dtype)[..., :64]
    both(counted, monkeypatch, lambda: attention.paged_attention_decode(wide, *args[1:]), 0)
    both(counted, monkeypatch, lambda: attention.paged_attention_decode(*args[:3], tables.long(), *args[4:]), 0)
    for wrong in ((q, k, v, tables, lens, 0.125, 8, 2, 64, block * 2), (q, k, v[:, :, :1], *args[3:]), (q, k.double(), *args[2:]),
                  (q, k, v, tables, lens[:0], *args[5:]), (q, k, v, tables, lens, 0.125, 4, 2, 64, block)):
        with pytest.raises(ValueError):
            attention.paged_attention_decode(*wrong)
    assert counted.taken == 0


def test_decodes_on_two_streams_without_a_workspace(counted):
    """Partial results of calls that run side by side do not meet; captured calls keep theirs in the graph's pool."""
    cases, streams = [], [torch.cuda.Stream() for _ in range(2)]
    for lengths, heads in (([9000, 4000, 7000], 8), ([6000, 8500], 4)):
        tables, (k, v), _ = paged(lengths, 16, 2, 64, torch.bfloat16)
        args = (normal(len(lengths), heads, 64), k, v, tables, torch.tensor(lengths, device=DEV), 0.125, heads, 2, 64, 16)
        own = torch.empty(attention.decode_workspace_bytes(len(lengths), heads, 64, tables.shape[1], 16), dtype=torch.uint8, device=DEV)
        cases.append((args, attention.paged_attention_decode(*args, workspace=own)))
    assert all(attention.paged_decode_plan(*(c[0][0].shape[0], c[0][6], 2, 64, c[0][3].shape[1], 16))[1] > 1 for c in cases)
    torch.cuda.synchronize()
    got = [[], []]
    for _ in range(20):
        for i, stream in enumerate(streams):
            with torch.cuda.stream(stream):
                got[i].append(attention.paged_attention_decode(*cases[i][0]))
    torch.cuda.synchronize()
    for results, (_, want) in zip(got, cases):
        assert all(torch.equal(r, want) for r in results)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        captured = attention.paged_attention_decode(*cases[0][0])
    for _ in range(3):
        captured.zero_()
        graph.replay()
        other = attention.paged_attention_decode(*cases[1][0])
        torch.cuda.synchronize()
        assert torch.equal(captured, cases[0][1]) and torch.equal(other, cases[1][1])
    assert counted.taken == 2 + 40 + 1 + 3


@pytest.mark.parametrize("lengths,block", [([5], 16), ([300, 1, 77], 32)])
def test_decode_int8(counted, monkeypatch, lengths, block):
    tables, (k, v), (ks, vs) = paged(lengths, block, 2, 128, None, int8=True)
    args = (normal(len(lengths), 4, 128), k, v, ks, vs, tables, torch.tensor(lengths, device=DEV), 0.1, 4, 2, 128, block)
    both(counted, monkeypatch, lambda: attention.paged_attention_decode_int8(*args), 1)
    for wrong in ((*args[:3], ks.half(), *args[4:]), (*args[:4], vs[:, :1], *args[5:]), (args[0], k.float(), *args[2:])):
        with pytest.raises(ValueError):
            attention.paged_attention_decode_int8(*wrong)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32, torch.int8])
def test_decode_int8_without_scales_is_refused(counted, dtype):
    """What is missing does not make the call one of the other operator's, whose caches would fit."""
    tables, (k, v), scales = paged([40, 17], 16, 2, 128, dtype, int8=dtype == torch.int8)
    ks, vs = scales or [torch.ones(k.shape[:3], device=DEV) for _ in range(2)]
    q, rest = normal(2, 4, 128, dtype=torch.bfloat16 if dtype == torch.int8 else dtype), (tables, torch.tensor([40, 17], device=DEV), 0.1, 4, 2, 128, 16)
    for given in ((None, None), (ks, None), (None, vs)):
        with pytest.raises((ValueError, AttributeError)):
            attention.paged_attention_decode_int8(q, k, v, *given, *rest)
        assert counted.calls.decode_int8(q, k, v, *given, *rest, None) is None
        assert given == (None, None) or counted.calls.decode(q, k, v, *given, *rest, None) is None
    assert counted.taken == 0


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("lengths", [[1], [40, 7], [900, 300]])
def test_prefill_and_store(counted, monkeypatch, dtype, lengths):
    rows, scale = sum(lengths), 0.125
    q, k, v = normal(rows, 8, 64, dtype=dtype), normal(rows, 2, 64, dtype=dtype), normal(rows + 1, 2, 64, dtype=dtype)[1:]
    cu = torch.tensor([0, *torch.tensor(lengths).cumsum(0).tolist()], dtype=torch.int32, device=DEV)
    for most in (max(lengths), 10 ** 6, None):
        both(counted, monkeypatch, lambda: attention.flash_attention_prefill(q, k, v, cu, scale, 8, 2, 64, max_seqlen=most), 1)
    both(counted, monkeypatch, lambda: attention.flash_attention_prefill(q, k, v, cu.long(), scale, 8, 2, 64, max_seqlen=max(lengths)), 0)
    both(counted, monkeypatch, lambda: attention.flash_attention_prefill(normal(rows, 2, 8, 64, dtype=dtype)[:, 0], k, v, cu, scale, 8, 2, 64),
         int(rows == 1))                                                   # (one row is dense)
    both(counted, monkeypatch, lambda: attention.flash_attention_prefill(q, k, v, cu, scale, 8, 2, 64, sink=torch.zeros(8, device=DEV)), 0)
    for wrong in ((q, k[:-1], v, cu), (q, k, v.double(), cu), (q[:, :4], k, v, cu)):
        with pytest.raises(ValueError):
            attention.flash_attention_prefill(*wrong, scale, 8, 2, 64)

    def stored(slots, key=k):
        caches = [torch.zeros(rows // 16 + 2, 16, 2, 64, dtype=dtype, device=DEV) for _ in range(2)]
        attention.store_kvcache(key, v, *caches, slots, 16)
        return torch.cat(caches)

    slots = torch.randperm(rows, generator=torch.Generator().manual_seed(1)).to(DEV)
    slots[0] = -1
    both(counted, monkeypatch, lambda: stored(slots), 1)
    both(counted, monkeypatch, lambda: stored(slots.int()), 0)
    both(counted, monkeypatch, lambda: stored(slots, normal(rows, 4, 64, dtype=dtype)[:, ::2]), 0)
    with pytest.raises((ValueError, AssertionError)):
        stored(slots[:-1])


@pytest.mark.parametrize("dtype,heads,kv,dim", [(torch.bfloat16, 8, 2, 64), (torch.float16, 6, 3, 128), (torch.float32, 8, 8, 64), (torch.float32, 2, 1, 128),
                                                (torch.bfloat16, 4, 1, 64), (torch.bfloat16, 4, 2, 96), (torch.bfloat16, 32, 8, 128)])
@pytest.mark.parametrize("lengths", [[1], [0, 31, 0], [129, 7], [700, 300, 40], [1900], [2000, 1500, 1400]])
def test_layer_stores_beside_its_prompts(counted, monkeypatch, dtype, heads, kv, dim, lengths):
    """Rows without a slot, slots past the cache, rows that end within a workgroup's portion, several ranges, kernels over whole rows, the two-group kernel."""
    rows = sum(lengths)
    q, k, v = normal(rows, heads, dim, dtype=dtype), normal(rows, kv, dim, dtype=dtype), normal(rows + 1, kv, dim, dtype=dtype)[1:]
    cu = torch.tensor([0, *torch.tensor(lengths).cumsum(0).tolist()], dtype=torch.int32, device=DEV)
    slots = torch.randperm(rows + 5, generator=torch.Generator().manual_seed(rows))[:rows]
    slots[rows // 2], slots[rows // 3] = -1, 10 ** 12
    slots = slots.to(DEV)
    layer = attention.Attention(heads, dim, num_kv_heads=kv, block_size=16)

    def forward(key=k, at=slots, most=max(lengths), caches=None):
        layer.k_cache, layer.v_cache = caches or [torch.zeros(rows // 16 + 1, 16, kv, dim, dtype=dtype, device=DEV) for _ in range(2)]
        set_context(True, cu_seqlens_q=cu, max_seqlen_q=most, slot_mapping=at)
        try:
            out = layer(q, key, v)
        finally:
            reset_context()
        return torch.cat([t.flatten() for t in (out, layer.k_cache, layer.v_cache)])

    for most in (max(lengths), 0):
        got = both(counted, monkeypatch, lambda: forward(most=most), 1)
    want = [torch.zeros(rows // 16 + 1, 16, kv, dim, dtype=dtype, device=DEV) for _ in range(2)]
    there = (slots >= 0) & (slots < want[0].shape[0] * 16)
    for cache, x in zip(want, (k, v)):
        cache.view(-1, kv, dim)[slots[there]] = x[there]
    assert torch.equal(got[rows * heads * dim:], torch.cat([t.flatten() for t in want]))
    both(counted, monkeypatch, lambda: forward(at=slots.int()), 1)         # (the attention alone)
    off = lambda: torch.zeros((rows // 16 + 1) * 16 * kv * dim + 1, dtype=dtype, device=DEV)[1:].view(-1, 16, kv, dim)
    both(counted, monkeypatch, lambda: forward(caches=[off(), off()]), 1)  # caches off 16 bytes: one after the other


@pytest.mark.parametrize("dtype,lengths,cached", [(torch.bfloat16, [200, 90], [150, 0]), (torch.float32, [700, 40], [640, 20]), (torch.bfloat16, [3000] * 8, [0] * 8),
                                                  (torch.float16, [9000], [5800])])                               # (its keys are split)
def test_prefill_over_a_prefix(counted, monkeypatch, dtype, lengths, cached):
    tables, (k, v), _ = paged(lengths, 16, 2, 64, dtype)
    new = [n - c for n, c in zip(lengths, cached)]
    cu = lambda x: torch.tensor([0, *torch.tensor(x).cumsum(0).tolist()], dtype=torch.int32, device=DEV)
    args = (normal(sum(new), 8, 64, dtype=dtype), k, v, tables, cu(new), cu(lengths), 0.125, 8, 2, 64, 16)
    both(counted, monkeypatch, lambda: attention.flash_attention_prefill_paged(*args, max_seqlen_k=max(lengths)), int(max(lengths) < 5000))
    both(counted, monkeypatch, lambda: attention.flash_attention_prefill_paged(*args), 0)
    both(counted, monkeypatch, lambda: attention.flash_attention_prefill_paged(*args, max_seqlen_k=max(lengths), key_splits=2 * (dtype != torch.float32)), 0)
    if max(lengths) == 700:                                                # no room for partial results
        monkeypatch.setattr(attention, "STAGED_PREFILL_MAX_BYTES", 16)
        both(counted, monkeypatch, lambda: attention.flash_attention_prefill_paged(*args, max_seqlen_k=max(lengths)), 0)


@pytest.mark.parametrize("shared", [False, True])
def test_windows(counted, monkeypatch, shared):
    rows = 150
    q, k, v = normal(rows, 8, 96)[..., :64], normal(rows, 2, 64), normal(rows, 3, 64)[:, :2]
    cu = torch.tensor([0, 70, rows], dtype=torch.int32, device=DEV)
    options = dict(slopes=torch.rand(8, device=DEV), positions=torch.arange(rows, device=DEV), temperature=(0.1, 16), gate=normal(rows, 8, 64)) if shared \
        else dict(v=v, gate=normal(rows, 8))

    def run(*change, **more):
        out = torch.zeros(rows, 8, 64, dtype=torch.bfloat16, device=DEV)
        window_prefill(out, *(change or (q, k, cu, cu, 0.125, 33)), **{**options, **more})
        return out

    both(counted, monkeypatch, run, 1)
    both(counted, monkeypatch, lambda: run(gate=None), 1)
    for change, more in (((q, k, cu.long(), cu, 0.125, 33), {}), ((q, k, cu, cu[:2], 0.125, 33), {}), ((q[:, :, :32], k, cu, cu, 0.125, 33), {}),
                         ((), dict(gate=normal(rows, 4))), ((), dict(slopes=torch.rand(7, device=DEV)))):
        with pytest.raises(ValueError):
            run(*change, **more)


def test_subclasses_and_modes_go_the_longer_way(counted):
    """What wants to see torch's operators, or is not a plain tensor, is left to them."""
    class Mine(torch.Tensor):
        pass

    class Seen(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            self.names = getattr(self, "names", []) + [str(func)]
            return func(*args, **(kwargs or {}))

    q, k = normal(40, 8, 64), normal(40, 2, 64)
    cu = torch.tensor([0, 40], dtype=torch.int32, device=DEV)
    want = attention.flash_attention_prefill(q, k, k, cu, 0.125, 8, 2, 64)
    assert counted.taken == 1
    got = attention.flash_attention_prefill(q.as_subclass(Mine), k, k, cu, 0.125, 8, 2, 64)
    assert type(got) is Mine and torch.equal(got.as_subclass(torch.Tensor), want)
    with Seen() as seen:
        assert torch.equal(attention.flash_attention_prefill(q, k, k, cu, 0.125, 8, 2, 64), want)
    assert counted.taken == 1 and any("empty_like" in n for n in seen.names)
    assert attention.flash_attention_prefill(torch.nn.Parameter(q), k, k, cu, 0.125, 8, 2, 64).requires_grad is False and counted.taken == 2


def _changed(t, rows):
    """A tensor that an operator converts or refuses: other types, device, layout, and of data other shapes, ``rows`` where the host knows their number."""
    yield from (None, t.cpu(), t.double(), t.to(torch.int32), torch.stack([t, t], -1)[..., 0])
    if t.dim() > 1:
        yield from (t.unsqueeze(0), t[..., :-1], t[..., :-1].contiguous(), t[:, :-1].contiguous())
        if rows:
            yield t[:-1]
        if t.is_floating_point():
            yield t.half()


def _operators():
    bf = dict(dtype=torch.bfloat16)
    tables, (k, v), _ = paged([40, 17], 16, 2, 64, torch.bfloat16)
    _, (k8, v8), (ks, vs) = paged([40, 17], 16, 2, 64, None, int8=True)
    lens, cu, cu_k = torch.tensor([40, 17], device=DEV), torch.tensor([0, 30, 39], dtype=torch.int32, device=DEV), torch.tensor([0, 40, 57], dtype=torch.int32, device=DEV)
    q, new_k, new_v, slots = normal(39, 4, 64, **bf), normal(39, 2, 64, **bf), normal(39, 2, 64, **bf) + 1, torch.arange(39, device=DEV)
    rest = (0.125, 4, 2, 64)

    def stored(*args):
        caches = [torch.zeros(4, 16, 2, 64, device=DEV, **bf) for _ in range(2)]
        attention.store_kvcache(*args[:2], *caches, args[2], 16)
        return torch.stack(caches)

    def layer(*args):
        a = attention.Attention(4, 64, num_kv_heads=2, block_size=16)
        a.k_cache, a.v_cache = [torch.zeros(4, 16, 2, 64, device=DEV, **bf) for _ in range(2)]
        set_context(True, cu_seqlens_q=args[3], max_seqlen_q=30, slot_mapping=args[4])
        try:
            return torch.cat([t.flatten() for t in (a(*args[:3]), a.k_cache, a.v_cache)])
        finally:
            reset_context()

    def window(*args):
        out = torch.zeros(39, 4, 64, device=DEV, **bf)
        window_prefill(out, *args[:4], 0.125, 20, v=args[4])
        return out

    return {
        "store": (stored, (new_k, new_v, slots)),
        "decode": (lambda *a: attention.paged_attention_decode(*a, *rest, 16), (q[:2], k, v, tables, lens)),
        "decode_int8": (lambda *a: attention.paged_attention_decode_int8(*a, *rest, 16), (q[:2], k8, v8, ks, vs, tables, lens)),
        "prefill": (lambda *a: attention.flash_attention_prefill(*a, *rest, max_seqlen=30), (q, new_k, new_v, cu)),
        "prefill_paged": (lambda *a: attention.flash_attention_prefill_paged(*a, *rest, 16, max_seqlen_k=40), (q, k, v, tables, cu, cu_k)),
        "layer": (layer, (q, new_k, new_v, cu, slots)),
        "window": (window, (q, new_k, cu, cu, new_v)),
    }


@pytest.mark.parametrize("name", ["store", "decode", "decode_int8", "prefill", "prefill_paged", "layer", "window"])
def test_both_ways_take_and_refuse_the_same(counted, monkeypatch, name):
    """Every argument changed by itself: what one way converts or refuses, and with which error, so does the other."""
    def outcome(f, args):
        try:
            return f(*args)
        except Exception as e:
            return type(e)

    f, args = _operators()[name]
    both(counted, monkeypatch, lambda: f(*args), 1)
    refused = 0
    for i in range(len(args)):
        for j, other in enumerate(_changed(args[i], name not in ("prefill_paged", "window"))):
            changed = (*args[:i], other, *args[i + 1:])
            a = outcome(f, changed)
            with monkeypatch.context() as m:
                m.setattr(_C, "calls", None)
                b = outcome(f, changed)
            refused += isinstance(a, type)
            assert (a is b) if isinstance(a, type) or isinstance(b, type) else torch.equal(a, b), (i, j, a, b)
    assert refused > len(args)
