"""Prefill over ranges of key tiles (mvllm_prefill_ranges) against the CPU oracle and the other kernels."""
import math

import pytest
import torch

import oracle
from helpers import error_stats, make_paged_prefill_case
from minivllm_amd import _C
from minivllm_amd.layers import attention

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
MAX_ABS_16, MEAN_ABS_16 = 2e-2, 2e-3                                   # the other forms' bounds: 16-bit weights and results


def _run(c, hq, hkv, d, bs, tiles, max_k, paged, sink=None):
    class Forced:
        def __getattr__(self, name):
            return getattr(_C.load(), name) if name != "mvllm_prefill_ranges_plan" else lambda *sizes: tiles
    out = torch.full_like(c["q_new"] if paged else c["q"], float("nan")).to(DEV)
    on = lambda name: c[name].to(DEV)
    q, k, v, tables, cu_k = (on("q_new"), on("k_cache"), on("v_cache"), on("block_tables"), on("cu_k")) if paged \
        else (on("q"), on("k"), on("v"), None, None)
    took = attention._prefill_ranges(Forced(), out, q, k, v, tables, on("cu_q") if paged else on("cu_k"), cu_k, len(c["cu_k"]) - 1, max_k,
                                     1 / math.sqrt(d), hq, hkv, d, bs if paged else 0, k.shape[0] if paged else 0, sink)
    assert took
    return out.cpu()


def _groups(c, hq, hkv, d, bs, tiles, max_k, paged, dtype=torch.bfloat16):
    """Groups of waves per range that ``_run`` of the same call runs on."""
    return _C.load().mvllm_prefill_ranges_groups(len(c["cu_k"]) - 1, len(c["q_new"] if paged else c["q"]), max_k, hq, hkv, d, bs if paged else 0,
                                                 _C.dtype_code(dtype), tiles)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("hq,hkv,d,bs,lengths,cached,tiles", [
    (8, 2, 128, 16, [128, 129, 127, 1], [64, 100, 126, 0], 2),         # a last tile that ends a range, starts one, falls short of it
    (8, 4, 128, 32, [160, 700], [96, 690], 2),                         # a range that only the later of two row tiles reaches
    (5, 5, 64, 48, [600, 300, 64], [470, 10, 63], 4),                  # one head per workgroup, row tiles over several waves
    (4, 2, 64, 256, [1000, 30], [0, 7], 6),                            # nothing cached: every row tile its own number of ranges
    (8, 2, 128, 16, [4200], [4190], 2),                                # 33 ranges
    (16, 8, 128, 16, [500, 200], [400, 150], 8),                       # whole: one range
])
@pytest.mark.parametrize("paged", [True, False])
def test_prefill_over_key_ranges(hq, hkv, d, bs, lengths, cached, tiles, paged, dtype):
    c = make_paged_prefill_case(61, lengths, cached, hq, hkv, d, bs, dtype=dtype)
    want = oracle.prefill_paged_oracle(c["q_new"].float(), torch.nan_to_num(c["k_cache"].float()), torch.nan_to_num(c["v_cache"].float()),
                                       c["block_tables"], c["cu_q"], c["cu_k"], 1 / math.sqrt(d), hq, hkv, d, bs)
    for bound in (max(lengths), max(1, max(lengths) - 150)):           # also a bound that is too low: the last range takes the rest
        got = _run(c, hq, hkv, d, bs, tiles, bound, paged)
        got = got if paged else got[c["new_rows"]]
        mx, mean = error_stats(got, want)
        assert torch.isfinite(got.float()).all() and mx <= MAX_ABS_16 and mean <= MEAN_ABS_16, (bound, mx, mean)


@pytest.mark.parametrize("new", [1, 31, 32, 33, 65, 100])
@pytest.mark.parametrize("hq,hkv,d,tiles", [(8, 2, 128, 4), (4, 2, 64, 2), (3, 3, 128, 4)])
def test_the_diagonal_at_every_place_of_a_tile(hq, hkv, d, tiles, new):
    """A wave's last tiles, one or two with the causal limit in them, the last of them whole or its first half: in the first or the second of the
    two buffers, first tile of a range or not, behind prefixes beside every multiple of 32 up to three tiles."""
    cached = [0, 1, 31, 32, 33, 63, 64, 65, 95, 96, 97, 127, 128, 129, 160, 192]
    c = make_paged_prefill_case(83 + new, [n + new for n in cached], cached, hq, hkv, d, 16, dtype=torch.bfloat16)
    want = oracle.prefill_paged_oracle(c["q_new"].float(), torch.nan_to_num(c["k_cache"].float()), torch.nan_to_num(c["v_cache"].float()),
                                       c["block_tables"], c["cu_q"], c["cu_k"], 1 / math.sqrt(d), hq, hkv, d, 16)
    for paged in (True, False):
        got = _run(c, hq, hkv, d, 16, tiles, max(cached) + new, paged)
        mx, mean = error_stats(got if paged else got[c["new_rows"]], want)
        assert mx <= MAX_ABS_16 and mean <= MEAN_ABS_16, (paged, mx, mean)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("hq,hkv,d,lengths,cached,tiles,groups", [
    (8, 2, 128, [5000, 2700, 64], [4900, 2650, 0], 40, (2, 1)),        # two ranges, one of an odd number of tiles, one of a single tile
    (8, 4, 64, [3400, 130, 0, 3], [3300, 70, 0, 0], 28, (2, 1)),
    (5, 5, 128, [3000, 1700], [2800, 1699], 24, (2, 1)),               # one head per workgroup
    (2, 1, 128, [2700, 40], [2000, 10], 14, (1, 2)),                   # packed: 14 tiles and 256 workgroups
    (3, 3, 64, [1900, 700, 0], [0, 0, 0], 14, (2, 2)),                 # ... one head per workgroup, two ranges and one
    (2, 1, 64, [2200, 900], [100, 0], 36, (2, 2)),                     # whole
])
@pytest.mark.parametrize("paged", [True, False])
def test_prefill_over_key_ranges_in_two_groups(hq, hkv, d, lengths, cached, tiles, groups, paged, dtype):
    """Few workgroups with long ranges: two groups of waves walk the halves of a range, whose sums meet in LDS.  groups: what these sizes run on, over a
    cache and packed."""
    c = make_paged_prefill_case(71, lengths, cached, hq, hkv, d, 16, dtype=dtype)
    want = oracle.prefill_paged_oracle(c["q_new"].float(), torch.nan_to_num(c["k_cache"].float()), torch.nan_to_num(c["v_cache"].float()),
                                       c["block_tables"], c["cu_q"], c["cu_k"], 1 / math.sqrt(d), hq, hkv, d, 16)
    assert _groups(c, hq, hkv, d, 16, tiles, max(lengths), paged, dtype) == groups[not paged]
    got = _run(c, hq, hkv, d, 16, tiles, max(lengths), paged)
    mx, mean = error_stats(got if paged else got[c["new_rows"]], want)
    assert torch.isfinite(got.float()).all() and mx <= MAX_ABS_16 and mean <= MEAN_ABS_16, (mx, mean)


@pytest.mark.parametrize("new", [1, 31, 32, 33, 65, 100])
@pytest.mark.parametrize("hq,hkv,d", [(8, 2, 128), (4, 2, 64), (3, 3, 128)])
def test_the_diagonal_at_every_place_of_a_tile_in_two_groups(hq, hkv, d, new):
    """As above with a bound of 64 tiles: from a single tile, which leaves the second group without one, to five, the limit in either group's last
    tile or before it; the sink counts once."""
    cached = [0, 1, 31, 32, 33, 63, 64, 65, 95, 96, 97, 127, 128, 129, 160, 192]
    c = make_paged_prefill_case(87 + new, [n + new for n in cached], cached, hq, hkv, d, 16, dtype=torch.bfloat16)
    want = oracle.prefill_paged_oracle(c["q_new"].float(), torch.nan_to_num(c["k_cache"].float()), torch.nan_to_num(c["v_cache"].float()),
                                       c["block_tables"], c["cu_q"], c["cu_k"], 1 / math.sqrt(d), hq, hkv, d, 16)
    for paged in (True, False):
        assert _groups(c, hq, hkv, d, 16, 64, 4096, paged) == 2
        got = _run(c, hq, hkv, d, 16, 64, 4096, paged)
        mx, mean = error_stats(got if paged else got[c["new_rows"]], want)
        assert mx <= MAX_ABS_16 and mean <= MEAN_ABS_16, (paged, mx, mean)
    sink = torch.randn(hq, generator=torch.Generator().manual_seed(1)).to(DEV)
    got = _run(c, hq, hkv, d, 16, 64, 4096, False, sink)
    whole = attention.flash_attention_prefill(*(c[n].to(DEV) for n in ("q", "k", "v", "cu_k")), d ** -0.5, hq, hkv, d, sink=sink).cpu()
    mx, mean = error_stats(got, whole.float())
    assert mx <= MAX_ABS_16 and mean <= MEAN_ABS_16, (mx, mean)


@pytest.mark.parametrize("lengths", [[0, 300, 0, 77], [200]])
def test_prefill_over_key_ranges_sinks_and_empty_sequences(lengths):
    """Against the kernel without ranges: the sink counts once, sequences without tokens have no rows."""
    c = make_paged_prefill_case(7, lengths, [0] * len(lengths), 8, 4, 128, 16, dtype=torch.bfloat16)
    sink = torch.randn(8, generator=torch.Generator().manual_seed(1)).to(DEV)
    got = _run(c, 8, 4, 128, 16, 2, max(lengths), False, sink)
    want = attention.flash_attention_prefill(*(c[n].to(DEV) for n in ("q", "k", "v", "cu_k")), 128 ** -0.5, 8, 4, 128, sink=sink).cpu()
    mx, mean = error_stats(got, want.float())
    assert mx <= MAX_ABS_16 and mean <= MEAN_ABS_16, (mx, mean)


@pytest.mark.parametrize("bound", [300, 32768, 2 ** 31 - 1, 2 ** 40])
def test_loose_bounds_cost_no_ranges(monkeypatch, bound):
    """The keys of a batch bound the caller's own bound: packed rows, or the places of the block tables."""
    c, asked, plan = make_paged_prefill_case(9, [300, 120], [200, 0], 8, 4, 128, 16, dtype=torch.bfloat16), [], attention._prefill_ranges_plan
    monkeypatch.setattr(attention, "_prefill_ranges_plan", lambda *a: asked.append(a[3]) or plan(*a))
    on = {n: c[n].to(DEV) for n in ("q", "k", "v", "q_new", "k_cache", "v_cache", "block_tables", "cu_q", "cu_k")}
    got = attention.flash_attention_prefill(on["q"], on["k"], on["v"], on["cu_k"], 128 ** -0.5, 8, 4, 128, max_seqlen=bound)
    paged = attention.flash_attention_prefill_paged(on["q_new"], on["k_cache"], on["v_cache"], on["block_tables"], on["cu_q"], on["cu_k"],
                                                    128 ** -0.5, 8, 4, 128, 16, min(bound, 2 ** 31 - 1))
    assert asked == [min(bound, 420), min(bound, 16 * c["block_tables"].shape[1])]
    want = attention.flash_attention_prefill(on["q"], on["k"], on["v"], on["cu_k"], 128 ** -0.5, 8, 4, 128)
    for a, b in ((got, want), (paged.cpu(), want.cpu()[c["new_rows"]])):
        mx, mean = error_stats(a.cpu(), b.cpu().float())
        assert mx <= MAX_ABS_16 and mean <= MEAN_ABS_16, (mx, mean)


def test_prefill_ranges_plan_and_rejections():
    lib = _C.load()
    bf, f32 = _C.dtype_code(torch.bfloat16), _C.dtype_code(torch.float32)
    plan = lib.mvllm_prefill_ranges_plan
    assert plan(2, 343, 3435, 16, 8, 128, 16, bf) in range(6, 20, 2)     # few rows behind many keys: ranges
    assert plan(2, 541, 275, 16, 8, 128, 0, bf) == 6                     # a small batch: whole (five tiles, an even number)
    assert plan(16, 16000, 2048, 32, 8, 128, 0, bf) == 0                 # the chip is full
    assert plan(65, 650, 4000, 16, 8, 128, 16, bf) == 0 and plan(1, 100, 4000, 16, 8, 128, 16, f32) == 0
    assert plan(1, 100, 4000, 16, 8, 80, 16, bf) == 0 and plan(1, 100, 4000, 16, 8, 128, 8, bf) == 0
    assert lib.mvllm_prefill_ranges_workspace_bytes(100, 640, 16, 128, 10) == 0
    assert lib.mvllm_prefill_ranges_workspace_bytes(100, 641, 16, 128, 10) == 2 * 100 * 16 * 129 * 4


@pytest.mark.parametrize("hq,hkv,d,bs,lengths,cached,tiles", [
    (8, 2, 128, 16, [64, 65, 63, 1], [32, 50, 62, 0], 1),              # a last tile that ends a range, starts one, falls short of it
    (8, 4, 64, 32, [160, 700], [96, 690], 3),                          # a range that only the later of two row tiles reaches
    (5, 5, 64, 48, [600, 300, 64], [470, 10, 63], 4),                  # one head per workgroup, row tiles over several waves
    (4, 2, 128, 256, [1000, 30], [0, 7], 5),                           # nothing cached: every row tile its own number of ranges
    (8, 2, 64, 16, [2040], [2030], 1),                                 # 64 ranges
    (16, 8, 64, 16, [500, 200], [400, 150], 16),                       # whole: one range
])
@pytest.mark.parametrize("paged", [True, False])
def test_fp32_prefill_over_key_ranges(hq, hkv, d, bs, lengths, cached, tiles, paged, monkeypatch):
    """fp32: against the oracle in 64 bits, 4e-6 of the results' root mean square (sums of up to 2000 fp32 products, weights by exp2 to 2^-21);
    rows that see nothing of a range, a bound that is too low, a sink against the kernel over whole rows."""
    c = make_paged_prefill_case(61, lengths, cached, hq, hkv, d, bs, dtype=torch.float32)
    want = oracle.prefill_paged_oracle(c["q_new"].double(), torch.nan_to_num(c["k_cache"].double()), torch.nan_to_num(c["v_cache"].double()),
                                       c["block_tables"], c["cu_q"], c["cu_k"], 1 / math.sqrt(d), hq, hkv, d, bs).double()
    monkeypatch.setattr(attention, "_prefill_ranges_plan", lambda lib, s, t, keys, hq, hkv, d, bs, code: (
        tiles, lib.mvllm_prefill_f32_ranges_workspace_bytes(t, keys, hq, d, tiles)))
    for bound in (max(lengths), max(1, max(lengths) - 150)):
        got = _run(c, hq, hkv, d, bs, tiles, bound, paged)
        got = got if paged else got[c["new_rows"]]
        assert torch.isfinite(got).all() and ((got.double() - want).norm() / want.norm()).item() <= 4e-6, bound
    if not paged:
        sink = torch.randn(hq, generator=torch.Generator().manual_seed(1)).to(DEV)
        got = _run(c, hq, hkv, d, bs, tiles, max(lengths), False, sink)
        whole = attention.flash_attention_prefill(*(c[n].to(DEV) for n in ("q", "k", "v", "cu_k")), d ** -0.5, hq, hkv, d, sink=sink).cpu()
        assert ((got - whole).norm() / whole.norm()).item() <= 2e-6


def test_fp32_ranges_plan_and_rejections():
    lib = _C.load()
    plan = lib.mvllm_prefill_f32_ranges_plan
    assert plan(3, 234, 1558, 16, 8, 64, 16) == 10                       # few rows behind many keys
    assert plan(12, 720, 1160, 16, 8, 64, 16) in (4, 5, 6) and plan(16, 1600, 2000, 32, 8, 64, 16) == 63      # places without rows in the other order
    assert plan(8, 1200, 150, 16, 8, 64, 0) == 0 and plan(8, 2400, 600, 32, 8, 64, 16) == 0      # short; the chip is full
    assert plan(65, 650, 4000, 16, 8, 64, 16) == 0 and plan(1, 100, 4000, 16, 8, 80, 16) == 0 and plan(1, 100, 4000, 16, 8, 64, 8) == 0
    keys = 2 ** 31 - 1                                                   # a bound that is none
    per = plan(1, 100, keys, 16, 8, 64, 16)
    assert -(-(-(-keys // 32)) // per) <= 64
    bad = lambda *a: lib.mvllm_prefill_f32_ranges(*a)
    q = torch.zeros(64, 8, 64, device=DEV)
    cu = torch.tensor([0, 64], dtype=torch.int32, device=DEV)
    p = q.data_ptr()
    args = lambda tiles, nbytes, dim=64, ws=p: (p, p, p, p, 0, 0, cu.data_ptr(), 0, 1, 64, 64, 8, 8, dim, 0, 0, 1.0, 0, tiles, ws, nbytes, 0)
    assert bad(*args(1, 0)) == -5 and bad(*args(1, 1 << 20, ws=0)) == -5 and bad(*args(0, 1 << 20)) == -3 and bad(*args(1, 1 << 20, dim=80)) == -4


@pytest.mark.parametrize("hq,hkv,d", [(8, 2, 64), (4, 2, 128), (3, 3, 64)])
@pytest.mark.parametrize("tiles", [1, 2, 4])
def test_fp32_ranges_with_fewer_keys_than_rows(hq, hkv, d, tiles, monkeypatch):
    """Paged sequences of more rows than keys: kernel and merge take the same row tiles for cut ones, and every row is written."""
    keys, rows = [64, 33, 200, 0, 300, 128], [300, 70, 65, 33, 310, 129]
    c = make_paged_prefill_case(29, keys, [0] * len(keys), hq, hkv, d, 16, dtype=torch.float32)
    c["q_new"] = torch.randn(sum(rows), hq, d, generator=torch.Generator().manual_seed(3))
    c["cu_q"] = torch.tensor([0, *torch.tensor(rows).cumsum(0).tolist()], dtype=torch.int32)
    monkeypatch.setattr(attention, "_prefill_ranges_plan", lambda lib, s, t, k, hq, hkv, d, bs, code: (
        tiles, lib.mvllm_prefill_f32_ranges_workspace_bytes(t, k, hq, d, tiles)))
    got = _run(c, hq, hkv, d, 16, tiles, max(keys), True)
    whole = attention.flash_attention_prefill_paged(*(c[n].to(DEV) for n in ("q_new", "k_cache", "v_cache", "block_tables", "cu_q", "cu_k")),
                                                    d ** -0.5, hq, hkv, d, 16).cpu()
    assert torch.isfinite(got).all() and ((got - whole).norm() / whole.norm()).item() <= 2e-6
