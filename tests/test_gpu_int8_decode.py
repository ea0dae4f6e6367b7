"""INT8 KV cache: store_kvcache_int8 then paged_attention_decode_int8 vs the CPU oracle.

The INT8 format is defined by this build (the reference has none): the oracle dequantises code*scale in
fp32 and runs the naive decode.  Tolerance: mean-abs 2e-3 and |err| <= 2e-2 + |want| * 2^-8 elementwise; the
second term is the rounding of the 16-bit output itself, which matters here because the 8-sigma outliers of
the INT8 workload make single outputs as large as 30 (one bf16 ulp at 16..32 is 0.125)."""
import math

import pytest
import torch

import oracle
from helpers import error_stats, half_step, make_paged_case
from minivllm_amd.layers.attention import paged_attention_decode_int8, paged_decode_partition, paged_decode_plan, store_kvcache_int8

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _quantised_case(seed, batch, ctx_lo, ctx_hi, hq, hkv, d, bs, dtype=torch.bfloat16, ctx_list=None):
    q, kc, vc, tables, ctx = make_paged_case(seed, batch, ctx_lo, ctx_hi, hq, hkv, d, bs, ctx_list=ctx_list)
    g = torch.Generator().manual_seed(seed + 100)
    kc[torch.rand(kc.shape, generator=g) < 0.01] *= 8.0          # 1 % outliers at 8 sigma
    vc[torch.rand(vc.shape, generator=g) < 0.01] *= 8.0
    nb = kc.shape[0]
    codes_k = torch.zeros(nb, bs, hkv, d, dtype=torch.int8, device=DEV)
    codes_v = torch.zeros_like(codes_k)
    sk = torch.zeros(nb, bs, hkv, device=DEV)
    sv = torch.zeros_like(sk)
    slots = torch.arange(nb * bs, device=DEV)
    store_kvcache_int8(kc.view(-1, hkv, d).to(dtype).to(DEV), vc.view(-1, hkv, d).to(dtype).to(DEV),
                       codes_k, codes_v, sk, sv, slots, bs)
    return q.to(dtype), codes_k, codes_v, sk, sv, tables, ctx


def _check(case, hq, hkv, d, bs, scale, ctx_dtype=torch.int64):
    """Max-abs 2e-2 / mean-abs 2e-3 against the fp32 oracle on the dequantised cache, with one allowance: the kernel's
    output is 16 bits wide, and these small cases (a handful of keys, 1 % of them 8-sigma outliers) have outputs of
    magnitude 4 to 10, where half a bf16 step alone (2^(floor(log2 |want|) - 8)) is 0.008 to 0.03.  That half step of the value is
    therefore taken off the difference before it is held against 2e-2.  The full-size configuration-4 test, whose
    outputs average thousands of keys, uses the bound as stated."""
    q, ck, cv, sk, sv, tables, ctx = case
    got = paged_attention_decode_int8(q.to(DEV), ck, cv, sk, sv, tables.to(DEV), ctx.to(ctx_dtype).to(DEV), scale,
                                      hq, hkv, d, bs).cpu()
    want = oracle.decode_int8_oracle(q.float(), ck.cpu(), cv.cpu(), sk.cpu(), sv.cpu(), tables, ctx, scale,
                                     hq, hkv, d, bs)
    mx, mean = error_stats(got, want)
    assert got.dtype == q.dtype and torch.isfinite(got).all()
    excess = ((got.float() - want).abs() - half_step(want, got.dtype)).max().item()
    assert excess <= 2e-2 and mean <= 2e-3, (mx, excess, mean)
    return got


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("hq,hkv,bs,ctx_hi", [(32, 8, 16, 700), (16, 8, 256, 1500), (8, 8, 32, 255), (6, 2, 48, 400),
                                              (32, 4, 16, 600), (16, 1, 32, 900), (24, 2, 16, 300), (5, 1, 64, 200)])
def test_int8_fast_path(dtype, hq, hkv, bs, ctx_hi):
    d = 128
    _check(_quantised_case(61, 7, 1, ctx_hi, hq, hkv, d, bs, dtype), hq, hkv, d, bs, 1 / math.sqrt(d))


@pytest.mark.parametrize("ctx_list", [[1, 2, 7, 8, 9, 15, 16, 17], [255, 256, 257, 1023, 1024, 1025]])
def test_int8_context_boundaries(ctx_list):
    hq, hkv, d, bs = 8, 2, 128, 16
    _check(_quantised_case(62, 0, 0, 0, hq, hkv, d, bs, ctx_list=ctx_list), hq, hkv, d, bs, 0.1, torch.int32)


@pytest.mark.parametrize("hq,hkv,d,bs", [(16, 16, 96, 16), (34, 2, 128, 16), (4, 2, 128, 8), (8, 4, 64, 8)])
def test_int8_generic_path(hq, hkv, d, bs):
    """head_dim 96 and block_size 8 run on the generic kernel (17 query heads per kv head: the MFMA kernel, two slices
    per kv head)."""
    _check(_quantised_case(63, 5, 1, 300, hq, hkv, d, bs), hq, hkv, d, bs, 1 / math.sqrt(d))


def test_int8_zero_context_and_missing_blocks():
    hq, hkv, d, bs = 8, 2, 128, 16
    q, ck, cv, sk, sv, tables, ctx = _quantised_case(64, 0, 0, 0, hq, hkv, d, bs, ctx_list=[40, 0, 100])
    sk[0].fill_(float("nan"))                                  # stale memory in a block nobody owns... 
    sv[0].fill_(float("nan"))
    owned = set(tables[tables >= 0].tolist())
    if 0 in owned:                                             # keep the poison only if block 0 is unowned
        sk[0].zero_()
        sv[0].zero_()
    got = paged_attention_decode_int8(q.to(DEV), ck, cv, sk, sv, tables.to(DEV), ctx.to(DEV), 0.09, hq, hkv, d, bs).cpu()
    assert torch.isfinite(got).all() and torch.count_nonzero(got[1]) == 0
    hole = tables.clone()
    hole[0, :] = -1
    got2 = paged_attention_decode_int8(q.to(DEV), ck, cv, sk, sv, hole.to(DEV), ctx.to(DEV), 0.09, hq, hkv, d, bs).cpu()
    assert torch.count_nonzero(got2[0]) == 0 and torch.equal(got2[2], got[2])


def test_config4_subset():
    """The INT8 workload's shape (B 128 is cut to 24 sequences here, ctx U[256,16384]) on the fast path."""
    hq, hkv, d, bs = 32, 8, 128, 16
    case = _quantised_case(65, 24, 256, 16384, hq, hkv, d, bs)
    _check(case, hq, hkv, d, bs, 1 / math.sqrt(d))


@pytest.mark.parametrize("hq,hkv,bs,d", [(32, 8, 16, 128), (16, 8, 256, 128), (16, 1, 32, 128), (24, 2, 16, 128),
                                         (5, 1, 64, 128), (16, 8, 16, 64), (12, 1, 32, 64), (8, 4, 256, 64),
                                         (40, 2, 16, 128), (71, 1, 32, 64)])
@pytest.mark.parametrize("form", ["one wave per head", "waves share a head", "waves share a head, one partition"])
def test_int8_both_grid_forms(hq, hkv, bs, d, form):
    """As test_both_grid_forms_vs_oracle of the 16-bit cache: the table width and the batch size pick the form."""
    batch = 7 if form == "waves share a head" else 64
    width = {"one wave per head": 32768, "waves share a head": 8192}.get(form, 4096) // bs * bs
    g = torch.Generator().manual_seed(66)
    ctx_list = torch.randint(1, 1301, (batch,), generator=g).tolist()
    ctx_list[2] = 1300
    q, ck, cv, sk, sv, tables, ctx = _quantised_case(67, 0, 0, 0, hq, hkv, d, bs, ctx_list=ctx_list)
    wide = torch.full((batch, width // bs), -1, dtype=torch.int32)
    wide[:, :tables.shape[1]] = tables
    part, parts, waves = paged_decode_plan(batch, hq, hkv, d, wide.shape[1], bs, q.dtype, int8_cache=True)
    if form == "one wave per head":
        assert waves == 1
    elif form == "waves share a head":
        assert waves > 1 and parts > 1
    else:
        assert waves > 1 and (parts == 1 or hkv < 8)
    scale = 1 / math.sqrt(d)
    got = paged_attention_decode_int8(q.to(DEV), ck, cv, sk, sv, wide.to(DEV), ctx.to(DEV), scale, hq, hkv, d, bs).cpu()
    want = oracle.decode_int8_oracle(q.float(), ck.cpu(), cv.cpu(), sk.cpu(), sv.cpu(), tables, ctx, scale, hq, hkv, d, bs)
    mx, mean = error_stats(got, want)
    excess = ((got.float() - want).abs() - half_step(want, got.dtype)).max().item()
    assert torch.isfinite(got).all() and excess <= 2e-2 and mean <= 2e-3, (mx, excess, mean)


@pytest.mark.parametrize("batch,width,d,bs,part,parts,spread,least", [
    (12, 2048, 128, 16, 384, 6, 5, 256), (20, 2016, 64, 48, 512, 4, 3, 256), (7, 8192, 128, 16, 512, 16, 16, 256), (7, 8192, 64, 16, 512, 16, 16, 256),
    (22, 6144, 128, 16, 768, 8, 8, 512), (16, 6144, 64, 256, 768, 8, 8, 512)])
def test_int8_partitions_as_long_as_the_contexts_ask_for(batch, width, d, bs, part, parts, spread, least):
    """As test_partitions_as_long_as_the_contexts_ask_for of the 16-bit cache."""
    sizes = (batch, 16, 8, d, width // bs, bs, torch.bfloat16, True)
    assert paged_decode_plan(*sizes) == (part, parts, 4)
    of = lambda ctx: paged_decode_partition(ctx, *sizes)
    assert of(1) == least < part == of(width) and of(spread * (least + 64)) == least + 64 and of(spread * (least + 64) + 1) > of(spread * (least + 64) - 64 * spread) == least
    edges = {n + by for n in (64, least, 2 * least, spread * least, spread * (least + 64), part, spread * part, parts * part) for by in (-1, 0, 1)}
    edges = sorted(n for n in edges | {1, 700, width - 1, width} if 0 < n <= width)
    for at in range(0, len(edges), batch):
        ctx_list = (edges[at:at + batch] + [129, 300] * batch)[:batch]
        q, ck, cv, sk, sv, tables, ctx = _quantised_case(at + d, 0, 0, 0, 16, 8, d, bs, ctx_list=ctx_list)
        wide = torch.full((batch, width // bs), -1, dtype=torch.int32)
        wide[:, :tables.shape[1]] = tables
        got = paged_attention_decode_int8(q.to(DEV), ck, cv, sk, sv, wide.to(DEV), ctx.to(DEV), d ** -0.5, 16, 8, d, bs).cpu()
        want = oracle.decode_int8_oracle(q.float(), ck.cpu(), cv.cpu(), sk.cpu(), sv.cpu(), tables, ctx, d ** -0.5, 16, 8, d, bs)
        mx, mean = error_stats(got, want)
        excess = ((got.float() - want).abs() - half_step(want, got.dtype)).max().item()
        assert torch.isfinite(got).all() and excess <= 2e-2 and mean <= 2e-3, (ctx_list, mx, excess, mean)


def test_config4_full_size_on_its_own_plan():
    """The INT8 workload in full: B 128, ctx U[256,16384], Hq32/Hkv8/D128, block 16, N(0,1) inputs with 1 % of
    the entries at 8 sigma, INT8 store then INT8 decode.  At this size the host picks the one-wave-per-head kernel
    with 16 partitions of 1024 tokens and the merge kernel (a smaller batch would take the other form).  The cache
    (2.2 GB of codes) is written on the device by the INT8 store in chunks; the oracle runs on picked sequences."""
    hq, hkv, d, bs, batch = 32, 8, 128, 16, 128
    scale = 1 / math.sqrt(d)
    g = torch.Generator().manual_seed(165)
    ctx = torch.randint(256, 16385, (batch,), generator=g)
    ctx[7], ctx[99] = 16384, 256                                   # both ends of the range are present
    need = [-(-int(c) // bs) for c in ctx.tolist()]
    nb = sum(need)
    perm = torch.randperm(nb, generator=g)
    tables = torch.full((batch, 16384 // bs), -1, dtype=torch.int32)
    at = 0
    for b, n in enumerate(need):
        tables[b, :n] = perm[at:at + n].to(torch.int32)
        at += n
    assert paged_decode_plan(batch, hq, hkv, d, tables.shape[1], bs, torch.bfloat16, int8_cache=True) == (1024, 16, 1)
    ck = torch.empty(nb, bs, hkv, d, dtype=torch.int8, device=DEV)
    cv = torch.empty_like(ck)
    sk = torch.empty(nb, bs, hkv, device=DEV)
    sv = torch.empty_like(sk)
    dg = torch.Generator(device=DEV).manual_seed(166)
    step = 4096                                                    # blocks per chunk: 64 K tokens, 134 MB of bf16 each
    for lo in range(0, nb, step):
        n = min(step, nb - lo) * bs
        kv = []
        for _ in range(2):
            x = torch.randn(n, hkv, d, generator=dg, device=DEV)
            x = torch.where(torch.rand(x.shape, generator=dg, device=DEV) < 0.01, x * 8.0, x)
            kv.append(x.to(torch.bfloat16))
        store_kvcache_int8(kv[0], kv[1], ck, cv, sk, sv, torch.arange(lo * bs, lo * bs + n, device=DEV), bs)
    q = torch.randn(batch, hq, d, generator=dg, device=DEV).to(torch.bfloat16)
    td, cd = tables.to(DEV), ctx.to(DEV)
    got = paged_attention_decode_int8(q, ck, cv, sk, sv, td, cd, scale, hq, hkv, d, bs).cpu()
    assert torch.isfinite(got).all()
    order = torch.argsort(ctx)
    pick = sorted({int(order[0]), int(order[1]), int(order[-1]), int(order[-2]), int(order[batch // 2]), 0, 64, 127})
    assert len(pick) >= 8
    for b in pick:
        ids = tables[b, :need[b]].long().to(DEV)
        table = torch.arange(need[b], dtype=torch.int32).unsqueeze(0)
        want = oracle.decode_int8_oracle(q[b:b + 1].cpu().float(), ck[ids].cpu(), cv[ids].cpu(), sk[ids].cpu(),
                                         sv[ids].cpu(), table, ctx[b:b + 1], scale, hq, hkv, d, bs)
        mx, mean = error_stats(got[b:b + 1], want)
        assert mx <= 2e-2 and mean <= 2e-3, (b, int(ctx[b]), mx, mean)    # the stated bound, no allowance
    # size-independent property over the whole batch: the output is linear in the V scales
    sv *= 2
    got2 = paged_attention_decode_int8(q, ck, cv, sk, sv, td, cd, scale, hq, hkv, d, bs).cpu()
    assert (got2.float() - 2 * got.float()).abs().max() <= 2e-2 + 2.0 ** -7 * got.float().abs().max()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("hq", [32, 8])
def test_int8_keys_as_operands_or_in_rows(dtype, hq):
    """Long tables: a batch of up to 2048 waves takes its keys as operands, a larger one in rows through LDS; same products in the same
    order, so the sequences of the smaller batch come out the same to the bit.  Contexts end at and beside tile and partition edges."""
    hkv, d, bs, scale = 8, 128, 16, 128 ** -0.5
    lens = [32768, 30001, 1, 17, 1024, 1025, 5007, 2048, 16]
    case = _quantised_case(67, 0, 0, 0, hq, hkv, d, bs, dtype, ctx_list=lens)
    few, many = (paged_decode_plan(n, hq, hkv, d, 2048, bs, int8_cache=True) for n in (8, 9))
    assert few == many and few[1] * 8 * hkv == 2048 and few[2] == 1            # one wave per kv head and partition
    whole = _check(case, hq, hkv, d, bs, scale)
    q, ck, cv, sk, sv, tables, ctx = case
    got = paged_attention_decode_int8(q[:8].to(DEV), ck, cv, sk, sv, tables[:8].to(DEV), ctx[:8].to(DEV), scale, hq, hkv, d, bs).cpu()
    assert torch.equal(got, whole[:8])
