"""The C-ABI library loads and exports every symbol include/minivllm_amd.h declares.
No compute calls: there is no GPU here."""
import ctypes
import os
import re

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HEADER = os.path.join(ROOT, "include", "minivllm_amd.h")


def _declared():
    text = open(HEADER).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(mvllm_[a-z0-9_]+)\s*\(", text)))


def _lib():
    from minivllm_amd import _C
    if not os.path.exists(_C.lib_path()):
        from minivllm_amd._build import build_library
        build_library(verbose=False)
    return _C


def test_header_declares_expected_entry_points():
    names = _declared()
    for n in ["mvllm_store_kvcache", "mvllm_store_kvcache_int8", "mvllm_paged_decode",
              "mvllm_paged_decode_int8", "mvllm_paged_decode_noalloc", "mvllm_paged_decode_workspace_bytes", "mvllm_paged_decode_plan", "mvllm_paged_decode_partition", "mvllm_prefill_plan", "mvllm_prefill_varlen",
              "mvllm_prefill_paged", "mvllm_prefill_paged_int8", "mvllm_prefill_paged_int8_staged", "mvllm_prefill_paged_staged", "mvllm_prefill_paged_staged_workspace_bytes", "mvllm_prefill_paged_split", "mvllm_prefill_paged_int8_split", "mvllm_prefill_paged_split_plan", "mvllm_prefill_paged_split_workspace_bytes", "mvllm_qk_norm_rope_store", "mvllm_sample_tokens", "mvllm_sample_tokens_dev_offset", "mvllm_decode_advance", "mvllm_sample_tokens_workspace_bytes",
              "mvllm_add_rms_norm", "mvllm_linear_small_m", "mvllm_norm_linear_small_m", "mvllm_linear_small_m_plan",
              "mvllm_linear_small_m_split", "mvllm_linear_small_m_split_bytes", "mvllm_prefill_ranges", "mvllm_prefill_ranges_plan", "mvllm_prefill_ranges_groups", "mvllm_prefill_store",
              "mvllm_prefill_ranges_workspace_bytes", "mvllm_mlstm_chunked_output",
              "mvllm_lm_head_sample", "mvllm_lm_head_sample_workspace_bytes",
              "mvllm_paged_decode_sink", "mvllm_prefill_varlen_sink", "mvllm_prefill_paged_sink",
              "mvllm_prefill_paged_split_sink", "mvllm_norm_conv", "mvllm_head_rope_store", "mvllm_head_unrotate_gate",
              "mvllm_chunk_decode_step", "mvllm_gate_linear", "mvllm_mlstm_recurrent", "mvllm_mlstm_output",
              "mvllm_mlstm_chunked", "mvllm_mlstm_chunked_workspace_bytes",
              "mvllm_stream_embed_norm", "mvllm_stream_norm", "mvllm_decay_memory_recurrent", "mvllm_decay_memory_chunked",
              "mvllm_decay_memory_chunked_workspace_bytes", "mvllm_gated_row_norm", "mvllm_latent_norm_store",
              "mvllm_head_linear", "mvllm_latent_decode", "mvllm_latent_decode_workspace_bytes", "mvllm_moe_route",
              "mvllm_moe_plan", "mvllm_moe_plan_bytes", "mvllm_moe_linear", "mvllm_moe_linear_shared", "mvllm_moe_linear_tiles",
              "mvllm_moe_route_softmax", "mvllm_moe_linear_clamped", "mvllm_gated_unit", "mvllm_stream_norm_identity", "mvllm_window_prefill",
              "mvllm_window_decode_workspace_bytes", "mvllm_window_decode", "mvllm_latent_rope_store", "mvllm_head_rope", "mvllm_copy_rows",
              "mvllm_head_norm_rope_store", "mvllm_window_decode_split", "mvllm_gelu_tanh", "mvllm_linear_small_m_gelu",
              "mvllm_post_norm", "mvllm_embed_rows", "mvllm_talk_prefill", "mvllm_talk_decode", "mvllm_talk_decode_workspace_bytes",
              "mvllm_silu_and_mul", "mvllm_version", "mvllm_status_string", "mvllm_calls_digest"]:
        assert n in names


def test_library_exports_every_declared_symbol():
    _C = _lib()
    raw = ctypes.CDLL(_C.lib_path())
    for name in _declared():
        assert hasattr(raw, name), f"{name} declared in the header but not exported"
    assert set(_C.SIGNATURES) == set(_declared())


def test_host_only_entry_points():
    _C = _lib()
    lib = _C.load()
    assert lib.mvllm_version() >= 1000
    assert lib.mvllm_status_string(-5).decode().startswith("workspace")
    # pure host arithmetic: (D + 2) floats per (seq, partition, head); partitions of 256..1024 tokens, at most 32
    # per sequence, shortened down to 64 tokens while batch * partitions < 1024
    assert lib.mvllm_paged_decode_workspace_bytes(1024, 16, 128, 16, 16) == 0        # 256 tokens: 1 partition
    assert lib.mvllm_paged_decode_workspace_bytes(8, 16, 128, 16, 16) == 8 * 4 * 16 * 130 * 4     # 4 x 64 tokens
    assert lib.mvllm_paged_decode_workspace_bytes(2, 4, 128, 64, 16) == 2 * 16 * 4 * 130 * 4      # 16 x 64 tokens
    assert lib.mvllm_paged_decode_workspace_bytes(256, 32, 128, 2048, 16) == 256 * 32 * 32 * 130 * 4


def test_prefill_ranges_take_any_bound():
    """A bound of the keys that is no bound at all is still one: counts do not overflow, the range grows with it."""
    lib = _lib().load()
    for keys in (4096, 2 ** 20, 2 ** 31 - 64, 2 ** 31 - 1):
        tiles, per = -(-keys // 64), lib.mvllm_prefill_ranges_plan(10, 500, keys, 16, 8, 128, 0, 1)
        ranges = -(-tiles // per)
        assert per % 2 == 0 and 2 <= ranges <= 64
        assert lib.mvllm_prefill_ranges_workspace_bytes(500, keys, 16, 128, per) == ranges * 500 * 16 * 129 * 4
        assert lib.mvllm_prefill_ranges_workspace_bytes(500, keys, 16, 128, 6) == -(-tiles // 6) * 500 * 16 * 129 * 4


def test_prefill_ranges_plan_looks_at_the_busiest_cu():
    """Equal sequences whose heavy row tiles meet on a CU stay with the other kernels, whatever their number; uneven ones, a single one and
    those that fit side by side go over."""
    plan = _lib().load().mvllm_prefill_ranges_plan
    heads, packed, paged = (16, 8, 128), (0, 1), (16, 1)
    assert plan(2, 2992, 1496, *heads, *packed) == 24 and plan(2, 3312, 1656, *heads, *packed) == 0    # 1.67 and 1.79 of the longest tile
    assert plan(3, 2928, 976, *heads, *packed) == 0 and plan(3, 3888, 1296, *heads, *packed) == 22     # 2.0 and 1.52
    assert plan(2, 3311, 1987, *heads, *packed) == 32 and plan(1, 3376, 3376, *heads, *packed) == 54   # uneven, one
    assert plan(5, 3120, 624, *heads, *packed) == 10                                                   # short: the start counts
    assert plan(3, 2382, 1588, *heads, *paged) == 26 and plan(4, 2352, 1176, *heads, *paged) == 0      # 1.80 and 1.90
    four = (32, 8, 64)
    assert plan(4, 1672, 758, *four, *paged) == 0 and plan(4, 2072, 758, *four, *paged) == 12          # 512 and 768 places of the other form
    assert plan(4, 472, 758, *four, *paged) == 12 and plan(8, 744, 758, *four, *paged) == 12           # one workgroup per CU
    assert plan(4, 1672, 1910, *four, *paged) == 30                                                    # long


def test_prefill_ranges_plan_keeps_ranges_where_whole_ones_go_elsewhere():
    """Few workgroups of heads of 64 over a cache: one range is another kernel's, so ranges are not given up for one in two groups."""
    plan = _lib().load().mvllm_prefill_ranges_plan
    for rows, seqs, keys, heads, tiles in [(552, 1, 1104, 16, 6), (799, 2, 1040, 8, 6), (324, 1, 1188, 16, 4), (228, 4, 928, 16, 4)]:
        kv = 8 if heads == 16 and rows != 324 else heads
        assert plan(seqs, rows, keys, heads, kv, 64, 16, 1) == tiles, (rows, seqs, keys)


def test_prefill_ranges_plan_of_odd_head_groups():
    """Row tiles of 128 in both forms: packed batches go over only where the other form's places pass the chip's 512, cached ones for its
    empty places, for alike tiles or for keys cut into ranges."""
    plan = _lib().load().mvllm_prefill_ranges_plan
    packed, paged = (0, 1), (16, 1)
    assert plan(10, 3320, 363, 12, 4, 128, *packed) == 0 and plan(5, 3820, 764, 14, 2, 128, *packed) == 0       # no more than 512 places
    assert plan(3, 1200, 400, 40, 8, 128, *packed) == 0                                                        # 480 places
    assert plan(4, 1120, 280, 40, 8, 128, *packed) == 6                                                        # 640 places, 480 workgroups
    assert plan(9, 1152, 128, 40, 8, 128, *packed) == 0                                                        # short: empty places cost nothing
    assert plan(1, 1000, 1000, 12, 4, 128, *packed) == 0
    assert plan(7, 378, 138, 40, 8, 128, *paged) == 4 and plan(10, 1630, 325, 12, 4, 128, *paged) == 0          # empty places, none
    assert plan(10, 1630, 1630, 12, 4, 128, *paged) == 26                                                      # most keys cached
    assert plan(2, 60, 300, 12, 4, 128, *paged) == 0 and plan(2, 60, 500, 12, 4, 128, *paged) == 8              # few, 5 and 8 tiles of keys
    assert 0 < plan(1, 100, 32768, 12, 4, 128, *paged) < 512
    assert plan(4, 1397, 700, 32, 8, 64, *paged) == 0 and plan(4, 1397, 1400, 32, 8, 64, *paged) == 22          # four heads: 352 of 512 places
    at64 = (8, 8, 64)
    assert plan(3, 5775, 1925, *at64, *packed) == 0 and plan(3, 5000, 2600, *at64, *packed) == 42              # equal and uneven
    assert plan(2, 3704, 3703, 16, 16, 64, *paged) == 0 and plan(2, 3704, 18500, 16, 16, 64, *paged) == 0      # 1.97; too many keys
    assert plan(10, 4700, 948, 16, 16, 64, *paged) == 16                                                       # 640 places


def test_prefill_ranges_plan_at_its_limits():
    """Which batches go over key ranges, on either side of each limit; all of them whole (one range of all tiles, an even number)."""
    plan = _lib().load().mvllm_prefill_ranges_plan
    packed, paged, four, two = (0, 1), (16, 1), (32, 8, 128), (16, 8, 128)
    assert plan(9, 1080, 120, *four, *packed) == 2 and plan(13, 1950, 150, *four, *packed) == 4                # four heads: up to 640 workgroups
    assert plan(7, 2300, 370, *four, *packed) == 6 and plan(7, 2400, 370, *four, *packed) == 0                 # 616 and 656
    assert plan(2, 1920, 960, *four, *packed) == 0 and plan(2, 1700, 960, *four, *packed) == 16                # 1.95 of the longest tile and 1.82
    assert plan(9, 2097, 233, *four, *packed) == 0                                                            # 3 of it
    assert plan(4, 2200, 1100, *four, *paged) == 18 and plan(2, 1627, 1631, *four, *paged) == 0                # behind halves: not two of them
    assert plan(1, 1500, 3000, *four, *paged) == 48 and plan(1, 1600, 3200, *four, *paged) == 0                # 384 and 408 of one sequence
    assert plan(4, 700, 3600, *four, *paged) == 58 and plan(8, 1200, 4000, *four, *paged) == 0                 # most keys cached: equal ones stay
    assert plan(1, 5800, 5800, *two, *packed) == 92 and plan(1, 6000, 6000, *two, *packed) == 0                # two heads: one sequence
    assert plan(16, 5900, 370, *two, *packed) == 6 and plan(16, 6900, 440, *two, *packed) == 0                 # 16 short ones
    assert plan(11, 4800, 900, *two, *paged) == 16 and plan(11, 5700, 900, *two, *paged) == 0                  # 688 and 800
    at64 = (32, 8, 64)
    assert plan(9, 1954, 334, *at64, *packed) == 6 and plan(3, 1344, 450, *at64, *packed) == 0                 # places without rows, none
    assert plan(2, 1800, 960, *at64, *packed) == 0 and plan(1, 1800, 1800, *at64, *packed) == 30               # two, one
    assert plan(16, 2720, 340, *at64, *paged) == 6 and plan(8, 4096, 1024, *at64, *paged) == 0                 # beyond 768 workgroups the same


def test_prefill_split_plan_is_host_arithmetic():
    """When a paged prefill is cut over its keys: few query tiles, at least 4096 keys, a shape the split form takes;
    and the workspace holds the ranges' tables, partial results and denominators."""
    _C = _lib()
    lib = _C.load()
    bf16, f32 = 1, 0
    plan = lib.mvllm_prefill_paged_split_plan
    assert plan(1, 128, 32768 + 128, 32, 8, 128, 256, bf16, 0) == 16          # 32 workgroups a range: 15 prefix ranges
    assert plan(1, 16, 32768 + 16, 32, 8, 128, 256, bf16, 0) == 17            # never more than 16 prefix ranges
    assert plan(2, 256, 4096 + 128, 32, 8, 128, 16, bf16, 0) == 5             # 1024 keys a range at least
    assert plan(2, 1024, 16384 + 512, 32, 8, 128, 256, bf16, 0) == 5          # a small batch is cut in 4 at least
    assert plan(16, 512, 4096 + 32, 32, 8, 128, 256, bf16, 0) == 0            # enough query tiles
    assert plan(1, 128, 4095, 32, 8, 128, 256, bf16, 0) == 0                  # too few keys
    assert plan(1, 128, 32768, 32, 8, 128, 256, f32, 0) == 0                  # fp32
    assert plan(1, 128, 32768, 32, 8, 128, 8, bf16, 0) == 0                   # blocks of 8 tokens
    assert plan(1, 128, 32768 + 128, 32, 8, 128, 256, bf16, 1) == 16          # INT8 cache: as the 16-bit one
    assert plan(1, 128, 32768, 32, 8, 80, 256, bf16, 1) == 0                  # ... but at head_dim 64 / 128 only
    assert plan(1, 128, 32768, 16, 8, 80, 256, bf16, 0) == 17                 # head_dim 80: 16 workgroups a range
    assert plan(8, 4096, 32768, 16, 8, 80, 256, bf16, 0) == 0                 # ... 576 of them fill the chip
    assert plan(1, 128, 32768, 16, 8, 72, 256, bf16, 0) == 17                 # head_dim 72: as 80
    assert plan(1, 128, 32768, 16, 8, 136, 256, bf16, 0) == 0                 # head_dim 136: not an LDS-tiled shape
    need = lib.mvllm_prefill_paged_split_workspace_bytes(1, 128, 32768 + 128, 32, 8, 128, 256, bf16, 16)
    partial = 16 * 128 * 32 * 128 * 2 + 16 * 128 * 32 * 4
    assert partial < need < partial + 16384
    assert lib.mvllm_prefill_paged_split_workspace_bytes(8, 128, 32768, 32, 8, 128, 256, bf16, 9) == 0   # 72 ranges


def test_decode_plan_in_narrow_tables():
    """(tokens per partition, partitions, waves) of 16-bit caches in tables of at most 2048 tokens: edges of every rule."""
    import torch
    from minivllm_amd.layers.attention import paged_decode_plan
    _lib().load()
    plan = lambda batch, tokens, kv=8, **kw: paged_decode_plan(batch, 4 * kv, kv, 128, tokens // 16, 16, **kw)
    assert plan(1, 512) == (512, 1, 8) and plan(1, 528) == (128, 5, 8)                # one partition whatever the batch, or parts
    assert plan(1, 2048) == (128, 16, 4) and plan(4, 2048) == (128, 16, 4)            # 512 workgroups at most ...
    assert plan(5, 2048) == (256, 8, 4) and plan(8, 1024) == (128, 8, 4)              # ... from then on 256 tokens
    assert plan(8, 1040) == (256, 5, 4) and plan(31, 2048) == (704, 3, 4)
    assert plan(32, 2048) == (2048, 1, 8) and plan(33, 2048) == (2048, 1, 4)          # one from 256 pairs on; eight waves up to 256 workgroups
    thin = lambda batch, tokens, d, block=16: paged_decode_plan(batch, 32, 8, d, tokens // block, block)
    assert thin(33, 2048, 64) == thin(63, 2048, 32) == thin(63, 2048, 104) == (2048, 1, 8)             # below 112 dims eight waves
    assert thin(33, 2048, 112) == thin(64, 2048, 64) == (2048, 1, 4) and thin(33, 512, 64) == (512, 1, 4)
    assert thin(33, 2048, 64, 8) == (1024, 2, 4) and thin(33, 2048, 128, 8) == (2048, 1, 4)            # blocks of less than a tile
    assert plan(31, 2064) == (704, 3, 4) and plan(33, 2064) == (1088, 2, 4)
    assert plan(1, 2048, int8_cache=True)[0] == 64 and plan(1, 2048, dtype=torch.float32)[0] == 64


def test_decode_partitions_of_a_sequence():
    """Their length follows the sequence's own where the plan says so, is never past the plan's, and never makes more of them than the workspace has."""
    import random
    import torch
    from minivllm_amd.layers.attention import paged_decode_partition, paged_decode_plan
    _lib().load()
    of = lambda ctx, batch, tokens, d=128, block=16, **kw: paged_decode_partition(ctx, batch, 32, 8, d, tokens // block, block, **kw)
    assert paged_decode_plan(12, 32, 8, 128, 128, 16) == (384, 6, 4)
    assert [of(n, 12, 2048) for n in (0, 1, 640, 641, 960, 961, 1600, 1601, 2048)] == [128, 128, 128, 192, 192, 256, 320, 384, 384]      # a fifth (512 / 96), in whole 64s
    assert paged_decode_plan(24, 32, 8, 128, 128, 16) == (704, 3, 4) and [of(n, 24, 2048) for n in (300, 1024, 1025, 2048)] == [512, 512, 576, 704]     # 512 at least
    assert of(1, 33, 2048) == 2048 and of(300, 64, 32768) == of(32768, 64, 32768) == 1024      # one partition, or one wave per head: the plan's
    wide = lambda batch, d, int8: of(100, batch, 6144, d, int8_cache=int8) < paged_decode_plan(batch, 32, 8, d, 384, 16, int8_cache=int8)[0]
    assert wide(24, 64, False) and wide(24, 128, False)                                # wide tables of INT8 caches up to 128 pairs of heads of 64, 176 of 128
    assert wide(16, 64, True) and not wide(17, 64, True) and wide(22, 128, True) and not wide(23, 128, True)
    assert of(100, 30, 2048, 64, int8_cache=True) < paged_decode_plan(30, 32, 8, 64, 128, 16, int8_cache=True)[0]
    assert of(100, 12, 2048, dtype=torch.float32) == of(2048, 12, 2048, dtype=torch.float32)
    rng, shorter = random.Random(3), 0
    for _ in range(3000):
        batch, tokens, kv = rng.randint(1, 80), 16 * rng.randint(1, 2000), rng.choice((1, 2, 8))
        sizes = (batch, 4 * kv, kv, rng.choice((32, 64, 128, 256)), tokens // 16, 16, rng.choice((torch.bfloat16, torch.float16, torch.float32)), rng.random() < 0.3)
        part, parts, waves = paged_decode_plan(*sizes)
        ctx = rng.randint(0, tokens)
        own = paged_decode_partition(ctx, *sizes)
        assert 0 < own <= part and -(-ctx // own) <= parts and (own == part or own % 64 == 0 and waves > 1)
        shorter += own < part
    assert shorter > 100
    for bad in (-1, 2049):
        with pytest.raises(ValueError):
            of(bad, 12, 2048)


def test_tiles_of_products_over_sorted_pairs():
    """Which tiles a product runs on: edges of every rule."""
    from minivllm_amd.layers.experts import moe_linear_tiles as tiles
    _lib().load()
    assert tiles(32, 8, 1536, 2048) == (32, 64) and tiles(33, 9, 1536, 2048) == (64, 64)          # one block of rows
    assert tiles(6, 64, 1536, 768) == (32, 64) and tiles(6, 64, 1536, 704) == (64, 128)           # K
    assert tiles(6, 64, 1536, 2048, (1, 64, 704)) == (64, 128) and tiles(6, 64, 1536, 2048, (1, 64, 768)) == (32, 64)
    assert tiles(4 * 8, 8, 512, 2048) == (32, 64) and tiles(4 * 8 + 1, 8, 512, 2048) == (64, 128) # pairs per expert
    assert tiles(1, 1, 160 * 128, 768) == (32, 64) and tiles(1, 1, 161 * 128, 768) == (64, 128)   # workgroups: up to 160,
    assert tiles(1, 1, 247 * 128, 768) == (64, 128) and tiles(1, 1, 248 * 128, 768) == (32, 64)   # ... from 248
    assert tiles(1, 1, 328 * 128, 768) == (32, 64) and tiles(1, 1, 329 * 128, 768) == (64, 128)
    assert tiles(1, 1, 384 * 128, 1024) == (32, 64) and tiles(1, 1, 385 * 128, 1024) == (64, 128)
    assert tiles(1, 1, 150 * 128, 1024, (1, 10 * 128, 1024)) == (32, 64) and tiles(1, 1, 150 * 128, 1024, (65, 6 * 128, 1024)) == (64, 128)
    assert tiles(48 * 64, 64, 1536, 2048) == (64, 128) and tiles(48 * 64 + 1, 64, 1536, 2048) == (256, 256)      # rows per expert, large tiles for every CU
    assert tiles(48 * 16 + 1, 16, 1024, 2048) == (128, 128) and tiles(384 * 16, 16, 1024, 2048) == (256, 256)
    with pytest.raises(ValueError):
        tiles(0, 1, 64, 64)


def test_decode_plan_is_host_arithmetic():
    """Which form a decode call takes, and that the split form never needs more workspace than is advertised."""
    import torch
    from minivllm_amd.layers.attention import paged_decode_plan
    lib = _lib().load()
    # one-wave-per-head form: large batch over a wide table (1024-token partitions)
    assert paged_decode_plan(256, 32, 8, 128, 2048, 16) == (1024, 32, 1)
    assert paged_decode_plan(64, 32, 8, 128, 2048, 16) == (1024, 32, 1)
    # small-batch form: 64 sequences x 8 kv heads in a 4096-token table are one partition each, four waves per head
    assert paged_decode_plan(64, 32, 8, 128, 256, 16) == (4096, 1, 4)
    assert paged_decode_plan(256, 32, 8, 128, 16, 256) == (4096, 1, 4)        # any batch while the table is <= 4096
    assert paged_decode_plan(1, 32, 8, 128, 2048, 16) == (1024, 32, 4)        # one long sequence: 256 workgroups
    for batch in (15, 16, 17):                                                # long partitions of one even round are no exception
        assert paged_decode_plan(batch, 32, 8, 128, 512, 16) == (512, 16, 4)
    for batch in (31, 32, 33):
        assert paged_decode_plan(batch, 32, 8, 128, 256, 16) == (512, 8, 4)
    # INT8 caches, and shapes outside the MFMA kernels
    assert paged_decode_plan(64, 32, 8, 128, 256, 16, int8_cache=True) == (4096, 1, 4)
    assert paged_decode_plan(256, 32, 8, 128, 256, 16, int8_cache=True) == (1024, 4, 1)     # large INT8 batch: first form
    assert paged_decode_plan(64, 16, 16, 64, 256, 16)[2] == 4                 # head_dim 64: MFMA kernels, both cache types
    assert paged_decode_plan(64, 16, 16, 64, 256, 16, int8_cache=True)[2] == 1      # 1024 (sequence, head) pairs: first form
    assert paged_decode_plan(64, 16, 16, 96, 256, 16, int8_cache=True)[2] == 0
    assert paged_decode_plan(64, 16, 16, 96, 256, 16)[2] == 4                 # 16-bit caches: also 96 dims (three 32-dim steps)
    assert paged_decode_plan(64, 16, 16, 80, 256, 16)[2] == 4 and paged_decode_plan(64, 16, 16, 112, 256, 16)[2] == 4   # ... and a partial last step
    assert paged_decode_plan(64, 16, 16, 72, 256, 16)[2] == 4 and paged_decode_plan(64, 16, 16, 120, 256, 16)[2] == 4   # any multiple of 8 from 32 to 128
    assert paged_decode_plan(64, 16, 16, 100, 256, 16)[2] == 0 and paged_decode_plan(64, 16, 16, 136, 256, 16)[2] == 0   # other head dims
    assert paged_decode_plan(64, 16, 16, 72, 256, 16, dtype=torch.float32)[2] == 0
    assert paged_decode_plan(64, 16, 8, 256, 256, 16)[2] == 4                 # 16-bit caches: also 256 and 32 dims
    assert paged_decode_plan(64, 16, 8, 32, 256, 16)[2] == 4
    assert paged_decode_plan(64, 16, 8, 256, 256, 16, int8_cache=True)[2] == 0
    assert paged_decode_plan(64, 16, 8, 256, 256, 16, dtype=__import__("torch").float32)[2] == 0
    assert paged_decode_plan(64, 32, 8, 128, 256, 16, dtype=torch.float32)[2] == 4       # fp32 caches: fp32 MFMA
    assert paged_decode_plan(64, 32, 8, 128, 256, 16, dtype=torch.float32, int8_cache=True)[2] == 0
    assert paged_decode_plan(8, 34, 2, 128, 64, 16)[2] == 4                   # 17 query heads per kv head: two slices each
    # the advertised workspace covers whatever form is chosen
    for batch in (1, 3, 16, 64, 200, 1000):
        for blocks, bs in ((16, 16), (64, 16), (300, 16), (2048, 16), (40, 256), (70000, 16)):
            for hkv in (1, 2, 8):
                part, parts, waves = paged_decode_plan(batch, 8 * hkv, hkv, 128, blocks, bs)
                assert part % 16 == 0 and parts == -(-blocks * bs // part) and 1 <= parts <= 32
                need = 0 if parts == 1 else batch * parts * 8 * hkv * 130 * 4
                assert need <= lib.mvllm_paged_decode_workspace_bytes(batch, 8 * hkv, 128, blocks, bs)


def test_prefill_plan_is_host_arithmetic():
    """Which kernel a prefill takes: 2 LDS-tiled MFMA, 1 16-row tile MFMA, 0 generic."""
    import torch
    from minivllm_amd.layers.attention import prefill_plan
    assert prefill_plan(32, 8, 128) == 2 and prefill_plan(16, 8, 64, dtype=torch.float16) == 2
    assert prefill_plan(32, 8, 128, block_size=16) == 2 and prefill_plan(32, 8, 128, block_size=8) == 0
    assert prefill_plan(32, 8, 128, dtype=torch.float32) == 2 and prefill_plan(16, 8, 64, 16, torch.float32) == 2     # fp32: its own LDS-tiled kernel
    assert prefill_plan(16, 8, 64, 8, torch.float32) == 0
    assert prefill_plan(8, 8, 256) == 2 and prefill_plan(8, 8, 32, block_size=32) == 2      # bf16 / fp16 only
    assert prefill_plan(8, 8, 256, dtype=torch.float32) == 0
    assert prefill_plan(6, 2, 80) == 2 and prefill_plan(6, 2, 96) == 2 and prefill_plan(6, 2, 96, dtype=torch.float32) == 0
    assert prefill_plan(6, 2, 112, block_size=16) == 2 and prefill_plan(6, 2, 112, block_size=8) == 0
    assert prefill_plan(6, 2, 72) == 2 and prefill_plan(6, 2, 40) == 2 and prefill_plan(6, 2, 48) == 2 and prefill_plan(6, 2, 100) == 0
    assert prefill_plan(6, 2, 120, block_size=32) == 2 and prefill_plan(6, 2, 72, dtype=torch.float32) == 0
    assert prefill_plan(6, 2, 136) == 0 and prefill_plan(6, 2, 24) == 0
    assert prefill_plan(32, 8, 128, 16, int8_cache=True) == 2
    assert prefill_plan(32, 8, 96, 16, int8_cache=True) == -1 and prefill_plan(32, 8, 128, 16, torch.float32, True) == -1
    assert prefill_plan(8, 8, 1024) == -1


def test_generic_kernel_warning_is_raised_once_per_shape():
    import warnings
    import torch
    from minivllm_amd.layers import attention
    attention._shapes_seen.clear()
    with warnings.catch_warnings(record=True) as seen:
        warnings.simplefilter("always")
        attention._warn_if_generic("decode", 16, 16, 100, 16, torch.bfloat16, False)
        attention._warn_if_generic("decode", 16, 16, 100, 16, torch.bfloat16, False)      # same shape: silent
        attention._warn_if_generic("prefill", 6, 2, 100, 0, torch.bfloat16, False)
        attention._warn_if_generic("decode", 32, 8, 128, 16, torch.bfloat16, False)      # MFMA kernel: silent
        attention._warn_if_generic("prefill", 32, 8, 128, 0, torch.bfloat16, False)
    assert len(seen) == 2 and all("generic kernel" in str(w.message) for w in seen)


def test_argument_validation_without_gpu():
    """Invalid arguments are rejected before any launch, so this is safe on CPU."""
    _C = _lib()
    lib = _C.load()
    assert lib.mvllm_store_kvcache(0, 0, 0, 0, 0, 4, 16, 2, 8, 7, 0) == -2      # bad dtype
    assert lib.mvllm_store_kvcache(0, 0, 0, 0, 0, 4, 16, 0, 8, 1, 0) == -3      # bad shape
    assert lib.mvllm_store_kvcache(0, 0, 0, 0, 0, 4, 16, 2, 8, 1, 0) == -1      # null pointers
    assert lib.mvllm_store_kvcache(0, 0, 0, 0, 0, 0, 16, 2, 8, 1, 0) == 0       # empty is a no-op
    assert lib.mvllm_store_kvcache_int8(0, 0, 0, 0, 0, 0, 0, 4, 16, 2, 12, 1, 0) == -4   # D % 8 != 0
    assert lib.mvllm_paged_decode(0, 0, 0, 0, 0, 4, 0, 1, 2, 6, 4, 128, 16, 8, 1.0, 1, 0, 0, 0) == -3  # Hq % Hkv
    noalloc = lib.mvllm_paged_decode_noalloc
    assert noalloc(0, 0, 0, 0, 0, 4, 0, 1, 2, 6, 4, 128, 16, 8, 1.0, 1, 0) == -3                       # Hq % Hkv
    assert noalloc(1, 1, 1, 1, 1, 2048, 1, 1, 256, 32, 8, 128, 16, 8, 1.0, 1, 0) == -5                 # beyond the static array: refused before any launch
    assert lib.mvllm_prefill_varlen(0, 0, 0, 0, 0, 0, 0, 4, 2, 128, 1.0, 1, 0) == 0      # empty batch
    assert lib.mvllm_prefill_varlen(0, 0, 0, 0, 0, 1, 5, 4, 2, 128, 1.0, 1, 0) == -1
    paged = lib.mvllm_prefill_paged
    #            out q kc vc tables MB cu_q cu_k S  T  Hq Hkv D   bs  NB scale dt stream
    assert paged(0, 0, 0, 0, 0, 4, 0, 0, 0, 0, 4, 2, 128, 16, 8, 1.0, 1, 0) == 0       # no sequences
    assert paged(0, 0, 0, 0, 0, 4, 0, 0, 1, 5, 4, 2, 128, 16, 8, 1.0, 1, 0) == -1      # null pointers
    assert paged(0, 0, 0, 0, 0, 4, 0, 0, 1, 5, 4, 3, 128, 16, 8, 1.0, 1, 0) == -3      # Hq % Hkv
    assert paged(0, 0, 0, 0, 0, 4, 0, 0, 1, 5, 4, 2, 128, 0, 8, 1.0, 1, 0) == -3       # block_size
    sample = lib.mvllm_sample_tokens
    assert sample(0, 0, 100, 0, 0, 1, 2, 0, 100, 1, 0, 0, 0) == 0        # empty batch
    assert sample(0, 0, 100, 0, 0, 1, 2, 4, 100, 1, 0, 0, 0) == -1       # null pointers
    assert sample(0, 0, 50, 0, 0, 1, 2, 4, 100, 1, 0, 0, 0) == -3        # row stride < vocab
    assert sample(0, 0, 100, 0, 0, 1, 2, 4, 100, 5, 0, 0, 0) == -2       # dtype
    ws = lib.mvllm_sample_tokens_workspace_bytes
    assert ws(64, 151936) == 64 * 8 * 8 and ws(1024, 151936) == 0 and ws(4, 1000) == 0 and ws(1, 151936) == 38 * 8
    norm = lib.mvllm_add_rms_norm
    assert norm(0, 0, 0, 0, 0, 1e-6, 0, 1024, 1024, 1024, 1, 0) == 0       # no rows
    assert norm(0, 0, 0, 0, 0, 1e-6, 4, 1024, 1024, 1024, 1, 0) == -1      # null pointers
    assert norm(0, 0, 0, 0, 0, 1e-6, 4, 1004, 1004, 1004, 1, 0) == -4      # hidden % 8
    assert norm(0, 0, 0, 0, 0, 1e-6, 4, 1024, 512, 1024, 1, 0) == -3       # stride < hidden
    act = lib.mvllm_silu_and_mul
    assert act(0, 0, 0, 3072, 6144, 1, 0) == 0
    assert act(0, 0, 2, 3072, 6144, 1, 0) == -1
    assert act(0, 0, 2, 3072, 3072, 1, 0) == -3                            # stride < 2 * width
    assert act(0, 0, 2, 3001, 6002, 1, 0) == -4                            # width not a multiple of 16 bytes
    lin = lib.mvllm_linear_small_m
    assert lin(0, 0, 0, 0, 1024, 0, 4096, 1024, 1, 0) == 0                 # no rows
    assert lin(0, 0, 0, 0, 1024, 4, 4096, 1024, 1, 0) == -1                # null pointers
    assert lin(16, 16, 16, 0, 1024, 65, 4096, 1024, 1, 0) == -4            # more than 64 rows: the library GEMM's
    assert lin(16, 16, 16, 0, 1024, 4, 4100, 1024, 1, 0) == -4             # N % 16
    assert lin(16, 16, 16, 0, 1000, 4, 4096, 1000, 1, 0) == -4             # K % 512
    assert lin(16, 16, 16, 0, 512, 4, 4096, 1024, 1, 0) == -3              # row stride < K
    assert lin(16, 16, 16, 0, 1024, 4, 4096, 1024, 0, 0) == -4             # fp32
    nl = lib.mvllm_norm_linear_small_m
    #    out res_out x res gamma eps w bias stride M N K glu dtype stream
    assert nl(0, 0, 0, 0, 0, 1e-6, 0, 0, 1024, 0, 4096, 1024, 0, 1, 0) == 0          # no rows
    assert nl(0, 0, 0, 0, 0, 1e-6, 0, 0, 1024, 4, 4096, 1024, 0, 1, 0) == -1         # null pointers
    assert nl(16, 0, 16, 16, 0, 1e-6, 16, 0, 1024, 4, 4096, 1024, 0, 1, 0) == -1     # a residual without gamma
    assert nl(16, 32, 32, 48, 64, 1e-6, 16, 0, 1024, 4, 4096, 1024, 0, 1, 0) == -3   # residual_out aliases x
    assert nl(16, 0, 16, 0, 0, 1e-6, 16, 0, 1024, 4, 4112, 1024, 1, 1, 0) == -4      # glu: N % 32
    plan = lib.mvllm_linear_small_m_plan
    w = ctypes.c_int(0)
    assert plan(16, 4096, 1024, 1, 0, 1, ctypes.byref(w)) == 0 and w.value == 4     # the engine's QKV projection
    assert plan(32, 6144, 1024, 1, 1, 1, ctypes.byref(w)) == 0 and w.value == 4     # gate/up with norm and SiLU
    assert plan(33, 4096, 1024, 1, 0, 1, ctypes.byref(w)) == 0 and w.value == 4     # 17 rows and more: a workgroup per 16 rows
    assert plan(64, 6144, 1024, 1, 1, 1, ctypes.byref(w)) == 0 and w.value == 4
    assert plan(33, 4096, 1024, 0, 0, 1, None) == 0                                 # plain: up to 64
    assert plan(16, 1024, 3072, 1, 0, 1, None) == -4                                # K / waves is not one burst
    assert plan(16, 1024, 2048, 1, 0, 1, ctypes.byref(w)) == 0 and w.value == 16    # 16 waves, 128 values each
    assert plan(32, 1024, 2048, 1, 0, 1, ctypes.byref(w)) == 0 and w.value == 8     # two row tiles: twice the workgroups, half the waves
    assert plan(16, 4096, 1024, 1, 0, 0, None) == -4 and plan(16, 4096, 1024, 1, 0, 9, None) == -2
    lm = lib.mvllm_lm_head_sample
    #   out hidden stride row_index weight temps seed offset offset_dev batch vocab K dtype ws ws_bytes stream
    assert lm(0, 0, 1024, 0, 0, 0, 0, 0, 0, 0, 151936, 1024, 1, 0, 0, 0) == 0                  # no rows
    assert lm(0, 0, 1024, 0, 0, 0, 0, 0, 0, 4, 151936, 1024, 1, 0, 0, 0) == -1                 # null pointers
    assert lm(8, 16, 1024, 0, 16, 8, 0, 0, 0, 65, 151936, 1024, 1, 0, 0, 0) == -4              # more than 64 rows
    assert lm(8, 16, 1024, 0, 16, 8, 0, 0, 0, 4, 151930, 1024, 1, 0, 0, 0) == -4               # vocab % 16
    assert lm(8, 16, 768, 0, 16, 8, 0, 0, 0, 4, 151936, 768, 1, 0, 0, 0) == -4                 # hidden size
    assert lm(8, 16, 1024, 0, 16, 8, 0, 0, 0, 4, 151936, 1024, 0, 0, 0, 0) == -4               # fp32
    assert lm(8, 16, 1024, 0, 16, 8, 0, 0, 0, 4, 151936, 1024, 1, 0, 0, 0) == -5               # no workspace
    wsb = lib.mvllm_lm_head_sample_workspace_bytes
    assert wsb(16, 1024) == 16 * 512 * 8 and wsb(64, 1024) == 64 * 256 * 8 and wsb(65, 1024) == 0
    adv = lib.mvllm_decode_advance
    assert adv(0, 0, 0, 0, 0, 0, 0, 0, 0, 0) == 0 and adv(0, 0, 0, 0, 0, 0, 0, 0, 4, 0) == -1
    assert adv(0, 0, 0, 0, 0, 0, 0, 0, -1, 0) == -3 and adv(8, 8, 8, 8, 8, 0, 8, 8, 4, 0) == -1     # host ids without the counter
    assert adv(8, 8, 8, 8, 8, 8, 8, 4, 4, 0) == -3                                                # host rows shorter than the batch + 1
    assert lib.mvllm_sample_tokens_dev_offset(8, 8, 100, 8, 1, 0, 4, 100, 1, 0, 0, 0) == -1       # no counter
    fused = lib.mvllm_qk_norm_rope_store
    #     q_out k_out v_out q k v | strides | gamma eps cos max_pos pos slots | caches scales int8 | T slots Hq Hkv D dt stream
    assert fused(0, 0, 0, 0, 0, 0, 512, 256, 256, 0, 1e-6, 0, 64, 0, 0, 0, 0, 0, 0, 0, 0, 0, 4, 2, 128, 1, 0) == 0   # no tokens
    assert fused(0, 0, 0, 0, 0, 0, 512, 256, 256, 0, 1e-6, 0, 64, 0, 0, 0, 0, 0, 0, 0, 3, 0, 4, 2, 128, 1, 0) == -1  # nulls
    assert fused(0, 0, 0, 0, 0, 0, 512, 256, 256, 0, 1e-6, 0, 64, 0, 0, 0, 0, 0, 0, 0, 3, 0, 4, 2, 100, 1, 0) == -4  # D % 8
    assert fused(0, 0, 0, 0, 0, 0, 100, 256, 256, 0, 1e-6, 0, 64, 0, 0, 0, 0, 0, 0, 0, 3, 0, 4, 2, 128, 1, 0) == -3  # stride < row
    assert fused(0, 0, 0, 0, 0, 0, 512, 256, 256, 0, 1e-6, 0, 64, 0, 0, 0, 0, 0, 0, 0, 3, 0, 4, 2, 128, 9, 0) == -2  # dtype
    with pytest.raises(ValueError):
        _C.check(-3, "x")
    with pytest.raises(RuntimeError):
        _C.check(700, "x")
