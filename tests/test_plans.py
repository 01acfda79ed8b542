"""Which kernel a product or an attention step is given: the decisions of ``ops/linear.py`` and ``ops/attention.py``
at the layer sizes of the 1.5B, 7B and 32B shapes.  Pure functions of the sizes: no GPU is touched."""
from vipera_rs_amd.ops.attention import decode_chunking
from vipera_rs_amd.ops.kernels import follow_stride, follow_sumsq_floats
from vipera_rs_amd.ops.linear import (gated_plan, gated_resident_fits, mid_plan, split_qkv_plan, streams_in_wave_order,
                                      streams_weights)

QKV_7B, O_7B, GATE_UP_7B, DOWN_7B, HEAD_7B = (4608, 3584), (3584, 3584), (37888, 3584), (3584, 18944), (152064, 3584)


def test_few_tokens_stream_the_weights_with_k_split_inside_a_workgroup():
    for n, k in (QKV_7B, O_7B, DOWN_7B, HEAD_7B):
        assert streams_in_wave_order(1, n, k) and streams_in_wave_order(4, n, k)
    assert streams_in_wave_order(16, *QKV_7B) and streams_in_wave_order(16, *O_7B)    # small weights: up to 16 tokens
    assert streams_in_wave_order(16, *QKV_7B, rotates=True) and not streams_in_wave_order(17, *QKV_7B)
    assert streams_in_wave_order(5, *DOWN_7B) and not streams_in_wave_order(6, *DOWN_7B)   # 68 M elements, few rows
    assert streams_in_wave_order(8, 1536, 8960) and not streams_in_wave_order(9, 1536, 8960)   # small, with a long K
    assert streams_in_wave_order(6, 2048, 11008) and not streams_in_wave_order(7, 2048, 11008)     # the 3B down projection
    assert streams_in_wave_order(6, 5120, 5120) and not streams_in_wave_order(7, 5120, 5120)
    assert not streams_in_wave_order(1, 5120, 27648) and not streams_in_wave_order(8, 5120, 27648)   # the 32B down projection
    assert streams_in_wave_order(1, 152064, 5120) and not streams_in_wave_order(8, *HEAD_7B)      # many rows: up to 4
    # 60 M elements and 4,096 rows or more: K goes over workgroups from the first token on
    assert not streams_in_wave_order(1, 5120, 13824) and not streams_in_wave_order(1, 8192, 8192)
    # q/k/v, whose second kernel costs more
    assert streams_in_wave_order(3, 10240, 8192, rotates=True) and not streams_in_wave_order(4, 10240, 8192, rotates=True)
    assert streams_in_wave_order(10, 7168, 5120, rotates=True) and not streams_in_wave_order(11, 7168, 5120, rotates=True)


def test_the_lds_shared_product_splits_k_where_rows_are_few():
    assert mid_plan(8, *DOWN_7B) == (4, 1)                 # 56 row blocks x 4 ranges fill 256 CUs
    assert mid_plan(64, *DOWN_7B) == (9, 2)                # many tokens and a long K: two tiles per wave, 28 row blocks x 9
    assert mid_plan(32, 5120, 27648) == (6, 2) and mid_plan(31, 5120, 27648) == (3, 1)
    assert mid_plan(64, 1536, 8960) == (10, 1)             # few rows: one tile per wave, 24 row blocks x 10
    assert mid_plan(32, 2048, 11008) == (8, 1) and mid_plan(8, 5120, 13824) == (3, 1)     # the 3B and 14B down projections
    assert mid_plan(8, *HEAD_7B) == (1, 1) and mid_plan(64, *HEAD_7B) == (1, 2)
    assert mid_plan(64, *QKV_7B) == (3, 1) and mid_plan(64, *O_7B) == (4, 1)
    ranges, _ = mid_plan(64, 2048, 1536)                   # 1.5B q/k/v: no range shorter than 512
    assert 1536 // ranges >= 512


def test_past_64_tokens_the_weights_are_streamed_where_tiles_would_be_few():
    for n, k in (QKV_7B, O_7B, DOWN_7B, HEAD_7B):
        assert streams_weights(64, n, k) and not streams_weights(129, n, k)
    for m in (65, 96, 128):                                # small weights only: the 7B output projection, the 1.5B widths
        assert streams_weights(m, *O_7B) and streams_weights(m, 2048, 1536) and streams_weights(m, 1536, 8960)
        assert not streams_weights(m, *DOWN_7B) and not streams_weights(m, *QKV_7B) and not streams_weights(m, *HEAD_7B)
        assert not streams_weights(m, 5120, 27648)
    assert mid_plan(65, 1536, 8960) == (8, 1) and mid_plan(96, *O_7B) == (4, 1) and mid_plan(128, 2048, 1536) == (4, 1)
    assert mid_plan(100, 1024, 320) == (1, 1)              # no range shorter than 256
    assert mid_plan(65, 896, 4864) == (8, 1)               # the 0.5B down projection


def test_the_gated_product_goes_resident_tiled_or_lds_shared():
    assert gated_resident_fits(16, *GATE_UP_7B) and not gated_resident_fits(17, *GATE_UP_7B)
    assert not gated_resident_fits(16, 55296, 5120)        # 32B: 16 tokens x 5120 do not fit a CU's LDS
    assert gated_resident_fits(8, 55296, 5120)
    assert not gated_resident_fits(8, 37888, 3584 + 64)    # K in whole chunks of 128 only
    assert gated_resident_fits(8, 9728, 896) and gated_plan(8, 9728, 896) == 0     # the 0.5B width: chunks of 128
    for m in (1, 8, 16):
        assert gated_plan(m, *GATE_UP_7B) == 0             # 18,944 outputs over 256 CUs: 72 or 76 each
    assert gated_plan(8, 17920, 1536) == 0                 # 1.5B: 8,960 outputs are 32 or 36 each, and the norm before it is free
    assert gated_plan(8, 55296, 5120) == 0
    assert gated_plan(17, *GATE_UP_7B) == 3 and gated_plan(64, *GATE_UP_7B) == 3   # past the resident kernel: tiled
    assert gated_plan(32, 59136, 8192) == 2 and gated_plan(33, 59136, 8192) == 3   # 72B: LDS-shared up to 32 tokens
    assert gated_plan(8, 59136, 8192) == 0
    assert gated_plan(24, 55296, 5120) == 3
    assert gated_plan(48, 17920, 1536) in (1, 2) and gated_plan(64, 17920, 1536) == 3
    assert gated_plan(8, *GATE_UP_7B, cus=304) == 0        # over 304 CUs: 60 or 64 outputs each
    assert gated_plan(8, *GATE_UP_7B, cus=500) == 0        # over 500: 36 or 40 each, 6 % above the mean
    assert gated_plan(8, 4096, 1024, cus=256) != 0         # 128 pairs over 256 CUs: half of them would have none


def test_q_k_v_rotates_in_the_kernel_that_adds_its_ranges_where_k_is_split():
    assert split_qkv_plan(64, *QKV_7B) == (3, 1) and split_qkv_plan(17, *QKV_7B) == (3, 1)
    assert split_qkv_plan(16, *QKV_7B) is None and split_qkv_plan(65, *QKV_7B) is None
    assert split_qkv_plan(32, 1024, 512) is None           # K too short to split
    # the widest models split from few tokens on, in two ranges where the rows alone would fill the CUs
    assert split_qkv_plan(8, 10240, 8192) == (2, 1) and split_qkv_plan(3, 10240, 8192) is None
    assert split_qkv_plan(16, 7168, 5120) == (2, 1) and split_qkv_plan(8, 7168, 5120) is None


def test_room_for_the_sums_of_squares():
    assert follow_stride(16) == 16 and follow_stride(17) == 64 and follow_stride(64) == 64
    assert follow_stride(65) == 128 and follow_stride(2048) == 2048
    for n in (16, 64, 1000, 3584, 8192):
        assert follow_sumsq_floats(n, 16) >= ((n + 7) // 8) * 16          # a workgroup per 8 columns, 16 tokens
        assert follow_sumsq_floats(n, 64) >= ((n + 1023) // 1024) * 64    # a workgroup per 1,024 columns, 64 tokens


def test_prompt_tiles_in_chunks_for_models_of_few_heads():
    from vipera_rs_amd.ops.attention import chunks_prompt_tiles
    one_prompt = sum(128 * t for t in range(1, 17))                     # positions that the 16 tiles of 2,048 tokens see
    assert chunks_prompt_tiles(16, 12, 2048, one_prompt, 256) is None   # 12 heads, one short prompt: the halved tiles
    assert chunks_prompt_tiles(16, 28, 2048, one_prompt, 256) is None   # 448 items: more than the CUs
    # four portions of 512 tokens that end at positions 1,000 to 8,000: 192 items, the deepest 125 steps long
    assert chunks_prompt_tiles(16, 12, 8000, 4 * (1000 + 3000 + 5000 + 8000), 256) == (25, 5)
    assert chunks_prompt_tiles(16, 12, 4096, 16 * 3900, 256) is None    # all about equally deep: nothing to balance
    assert chunks_prompt_tiles(0, 12, 0, 0, 256) is None


def test_decode_attention_chunks():
    assert decode_chunking(4096, 8, 4, 1) == (256, 16)     # 8 requests x 4 key heads x 16 chunks = 512 waves
    assert decode_chunking(4096, 64, 4, 1) == (1024, 4)
    assert decode_chunking(4096, 1, 4, 1) == (128, 32)     # never below 128 positions a chunk
    assert decode_chunking(100, 1, 4, 1) == (128, 1)
    # many requests at long contexts: longer chunks while they still make 2,048 waves
    assert decode_chunking(32768, 64, 4, 1) == (4096, 8) and decode_chunking(16384, 64, 4, 1) == (2048, 8)
    assert decode_chunking(8192, 64, 4, 1) == (1024, 8) and decode_chunking(32768, 16, 4, 1) == (1024, 32)
    assert decode_chunking(32768, 64, 2, 1) == (2048, 16)
    chunk, chunks = decode_chunking(1 << 20, 1, 1, 1)      # never more than 128 chunks
    assert chunks <= 128 and chunk * chunks >= 1 << 20 and chunk % 32 == 0


def test_decode_attention_counts_the_entries_by_the_positions_they_hold():
    assert decode_chunking(4096, 8, 4, 1, 8 * 4096) == decode_chunking(4096, 8, 4, 1)      # all full: as without
    assert decode_chunking(16384, 64, 4, 1, 301000) == (1024, 16)      # 64 requests that fill 18 %: no long chunks
    assert decode_chunking(8192, 16, 4, 1, 70000) == (512, 16)         # as 9 full ones
    assert decode_chunking(8192, 8, 4, 1, 8 * 4100) == (256, 32)       # a little past a context bucket's half
    assert decode_chunking(4096, 8, 4, 1, 1) == decode_chunking(4096, 1, 4, 1)             # never fewer than one entry
    assert decode_chunking(4096, 8, 4, 1, 10 ** 9) == decode_chunking(4096, 8, 4, 1)       # nor more than there are


def test_decode_attention_chunks_cover_every_length_for_any_batch():
    import random
    rng = random.Random(5)
    for _ in range(3000):
        longest = rng.choice([1, 31, 32, 33, 100, 1000, 4096, 8191, 40000, rng.randrange(1, 1 << 21)])
        entries = rng.choice([1, 2, 7, 8, 63, 64, 200, 256])
        kv_heads, head_blocks = rng.choice([1, 2, 4, 8]), rng.choice([1, 2])
        total = rng.choice([0, 1, longest, rng.randrange(1, entries * longest + 1), entries * longest, 10 * entries * longest])
        chunk, chunks = decode_chunking(longest, entries, kv_heads, head_blocks, total)
        assert chunk % 32 == 0 and chunk >= 128 and 1 <= chunks <= 128, (longest, entries, total)
        assert chunk * chunks >= longest and chunk * (chunks - 1) < longest, (longest, entries, total)
        # fewer positions in all never make the chunks longer
        if total:
            assert chunk <= decode_chunking(longest, entries, kv_heads, head_blocks)[0]


def test_a_captured_step_is_chosen_by_the_share_of_its_context_bucket_that_is_filled():
    from vipera_rs_amd.engine.graphs import FILL_CLASSES, fill_class
    assert FILL_CLASSES == (1.0, 0.5, 0.25)
    assert fill_class(8 * 4096, 8, 4096) == 0 and fill_class(8 * 3000, 8, 4096) == 0
    assert fill_class(8 * 4100, 8, 8192) == 1              # equal lengths just past a bucket's edge
    assert fill_class(301000, 64, 16384) == 2 and fill_class(8, 8, 256) == 2


def test_one_workgroup_takes_all_chunks_of_a_request_and_key_head_where_those_fill_the_gpu():
    from vipera_rs_amd.ops.attention import joins_decode_chunks
    assert joins_decode_chunks(4, 64, 4, 1, 256) and joins_decode_chunks(4, 128, 4, 1, 256)
    assert not joins_decode_chunks(16, 8, 4, 1, 256)        # 32 pairs for 256 CUs
    assert not joins_decode_chunks(16, 64, 4, 1, 256)       # more chunks than a workgroup has waves
    # a few more pairs than CUs: the CUs with two workgroups would set the time
    assert not joins_decode_chunks(4, 72, 4, 1, 256) and not joins_decode_chunks(4, 40, 8, 1, 256)
    assert not joins_decode_chunks(4, 96, 4, 1, 256) and joins_decode_chunks(4, 112, 4, 1, 256)
    # heads wider than 128 keep a workgroup per chunk: one wave a SIMD, with room for their sums
    assert joins_decode_chunks(4, 64, 4, 1, 256, 128) and joins_decode_chunks(4, 64, 4, 1, 256, 112)
    assert not joins_decode_chunks(4, 64, 4, 1, 256, 160) and not joins_decode_chunks(4, 64, 4, 1, 256, 256)


def test_prompt_tiles_are_halved_between_sixteen_waves_only_where_a_cu_would_be_left_with_one_workgroup():
    from vipera_rs_amd.ops.attention import halves_prompt_tiles
    reach = [128 * (t + 1) for t in range(16)]                       # one prompt of 2,048 tokens
    assert halves_prompt_tiles(16, 28, max(reach), sum(reach), 256)  # 448 items, the longest 1.9 times the mean
    even = [1536 + 128 * (t + 1) for t in range(4)] * 4              # four portions of 512 tokens at position 1,536
    assert not halves_prompt_tiles(16, 28, max(even), sum(even), 256)
    assert halves_prompt_tiles(4, 28, 512, 1280, 256)                # fewer items than CUs
    long = [128 * (t + 1) for t in range(64)]                        # 8,192 tokens: several rounds of workgroups
    assert not halves_prompt_tiles(64, 28, max(long), sum(long), 256)
    assert not halves_prompt_tiles(0, 28, 0, 0, 256)


def test_the_cut_of_a_32_bit_product_is_asked_for_once_for_a_size(monkeypatch):
    from vipera_rs_amd.ops import kernels
    asked, real = [], kernels._fn
    monkeypatch.setattr(kernels, "_fn", lambda *args, **named: asked.append(args[1]) or real(*args, **named))
    first = kernels._gemm_generic_parts(77, 1155, 899)
    assert asked == ["vk_gemm_generic_workspace"] and first == kernels._gemm_generic_parts(77, 1155, 899) and len(asked) == 1


def test_an_aligned_32_bit_product_asks_for_the_memory_that_its_form_writes():
    from vipera_rs_amd.ops.kernels import _gemm_direct_parts, _gemm_generic_parts
    assert _gemm_generic_parts(333, 1152, 896) == 4 * 333 * 1152 and _gemm_direct_parts(333, 1152, 896) == 0       # one slab
    assert _gemm_generic_parts(64, 1536, 8960) == 35 * 64 * 1536 and _gemm_direct_parts(64, 1536, 8960) == 9 * 64 * 1536
    assert _gemm_generic_parts(65, 17930, 1540) == 2 * 65 * 17930 and _gemm_direct_parts(65, 17930, 1540) == 0     # walks all of K
    assert _gemm_generic_parts(2048, 9728, 8960) == 0 == _gemm_direct_parts(2048, 9728, 8960)


def test_a_gated_32_bit_product_is_one_launch_where_that_is_faster():
    """us of product and gate in two launches and in one."""
    from vipera_rs_amd.ops.kernels import _gemm_gated_takes as takes, gemm_generic_gated_pays as pays
    for slower in ((400, 4096, 1024), (494, 2148, 948),          # 75 and 83, 51 and 61: 4.5 and 2.9 tiles of 48 x 64 a CU
                   (441, 3396, 932), (550, 9720, 968),           # 67 and 75, 206 and 228: 2.9 and 10.7 of 64 x 64
                   (231, 6056, 956)):                            # 74 and 76: 4.9 of 48 x 48
        assert takes(*slower) and not pays(*slower)
    for faster in ((333, 4864, 896), (17, 4864, 896), (130, 4864, 896), (65, 8960, 1536), (512, 4096, 1024),     # 68 and 65, 16 and 14, 34 and 32, ...
                   (138, 10328, 948), (635, 5812, 992), (742, 1688, 988)):          # 3.8 of 48 x 64, 7.1 of 64 x 64, 6.6 of 48 x 32
        assert takes(*faster) and pays(*faster)
    assert not pays(65, 12, 1028) and not takes(65, 12, 1028)


def test_past_128_tokens_small_tiles_carry_out_a_128x128_plan_unless_its_tiles_fill_the_gpu():
    """The tiling and the ranges of K.  Tilings 9: 128x128, 13: 64x64 with K split, 14: 64x64 that walk K, 15: 128x64 that walk K."""
    from vipera_rs_amd.ops.kernels import gemm_bf16_tile_plan as plan
    assert plan(512, 2048, 2048) == (14, 1) and plan(512, 1057, 2048) == (14, 4) and plan(512, 64, 2048) == (13, 4)
    assert plan(512, 2576, 2048) == (15, 1) and plan(700, 5120, 2048) == (15, 1)           # more than a 64x64 tile a CU
    assert plan(2819, 768, 1280, gated=True) == (15, 1) and plan(300, 1024, 768, gated=True) == (14, 1)
    # as many ranges as fill the CUs with 128x128 tiles: these stay, or walk K where it has four
    assert plan(330, 7488, 7168) == (9, 2) and plan(353, 3168, 6400) == (9, 4) and plan(301, 4288, 6848) == (9, 4)
    assert plan(1879, 256, 8192) == (9, 8) and plan(953, 512, 6400) == (9, 8) and plan(468, 1792, 4352) == (14, 4)
    assert plan(161, 1792, 10496) == (13, 8)       # 256 tokens' worth of 128x128 tiles for 161
    # one 128x128 tile a CU at the most, however long K is
    assert all(plan(700, 5120, k, gated=True) == (15, 1) for k in (1024, 8192, 12288)) and plan(277, 10880, 4096, gated=True) == (15, 1)
    assert plan(277, 10976, 4096, gated=True) == (9, 1) and plan(270, 13312, 8192, gated=True) == (9, 1)
    assert plan(512, 2048, 2040)[0] == 0           # no whole steps of 64


def test_a_plan_of_one_range_takes_the_tile_of_the_least_rounds():
    """16: 192x64, 17: 128x128 of three stages, 18 and 19: 192x128 of three and two, 20: 192x192."""
    from vipera_rs_amd.ops.kernels import gemm_bf16_tile_carried_out as carried, gemm_bf16_tile_plan as plan
    assert carried(1396, 1536, 1536) == 16 and carried(783, 4096, 2048) == 17 and carried(1000, 4608, 3584) == 18
    assert carried(2048, 4608, 3584, output_bytes=2) == 19 and carried(311, 22016, 2048, gated=True) == 20
    assert carried(2048, 37888, 3584, gated=True) == 5 and carried(2048, 3584, 18944) == 7 and carried(1000, 2048, 1536) == 15
    for sizes in ((100, 4608, 3584), (512, 2048, 2048), (330, 7488, 7168), (1396, 1536, 8960), (700, 4096, 2040)):
        assert carried(*sizes) == plan(*sizes)[0]       # up to 128 tokens, 64x64 tiles, ranges, no whole steps of 64


def test_256x128_tiles_with_few_last_tokens_keep_their_deep_ranges():
    """7: 256x128, 18: 192x128; us of either."""
    from vipera_rs_amd.ops.kernels import gemm_bf16_tile_carried_out as carried
    assert carried(575, 2048, 11008) == 7 and carried(572, 2048, 8192) == 7            # 45.2 and 47.7, 35.7 and 39.0: 63 tokens in the last tile
    assert carried(1315, 2048, 11008) == 7 and carried(940, 3072, 8192) == 7           # 74.4 and 80.1, 62.3 and 64.5
    assert carried(649, 4096, 14336) == 18 and carried(1241, 1792, 7168) == 18         # 98.4 and 83.0, 56.3 and 46.2
    assert carried(575, 2560, 10240) == 18 and carried(575, 2048, 4096) == 18          # 47.0 and 45.4: 240 tiles; 27.0 and 25.6: ranges of 1,024
    assert carried(134, 3584, 18944) == 18 and carried(1032, 2560, 10240) == 18        # 46.9 and 44.5: a single tile of tokens; 69 and 62
    assert carried(945, 1536, 8960) == 18                                              # 42.2 and 39.8


def test_split_small_tiles_give_way_where_the_larger_ones_are_faster():
    """13: 64x64 with K split, 16: 192x64, 17: 128x128; us of the small tiles and of those picked, or of 17 where they stay."""
    from vipera_rs_amd.ops.kernels import gemm_bf16_tile_carried_out as carried
    assert carried(204, 1152, 6912) == 13 and carried(250, 1152, 6912) == 13      # 18.2 and 18.7, 19.6 and 19.8: 576 small tiles
    assert carried(204, 1280, 5120) == 17 and carried(204, 2560, 4096) == 17      # 16.9 and 16.8, 20.1 and 19.0: 640
    assert carried(319, 896, 4864) == 16 and carried(572, 512, 8192) == 16        # 15.0 and 14.9, 17.9 and 17.2: 560 and 576
    assert carried(200, 1024, 4096) == 13                                         # 512, two a CU
    # 14: 64x64 that walk K
    assert carried(771, 896, 4864) == 14 and carried(797, 1024, 8192) == 17       # 17.5 and 19.4, 32.3 and 27.5
    assert carried(568, 1536, 8960) == 17 and carried(133, 3584, 3584) == 16      # 42.2 and 30.2, 17.6 and 16.9


def _walked(reach, tokens, window, keep_first=0):
    """Steps that the kernel's walk makes of a tile of so many tokens whose last one sees ``reach`` positions (TileWalk)."""
    pos = reach - tokens
    first = (max(pos + 1 - window, 0) if window > 0 else pos - pos % -window if window < 0 else 0) // 64 * 64
    kept = min((keep_first + 63) // 64, first // 64)
    return kept + (reach - first + 63) // 64


def test_the_steps_of_a_prompt_tile_are_those_of_the_kernels_walk():
    from vipera_rs_amd.ops.attention import prompt_tile_steps
    for window, keep in ((0, 0), (1, 0), (64, 0), (100, 7), (512, 64), (512, 65), (512, 4000), (2048, 300), (-64, 0), (-100, 0), (-512, 0)):
        for reach in (*range(1, 420), *range(1000, 1200), *range(30000, 30200)):
            steps = prompt_tile_steps(reach, window, keep)
            assert steps == _walked(reach, min(reach, 128), window, keep)
            assert steps >= max(_walked(reach, n, window, keep) for n in range(1, min(reach, 128) + 1))


def test_cut_prompt_tiles_ask_for_no_more_than_their_walks():
    """Workgroups and memory are those of the longest walk through the window, and 512 MB of partial results at the most."""
    import random
    from vipera_rs_amd.ops.attention import cut_prompt_tiles
    portion = lambda first, n: [first + min(off + 128, n) for off in range(0, n, 128)]
    for window, heads in ((2048, 16), (-2048, 16), (4096, 16), (2048, 8), (1024, 4)):
        for first in (3000, 30000, 120000):
            for dim in (64, 128, 256):
                plan = cut_prompt_tiles(portion(first, 512), heads, dim, window, 256)
                assert plan is None or 4 * heads * plan[1] <= 2 * 256, (window, heads, first, dim, plan)
    rng = random.Random(7)
    for _ in range(600):
        tiles = sorted(rng.randrange(128, rng.choice([400, 4000, 130000])) for _ in range(rng.randrange(1, 120)))
        heads, window, dim = rng.choice([1, 2, 14]), rng.choice([0, 0, 700, 5000, -3000]), rng.choice([64, 128, 256])
        keep = rng.choice([0, 4, 1000]) if window > 0 else 0
        plan = cut_prompt_tiles(tiles, heads, dim, window, 256, keep)
        if plan is not None:
            longest = max(_walked(t, 128, window, keep) for t in tiles)
            assert plan[1] == -(-longest // plan[0]) and len(tiles) * heads * plan[1] * 128 * (dim + 4) * 4 <= 512 << 20


def test_the_chunk_of_cut_prompt_tiles_is_the_best_of_all():
    import random
    from vipera_rs_amd.ops.attention import PROMPT_COSTS, PROMPT_PARTIAL_BYTES, cut_prompt_tiles, prompt_tile_steps
    rng = random.Random(11)
    plans = 0
    for _ in range(500):
        tiles = sorted(rng.randrange(1, rng.choice([600, 3000, 30000])) for _ in range(rng.randrange(1, rng.choice([6, 60]))))
        heads, window, dim, cus = rng.choice([1, 3, 12]), rng.choice([0, 0, 2500, -4000]), rng.choice([64, 128, 256]), rng.choice([256, 304])
        steps, items = [prompt_tile_steps(t, window) for t in tiles], len(tiles) * heads
        (alone, beside), one, two = PROMPT_COSTS[dim]
        best, want = 0.9 * (alone * max(steps) + beside), None
        for chunk in range(4, max(steps) if items <= cus else 0):
            groups = heads * sum(-(-s // chunk) for s in steps)
            cost = one if groups <= cus else two if groups <= 1.7 * cus else None
            most = -(-max(steps) // chunk)
            if cost is None or items * most * 128 * (dim + 4) * 4 > PROMPT_PARTIAL_BYTES:
                continue
            us = cost[0] * chunk + cost[1] + cost[2] * groups
            if us < best:
                best, want = us, (chunk, most)
        assert cut_prompt_tiles(tiles, heads, dim, window, cus) == want
        plans += want is not None
    assert plans > 100


def test_a_cut_of_prompt_tiles_is_found_in_a_few_looks_however_deep(monkeypatch):
    from vipera_rs_amd.ops import attention
    looks = []
    counted = attention._cut_workgroups
    monkeypatch.setattr(attention, "_cut_workgroups", lambda *a: looks.append(1) or counted(*a))
    for reach in (500, 2048, 8192, 32768, 131072):
        for tiles, heads, dim in ((16, 14, 64), (4, 12, 128), (16, 1, 128), (19, 4, 256), (1, 28, 128)):
            looks.clear()
            attention.cut_prompt_tiles([max(128, reach - 128 * i) for i in range(tiles)], heads, dim, 0, 256)
            assert len(looks) <= 40, (reach, tiles, heads, dim, len(looks))


def test_prompt_tiles_of_known_lengths_are_cut_where_it_pays():
    """Chunks as long as one another are few enough to run at once, never leave a position out and never outnumber what was
    allowed for."""
    import random
    from vipera_rs_amd.ops.attention import cut_prompt_tiles
    reaches = lambda *portions: [first + min(off + 128, n) for first, n in portions for off in range(0, n, 128)]
    assert cut_prompt_tiles(reaches((1194, 512), (2389, 456), (3584, 399)), 12, 128, 0, 256) == (16, 4)
    assert cut_prompt_tiles(reaches((1900, 100)), 14, 64, 0, 256) == (4, 8)
    assert cut_prompt_tiles(reaches((0, 1000), (0, 834)), 16, 128, 0, 256) is None
    assert cut_prompt_tiles(reaches((0, 2048)), 28, 128, 0, 256) is None                   # more items than CUs
    assert cut_prompt_tiles(reaches((3000, 200)), 12, 96, 0, 256) is None and cut_prompt_tiles([], 12, 128, 0, 256) is None
    assert cut_prompt_tiles(reaches((8000, 200)), 12, 128, 100, 256) is None               # a window of 100: short walks
    rng = random.Random(3)
    for _ in range(300):
        tiles = sorted(rng.randrange(1, rng.choice([200, 2000, 30000])) for _ in range(rng.randrange(1, 20)))
        heads, window = rng.choice([1, 8, 14, 28]), rng.choice([0, 0, 512, -512])
        plan = cut_prompt_tiles(tiles, heads, rng.choice([64, 128, 256]), window, 256)
        if plan is not None:
            chunk, most = plan
            assert chunk >= 4 and chunk * most >= max(_walked(t, n, window) for t in tiles for n in (1, 64, 127, 128) if n <= t)
            if not window:
                assert heads * sum(-(-t // (64 * chunk)) for t in tiles) <= 2 * 256


def test_few_requests_of_short_contexts_take_short_chunks():
    from vipera_rs_amd.ops.attention import short_decode_plan
    assert short_decode_plan(512, 1, 2, 1, 64) == (64, 8, True) and short_decode_plan(513, 1, 2, 1, 64) == (32, 17, False)
    assert short_decode_plan(256, 8, 4, 1, 128) == (32, 8, True) and short_decode_plan(512, 8, 4, 1, 128) == (32, 16, False)
    assert short_decode_plan(1024, 8, 4, 1, 128) == (64, 16, False) and short_decode_plan(2048, 8, 4, 1, 128) is None
    assert short_decode_plan(4096, 1, 4, 1, 128) == (64, 64, False) and short_decode_plan(4097, 1, 4, 1, 128) is None
    assert short_decode_plan(512, 80, 2, 1, 64) is None and short_decode_plan(300, 1, 2, 1, 256) is None
    for length in range(1, 4500, 7):
        for entries, kv, dim in ((1, 2, 64), (3, 4, 128), (40, 2, 64)):
            plan = short_decode_plan(length, entries, kv, 1, dim)
            if plan is not None:
                chunk, chunks, join = plan
                assert chunk % 32 == 0 and chunk * chunks >= length and (chunks <= 8 if join else chunks <= 64)


def test_attention_keeps_the_order_of_its_sums_in_every_model_that_may_route():
    from types import SimpleNamespace
    import gilidra_helpers
    import helpers
    import lurirax_helpers
    import muzasun_helpers
    import rebidra_helpers
    import zeladra_helpers
    import zulesun_helpers
    from vipera_rs_amd.config import config_from_dict
    from vipera_rs_amd.models.decoder import routes_tokens
    from vipera_rs_amd.parts import FeedForward, register_ffn, unregister
    seen = set()
    for data in (helpers.CONFIG_B, gilidra_helpers.G1, gilidra_helpers.G2, lurirax_helpers.L1, lurirax_helpers.L2, muzasun_helpers.M1,
                 muzasun_helpers.M2, rebidra_helpers.R1, rebidra_helpers.R2, zeladra_helpers.Z1, zulesun_helpers.Z1):
        config = config_from_dict(data)
        routed = any(spec.ffn is not None and "experts" in spec.ffn.params for spec in config.layer_specs())
        assert routes_tokens(config) == routed, config.architecture
        seen.add(routed)
    assert seen == {True, False}

    class Unsaid(FeedForward):
        pass

    register_ffn("unsaid", Unsaid)
    try:
        layers = [SimpleNamespace(ffn=SimpleNamespace(kind=kind)) for kind in ("gated_mlp", "mlp", "none")] + [SimpleNamespace(ffn=None)]
        assert not routes_tokens(SimpleNamespace(layer_specs=lambda: layers))
        assert routes_tokens(SimpleNamespace(layer_specs=lambda: layers + [SimpleNamespace(ffn=SimpleNamespace(kind="unsaid"))]))
    finally:
        unregister("ffn", "unsaid")
