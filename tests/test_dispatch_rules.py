"""Launch decisions that are made on the host, as far as they are plain arithmetic (no GPU)."""
import inspect

from ferrox_amd import ops


def splits(n_items, n_heads, n_kv_heads, max_kv_len, cus=256):
    chunk = ops.decode_attention_chunk(n_items, n_heads, n_kv_heads, max_kv_len, cus)
    assert chunk % 64 == 0 and chunk >= 64
    return -(-max_kv_len // chunk)


def test_decode_attention_chunks_fill_the_gpu_and_avoid_partial_rounds():
    # few (sequence, kv head) pairs: chunks enough for about eight waves a CU
    assert splits(1, 16, 16, 2560) >= 12
    assert splits(8, 16, 16, 2560) == 2
    assert splits(8, 28, 4, 2560) == 8
    # as many pairs as CUs, or a whole number of rounds of them: one chunk, no merge launch
    for n in (16, 32, 64):
        assert splits(n, 16, 16, 2560) == 1
    assert splits(128, 28, 4, 2560) == 1
    # a last round far from full (steps recorded for 24, 40, 48 and 56 sequences of 16 kv heads): eight chunks
    for n in (24, 40, 48, 56):
        assert splits(n, 16, 16, 2560) == 8
    assert splits(80, 28, 4, 2560) == 8
    # short sequences have too few tiles to cut, and from four pairs a CU on one chunk is level with the rest
    assert splits(24, 16, 16, 512) == 1
    for n in (72, 96, 128, 256):
        assert splits(n, 16, 16, 2560) == 1
    # another GPU: the same decisions by its own number of CUs
    assert splits(8, 16, 16, 2560, cus=128) == 1 and splits(12, 16, 16, 2560, cus=128) == 8


def test_chunks_of_the_widest_heads_are_one_round_of_the_simds():
    chunk = lambda n, kv, hd=256, cus=256: ops.decode_attention_chunk(n, 16, 1, kv, cus, hd)
    assert chunk(1, 40) == chunk(8, 2060) == chunk(16, 2060) == chunk(32, 1030) == chunk(32, 2048) == 64
    assert chunk(32, 2060) == chunk(64, 2048) == 128 and chunk(64, 2060) == 192 and chunk(8, 2060, cus=64) == 128
    for n in (1, 8, 100, 1024, 5000):
        for kv in (1, 64, 65, 2060, 30000):
            c = chunk(n, kv)
            assert c % 64 == 0 and c >= 64 and (c == 64 or n * -(-kv // c) <= 1024 or c >= kv)


def test_chunks_of_the_widest_heads_without_items_or_keys():
    for hd in (64, 128, 192, 256):
        assert ops.decode_attention_chunk(0, 16, 1, 2060, 256, hd) >= 64 and ops.decode_attention_chunk(0, 16, 1, 0, 256, hd) == 64
        assert ops.decode_attention_chunk(8, 16, 1, 0, 256, hd) == 64 and ops.decode_attention_chunk(8, 16, 16, 0, 256, hd) == 64


def test_chunks_of_wide_heads_on_the_kernel_for_any_shape():
    """A wave per head there: eight or nine waves a CU, however few kv heads there are."""
    rule = lambda n, nh, nkv, kv, span=0: ops.decode_attention_chunk(n, nh, nkv, kv, 256, 512, span, True)
    assert rule(32, 16, 1, 2060) == rule(32, 16, 16, 2060) == 576 and rule(8, 16, 1, 8200) == 512 and rule(8, 16, 16, 2060) == 128
    assert rule(1, 16, 1, 2060) == 64 and rule(5000, 16, 1, 100) == 128 and rule(0, 16, 1, 0) == rule(0, 16, 1, 500) == rule(8, 16, 1, 0) == 64
    assert rule(1, 16, 1, 30000, 1024) == 64 and rule(8, 16, 1, 30000, 1024) == 256 and rule(8, 16, 1, 500, 1024) == rule(8, 16, 1, 500)
    for n in (1, 8, 100):
        for kv in (500, 8200, 30000):
            for span in (0, 64, 1024):
                c = rule(n, 16, 4, kv, span)
                assert c % 64 == 0 and -(-kv // c) <= max(1, 2304 // (16 * n), 1024 // (4 * n))


def test_chunks_of_the_widest_heads_by_the_keys_that_a_query_sees():
    """No more chunks than a span of keys touches tiles, wherever it begins, and chunks that cover the sequence; the same without a span that is shorter."""
    rule = ops.decode_attention_chunk
    for n in (1, 8, 16, 100, 1024):
        for kv in (1, 64, 500, 2060, 30000):
            for span in (1, 2, 64, 65, 66, 128, 1024, 5000, 50000):
                c, whole = rule(n, 16, 1, kv, 256, 256, span), rule(n, 16, 1, kv, 256, 256)
                chunks = -(-kv // c)
                touched = max(-(-(first % 64 + span) // 64) for first in range(64))
                assert c % 64 == 0 and c >= whole and chunks <= max(1, min(touched, -(-kv // whole))) and chunks * c >= kv
                assert span < kv or c == whole
    assert -(-30000 // rule(8, 16, 1, 30000, 256, 256, 1024)) == 17 and rule(8, 16, 1, 30000, 256, 256) == 256


def test_chunks_of_wide_heads_with_few_query_heads_a_kv_head():
    """3 to 7 query heads a kv head take the chunks of narrower heads where those hold three tiles or more and fill the CUs, and so does one chunk a sequence."""
    wide = lambda n, nh, nkv, kv, span=0: ops.decode_attention_chunk(n, nh, nkv, kv, 256, 256, span)
    narrow = lambda n, nh, nkv, kv: ops.decode_attention_chunk(n, nh, nkv, kv, 256)
    for n, nh, nkv, kv in ((1, 16, 4, 8200), (5, 16, 4, 2060), (10, 16, 4, 8200), (12, 28, 4, 8200), (64, 16, 4, 500), (32, 16, 8, 2060), (14, 16, 16, 2060)):
        assert wide(n, nh, nkv, kv) == narrow(n, nh, nkv, kv) >= 192
    assert wide(1, 16, 4, 2060) == wide(4, 16, 4, 1030) == wide(14, 16, 4, 1030) == 64      # two tiles or fewer; blocks for 7/8 of the CUs
    assert wide(36, 16, 4, 8200) == 1216 and wide(9, 16, 16, 2060) == 320 and wide(33, 16, 8, 500) == 192 and wide(1, 16, 16, 8200) == 192
    assert wide(1, 16, 4, 30000, 1024) == 1792 and wide(8, 16, 4, 30000, 1024) == narrow(8, 16, 4, 30000)


def test_half_sets_of_weight_rows_where_the_busiest_cu_fetches_less():
    from ferrox_amd.csrc.build import load_library
    rule = lambda m, n, dual=0, sets=None, cus=256: bool(load_library("gemm").fx_gemm_half_sets(
        m, n, dual, sets or (2 if dual or -(-n // 32) >= 160 else 1), cus))
    for m in (1, 8, 16):
        assert rule(m, 2048) and rule(m, 256) and rule(m, 1408, 1) and rule(m, 5632, 1) and not rule(m, 2560) and not rule(m, 4096)
        assert not rule(m, 2064) and not rule(m, 2048, cus=128)
    assert rule(1, 6144) and not rule(8, 6144) and not rule(16, 6144) and not rule(17, 2048)


def test_half_sets_beyond_one_round_of_the_cus_only_where_they_were_ahead():
    from ferrox_amd.csrc.build import load_library
    rule = lambda m, n, dual=0, cus=256: bool(load_library("gemm").fx_gemm_half_sets(m, n, dual, 2 if dual or -(-n // 32) >= 160 else 1, cus))
    for m in (1, 2):
        assert rule(m, 6144) and rule(m, 9216) and not any(rule(m, n) for n in (12288, 18432, 20480, 50257, 151936))
    for m in (3, 5, 16):
        assert not any(rule(m, n) for n in (4608, 5632, 9216, 12288, 50257)) and rule(m, 2048)
    for m in (1, 4, 16):
        assert rule(m, 4608, 1) and rule(m, 6144, 1) and not any(rule(m, n, 1) for n in (9216, 18432, 50257))
    assert rule(1, 5120, cus=128) and not rule(1, 6144, cus=128) and not rule(1, 6144, 1, cus=128)


def test_weights_of_the_rotating_product_leave_first_with_sums_of_one_batch_and_k_or_rows_enough():
    from ferrox_amd.csrc.build import load_library
    rule = lambda m, k, sums=None: bool(load_library("gemm").fx_qkv_rope_weights_first(m, k, -(-k // 256) if sums is None else sums))
    assert rule(1, 2048) and rule(16, 2048) and rule(1, 1032) and rule(16, 1024) and not rule(17, 2048) and not rule(15, 1024) and not rule(16, 768)
    assert not rule(16, 2048, 0) and not rule(16, 2056) and not rule(16, 3584) and rule(16, 3584, 8)


def test_row_tiles_of_the_rotating_product():
    """The fewest row tiles a block that keep its blocks within one round of the CUs, or else one block for all rows."""
    from ferrox_amd.csrc.build import load_library
    rule = lambda m, groups, cus=256: load_library("gemm").fx_qkv_rope_row_tiles(m, groups, cus)
    assert [rule(m, 192) for m in (1, 16, 17, 32, 33, 48, 49, 64)] == [1, 1, 2, 2, 3, 3, 4, 4]
    assert [rule(m, 128) for m in (16, 17, 32, 33, 48, 49, 64)] == [1, 1, 1, 2, 2, 2, 2]
    assert [rule(m, 64) for m in (17, 33, 49, 64)] == [1, 1, 1, 1] and [rule(m, 85) for m in (33, 48, 49, 64)] == [1, 1, 2, 2]
    assert rule(64, 192, 1024) == 1 and rule(64, 300) == 4 and rule(16, 300) == 1


def test_a_block_per_row_tile_while_such_blocks_are_one_a_cu():
    """The product of 33 to 128 plain rows: beyond 64 rows a second round of blocks is behind two row tiles a block."""
    from ferrox_amd.csrc.build import load_library
    rule = lambda m, n, cus=256: bool(load_library("gemm").fx_gemm_row_tile_blocks(m, n, cus))
    assert not rule(32, 64) and rule(33, 64) and rule(128, 64) and not rule(129, 64)
    assert rule(61, 1280) and not rule(61, 1296) and rule(40, 1696)
    assert rule(96, 672) and not rule(96, 688) and not rule(96, 768) and rule(128, 512) and not rule(128, 528)
    assert rule(128, 1024, cus=512) and not rule(128, 512, cus=128)


def test_tiles_of_plain_products():
    """One round of 128 x 128 tiles in two stages goes two to a CU; more rounds go to the tiles that share the work most
    evenly, and to two stages only in place of 128 x 128 in four."""
    from ferrox_amd.csrc.build import load_library
    tile = lambda m, n, k=2048, dual=0, cus=256: load_library("gemm").fx_gemm_plain_tile(m, n, k, dual, cus)
    assert tile(512, 2048) == 464 and tile(513, 2048) == 4128 and tile(1024, 2048) == 4128
    assert tile(512, 2048, dual=1) == 4128                               # no 64 x 64 of two matrices
    assert tile(768, 6144) == tile(1280, 6144) == tile(2432, 2048) == tile(4096, 2048) == 8128
    assert tile(16384, 512) == tile(14336, 512, 8192) == 8128 and tile(16384, 512, 4096) == 128
    # four rounds' worth of 128 x 128, nearly full
    assert tile(2560, 6144) == tile(7680, 2048) == tile(8192, 2048) == 256
    assert tile(3456, 4608, 3584) == tile(4480, 3584, 3584) == tile(2048, 4096, dual=1) == 256
    assert tile(2688, 6144) == tile(1337, 5632, dual=1) == 8128
    assert tile(2048, 5632, dual=1) == 12 and tile(4096, 6144) == 192
    assert tile(4096, 2048, cus=128) == tile(8192, 2048)


def test_tiles_twice_as_wide():
    """128 x 256 in place of 128 x 128 while they are one round of the CUs, or nearly whole rounds."""
    from ferrox_amd.csrc.build import load_library
    rule = lambda m, n, dual=0, cus=256: bool(load_library("gemm").fx_gemm_twice_as_wide(m, n, dual, cus))
    assert rule(1000, 6144) and rule(3001, 2048) and rule(512, 5632, 1) and rule(1337, 5632, 1)
    assert not rule(1000, 5632, 1) and rule(4096, 2048) and not rule(4097, 2048) and not rule(4096, 2048, cus=192)


def test_tiles_of_96_rows():
    """In place of 128 rows while tiles of 96 are one round of the CUs too."""
    from ferrox_amd.csrc.build import load_library
    rule = lambda m, n, tile, dual=0, cus=256: bool(load_library("gemm").fx_gemm_lower_tiles(m, n, tile, dual, cus))
    assert rule(1337, 2048, 64) and rule(1536, 2048, 64) and not rule(1537, 2048, 64) and rule(1337, 4096, 8256)
    assert not rule(1000, 6144, 8256) and rule(512, 2816, 8256, 1) and not rule(512, 5632, 8256, 1)
    assert not rule(1337, 2048, 8128) and not rule(1337, 2048, 256) and not rule(1337, 2048, 64, cus=200)


def test_long_sums_of_one_round_of_tiles_take_the_ring():
    """128 x 128 tiles that are one round of the CUs: quarters, but the ring of four stages for a long K."""
    from ferrox_amd.csrc.build import load_library
    tile = lambda m, n, k: load_library("gemm").fx_gemm_plain_tile(m, n, k, 0, 256)
    rule = lambda m, n, k: bool(load_library("gemm").fx_gemm_ring_of_four(tile(m, n, k), k))
    assert rule(1000, 3584, 20480) and rule(800, 3584, 16384) and rule(1500, 2048, 20480)
    assert not rule(1000, 3584, 14336) and not rule(300, 3584, 20480) and not rule(1500, 3584, 20480)


def test_items_on_waves_of_32_queries():
    from ferrox_amd.csrc.build import load_library
    rule = lambda blocks, cus=256: load_library("attention").fx_attn_rows32(blocks, cus)
    assert rule(1) == rule(191) == 0 and rule(192) == rule(768) == 2 and rule(769) == rule(5000) == 1
    assert rule(95, 128) == 0 and rule(192, 128) == 2 and rule(385, 128) == 1


def test_items_on_waves_of_32_queries_under_a_mask():
    """Short spans stay on waves of 16; even work takes one group from a block a CU on."""
    from ferrox_amd.csrc.build import load_library
    rule = lambda blocks, span, tokens, cus=256, chunked=0: load_library("attention").fx_attn_rows32_masked(blocks, cus, span, chunked, tokens)
    for blocks, tokens in ((1, 128), (191, 1536), (192, 1536), (256, 2048), (336, 1536), (512, 4096), (896, 4096), (5000, 20000)):
        assert rule(blocks, 1, tokens) == rule(blocks, 768, tokens) == rule(blocks, 1024, tokens, chunked=1) == 0
    assert rule(191, 4096, 1536) == 0 and rule(192, 1024, 1536) == rule(256, 1024, 2048) == 0 and rule(256, 1025, 2048) == rule(256, 40000, 2048) == 2
    assert rule(257, 769, 2112) == rule(511, 40000, 4096) == rule(512, 1024, 4096) == rule(512, 3072, 4096) == rule(640, 40000, 5120) == rule(769, 40000, 6000) == 1
    assert rule(512, 3073, 4096) == rule(639, 40000, 5120) == 2 and rule(400, 2049, 4096, cus=128) == 1 and rule(256, 3073, 4096, cus=128) == 2
    assert rule(256, 2048, 2048, chunked=1) == 0 and rule(256, 2049, 2048, chunked=1) == rule(336, 1536, 1536, chunked=1) == rule(512, 4096, 4096, chunked=1) == 2
    assert rule(512, 1536, 4096, chunked=1) == rule(640, 8192, 4096, chunked=1) == rule(900, 8192, 4096, chunked=1) == 1


def test_every_item_and_head_of_a_prompt_has_its_block():
    """Numbers of heads that eight XCDs share evenly and not, of items on both sides of eight: every pair once, last items first, an XCD's share of
    the work of a causal prompt within a row of its heads' mean."""
    from ferrox_amd.csrc.build import load_library
    place = load_library("attention").fx_attn_block_place
    for nh in (1, 3, 8, 16, 28, 71):
        for n in (1, 7, 8, 9, 33):
            for paired in (0, 1):
                pairs, b, work = [], 0, [0] * 8
                while (p := place(b, nh, n, paired)) != -2:
                    if p >= 0:
                        pairs.append(p)
                        work[b % 8] += p // nh + 1
                    b += 1
                assert sorted(pairs) == list(range(nh * n)) and b - nh * n < 64 * -(-nh // 8)
                assert max(work) <= sum(work) / 8 + n + 8
            for xcd in range(8):
                own = [place(c, nh, n, 0) // nh for c in range(xcd, b, 8) if place(c, nh, n, 0) >= 0]
                assert own == sorted(own, reverse=True)


def test_tiles_of_sorted_rows():
    """Average shares up to 20 rows go to tiles of 64, up to 104 to tiles whose loop an expert's own share decides (even shares lose
    with tiles in quarters there, crowded ones with a ring), more to tiles of 192 or 256."""
    from ferrox_amd.csrc.build import load_library
    tile = lambda share, n=2816, experts=60, dual=1, cus=256: load_library("gemm").fx_gemm_grouped_tile(share, share * experts, n, experts, dual, cus)
    assert tile(4) == tile(20) == 4 and tile(21) == tile(37) == tile(104) == tile(37, 2048, dual=0) == 1256
    assert tile(105) == tile(113) == tile(128) == tile(176) == 12 and tile(193) == 256


def test_the_chunk_rule_leaves_the_callers_arguments_alone():
    """The rule counts waves per block; it once did so in a variable named like the `waves` argument of
    `attention_decode`, which then reached the launch instead of the caller's value."""
    src = inspect.getsource(ops.attention_decode)
    body = src[src.index('"""', src.index('"""') + 3):]
    assert "waves =" not in body and "waves=" not in body.replace("int(waves)", "")
    assert "int(waves)" in body


def test_float32_products_from_parts_by_the_weights_alone():
    """Whole steps of 32 k, sums of 1,024 and more, weights of more than a million numbers; the router's product, whose rows stand where weights do, is left out of the
    rule: no number of tokens changes how its float32 operands are multiplied."""
    from types import SimpleNamespace
    import torch
    from ferrox_amd import ops
    from ferrox_amd.csrc.build import load_library
    from ferrox_amd.parts.moe import SparseMoE
    rule = load_library("gemm").fx_gemm_f32_split
    assert rule(2048, 2048) and rule(6144, 2048) and rule(1408, 2048) and rule(151936, 2048) and rule(1025, 1024) and not rule(1024, 1024)
    assert not rule(2048, 2056) and not rule(4096, 992) and not rule(60, 2048) and not rule(256, 2048)
    asked = []

    def gemm(a, w, *, f32_instruction=False, **kw):
        asked.append((tuple(a.shape), tuple(w.shape), f32_instruction))
        return torch.zeros(a.shape[0], w.shape[0])

    moe, plain_gemm = SparseMoE(2048, 60, 4, 1408, True), ops.gemm
    moe.router = torch.zeros(60, 2048)
    try:
        ops.gemm = gemm
        for T in (1, 64, 65, 511, 512, 700, 4096):
            assert moe._logits(torch.zeros(T, 2048)).shape == (T, 60)
            rows, weights, instruction = asked.pop()
            assert instruction or not rule(weights[0], weights[1]), T
    finally:
        ops.gemm = plain_gemm


def test_values_go_out_in_windows_of_64_tokens_from_a_number_of_them_on():
    """Two million bfloat16 values or half a million float32 ones, where 16-byte pieces of rows and of pages fit; a block of 64 tokens takes 4 G pieces of G elements."""
    import ctypes
    from ferrox_amd.csrc.build import load_library
    rule = load_library("elementwise").fx_many_value_blocks
    rule.restype = ctypes.c_long
    rule.argtypes = [ctypes.c_long] + [ctypes.c_int] * 4 + [ctypes.c_void_p, ctypes.c_long, ctypes.c_void_p]
    f32, bf16 = 0, 1
    assert rule(1024, 16, 128, 64, bf16, 4096, 6144, 4096) == 16 * 8 and rule(1023, 16, 128, 64, bf16, 4096, 6144, 4096) == 0
    assert rule(256, 16, 128, 64, f32, 4096, 6144, 4096) == 4 * 32 and rule(255, 16, 128, 64, f32, 4096, 6144, 4096) == 0
    assert rule(2048, 11, 136, 16, bf16, 4096, 6144, 4096) == 32 * 6                    # (187 pieces of 8, 32 a block)
    for bs, vd, ldv, v, pages in ((20, 128, 6144, 4096, 4096), (64, 132, 6144, 4096, 4096), (64, 128, 6148, 4096, 4096), (64, 128, 6144, 4104, 4096), (64, 128, 6144, 4096, 4104)):
        assert rule(4096, 16, vd, bs, bf16, v, ldv, pages) == 0
    assert rule(4096, 16, 132, 20, f32, 4096, 6148, 4096) > 0


def test_tiles_of_float32_products_from_parts():
    """Up to 32 rows tiles of 32; up to 64 rows one row tile, or two of 32 where those are one block a CU, while one row tile's blocks are; beyond that by what the CU with the most
    blocks takes."""
    from ferrox_amd.csrc.build import load_library
    rule = lambda m, n, dual=0, cus=256: load_library("gemm").fx_gemm_f32_split_tile(m, n, dual, cus)
    assert [rule(m, 6144) for m in (1, 32)] == [32, 32]
    assert [rule(m, n) for m in (33, 64) for n in (2048, 8192, 8256, 16384)] == [32, 32, 64, 64] * 2
    assert [rule(m, n, 1) for m in (33, 64) for n in (4096, 4128, 8192)] == [32, 64, 64] * 2
    assert [rule(m, n) for m in (33, 64) for n in (16448, 40960)] == [48, 48, 64, 64]
    assert rule(65, 2048) == 32 and rule(700, 6144) == 144 and rule(700, 2048) == 48 and rule(700, 1024) == 48


def test_which_products_of_few_rows_share_a_launch():
    """A gate/up product or one that is stored in float32, in half sets of weight rows by four waves, beside one that is stored; a switch that gives the first another kernel
    leaves both to launches of their own."""
    from ferrox_amd import debug
    from ferrox_amd.csrc.build import load_library
    lib = load_library("gemm")
    stored, stored_f32, added, gated = 0, 1, 2, 3
    pairs = lambda m, epi, n, k, epi2=stored_f32, n2=1024, k2=2048: bool(lib.fx_gemm_pairs(m, epi, n, k, epi2, n2, k2, 256))
    assert all(pairs(m, gated, 5632, 2048) and pairs(m, stored_f32, 2048, 5632, stored, 4096, 768) for m in (1, 5, 16))
    assert not any(pairs(m, gated, 5632, 2048) for m in (0, 17, 64))
    assert not pairs(8, added, 2048, 5632) and not pairs(8, stored, 2048, 5632) and not pairs(8, gated, 5632, 2048, added) and not pairs(8, gated, 5632, 2048, gated)
    assert not pairs(8, gated, 5632, 2052) and not pairs(8, gated, 5632, 2048, stored, 1024, 2044) and not pairs(8, gated, 5632, 2048, stored, 65536)
    assert pairs(4, gated, 5632, 4096) and not pairs(5, gated, 5632, 4096)                # (four pieces on their way)
    for m, n, dual, sets in ((8, 5632, 1, 2), (8, 2048, 0, 1), (8, 24576, 0, 2), (16, 40960, 1, 2)):       # as the rule for half sets has it
        assert pairs(m, gated if dual else stored_f32, n, 2048) == bool(lib.fx_gemm_half_sets(m, n, dual, sets, 256))
    for key, value in (("skinny_half", 0), ("skinny_waves", 8)):
        with debug.kernel_switch("gemm", key, value):
            assert not pairs(8, gated, 5632, 2048) and not pairs(8, stored_f32, 2048, 5632, stored, 4096, 768)


def test_waves_that_walk_many_tiles_of_keys():
    """16 tiles of 64 keys and more a wave, by the longest sequence that a launch can have; of heads of up to 64 five."""
    import ctypes
    from ferrox_amd.csrc.build import load_library
    rule = load_library("attention").fx_attn_wave_walks
    rule.argtypes = [ctypes.c_long, ctypes.c_int, ctypes.c_int]
    assert [rule(keys, waves, 128) for keys, waves in ((960, 1), (961, 1), (2560, 1), (2560, 2), (2560, 4), (4032, 4), (4033, 4))] == [0, 1, 1, 1, 0, 0, 1]
    assert [rule(keys, waves, 64) for keys, waves in ((256, 1), (257, 1), (512, 2), (577, 2), (2560, 8), (2561, 8))] == [0, 1, 0, 1, 1, 1]
