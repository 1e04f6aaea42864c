"""The host-side rules that choose kernels and how they cut their work (no GPU needed)."""
import ctypes

import pytest

from qil_amd import ops


@pytest.fixture(scope='module')
def lib():
    """The kernel library's planners are host code: they run without a GPU once the library is built."""
    try:
        return ops.library.load()
    except ops.library.KernelLibraryError as error:
        pytest.skip(f'kernel library not available here: {error}')


def test_row_kernel_parts_scale_with_the_work():
    """One row of 2,048 keys is cut into parts of 64 keys, eight rows into parts of 128, sixty-four into parts of
    512; never below 64 or above 512, and a power of two."""
    kv_heads = 8
    assert ops._rows_part(1, kv_heads, 2048) == 64
    assert ops._rows_part(8, kv_heads, 2048) == 128
    assert ops._rows_part(8, kv_heads, 2100) == 128
    assert ops._rows_part(8, kv_heads, 8192) == 512
    assert ops._rows_part(64, kv_heads, 2048) == 512
    assert ops._rows_part(1, 1, 5) == 64
    assert ops._rows_part(128, 8, 100000) == 512
    last = 0
    for context in range(1, 40000, 977):
        part = ops._rows_part(4, 2, context)
        assert part in (64, 128, 256, 512) and part >= last
        last = part


def test_decode_parts_cover_the_context():
    for rows, kv_heads, context in ((1, 8, 2048), (8, 8, 2048), (64, 8, 2048), (3, 1, 70000), (16, 4, 17), (1, 2, 1)):
        part, parts = ops._decode_parts(rows, kv_heads, context)
        assert part % 64 == 0 and ops.DECODE_MIN_PART <= part <= ops.DECODE_MAX_PART
        assert parts >= 1 and part * parts >= context and part * (parts - 1) < context


def test_decode_parts_fill_their_rounds_of_blocks():
    """More blocks than CUs run in rounds: where one part a row would leave the last round mostly empty the context
    is cut so that the rounds fill; where the rounds are full anyway, or the context is short, it stays whole."""
    kv_heads = 8
    assert ops._decode_parts(32, kv_heads, 2048) == (2048, 1)         # 256 blocks: one round
    assert ops._decode_parts(33, kv_heads, 2048) == (512, 4)          # 264 blocks -> 1,056: 5 rounds, 82 % full
    assert ops._decode_parts(40, kv_heads, 2048) == (1024, 2)
    assert ops._decode_parts(48, kv_heads, 2048) == (2048, 1)         # 384 blocks: the second round is half full
    assert ops._decode_parts(64, kv_heads, 2048) == (2048, 1)
    assert ops._decode_parts(65, kv_heads, 2048) == (1024, 2)
    assert ops._decode_parts(33, kv_heads, 8192) == (1216, 7)         # long parts: filled to 90 %
    assert ops._decode_parts(33, kv_heads, 700) == (704, 1)           # too short to cut
    for rows in range(1, 300, 7):
        for context in (1, 300, 2048, 5000, 40000, 131072):
            part, parts = ops._decode_parts(rows, kv_heads, context)
            assert part % 64 == 0 and ops.DECODE_MIN_PART <= part <= ops.DECODE_MAX_PART
            assert parts >= 1 and part * parts >= context and part * (parts - 1) < context


def test_products_of_257_to_512_rows_go_to_blocks_of_rows_where_the_library_is_slow(lib):
    down, qkv, gate_up = (4096, 12288), (6144, 4096), (24576, 4096)
    assert lib.qil_gemm_bf16_mid_rows_takes(512, *down) and lib.qil_gemm_bf16_mid_rows_takes(257, *down)
    assert lib.qil_gemm_bf16_mid_rows_takes(300, *qkv) and not lib.qil_gemm_bf16_mid_rows_takes(400, *qkv)
    assert not lib.qil_gemm_bf16_mid_rows_takes(300, *gate_up)
    assert not lib.qil_gemm_bf16_mid_rows_takes(256, *down) and not lib.qil_gemm_bf16_mid_rows_takes(513, *down)
    assert not lib.qil_gemm_bf16_mid_rows_takes(300, 4100, 4096) and not lib.qil_gemm_bf16_mid_rows_takes(300, 4096, 4000)
    for rows in (257, 300, 512):                              # the plan of such a product: whole stages, 4 or more a split
        splits = lib.qil_gemm_bf16_mid_splits(rows, *down)
        assert 1 <= splits <= 16 and (12288 // 64) % splits == 0 and 12288 // 64 // splits >= 4
    assert lib.qil_gemm_bf16_mid_splits(1025, *down) == 0


def test_float32_products_split_k_to_fill_the_chip(lib):
    """Up to 16 rows and 17 to 64 rows are whole-line kernels with K in whole stages of 64 columns, three or more a
    split; the blocks of 128 columns times the splits stay within the CUs where they can."""
    for rows in (1, 16, 17, 64):
        for n, k in ((4096, 4096), (6144, 4096), (1024, 3072), (24576, 4096), (130, 192)):
            splits = lib.qil_gemm_f32_splits(rows, n, k)
            assert splits >= 1 and k % (64 * splits) == 0 and k // (64 * splits) >= 3, (rows, n, k, splits)
    assert lib.qil_gemm_f32_splits(20, 4096, 4096) == 8        # 32 blocks of columns x 8 = 256
    assert lib.qil_gemm_f32_splits(20, 24576, 4096) == 1       # 192 blocks of columns already
    assert lib.qil_gemm_f32_splits(20, 4096, 100) >= 1         # no whole stage: another kernel, still a valid answer


def test_general_tile_kernel_cuts_the_keys_of_few_row_tiles(lib):
    part = ctypes.c_int(0)
    float32, bfloat16 = 0, 1
    # one portion of 128 rows, 16 heads in 8 groups: 32 blocks of row tiles -> parts of 128 keys
    assert lib.qil_attn_tile_key_parts(1, 128, 16, 8, 128, 2048, float32, ctypes.byref(part)) == 16 and part.value == 128
    assert lib.qil_attn_tile_key_parts(1, 128, 16, 8, 128, 2700, float32, ctypes.byref(part)) == 22 and part.value == 128
    # a whole prompt of 2,048 rows fills the chip by itself; a short context is not worth cutting
    assert lib.qil_attn_tile_key_parts(1, 2048, 16, 8, 128, 2048, float32, ctypes.byref(part)) == 1
    assert lib.qil_attn_tile_key_parts(1, 128, 16, 8, 128, 400, float32, ctypes.byref(part)) == 1
    for context in (512, 1000, 5000, 40000):
        for dtype in (float32, bfloat16):
            parts = lib.qil_attn_tile_key_parts(2, 64, 8, 2, 96, context, dtype, ctypes.byref(part))
            if parts > 1:
                assert part.value % 64 == 0 and part.value >= 128 and parts <= 32
                assert part.value * parts >= context > part.value * (parts - 1)


def test_narrow_products_of_many_rows_are_whole(lib):
    """Partial sums only of what a norm or a join reads once: not of factors that a scan reads again and again."""
    for rows in (513, 700, 2048):
        for columns in (32, 64, 288, 992):
            assert lib.qil_gemm_bf16_wide_splits(rows, columns, 4096, 1) in (0, 1)
        assert lib.qil_gemm_bf16_wide_splits(rows, 32, 1024, 1) == lib.qil_gemm_bf16_wide_splits(rows, 32, 1024, 0)
    assert lib.qil_gemm_bf16_wide_splits(700, 1024, 3072, 1) > 1


def test_a_products_rounds_are_those_of_the_fullest_xcd(lib):
    """243 blocks of 128 x 128 whose last patch of columns is nearly empty: 34 of them on XCDs of 32 CUs, two rounds.
    Where the patches are whole (48 bands of columns) every XCD has 30."""
    assert lib.qil_gemm_bf16_wide_splits(640, 6528, 1024, 0) == 1            # (short enough for two rounds)
    assert lib.qil_gemm_bf16_wide_splits(257, 10304, 2048, 0) == 0
    assert lib.qil_gemm_bf16_wide_splits(600, 6400, 2048, 0) == 0 and lib.qil_gemm_bf16_wide_splits(600, 6144, 2048, 0) == 1


def test_products_of_steps_that_a_graph_may_replay(lib):
    """Up to 512 rows only products that are level with the library's on the GPU: not few blocks with a long K, and no
    partial sums.  From 513 rows on the host's time for a library product counts too."""
    for rows in (257, 300, 400, 512):
        for columns, k in ((2048, 2048), (1024, 2048), (1024, 1024), (3072, 1536), (2112, 2048)):
            assert lib.qil_gemm_bf16_wide_splits(rows, columns, k, 1) == 0
        assert lib.qil_gemm_bf16_wide_splits(rows, 8192, 1024, 1) == 1
        assert lib.qil_gemm_bf16_wide_gated_wanted(rows, 3072, 1024) and not lib.qil_gemm_bf16_wide_gated_wanted(rows, 1024, 2048)
    assert lib.qil_gemm_bf16_wide_splits(513, 2048, 2048, 0) == 1 and lib.qil_gemm_bf16_wide_splits(513, 1024, 1024, 1) > 1
    assert lib.qil_gemm_bf16_wide_gated_wanted(513, 1024, 2048)


def test_whole_products_of_few_rows_that_cannot_split_k(lib):
    """A K of an odd number of stages of 128 runs with K split over the waves only where the columns alone fill the chip, or
    where the other kernel does not take it (up to 8 rows and more than 33 stages)."""
    for rows in (1, 8, 16):
        for columns in (32, 1024, 4096):
            for k in (1152, 1408, 3200, 4224):
                assert not lib.qil_gemm_bf16_whole_takes(rows, columns, k)
            assert lib.qil_gemm_bf16_whole_takes(rows, columns, 1280) and lib.qil_gemm_bf16_whole_takes(rows, columns, 2304)
            assert lib.qil_gemm_bf16_whole_takes(rows, columns, 4480) == (rows <= 8)
        assert lib.qil_gemm_bf16_whole_takes(rows, 4112, 1152) and lib.qil_gemm_bf16_whole_takes(rows, 12288, 4480)


def test_small_float32_products_take_narrow_blocks(lib):
    """Blocks of 4 waves where those fill more CUs and the weights are at most 16 MB, else of 8 (or 16 for one full round)."""
    waves = lambda rows, n, k: lib.qil_gemm_f32_waves(rows, n, k, lib.qil_gemm_f32_splits(rows, n, k))
    for rows in (1, 4, 16):
        assert waves(rows, 4096, 1024) == waves(rows, 1024, 2048) == waves(rows, 1024, 3072) == 4
        assert waves(rows, 4096, 1088) == 8                        # a stage more than 16 MB
        assert waves(rows, 6144, 1024) == 8
    assert lib.qil_gemm_f32_splits(4, 1024, 3072) == 12


def test_decode_attention_refuses_caches_of_other_types():
    """Its kernels read bfloat16 and float32 pages; caches of another type of two bytes must not be taken for bfloat16 ones."""
    import torch
    d, rows = 64, 2
    for dtype in (torch.float16, torch.float64, torch.int16):
        k, v = torch.zeros(3, 1, 16, d, dtype=dtype), torch.zeros(3, 1, d, 16, dtype=dtype)
        with pytest.raises(ops.UnsupportedShape):
            ops.decode_attention(ops.Partials(torch.zeros(1, rows, 3 * d)), heads=1, kv_heads=1, head_dim=d, q_weight=None,
                                 k_weight=None, eps=1e-6, rotation=None, positions=torch.zeros(rows, dtype=torch.int32), writes=False,
                                 k_cache=k, v_cache=v, page_size=16, block_tables=torch.zeros(rows, 1, dtype=torch.int32),
                                 row_seq=torch.zeros(rows, dtype=torch.int32), max_context=1, scale=1.0, window=None)


def test_adds_are_told_how_many_pieces_their_array_holds(lib):
    """Groups of 8 columns leave twice the pieces of groups of 16: an array sized for the other number is refused before
    anything is launched (the addresses are never read)."""
    for m, n, k in ((1, 1024, 3072), (8, 2048, 6144), (9, 1024, 3072), (8, 1024, 2048)):
        pieces = lib.qil_gemm_bf16_add_pieces(m, n, k)
        assert pieces in (n // 16, n // 8)
        for other in (0, n // 16 + n // 8 - pieces, pieces + 1):
            assert lib.qil_gemm_bf16_add_in_pieces(16, 16, 16, 16, other, m, n, k, None) == -1


def test_queries_in_the_latents_space_need_a_rotated_part():
    """Pairs of elements are turned: none, or an odd number of them, is refused as ever."""
    import torch
    for rot in (0, 1, 7):
        with pytest.raises(RuntimeError, match='size not taken'):
            ops.latent_query(torch.zeros(2, 3 * (8 + rot)), torch.zeros(3, 8, 16), heads=3, dim=8, rot=rot, rank=16,
                             frequencies=torch.zeros(rot // 2), positions=torch.zeros(2, dtype=torch.int32))


def test_gate_functions_inside_products_of_many_rows():
    """Where a function other than silu joins a product of more than 256 rows: 2,048 to 4,096 columns, and a short K or more rows
    than a graph replays."""
    assert ops._wide_function_wanted(300, 2048, 1024) and ops._wide_function_wanted(512, 3072, 1024)
    assert not ops._wide_function_wanted(400, 1536, 1024) and not ops._wide_function_wanted(300, 512, 512)
    assert not ops._wide_function_wanted(450, 2048, 2048) and ops._wide_function_wanted(600, 2048, 2048)
    assert not ops._wide_function_wanted(600, 1024, 2048) and not ops._wide_function_wanted(257, 6144, 1024)


def test_gate_functions_inside_products_of_few_rows():
    """A short K, or more columns with it: what a long K loses when a block's waves share it instead of blocks."""
    assert ops._few_function_wanted(1, 48, 256) and ops._few_function_wanted(8, 10240, 5120) and ops._few_function_wanted(16, 10240, 4096)
    assert not ops._few_function_wanted(8, 2048, 4096) and not ops._few_function_wanted(8, 6144, 8192)
    assert not ops._few_function_wanted(9, 5120, 4096) and not ops._few_function_wanted(16, 8192, 4096)


def test_float32_decode_parts_and_kernels():
    """Two blocks a CU with heads of 128, four with heads of 64; groups of one head on the matrix cores where the work is less than
    a round of blocks or many rounds (heads of 128), or not just more than one (heads of 64); other groups always."""
    assert ops._matrix_part(8, 8, 128, 2048) == 256 and ops._matrix_part(8, 8, 64, 2048) == 128
    assert ops._matrix_part(1, 8, 128, 512) == 64 and ops._matrix_part(64, 8, 128, 8192) == 512
    assert ops._matrix_part(33, 8, 128, 1000) == 256          # 1,056 blocks, not 528
    for rows, kv_heads, places in ((1, 8, 100), (16, 16, 300), (33, 2, 4000), (64, 8, 16000)):
        assert ops._matrix_attention_wanted(rows, 2 * kv_heads, kv_heads, 128, places)
        assert ops._matrix_attention_wanted(rows, 2 * kv_heads, kv_heads, 64, places)
    assert ops._matrix_attention_wanted(33, 2, 2, 128, 300) and ops._matrix_attention_wanted(48, 16, 16, 128, 1000)
    assert not ops._matrix_attention_wanted(33, 16, 16, 128, 20) and not ops._matrix_attention_wanted(16, 16, 16, 128, 300) and not ops._matrix_attention_wanted(33, 16, 16, 128, 520)
    assert not ops._matrix_attention_wanted(33, 4, 4, 64, 2048) and ops._matrix_attention_wanted(24, 4, 4, 64, 2048)


def test_prompt_attention_in_two_groups_of_waves_by_the_keys_a_block_passes(lib):
    """Not by the rows that come in: a portion behind a history passes all of its keys."""
    waves = lambda seqs, rows, keys, heads=16, window=0: lib.qil_attn_prompt_waves(seqs, rows, keys, heads, 8, window)
    for heads in (16, 32):
        for rows, keys in ((33, 633), (64, 764), (64, 964), (128, 628), (256, 756), (400, 900)):
            assert waves(1, rows, keys, heads) == 16 and waves(1, rows, keys, heads, 100) == 4
        for rows, keys in ((33, 33), (64, 64), (64, 264), (128, 428), (256, 456), (400, 400)):
            assert waves(1, rows, keys, heads) == 4
    assert waves(3, 300, 900, 32) == 16 and waves(3, 301, 301) == 4 and waves(2, 900, 900) == 16 and waves(2, 600, 600, 32) == 4
    assert waves(1, 1000, 1000, 32) == 16 and waves(1, 2300, 2300) == 16 and waves(1, 2900, 2900) == 4 and waves(1, 2048, 2048, 32) == 4
    assert waves(8, 128, 1128, 32) == 16 and waves(4, 256, 1756, 32) == 16        # as many blocks as CUs, too many to cut the keys
