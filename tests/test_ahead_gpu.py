"""Few-row kernels that ask for their weights ahead of their operand's arrival: the edges of the rules and of the loads."""
import pytest
import torch

import kernel_refs as refs
from test_kernels_gpu import Rot, build_cache

pytestmark = pytest.mark.gpu


@pytest.fixture(scope='module')
def ops():
    from qil_amd import ops
    ops.library.load()
    return ops


def rand(*shape, dtype=torch.float32, scale=1.0, seed=0):
    g = torch.Generator().manual_seed(seed + sum(shape))
    return (torch.randn(*shape, generator=g) * scale).to(dtype).cuda()


# blocks of four and of eight waves; one turn of parts (4), a second one (5) and a third batch of maxima (21); a piece of A a thread
# and more; a window that leaves the first parts without keys
@pytest.mark.parametrize('m', [1, 4, 5, 8, 16])
@pytest.mark.parametrize('parts', [1, 4, 5, 21])
@pytest.mark.parametrize('n,heads,d,window', [(1024, 16, 128, 0), (64, 6, 64, 0), (4096, 32, 128, 40)])
def test_products_behind_the_merge(ops, m, parts, n, heads, d, window):
    """The parts past a row's keys hold NaN, which nothing may read into a sum.  The operand is rounded to bfloat16 (2^-9 of each of k
    terms) and multiplied in float32."""
    lib, part = ops.library.load(), 32
    k, splits = heads * d, ops.library.load().qil_gemm_bf16_splits(m, n, heads * d)
    assert lib.qil_gemm_bf16_unmerged_takes(m, n, heads, d, splits)
    positions = torch.tensor([(r * 37 + 5) % (parts * part) for r in range(m - 1)] + [parts * part - 1], dtype=torch.int32).cuda()
    acc, top, total = rand(m, heads, parts, d), rand(m, heads, parts, seed=1), rand(m, heads, parts, seed=2).abs() + 1
    index = torch.arange(parts, device='cuda')
    last = positions // part
    first = (positions + 1 - window).clamp(min=0) // part if window else torch.zeros_like(last)
    live = (index >= first[:, None]) & (index <= last[:, None])
    weights = torch.where(live[:, None], top.double(), -torch.inf).softmax(-1)           # exp(m_p - max) over its sum
    divisor = (weights * total.double().where(live[:, None], 0)).sum(-1)
    want = (weights[..., None] * acc.double()).sum(2) / divisor[..., None]
    workspace = torch.cat([acc.where(live[:, None, :, None], torch.nan).flatten(), top.where(live[:, None], torch.nan).flatten(),
                           total.where(live[:, None], torch.nan).flatten()])
    w = rand(n, k, dtype=torch.bfloat16, scale=k ** -0.5, seed=3)
    out = torch.empty(splits, m, n, device='cuda')
    assert lib.qil_gemm_bf16_unmerged(workspace.data_ptr(), positions.data_ptr(), w.data_ptr(), out.data_ptr(), m, n, heads, d,
                                      window, part, parts, splits, torch.cuda.current_stream().cuda_stream) == 0
    rounded = want.reshape(m, k).to(torch.float32).to(torch.bfloat16).double()
    # (a value that lies at a rounding's edge may go either way: one in a few hundred, 2^-8 of its size and 1 / sqrt(k) of the row's)
    torch.testing.assert_close(out.double().sum(0), rounded @ w.double().t(), atol=2.0 ** -8 * 4 * k ** -0.5 * want.abs().max().item(), rtol=1e-5)


# a thread's first and second piece of A and more; one and two rows a wave; pieces of 8 and of 16 columns, more than 256 of them in blocks
# of four and of eight waves, more than 512
@pytest.mark.parametrize('m', [1, 4, 5, 8, 9, 16])
@pytest.mark.parametrize('n,k,columns', [(4096, 1024, 8), (64, 384, 16), (6144, 4096, 16), (512, 4608, 16), (512, 2560, 8), (6144, 2560, 8),
                                         (7168, 5120, 16), (512, 5120, 8)])
def test_products_behind_the_norm(ops, m, n, k, columns):
    """As above, with the operand as the norm rounds it: the row over its root mean square, then the weight."""
    lib = ops.library.load()
    splits = lib.qil_gemm_bf16_splits(m, n, k)
    if not lib.qil_gemm_bf16_normed_takes(m, n, k, splits):
        pytest.skip('not a size of this kernel')
    stream, weight = rand(m, k, scale=3.0), 1 + 0.1 * rand(k, seed=1)
    squares = stream.square().reshape(m, k // columns, columns).sum(-1).t().contiguous()
    normed = (stream.double() / torch.sqrt(stream.double().square().mean(-1, keepdim=True) + 1e-6)).float().bfloat16().float() * weight
    w = rand(n, k, dtype=torch.bfloat16, scale=k ** -0.5, seed=2)
    out = torch.empty(splits, m, n, device='cuda')
    assert lib.qil_gemm_bf16_normed(stream.data_ptr(), weight.data_ptr(), squares.data_ptr(), k // columns, 1e-6, w.data_ptr(),
                                    out.data_ptr(), m, n, k, splits, torch.cuda.current_stream().cuda_stream) == 0
    torch.testing.assert_close(out.double().sum(0), normed.bfloat16().double() @ w.double().t(),
                               atol=2.0 ** -8 * 4 * k ** -0.5 * normed.abs().max().item(), rtol=1e-5)


# rows of A that the waves share unevenly, a last piece of A that half of the lanes load, waves with two stages and with more
@pytest.mark.parametrize('m', [1, 3, 8, 9, 16])
@pytest.mark.parametrize('inner,k', [(3072, 1024), (48, 256), (768, 640), (4096, 4096), (6144, 2176), (12288, 4096)])
def test_gated_products_of_few_rows(ops, m, inner, k):
    """silu(gate) * up of float32 sums of k products, rounded once.  (What stands in LDS past the rows is whatever ran before.)"""
    assert m > 8 or ops.library.load().qil_gemm_bf16_gated_takes(m, inner, k, 1)       # (more rows of a long k do not fit LDS)
    x, w = rand(m, k, dtype=torch.bfloat16), rand(2 * inner, k, dtype=torch.bfloat16, seed=1, scale=k ** -0.5)
    y = x.double() @ w.double().t()
    want = torch.nn.functional.silu(y[:, :inner]) * y[:, inner:]
    got = ops.gated_linear(x, ops.interleave_gate_up(w[:inner].contiguous(), w[inner:].contiguous()), interleaved=True)
    torch.testing.assert_close(got.double(), want, atol=3e-5 * want.abs().max().item(), rtol=2.0 ** -8)


# groups of 8 and of 16 columns, one group a block and several, one wave and eight a group, a block that holds groups past the end
@pytest.mark.parametrize('m', [1, 5, 8, 9, 16])
@pytest.mark.parametrize('n,k', [(1024, 3072), (512, 1024), (16, 384), (4112, 1152), (4096, 4096), (80, 3200)])
def test_products_that_add_into_the_stream(ops, m, n, k):
    """Float32 sums of k products; the pieces of the squares are those of the stream as it is afterwards."""
    lib = ops.library.load()
    x, w = rand(m, k, dtype=torch.bfloat16), rand(n, k, dtype=torch.bfloat16, seed=1, scale=k ** -0.5)
    stream = rand(m, n, seed=2)
    want = stream.double() + x.double() @ w.double().t()
    pieces = lib.qil_gemm_bf16_add_pieces(m, n, k)
    squares = torch.empty(pieces, m, device='cuda')
    assert lib.qil_gemm_bf16_add_in_pieces(x.data_ptr(), w.data_ptr(), stream.data_ptr(), squares.data_ptr(), pieces, m, n, k,
                                           torch.cuda.current_stream().cuda_stream) == 0
    torch.testing.assert_close(stream.double(), want, atol=3e-6 * want.abs().max().item(), rtol=0)
    torch.testing.assert_close(squares.double(), stream.double().square().reshape(m, pieces, n // pieces).sum(-1).t(), atol=0, rtol=1e-6)


# groups of fifteen heads (more LDS than a kernel has without asking) and of one; pages whose size is no power of two; four sums at a
# time and a fifth; neither norm nor rotation; new keys at every place of a step's lanes, in a block's first and last step
@pytest.mark.parametrize('d,heads,kv_heads,page_size', [(128, 15, 1, 16), (128, 16, 8, 24), (64, 4, 4, 8), (64, 16, 1, 40)])
@pytest.mark.parametrize('splits,plain,window', [(2, False, None), (5, False, 40), (1, True, None)])
def test_decode_attention_that_makes_its_queries(ops, d, heads, kv_heads, page_size, splits, plain, window):
    """Keys and values in the pages bit for bit those of the q/k kernel; the result against the float32 reference, one rounding to
    bfloat16 and its neighbour."""
    lengths = [1, 2, 31, 32, 33, 40, 100, 255, 256, 257, 300, 517]
    dtype, rows = torch.bfloat16, len(lengths)
    k_cache, v_cache, table, _ = build_cache(lengths, page_size, kv_heads, d, dtype)
    positions = torch.tensor([n - 1 for n in lengths], dtype=torch.int32).cuda()
    row_seq = torch.arange(rows, dtype=torch.int32).cuda()
    sizes = dict(heads=heads, kv_heads=kv_heads, head_dim=d)
    step = dict(page_size=page_size, block_tables=table, row_seq=row_seq, positions=positions, max_context=max(lengths),
                scale=d ** -0.5, window=window, **sizes)
    rest = dict(cu_seqlens=None, seq_starts=None, single_rows=None, n_seqs=rows, max_query=1)
    slots = (table[row_seq.long(), (positions // page_size).long()] * page_size + positions % page_size).to(torch.int32)
    qkv = ops.Partials(rand(splits, rows, (heads + 2 * kv_heads) * d, scale=splits ** -0.5, seed=21))
    norms = dict(q_weight=None, k_weight=None, eps=0.0, rotation=None) if plain else \
        dict(q_weight=1 + 0.1 * rand(d, seed=22), k_weight=1 + 0.1 * rand(d, seed=23), eps=1e-6, rotation=Rot(d, 10000.0, max(lengths), d))
    k_fused, v_fused = k_cache.clone(), v_cache.clone()
    fused = ops.decode_attention(qkv, writes=True, k_cache=k_fused, v_cache=v_fused, **norms, **step)
    q = ops.qk_norm_rope_store(qkv, positions=positions, slots=slots, k_cache=k_cache, v_cache=v_cache, page_size=page_size,
                               dtype=dtype, **norms, **sizes)
    assert torch.equal(k_fused.view(torch.int16), k_cache.view(torch.int16))
    assert torch.equal(v_fused.view(torch.int16), v_cache.view(torch.int16))
    want = refs.paged_attention(q, k_cache=k_cache, v_cache=v_cache, **step, **rest).float()
    torch.testing.assert_close(fused.float(), want, atol=2.0 ** -8, rtol=2.0 ** -7)


# blocks of four waves with a piece of A a thread and with more, of eight and of sixteen; one turn of parts (16) or sums (4) and a second
@pytest.mark.parametrize('m', [1, 3, 4, 5, 9, 16])
@pytest.mark.parametrize('n,heads,d,parts', [(1024, 16, 128, 16), (1024, 16, 128, 17), (96, 6, 64, 3), (6144, 32, 128, 4)])
def test_float32_products_behind_the_merge(ops, m, n, heads, d, parts):
    """The parts past a row's keys hold NaN.  Float32 sums of k products."""
    lib, part, k = ops.library.load(), 64, heads * d
    splits = lib.qil_gemm_f32_splits(m, n, k)
    if not lib.qil_gemm_f32_unmerged_takes(m, n, heads, d, splits):
        pytest.skip('not a size of this kernel')
    positions = torch.tensor([(r * 71 + 5) % (parts * part) for r in range(m - 1)] + [parts * part - 1], dtype=torch.int32).cuda()
    acc, top, total = rand(m, heads, parts, d), rand(m, heads, parts, seed=1), rand(m, heads, parts, seed=2).abs() + 1
    live = torch.arange(parts, device='cuda') <= (positions // part)[:, None]
    weights = torch.where(live[:, None], top.double(), -torch.inf).softmax(-1)
    want = (weights[..., None] * acc.double()).sum(2) / (weights * total.double()).sum(-1)[..., None]
    workspace = torch.cat([acc.where(live[:, None, :, None], torch.nan).flatten(), top.where(live[:, None], torch.nan).flatten(),
                           total.where(live[:, None], torch.nan).flatten()])
    w = rand(n, k, scale=k ** -0.5, seed=3)
    out = torch.empty(splits, m, n, device='cuda')
    assert lib.qil_gemm_f32_unmerged(workspace.data_ptr(), positions.data_ptr(), w.data_ptr(), out.data_ptr(), m, n, heads, d, 0,
                                     part, parts, splits, torch.cuda.current_stream().cuda_stream) == 0
    want = want.reshape(m, k) @ w.double().t()
    torch.testing.assert_close(out.double().sum(0), want, atol=3e-6 * want.abs().max().item(), rtol=0)


@pytest.mark.parametrize('m', [1, 3, 4, 5, 9, 16])
@pytest.mark.parametrize('n,k,sums', [(1024, 3072, 4), (1024, 3072, 5), (64, 192, 1), (4096, 12288, 2)])
@pytest.mark.parametrize('interleaved', [False, True])
def test_float32_products_of_few_rows(ops, m, n, k, sums, interleaved):
    """Behind the activation, and of an operand as it is.  Float32 sums of k products."""
    lib, stream = ops.library.load(), torch.cuda.current_stream().cuda_stream
    splits = lib.qil_gemm_f32_splits(m, n, k)
    w, parts = rand(n, k, scale=k ** -0.5, seed=3), rand(sums, m, 2 * k, scale=sums ** -0.5)
    out = torch.empty(splits, m, n, device='cuda')
    total = parts.double().sum(0)
    gate, up = (total.reshape(m, k // 16, 2, 16).unbind(2) if interleaved else total.reshape(m, 2, k).unbind(1))
    operand = (torch.nn.functional.silu(gate) * up).reshape(m, k)
    if lib.qil_gemm_f32_gated_takes(m, n, k, int(interleaved), splits):
        assert lib.qil_gemm_f32_gated(parts.data_ptr(), sums, int(interleaved), w.data_ptr(), out.data_ptr(), m, n, k, splits, stream) == 0
        want = operand @ w.double().t()
        torch.testing.assert_close(out.double().sum(0), want, atol=3e-6 * want.abs().max().item(), rtol=0)
    x = operand.float()
    assert lib.qil_gemm_f32(x.data_ptr(), w.data_ptr(), None, out.data_ptr(), m, n, k, splits, stream) == 0
    want = x.double() @ w.double().t()
    torch.testing.assert_close(out.double().sum(0), want, atol=3e-6 * want.abs().max().item(), rtol=0)


def behind_parts(ops, m, n, heads, d, parts, window):
    """(an unmerged operand, its merged rows in float64, the product's weights); the parts past a row's keys hold NaN."""
    part, k = 32, heads * d
    positions = torch.tensor([(r * 37 + 5) % (parts * part) for r in range(m - 1)] + [parts * part - 1], dtype=torch.int32).cuda()
    index, last = torch.arange(parts, device='cuda'), positions // part
    first = (positions + 1 - window).clamp(min=0) // part if window else torch.zeros_like(last)
    live = ((index >= first[:, None]) & (index <= last[:, None]))[:, None].expand(m, heads, parts)
    acc, top, total = rand(m, heads, parts, d), rand(m, heads, parts, seed=1), rand(m, heads, parts, seed=2).abs() + 1
    workspace = torch.cat([acc.where(live[..., None], torch.nan).flatten(), top.where(live, torch.nan).flatten(), total.where(live, torch.nan).flatten()])
    w = rand(n, k, dtype=torch.bfloat16, scale=k ** -0.5, seed=3)
    make = lambda: ops.Unmerged(workspace, positions, torch.empty(m, k, dtype=torch.bfloat16, device='cuda'), heads=heads, head_dim=d, window=window,
                                part=part, parts=parts)
    return make(), make().merge().double(), w


# one turn of pieces a thread and more, one to four stages a wave, two parts to four; a window that leaves the first part without keys
SECOND_NORM = [(1024, 16, 128, 2, 0), (2048, 16, 64, 4, 0), (1024, 32, 128, 4, 40), (1024, 16, 128, 16, 0)]


# ... one block of 8 columns; more rows, parts and columns than the kernel takes, and heads * d that is no multiple of 1,024
@pytest.mark.parametrize('m', [1, 2, 3, 4, 5])
@pytest.mark.parametrize('n,heads,d,parts,window', SECOND_NORM + [(8, 24, 128, 3, 0), (1024, 16, 128, 5, 0), (4096, 32, 128, 2, 0), (1024, 6, 128, 2, 0)])
def test_products_behind_the_merge_that_add_into_the_stream(ops, m, n, heads, d, parts, window):
    """Where the rule refuses, partial sums come back and the stream is as it was.  Float32 sums of k products."""
    lib = ops.library.load()
    taken = m <= 4 and m * parts <= 16 and n <= 2048 and heads * d % 1024 == 0
    assert lib.qil_gemm_bf16_unmerged_add_takes(m, n, heads, d, parts) == taken
    operand, merged, w = behind_parts(ops, m, n, heads, d, parts, window)
    stream = rand(m, n, seed=4)
    before, want = stream.clone(), stream.double() + merged @ w.double().t()
    added = ops.linear(operand, w, partials=True, add_to=stream)
    if taken:
        assert isinstance(added, ops.Added)
        torch.testing.assert_close(added.squares.double(), stream.double().square().reshape(m, n // 8, 8).sum(-1).t(), atol=0, rtol=1e-6)
        got = stream.double()
    else:
        assert isinstance(added, ops.Partials) and torch.equal(stream, before)
        got = before.double() + added.tensor.double().sum(0)
    torch.testing.assert_close(got, want, atol=3e-6 * want.abs().max().item(), rtol=0)


@pytest.mark.parametrize('m', [1, 2, 3, 4])
@pytest.mark.parametrize('n,heads,d,parts,window', [case for case in SECOND_NORM if case[3] <= 4])
@pytest.mark.parametrize('inner', [3072, 48])
def test_second_norm_without_a_kernel(ops, m, n, heads, d, parts, window, inner):
    """The product behind the merge adds into the stream, the gated product behind it makes the norm: against the norm's kernel."""
    operand, _, w = behind_parts(ops, m, n, heads, d, parts, window)
    stream = rand(m, n, seed=4)
    added = ops.linear(operand, w, partials=True, add_to=stream)
    weight, gate_up = 1 + 0.1 * rand(n, seed=5), rand(2 * inner, n, dtype=torch.bfloat16, scale=n ** -0.5, seed=6)
    assert ops.library.load().qil_gemm_bf16_gated_normed_takes(m, inner, n)
    lazy = ops.Normed(stream, weight, 1e-6, torch.bfloat16, added)
    got = ops.gated_linear(lazy, gate_up, torch.bfloat16, interleaved=True)
    want = ops.gated_linear(lazy.materialize(), gate_up, torch.bfloat16, interleaved=True)
    # (an operand at a rounding's edge may go either way)
    torch.testing.assert_close(got.double(), want.double(), atol=2.0 ** -8 * 4 * n ** -0.5 * want.abs().max().item(), rtol=2.0 ** -8)


# one and two rows a wave in blocks of one wave, of two and of four; blocks of several pairs of tiles, of which the last has too few
@pytest.mark.parametrize('inner,k,most', [(48, 1152, 2), (48, 1280, 4), (48, 1024, 8), (6160, 2048, 16)])
def test_gated_products_behind_the_norm(ops, inner, k, most):
    """silu(gate) * up of the norm of a stream whose rows' squares are there in pieces of 8 columns; the operand as the norm rounds it."""
    lib = ops.library.load()
    assert not lib.qil_gemm_bf16_gated_normed_takes(most + 1, inner, k)
    w, weight = rand(2 * inner, k, dtype=torch.bfloat16, seed=1, scale=k ** -0.5), 1 + 0.1 * rand(k, seed=2)
    interleaved = ops.interleave_gate_up(w[:inner].contiguous(), w[inner:].contiguous())
    for m in sorted({1, most // 2, most // 2 + 1, most}):
        assert lib.qil_gemm_bf16_gated_normed_takes(m, inner, k)
        stream = rand(m, k, scale=3.0)
        squares = stream.square().reshape(m, k // 8, 8).sum(-1).t().contiguous()
        out = torch.empty(m, inner, dtype=torch.bfloat16, device='cuda')
        assert lib.qil_gemm_bf16_gated_normed(stream.data_ptr(), weight.data_ptr(), squares.data_ptr(), k // 8, 1e-6, interleaved.data_ptr(),
                                              out.data_ptr(), m, inner, k, torch.cuda.current_stream().cuda_stream) == 0
        normed = (stream.double() / torch.sqrt(stream.double().square().mean(-1, keepdim=True) + 1e-6)).float().bfloat16().float() * weight
        y = normed.bfloat16().double() @ w.double().t()
        want = torch.nn.functional.silu(y[:, :inner]) * y[:, inner:]
        # (an operand at a rounding's edge may go either way)
        torch.testing.assert_close(out.double(), want, atol=2.0 ** -8 * 4 * k ** -0.5 * want.abs().max().item(), rtol=2.0 ** -8)


# one row more and less than a tile of 32 (64 with groups of two heads), keys in one piece (543 rows) and in parts (1,057 without a
# window or sinks: fewer blocks than CUs), two sequences of which one is short, a history ahead of the rows, a window; sinks
@pytest.mark.parametrize('heads,kv_heads,d', [(16, 8, 128), (16, 4, 128), (8, 2, 64), (6, 2, 96)])
@pytest.mark.parametrize('rows,starts,window', [([543], [0], None), ([1057], [0], None), ([65, 33], [40, 0], None), ([1057], [0], 100), ([31], [300], None)])
@pytest.mark.parametrize('sink', [False, True])
def test_prompt_attention_of_odd_lengths(ops, heads, kv_heads, d, rows, starts, window, sink):
    """Tiles of keys that a not quite full tile of rows sees whole are not masked: against the float32 reference, one rounding to
    bfloat16 and its neighbour."""
    lengths = [r + s for r, s in zip(rows, starts)]
    k_cache, v_cache, table, _ = build_cache(lengths, 16, kv_heads, d, torch.bfloat16)
    q = rand(sum(rows), heads * d, dtype=torch.bfloat16, seed=7)
    ints = lambda values: torch.tensor(values, dtype=torch.int32).cuda()
    step = dict(heads=heads, kv_heads=kv_heads, head_dim=d, page_size=16, block_tables=table, scale=d ** -0.5, window=window,
                row_seq=ints([i for i, r in enumerate(rows) for _ in range(r)]),
                positions=ints([s + j for r, s in zip(rows, starts) for j in range(r)]), max_context=max(lengths),
                cu_seqlens=ints([sum(rows[:i]) for i in range(len(rows) + 1)]), seq_starts=ints(starts),
                single_rows=torch.empty(0, dtype=torch.int32).cuda(), n_seqs=len(rows), max_query=max(rows),
                sinks=rand(heads, seed=8) if sink else None)
    got = ops.paged_attention(q, k_cache=k_cache, v_cache=v_cache, **step)
    want = refs.paged_attention(q, k_cache=k_cache, v_cache=v_cache, **step)
    torch.testing.assert_close(got.float(), want.float(), atol=2.0 ** -8, rtol=2.0 ** -7)


@pytest.mark.parametrize('heads,rows,waves', [(16, 2273, 16), (32, 1505, 4), (16, 607, 16)])
def test_prompt_attention_of_many_blocks(ops, heads, rows, waves):
    """Keys in one piece behind a last tile of rows that is not full: 288 blocks of two groups of waves, 384 of four waves, and 80 of
    two groups.  As above."""
    lib, kv_heads, d = ops.library.load(), 8, 128
    k_cache, v_cache, table, _ = build_cache([rows], 16, kv_heads, d, torch.bfloat16)
    q = rand(rows, heads * d, dtype=torch.bfloat16, seed=7)
    ints = lambda values: torch.tensor(values, dtype=torch.int32).cuda()
    assert ops.tile_key_parts(lib, q.dtype, 1, rows, heads, kv_heads, d, 16, table.shape[1], rows)[1] == 1
    assert lib.qil_attn_prompt_waves(1, rows, rows, heads, kv_heads, 0) == waves
    step = dict(heads=heads, kv_heads=kv_heads, head_dim=d, page_size=16, block_tables=table, scale=d ** -0.5, window=None,
                row_seq=ints([0] * rows), positions=ints(range(rows)), max_context=rows, cu_seqlens=ints([0, rows]), seq_starts=ints([0]),
                single_rows=ints([]), n_seqs=1, max_query=rows)
    got = ops.paged_attention(q, k_cache=k_cache, v_cache=v_cache, **step)
    want = refs.paged_attention(q, k_cache=k_cache, v_cache=v_cache, **step)
    torch.testing.assert_close(got.float(), want.float(), atol=2.0 ** -8, rtol=2.0 ** -7)


@pytest.mark.parametrize('rows,starts,told,waves', [([64], [700], None, 16), ([300, 300], [600, 600], None, 16), ([64], [100], None, 4),
                                                    ([64, 1], [700, 900], None, 4), ([64, 1], [700, 900], 764, 16), ([64, 1], [100, 900], 164, 4),
                                                    ([256] * 8, [800] * 8, None, 16)])
def test_block_shape_of_portions_behind_a_history(ops, rows, starts, told, waves):
    """By the keys the portion passes, where they are known (without ``tile_context`` a row alone may be the one with the longest
    context)."""
    lib, heads, kv_heads, d = ops.library.load(), 16, 8, 128
    lengths = [r + s for r, s in zip(rows, starts)]
    k_cache, v_cache, table, _ = build_cache(lengths, 16, kv_heads, d, torch.bfloat16)
    q = rand(sum(rows), heads * d, dtype=torch.bfloat16, seed=7)
    ints = lambda values: torch.tensor(values, dtype=torch.int32).cuda()
    step = dict(heads=heads, kv_heads=kv_heads, head_dim=d, page_size=16, block_tables=table, scale=d ** -0.5, window=None,
                row_seq=ints([i for i, r in enumerate(rows) for _ in range(r)]),
                positions=ints([s + j for r, s in zip(rows, starts) for j in range(r)]), max_context=max(lengths),
                cu_seqlens=ints([sum(rows[:i]) for i in range(len(rows) + 1)]), seq_starts=ints(starts),
                single_rows=ints([sum(rows[:i]) for i, r in enumerate(rows) if r == 1]), n_seqs=len(rows), max_query=max(rows), tile_context=told)
    got = {}
    for shape in (0, 4, 16):
        lib.qil_attn_tile_waves(shape)
        try:
            got[shape] = ops.paged_attention(q, k_cache=k_cache, v_cache=v_cache, **step)
        finally:
            lib.qil_attn_tile_waves(0)
    assert torch.equal(got[0], got[waves]) and not torch.equal(got[0], got[20 - waves])       # (sums in another order)


@pytest.mark.parametrize('heads,kv_heads,d,dtype', [(16, 8, 128, torch.bfloat16), (32, 8, 128, torch.bfloat16), (8, 2, 64, torch.bfloat16),
                                                    (6, 2, 96, torch.bfloat16), (4, 2, 128, torch.float32)])
@pytest.mark.parametrize('told', [None, 1030])
@pytest.mark.parametrize('first', [None, 1])
def test_parts_of_a_portion_beside_a_row_of_a_longer_context(ops, heads, kv_heads, d, dtype, told, first):
    """40 rows behind 990 keys beside a row alone behind 2,600: whether the keys' parts are made for the portion's own context or
    for the row's, and whether the merge takes the row too or the portion's rows only.  Against the float32 reference: bfloat16 one
    rounding and its neighbour, float32 sums of a thousand weighted values of size one in another order."""
    rows, starts = [40, 1], [990, 2600]
    lengths = [r + s for r, s in zip(rows, starts)]
    k_cache, v_cache, table, _ = build_cache(lengths, 16, kv_heads, d, dtype)
    q = rand(sum(rows), heads * d, dtype=dtype, seed=7)
    ints = lambda values: torch.tensor(values, dtype=torch.int32).cuda()
    step = dict(heads=heads, kv_heads=kv_heads, head_dim=d, page_size=16, block_tables=table, scale=d ** -0.5, window=None,
                row_seq=ints([i for i, r in enumerate(rows) for _ in range(r)]),
                positions=ints([s + j for r, s in zip(rows, starts) for j in range(r)]), max_context=max(lengths),
                cu_seqlens=ints([sum(rows[:i]) for i in range(len(rows) + 1)]), seq_starts=ints(starts),
                single_rows=ints([rows[0]]), n_seqs=len(rows), max_query=max(rows))
    got = ops.paged_attention(q, k_cache=k_cache, v_cache=v_cache, tile_context=told, tile_seqs=first, **step)
    want = refs.paged_attention(q, k_cache=k_cache, v_cache=v_cache, **step)
    tolerance = dict(atol=2.0 ** -8, rtol=2.0 ** -7) if dtype == torch.bfloat16 else dict(atol=2e-6, rtol=2e-5)
    torch.testing.assert_close(got.float(), want.float(), **tolerance)
