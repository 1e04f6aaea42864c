"""Kernels of steps with few rows (norms with the row in registers, products whose result has to be whole, small gated ones, the
row attention's values), the gate of four elements a thread and the convolution of long sequences."""
import pytest
import torch

import kernel_refs as refs
from test_kernels_gpu import build_cache

pytestmark = pytest.mark.gpu


@pytest.fixture(scope='module')
def ops():
    from qil_amd import ops
    ops.library.load()
    return ops


def rand(*shape, dtype=torch.float32, scale=1.0, seed=0):
    g = torch.Generator().manual_seed(seed + sum(shape))
    return (torch.randn(*shape, generator=g) * scale).to(dtype).cuda()


# a width at each edge of the register shapes, one that no thread fills, one beyond them and one that is no multiple of four
@pytest.mark.parametrize('width', [4, 256, 260, 1024, 2044, 2048, 4096, 8192, 8196, 1002])
@pytest.mark.parametrize('centre', [True, False])
@pytest.mark.parametrize('kind', ['none', 'bfloat16', 'partials', 'float32'])
def test_norms_with_the_row_in_registers(ops, width, centre, kind):
    """Against the reference in float64: sums of `width` float32 terms are off by about 2^-24 sqrt(width) of the row's size, the
    result is rounded once.  The stream's sum is the same float32 sum, split by split, to one rounding of the scaled delta."""
    n, dtype = 3, torch.float32 if kind == 'float32' else torch.bfloat16
    stream = rand(n, width, scale=2.0) + 5.0                 # a mean to be removed
    weight, bias = 1 + 0.2 * rand(width, seed=2), rand(width, seed=3)
    delta = {'none': None, 'bfloat16': rand(n, width, dtype=torch.bfloat16, seed=4), 'float32': rand(n, width, seed=4),
             'partials': ops.Partials(rand(5, n, width, seed=5))}[kind]
    value = 0.0 if delta is None else (delta.tensor.double().sum(0) if kind == 'partials' else delta.double())
    total = stream.double() + 0.5 * value
    centred = total - total.mean(-1, keepdim=True) if centre else total
    want = centred / torch.sqrt(centred.square().mean(-1, keepdim=True) + 1e-5) * weight.double() + bias.double()
    rows = torch.tensor([2, 0], dtype=torch.int32).cuda()
    close = dict(atol=2e-5, rtol=2e-5) if dtype == torch.float32 else dict(atol=2e-4, rtol=2.0 ** -8)
    before = stream.clone()
    some = ops.rows_norm(stream, delta, rows, weight, 1e-5, dtype, centre=centre, delta_scale=0.5, bias=bias)
    assert torch.equal(stream, before)
    got = ops.add_norm(stream, delta, weight, 1e-5, dtype, centre=centre, delta_scale=0.5, bias=bias)
    torch.testing.assert_close(got.double(), want, **close)
    assert torch.equal(some, got[rows.long()])
    torch.testing.assert_close(stream.double(), total, atol=1e-5, rtol=2.0 ** -22)


@pytest.mark.parametrize('m', [1, 8, 9, 16])
@pytest.mark.parametrize('n,k', [(16, 1024), (3072, 1536), (2064, 6144), (16384, 1152)])
def test_whole_products_of_few_rows(ops, m, n, k):
    """One rounding of a float32 sum of k terms of size one (3e-6 of the largest covers 6,144 of them)."""
    assert ops.library.load().qil_gemm_bf16_whole_takes(m, n, k)
    x, w = rand(m, k, dtype=torch.bfloat16), rand(n, k, dtype=torch.bfloat16, seed=1, scale=k ** -0.5)
    want = x.double() @ w.double().t()
    got = ops.linear(x, w)
    assert got.dtype == torch.bfloat16
    torch.testing.assert_close(got.double(), want, atol=3e-6 * want.abs().max().item(), rtol=2.0 ** -8)


@pytest.mark.parametrize('m', [1, 8, 16])
@pytest.mark.parametrize('inner,k', [(3072, 1024), (16, 256), (4096, 4096), (4096, 384), (48, 640)])
def test_small_gated_products(ops, m, inner, k):
    """Fewer pairs of tiles than CUs: a block each.  As above, through silu(gate) * up."""
    x, w = rand(m, k, dtype=torch.bfloat16), rand(2 * inner, k, dtype=torch.bfloat16, seed=1, scale=k ** -0.5)
    y = x.double() @ w.double().t()
    want = torch.nn.functional.silu(y[:, :inner]) * y[:, inner:]
    got = ops.gated_linear(x, ops.interleave_gate_up(w[:inner].contiguous(), w[inner:].contiguous()), interleaved=True)
    torch.testing.assert_close(got.double(), want, atol=3e-5 * want.abs().max().item(), rtol=2.0 ** -8)


# every way the waves share a head's elements: one run of 32 for four waves, two, three (a wave idles), four, more than four;
# every head tile; a part of one key, parts that end inside a run of keys, and keys behind a window
@pytest.mark.parametrize('d', [8, 32, 64, 96, 128, 136, 256])
@pytest.mark.parametrize('heads,kv_heads', [(2, 2), (4, 2), (6, 2), (16, 2)])
def test_rows_attention_shares_out_the_values(ops, monkeypatch, d, heads, kv_heads):
    """Float32 rows against float64: weights and values of size one over 600 keys, sums off by a few 1e-6."""
    lengths, page_size = [1, 17, 256, 600], 16
    k_cache, v_cache, table, _ = build_cache(lengths, page_size, kv_heads, d, torch.float32)
    positions = torch.tensor([n - 1 for n in lengths], dtype=torch.int32).cuda()
    q = rand(len(lengths), heads * d, seed=5)
    for window in (None, 40):
        step = dict(heads=heads, kv_heads=kv_heads, head_dim=d, page_size=page_size, block_tables=table, scale=d ** -0.5,
                    row_seq=torch.arange(len(lengths), dtype=torch.int32).cuda(), positions=positions, max_context=max(lengths),
                    window=window, cu_seqlens=None, seq_starts=None, single_rows=None, n_seqs=len(lengths), max_query=1)
        got = ops.paged_attention(q, k_cache=k_cache, v_cache=v_cache, **step)
        want = refs.paged_attention(q.double(), k_cache=k_cache.double(), v_cache=v_cache.double(), accumulate=torch.float64, **step)
        torch.testing.assert_close(got.double(), want.double(), atol=1e-5, rtol=1e-5)


# long parts, whose head sizes decide whether the waves share out elements or keys, and how many runs of keys they ask for
@pytest.mark.parametrize('d', [32, 64, 80, 128, 160, 192])
@pytest.mark.parametrize('heads,kv_heads', [(2, 2), (4, 2), (8, 2), (16, 2)])
def test_rows_attention_with_long_parts(ops, monkeypatch, d, heads, kv_heads):
    """Parts of 512 keys, one of a key and one that is not whole.  Float32 rows against float64 as above, over 1,300 keys."""
    monkeypatch.setattr(ops, 'ATTENTION_PART', 512)
    lengths, page_size = [1, 513, 1300, 512], 16
    k_cache, v_cache, table, _ = build_cache(lengths, page_size, kv_heads, d, torch.float32)
    positions = torch.tensor([n - 1 for n in lengths], dtype=torch.int32).cuda()
    q = rand(len(lengths), heads * d, seed=6)
    step = dict(heads=heads, kv_heads=kv_heads, head_dim=d, page_size=page_size, block_tables=table, scale=d ** -0.5,
                row_seq=torch.arange(len(lengths), dtype=torch.int32).cuda(), positions=positions, max_context=max(lengths),
                window=None, cu_seqlens=None, seq_starts=None, single_rows=None, n_seqs=len(lengths), max_query=1)
    got = ops.paged_attention(q, k_cache=k_cache, v_cache=v_cache, **step)
    want = refs.paged_attention(q.double(), k_cache=k_cache.double(), v_cache=v_cache.double(), accumulate=torch.float64, **step)
    torch.testing.assert_close(got.double(), want.double(), atol=1e-5, rtol=1e-5)


# widths the four-element kernel takes and does not, a gate that starts between its loads, an input that is not aligned
@pytest.mark.parametrize('columns,offset,width,shift', [(1024, 4, 1028, 0), (4, 0, 4, 0), (1024, 2, 1028, 0), (30, 4, 64, 0), (64, 4, 70, 0),
                                                        (64, 4, 68, 1)])
@pytest.mark.parametrize('kind', ['bfloat16', 'partials', 'float32'])
def test_gate_of_four_elements(ops, columns, offset, width, shift, kind):
    """The sigmoid to a few float32 roundings, then one rounding of the product."""
    n, dtype = 5, torch.float32 if kind == 'float32' else torch.bfloat16
    x = rand(n * columns + shift, dtype=dtype)[shift:].view(n, columns)
    source = ops.Partials(rand(3, n, width, seed=1)) if kind == 'partials' else rand(n, width, dtype=dtype, seed=1)
    logits = (source.tensor.double().sum(0) if kind == 'partials' else source.double())[:, offset:offset + columns]
    got = ops.sigmoid_gate(x, source, offset=offset)
    torch.testing.assert_close(got.double(), x.double() * torch.sigmoid(logits), atol=1e-6, rtol=2e-6 if kind == 'float32' else 2.0 ** -8)


# rows whose last group is not whole; sequences that start at the edge of a group, inside one, next to each other, with fewer
# rows than the state holds, that begin or continue (from a state shorter than three inputs too); passed columns or none
@pytest.mark.parametrize('counts,starts', [([513], [0]), ([301, 8, 1, 2, 3, 250], [0, 5, 1, 0, 2, 7]), ([520, 505], [2, 0]),
                                           ([256, 2, 256], [9, 1, 0])])
@pytest.mark.parametrize('channels,passed', [(1024, 64), (1032, 0), (8, 8)])
def test_convolution_of_long_sequences(ops, counts, starts, channels, passed):
    """Against the reference in float32: four products of size one and a silu, then one rounding; the state is the inputs."""
    n, width, n_seqs = sum(counts), channels + passed + 8, len(counts)
    x = rand(n, width, dtype=torch.bfloat16)
    weight, bias = rand(4, channels, seed=1), rand(channels, seed=2)
    state = rand(8, 3, channels, seed=3)
    for s, start in enumerate(starts):                        # what lies before a sequence's first position is never read
        state[s + 1, :max(3 - start, 0)] = float('nan')
    step = dict(cu_seqlens=torch.tensor([0] + counts).cumsum(0).to(torch.int32), seq_starts=torch.tensor(starts, dtype=torch.int32),
                seq_slots=torch.arange(1, n_seqs + 1, dtype=torch.int32),
                row_seq=torch.arange(n_seqs, dtype=torch.int32).repeat_interleave(torch.tensor(counts)))
    sizes = dict(columns=channels, n_seqs=n_seqs, activation='silu', out_dtype=torch.bfloat16, pass_from=channels + 8 if passed else 0,
                 passed=passed)
    state_c = state.cpu()
    want = refs.channel_conv(x.cpu(), weight.cpu(), bias.cpu(), state=state_c, **step, **sizes)
    got = ops.channel_conv(x, weight, bias, state=state, **{k: v.cuda() for k, v in step.items()}, **sizes)
    if passed:
        assert torch.equal(got[1].cpu(), want[1])
        got, want = got[0], want[0]
    torch.testing.assert_close(got.cpu().float(), want.float(), atol=2e-6, rtol=2.0 ** -7)
    assert torch.equal(state.cpu().nan_to_num(7.0), state_c.nan_to_num(7.0))


# eight rows: K split over a block's waves where the operands lie on 16 bytes; 600: a block kernel of this library's
@pytest.mark.parametrize('m', [8, 600])
@pytest.mark.parametrize('shifted', ['x', 'weight', 'both'])
def test_products_of_views_at_odd_offsets(ops, m, shifted):
    """Contiguous views that begin between two multiples of 16 bytes are taken as they always were: whole results, and the
    gated product of many rows, against float64.  (One rounding of the sums; through the gate the products' own rounding to
    bfloat16 too, 2^-8 of values up to the largest sum.)"""
    n, k = 2048, 1024
    lib = ops.library.load()
    assert lib.qil_gemm_bf16_whole_takes(8, n, k) and lib.qil_gemm_bf16_wide_splits(600, n, k, 0) and \
        lib.qil_gemm_bf16_wide_gated_wanted(600, n // 2, k)
    view = lambda rows, columns, name, **kw: rand(rows * columns + 8, dtype=torch.bfloat16, **kw)[
        1 if shifted in (name, 'both') else 0:][:rows * columns].view(rows, columns)
    x, w = view(m, k, 'x'), view(n, k, 'weight', seed=1, scale=k ** -0.5)
    assert (x.data_ptr() | w.data_ptr()) % 16
    want = x.double() @ w.double().t()
    got = ops.linear(x, w)
    assert isinstance(got, torch.Tensor) and got.dtype == torch.bfloat16
    torch.testing.assert_close(got.double(), want, atol=3e-6 * want.abs().max().item(), rtol=2.0 ** -8)
    if m > 16:
        at = torch.arange(n).view(-1, 2, 16)                 # gate and up rows in turns of 16
        gate, up = want[:, at[:, 0].reshape(-1).cuda()], want[:, at[:, 1].reshape(-1).cuda()]
        gated = ops.gated_linear(x, w, interleaved=True)
        torch.testing.assert_close(gated.double(), torch.nn.functional.silu(gate) * up,
                                   atol=2.0 ** -7 * want.abs().max().item(), rtol=2.0 ** -6)


@pytest.mark.parametrize('d,heads,kv_heads', [(32, 8, 8), (48, 8, 4), (64, 16, 8), (80, 16, 4), (96, 8, 4)])
@pytest.mark.parametrize('lengths,window', [([320], None), ([2049, 1, 33, 545, 1024, 1056, 1300, 2017] * 2, None), ([700, 289, 5, 2000] * 6, 256)])
def test_decode_attention_with_two_steps_in_flight(ops, d, heads, kv_heads, lengths, window):
    """Launches of at most a block a CU whose waves have several steps of 32 keys, an even and an odd number of them, none for
    some waves: against the float32 reference, one rounding to bfloat16 and its neighbour (2^-7), values of size one."""
    lengths = lengths * (256 // kv_heads) if len(lengths) == 1 else lengths
    dtype, rows, page_size = torch.bfloat16, len(lengths), 16
    k_cache, v_cache, table, _ = build_cache(lengths, page_size, kv_heads, d, dtype)
    step = dict(heads=heads, kv_heads=kv_heads, head_dim=d, k_cache=k_cache, v_cache=v_cache, page_size=page_size, block_tables=table,
                row_seq=torch.arange(rows, dtype=torch.int32).cuda(), positions=torch.tensor([n - 1 for n in lengths], dtype=torch.int32).cuda(),
                cu_seqlens=None, seq_starts=None, single_rows=None, n_seqs=rows, max_query=1, max_context=max(lengths), scale=d ** -0.5,
                window=window)
    part, parts = ops._decode_parts(rows, kv_heads, ops._places(max(lengths), window, 0))
    assert rows * kv_heads * parts <= 256 and part > 32 * ops.DECODE_WAVES
    q = rand(rows, heads * d, dtype=dtype, seed=5)
    got = ops.paged_attention(q, **step)
    torch.testing.assert_close(got.float(), refs.paged_attention(q, **step).float(), atol=2.0 ** -8, rtol=2.0 ** -7)
