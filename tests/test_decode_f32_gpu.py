"""The float32 decode attention on the matrix cores, around its steps and parts, against float64."""
import pytest
import torch

import kernel_refs as refs
from test_kernels_gpu import Rot, build_cache, rand

pytestmark = pytest.mark.gpu


@pytest.fixture(scope='module')
def ops():
    from qil_amd import ops
    ops.library.load()
    return ops


def task(lengths, page_size, heads, kv_heads, d, **more):
    rows = len(lengths)
    k_cache, v_cache, table, _ = build_cache(lengths, page_size, kv_heads, d, torch.float32)
    positions = torch.tensor([n - 1 for n in lengths], dtype=torch.int32).cuda()
    step = dict(heads=heads, kv_heads=kv_heads, head_dim=d, page_size=page_size, block_tables=table, scale=d ** -0.5,
                row_seq=torch.arange(rows, dtype=torch.int32).cuda(), positions=positions, max_context=max(lengths), window=None)
    step.update(more)
    return k_cache, v_cache, step, dict(cu_seqlens=None, seq_starts=None, single_rows=None, n_seqs=rows, max_query=1)


# A score is a float32 sum of d products of N(0, 1) elements times d^-1/2: within 1e-6 of a size-one score, so a weight within
# 1e-6 of itself; the weighted values are a float32 sum on top.  1e-5 as in the row kernel's tests.
NEAR = dict(atol=1e-5, rtol=1e-5)

# keys around a wave's step (16), a part (64), two parts and a page; groups of one head, of an odd number and of all 16 columns
LENGTHS = [[1, 15, 16, 17], [63, 64, 65, 300], [2, 1500]]


@pytest.mark.parametrize('lengths', LENGTHS)
@pytest.mark.parametrize('d,heads,kv_heads', [(128, 2, 2), (128, 10, 2), (128, 16, 2), (64, 32, 2), (64, 3, 1)])
@pytest.mark.parametrize('page_size', [4, 16, 24])
def test_rows_alone(ops, lengths, d, heads, kv_heads, page_size):
    assert ops.library.load().qil_attn_decode_f32_takes(heads, kv_heads, d, page_size, 0, 0)
    k_cache, v_cache, step, rest = task(lengths, page_size, heads, kv_heads, d)
    q = rand(len(lengths), heads * d, seed=5)
    got = ops.paged_attention(q, k_cache=k_cache, v_cache=v_cache, **step, **rest)
    want = refs.paged_attention(q.double(), k_cache=k_cache.double(), v_cache=v_cache.double(), accumulate=torch.float64, **step, **rest)
    torch.testing.assert_close(got.double(), want.double(), **NEAR)


# a window that begins inside a step, kept keys with a hole behind them, slopes, sinks and a cap
@pytest.mark.parametrize('more', [dict(window=40), dict(window=1), dict(window=50, keep_first=5), dict(softcap=5.0), 'slopes', 'sinks'])
@pytest.mark.parametrize('lengths', LENGTHS)
def test_masks_and_scores(ops, lengths, more):
    heads, kv_heads, d = 8, 2, 128
    if more == 'slopes':
        more = dict(slopes=torch.tensor([2.0 ** (-h - 1) for h in range(heads)]).cuda())
    elif more == 'sinks':
        more = dict(sinks=rand(heads, seed=3))
    k_cache, v_cache, step, rest = task(lengths, 16, heads, kv_heads, d, **more)
    q = rand(len(lengths), heads * d, seed=6)
    got = ops.paged_attention(q, k_cache=k_cache, v_cache=v_cache, **step, **rest)
    plain = {k: v.double() if k in ('slopes', 'sinks') else v for k, v in step.items()}
    want = refs.paged_attention(q.double(), k_cache=k_cache.double(), v_cache=v_cache.double(), accumulate=torch.float64, **plain, **rest)
    torch.testing.assert_close(got.double(), want.double(), **NEAR)


# a wave makes four heads (d 128) or eight (d 64): groups of one wave, of several, and one head less than whole;
# norms and rotations as the parts ask for them; a reader of another layer's cache
@pytest.mark.parametrize('lengths', LENGTHS)
@pytest.mark.parametrize('d,heads,kv_heads,splits', [(128, 4, 2, 3), (128, 15, 1, 5), (64, 16, 1, 1), (128, 2, 2, 8)])
@pytest.mark.parametrize('form', ['norms', 'bare', 'frequencies'])
def test_queries_made_inside(ops, lengths, d, heads, kv_heads, splits, form):
    """The same bits as the kernel for norms and rotations followed by the attention of its queries, in the caches too."""
    k_cache, v_cache, step, rest = task(lengths, 16, heads, kv_heads, d)
    rows, positions, table = len(lengths), step['positions'], step['block_tables']
    slots = (table[step['row_seq'].long(), (positions // 16).long()] * 16 + positions % 16).to(torch.int32)
    qkv = ops.Partials(rand(splits, rows, (heads + 2 * kv_heads) * d, scale=splits ** -0.5, seed=7))
    made = dict(q_weight=None, k_weight=None, eps=1e-6, rotation=None)
    if form != 'bare':
        made.update(q_weight=1 + 0.1 * rand(d, seed=22), k_weight=1 + 0.1 * rand(d, seed=23), rotation=Rot(d, 10000.0, max(lengths), d))
    if form == 'frequencies':
        from qil_amd.parts import RotaryFrequencies
        made.update(rotation=RotaryFrequencies(d, 10000.0, device='cuda').rotation())
    sizes = dict(heads=heads, kv_heads=kv_heads, head_dim=d)
    assert ops.decode_attention_takes(qkv, page_size=16, rotation=made['rotation'], dtype=torch.float32, **sizes)
    k_two, v_two = k_cache.clone(), v_cache.clone()
    got = ops.decode_attention(qkv, writes=True, k_cache=k_cache, v_cache=v_cache, **made, **step)
    q = ops.qk_norm_rope_store(qkv, positions=positions, slots=slots, k_cache=k_two, v_cache=v_two, page_size=16, dtype=torch.float32,
                               **made, **sizes)
    want = ops.paged_attention(q, k_cache=k_two, v_cache=v_two, **step, **rest)
    assert torch.equal(got, want)
    assert torch.equal(k_cache.view(torch.int32), k_two.view(torch.int32)) and torch.equal(v_cache.view(torch.int32), v_two.view(torch.int32))
    exact = refs.paged_attention(q.double(), k_cache=k_two.double(), v_cache=v_two.double(), accumulate=torch.float64, **step, **rest)
    torch.testing.assert_close(got.double(), exact.double(), **NEAR)


def test_caches_at_other_addresses(ops):
    """Caches that do not begin at a multiple of 16 bytes stay with the row kernel."""
    heads, kv_heads, d, lengths = 4, 2, 64, [33, 200]
    k_cache, v_cache, step, rest = task(lengths, 16, heads, kv_heads, d)
    shifted = torch.empty(k_cache.numel() + 1, device='cuda')[1:].view(k_cache.shape).copy_(k_cache)
    q = rand(2, heads * d, seed=5)
    got = ops.paged_attention(q, k_cache=shifted, v_cache=v_cache, **step, **rest)
    want = refs.paged_attention(q.double(), k_cache=k_cache.double(), v_cache=v_cache.double(), accumulate=torch.float64, **step, **rest)
    torch.testing.assert_close(got.double(), want.double(), **NEAR)
