"""The decode attention's plan: rows of different lengths cut into parts of one size that the GPU chooses."""
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


# one long row beside short ones, rows at the edges of steps and parts, more rows than lanes of a wave, a part a row
@pytest.mark.parametrize('lengths,blocks', [([5000, 1, 33, 257], 32), ([1], 2), ([31, 32, 33, 64, 65], 5), ([2049] * 8, 32),
                                            ([37 * i % 900 + 1 for i in range(100)], 128), ([513, 4096], 3)])
def test_a_plan_covers_every_key_once(ops, lengths, blocks):
    """The smallest part (a multiple of 32 keys, 256 at least) with which all rows fit the blocks, restated on the host."""
    positions = torch.tensor([n - 1 for n in lengths], dtype=torch.int32).cuda()
    plan = torch.full((1 + blocks,), 12345, dtype=torch.int32, device='cuda')
    stream = torch.cuda.current_stream().cuda_stream
    assert ops.library.load().qil_attn_plan(positions.data_ptr(), None, len(lengths), blocks, 256, plan.data_ptr(), stream) == 0
    size, *jobs = plan.tolist()
    cut = lambda part: sum(-(-n // part) for n in lengths)
    assert size % 32 == 0 and size >= 256 and cut(size) <= blocks and (size == 256 or cut(size - 32) > blocks)
    want = [row << 16 | part for row, n in enumerate(lengths) for part in range(-(-n // size))]
    assert jobs == want + [-1] * (blocks - len(want))
    assert ops.library.load().qil_attn_plan(positions.data_ptr(), None, len(lengths), len(lengths) - 1, 256, plan.data_ptr(),
                                            stream) == -1                      # a row needs a block


@pytest.mark.parametrize('lengths', [[3000, 1, 255, 256, 257], [700, 90], [2049] * 4])
@pytest.mark.parametrize('d,heads,kv_heads,page_size', [(128, 32, 8, 16), (64, 16, 8, 8)])
def test_planned_attention(ops, monkeypatch, lengths, d, heads, kv_heads, page_size):
    """With a plan: the row kernel's task alone (merged, and merged by the product behind it) and the kernel that makes its
    queries itself, against the float32 reference; one rounding to bfloat16 and its neighbour (2^-7), values of size one."""
    monkeypatch.setattr(ops, 'PLAN_FEWEST_KEYS', 1)
    dtype, rows = torch.bfloat16, len(lengths)
    k_cache, v_cache, table, _ = build_cache(lengths, page_size, kv_heads, d, dtype)
    positions = torch.tensor([n - 1 for n in lengths], dtype=torch.int32).cuda()
    row_seq = torch.arange(rows, dtype=torch.int32).cuda()
    sizes = dict(heads=heads, kv_heads=kv_heads, head_dim=d)
    step = dict(page_size=page_size, block_tables=table, row_seq=row_seq, positions=positions, max_context=max(lengths),
                scale=d ** -0.5, window=None, **sizes)
    rest = dict(cu_seqlens=None, seq_starts=None, single_rows=None, n_seqs=rows, max_query=1)
    slots = (table[row_seq.long(), (positions // page_size).long()] * page_size + positions % page_size).to(torch.int32)
    qkv = ops.Partials(rand(2, rows, (heads + 2 * kv_heads) * d, scale=0.7, seed=21))
    norms = dict(q_weight=(1 + 0.1 * rand(d, seed=22)), k_weight=(1 + 0.1 * rand(d, seed=23)), eps=1e-6,
                 rotation=Rot(d, 10000.0, max(lengths), d))
    k_fused, v_fused = k_cache.clone(), v_cache.clone()
    plans = {}
    fused = ops.decode_attention(qkv, writes=True, k_cache=k_fused, v_cache=v_fused, unmerged=True, plans=plans, **norms, **step)
    assert len(plans) == 1 and isinstance(fused, ops.Unmerged) and fused.part == 0
    q = ops.qk_norm_rope_store(qkv, positions=positions, slots=slots, k_cache=k_cache, v_cache=v_cache, page_size=page_size,
                               dtype=dtype, **norms, **sizes)
    want = refs.paged_attention(q, k_cache=k_cache, v_cache=v_cache, **step, **rest).float()
    alone = ops.paged_attention(q, k_cache=k_cache, v_cache=v_cache, plans=plans, **step, **rest)
    lazy = ops.paged_attention(q, k_cache=k_cache, v_cache=v_cache, plans=plans, unmerged=True, **step, **rest)
    w = rand(256, heads * d, dtype=dtype, seed=4, scale=(heads * d) ** -0.5)
    product = ops.linear(lazy, w, partials=True)
    for got in (alone, fused.merge()):
        torch.testing.assert_close(got.float(), want, atol=2.0 ** -8, rtol=2.0 ** -7)
    assert torch.equal(alone, fused.merge()) and len(plans) == 1
    if isinstance(product, ops.Partials):
        torch.testing.assert_close(product.sum(), alone.float() @ w.float().t(), atol=2e-5, rtol=1e-4)


def test_no_plan_behind_a_window_or_for_many_rows(ops):
    assert ops._decode_shares(8, 8, 9000, 512, None, None, {})[3] is None
    assert ops._decode_shares(17, 8, 9000, 0, None, None, {})[3] is None       # 32 blocks a kv head: fewer than two a row
    assert ops._decode_shares(1, 8, 40000, 0, None, None, {})[3] is None       # one row: the context's bucket says enough
    assert ops._decode_shares(8, 8, 2048, 0, None, None, {})[3] is None        # few keys
