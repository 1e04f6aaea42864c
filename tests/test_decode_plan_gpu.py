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


@pytest.mark.parametrize('order', [[0, 1, 2, 3], [2, 0, 3, 1]])
def test_planned_rows_beside_a_portion(ops, monkeypatch, order):
    """Single rows behind the seven rows of a portion, listed in any order: plan, partial results and merge go through the
    list.  The bound is that of ``test_planned_attention``."""
    monkeypatch.setattr(ops, 'PLAN_FEWEST_KEYS', 1)
    dtype, d, heads, kv_heads, page_size, portion = torch.bfloat16, 64, 8, 2, 8, 7
    lengths = [40, 2500, 1, 300, 257]                        # the portion's sequence first
    k_cache, v_cache, table, _ = build_cache(lengths, page_size, kv_heads, d, dtype)
    ints = lambda values: torch.tensor(values, dtype=torch.int32).cuda()
    positions = ints(list(range(lengths[0] - portion, lengths[0])) + [n - 1 for n in lengths[1:]])
    row_seq = ints([0] * portion + [1, 2, 3, 4])
    q = rand(portion + 4, heads * d, dtype=dtype, seed=5)
    common = dict(heads=heads, kv_heads=kv_heads, head_dim=d, k_cache=k_cache, v_cache=v_cache, page_size=page_size, block_tables=table,
                  row_seq=row_seq, positions=positions, n_seqs=5, max_query=portion, max_context=max(lengths), scale=d ** -0.5, window=None)
    want = refs.paged_attention(q, cu_seqlens=None, seq_starts=None, single_rows=None, **common).float()
    plans = {}
    for _ in range(2):                                       # a second layer reads the same plan
        got = ops.paged_attention(q, cu_seqlens=ints([0, portion, portion + 1, portion + 2, portion + 3, portion + 4]),
                                  seq_starts=ints([lengths[0] - portion] + [n - 1 for n in lengths[1:]]),
                                  single_rows=ints([portion + i for i in order]), tile_seqs=1, plans=plans, **common)
        torch.testing.assert_close(got.float(), want, atol=2.0 ** -8, rtol=2.0 ** -7)
    assert len(plans) == 1


@pytest.mark.parametrize('sinks', [False, True])
@pytest.mark.parametrize('gated', [False, True])
def test_planned_parts_meet_sinks_and_an_output_gate(ops, monkeypatch, sinks, gated):
    """The merges that read a plan's part size: with and without a plan the same sums over keys cut elsewhere, rounded once to
    bfloat16 (2^-7 for its neighbour)."""
    monkeypatch.setattr(ops, 'PLAN_FEWEST_KEYS', 1)
    dtype, d, heads, kv_heads, page_size, lengths = torch.bfloat16, 64, 16, 8, 8, [3000, 5, 700, 257]
    rows = len(lengths)
    k_cache, v_cache, table, _ = build_cache(lengths, page_size, kv_heads, d, dtype)
    positions = torch.tensor([n - 1 for n in lengths], dtype=torch.int32).cuda()
    sink = rand(heads, seed=7, scale=2.0) if sinks else None
    qkv = ops.Partials(rand(2, rows, (heads + 2 * kv_heads) * d, scale=0.7, seed=21))
    gate = rand(rows, heads * d, dtype=dtype, seed=9) if gated else None
    step = dict(heads=heads, kv_heads=kv_heads, head_dim=d, page_size=page_size, block_tables=table,
                row_seq=torch.arange(rows, dtype=torch.int32).cuda(), positions=positions, max_context=max(lengths), scale=d ** -0.5,
                window=None, sinks=sink)
    fused = dict(q_weight=None, k_weight=None, eps=1e-6, rotation=None, writes=True, gate=gate)
    got, cut = [], []
    for plans in (None, {}):
        k, v = k_cache.clone(), v_cache.clone()
        got.append(ops.decode_attention(qkv, k_cache=k, v_cache=v, plans=plans, **fused, **step))
        cut.append(plans)
        q = rand(rows, heads * d, dtype=dtype, seed=11)
        got.append(ops.paged_attention(q, k_cache=k, v_cache=v, cu_seqlens=None, seq_starts=None, single_rows=None, n_seqs=rows,
                                       max_query=1, plans=plans, **step))
    assert len(cut[1]) == 1
    for planned, plain in ((got[2], got[0]), (got[3], got[1])):
        assert planned.dtype == dtype and torch.isfinite(planned.float()).all()
        torch.testing.assert_close(planned.float(), plain.float(), atol=2.0 ** -8, rtol=2.0 ** -7)


def test_a_captured_plan_follows_the_rows_as_they_grow(ops, monkeypatch):
    """Decode steps of four rows replayed from one graph while their lengths move the plan's part size on: the bits of a
    runner that launches its kernels one by one, whose plans are made anew each step, and logits that differ from those
    without plans by bfloat16's roundings only."""
    from qil_amd import Qwen3, ModelRunner
    import plain_qwen3 as plain
    monkeypatch.setattr(ops, 'PLAN_FEWEST_KEYS', 1)
    monkeypatch.setattr(ops, 'PLAN_MIN_PART', 32)
    config = dict(plain.TINY_B, num_attention_heads=8, num_key_value_heads=2, head_dim=64, hidden_size=512, max_position_embeddings=1024)
    monkeypatch.setattr(ops, 'PLAN_BLOCKS', 2 * 12)          # 12 blocks a kv head: 4 rows of up to 512 keys do not fit with parts of 32
    model = Qwen3.from_config(config, seed=3, dtype=torch.bfloat16, device='cuda:0')
    lengths, steps = [150, 90, 60, 30], 45
    tokens = torch.randint(0, config['vocab_size'], (4, 300), generator=torch.Generator().manual_seed(1)).tolist()
    sizes, real = [], ops._decode_shares

    def shares(*args):
        result = real(*args)
        sizes.append(result[3])
        return result

    def run(graphs, eager_sizes=None):
        runner = ModelRunner(model, num_pages=4 * 38, page_size=8, max_requests=4, graphs=True)
        for r in range(4):
            runner.admit(r)
        runner.step([(r, tuple(tokens[r][:n]), ()) for r, n in enumerate(lengths)])
        if not graphs:                                       # (the prompts' step the same in both)
            runner.graphs = None
        out = []
        for i in range(steps):
            out.append(runner.step([(r, (tokens[r][n + i],), (0,)) for r, n in enumerate(lengths)]).clone())
            if eager_sizes is not None:
                assert sizes[-1] is not None
                eager_sizes.append(int(sizes[-1][0]))
        if graphs:
            assert runner.graphs.captures == 1 and runner.graphs.replays == steps
        return torch.stack(out)

    monkeypatch.setattr(ops, '_decode_shares', shares)
    eager_sizes = []
    launched = run(False, eager_sizes)
    assert len(set(eager_sizes)) >= 2, eager_sizes
    assert torch.equal(run(True), launched)
    monkeypatch.setattr(ops, 'PLAN_FEWEST_KEYS', 1 << 40)
    without = run(True)
    assert (launched - without).norm() < 0.02 * without.norm()


def test_no_plan_behind_a_window_or_for_many_rows(ops):
    assert ops._decode_shares(8, 8, 9000, 512, None, None, {})[3] is None
    assert ops._decode_shares(17, 8, 9000, 0, None, None, {})[3] is None       # 32 blocks a kv head: fewer than two a row
    assert ops._decode_shares(1, 8, 40000, 0, None, None, {})[3] is None       # one row: the context's bucket says enough
    assert ops._decode_shares(8, 8, 2048, 0, None, None, {})[3] is None        # few keys
