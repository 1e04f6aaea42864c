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


@pytest.mark.parametrize('moved', ['k', 'v', 'q_weight', 'k_weight', 'bias', 'cos', 'part'])
def test_steps_with_operands_at_other_addresses(ops, monkeypatch, moved):
    """A float32 step of an attention part, one operand beginning between multiples of 16 bytes (or parts of the keys that are
    no whole steps): not the kernel that makes its queries itself, and the same results and cache."""
    from qil_amd.cache.manager import KVView
    from qil_amd.engine.batch import StepContext
    from qil_amd.parts import Attention, Rotary
    heads, kv_heads, d, width, lengths = 4, 2, 64, 512, [33, 200, 1]
    rotary = Rotary(d, 10000.0, 256, device='cuda')
    extended = dict(bias=True, gate=True) if moved == 'bias' else dict(bias=False)
    part = Attention(width=width, heads=heads, kv_heads=kv_heads, head_dim=d, qk_norm_eps=1e-6, scale=d ** -0.5, position=rotary,
                     dtype=torch.float32, **extended)
    for index, (name, spec) in enumerate(part.param_specs().items()):
        part.set_param(name, rand(*spec.shape, scale=spec.shape[-1] ** -0.5, seed=30 + index))
    part.finalize()
    k_cache, v_cache, step, rest = task(lengths, 16, heads, kv_heads, d)
    rows, positions, table = len(lengths), step['positions'], step['block_tables']
    slots = (table[step['row_seq'].long(), (positions // 16).long()] * 16 + positions % 16).to(torch.int32)
    single = dict(cu_seqlens=torch.arange(rows + 1, dtype=torch.int32).cuda(), seq_starts=positions, seq_slots=None, single_rows=None)
    ctx = StepContext(n_tokens=rows, n_seqs=rows, n_logit_rows=0, token_ids=None, positions=positions, row_seq=step['row_seq'],
                      logit_rows=None, max_query=1, max_context=max(lengths), **single)
    h = rand(rows, width, seed=41)
    asked = []
    plain = ops.decode_attention
    monkeypatch.setattr(ops, 'decode_attention', lambda *a, **kw: (asked.append(1), plain(*a, **kw))[1])

    def shifted(tensor):
        return torch.empty(tensor.numel() + 1, dtype=tensor.dtype, device='cuda')[1:].view(tensor.shape).copy_(tensor)

    def attend(k, v):
        view = KVView(k=k, v=v, page_size=16, writes=True, group=0, block_tables=table, slots=slots)
        out = part.forward(h, ctx, view)
        return (out.sum() if isinstance(out, ops.Partials) else out), k, v
    want = attend(k_cache.clone(), v_cache.clone())
    assert asked
    asked.clear()
    k, v = (shifted(c) if moved == name else c.clone() for c, name in ((k_cache, 'k'), (v_cache, 'v')))
    if moved in ('q_weight', 'k_weight'):
        part.p[moved[0] + '_norm.weight'] = shifted(part.p[moved[0] + '_norm.weight'])
    elif moved == 'bias':
        part.b_qkv_own = shifted(part.b_qkv_own)
    elif moved == 'cos':
        rotation = rotary.rotation()
        monkeypatch.setattr(rotary, 'rotation', lambda: type(rotation)(shifted(rotation.cos), rotation.sin, rotation.rot_dim))
    elif moved == 'part':
        monkeypatch.setattr(ops, 'ATTENTION_PART', 48)
    got = attend(k, v)
    assert not asked
    for a, b in zip(got, want):
        torch.testing.assert_close(a, b, equal_nan=True, **NEAR)


# groups of one head on both sides of the lines between the kernels, and parts of every size (64 to 512 keys)
@pytest.mark.parametrize('heads,kv_heads,d,lengths', [(16, 16, 128, [60] * 41), (16, 16, 128, [60, 33] * 21), (4, 4, 64, [2048, 700, 9] * 11),
                                                      (8, 8, 128, [1500] * 62 + [7]), (8, 8, 128, [1500] * 63), (16, 8, 128, [2048, 100, 1999] * 3),
                                                      (4, 1, 64, [9000, 64, 8000])])
def test_rows_alone_where_their_kernel_changes(ops, heads, kv_heads, d, lengths):
    k_cache, v_cache, step, rest = task(lengths, 16, heads, kv_heads, d)
    q = rand(len(lengths), heads * d, seed=5)
    got = ops.paged_attention(q, k_cache=k_cache, v_cache=v_cache, **step, **rest)
    want = refs.paged_attention(q.double(), k_cache=k_cache.double(), v_cache=v_cache.double(), accumulate=torch.float64, **step, **rest)
    torch.testing.assert_close(got.double(), want.double(), **NEAR)
