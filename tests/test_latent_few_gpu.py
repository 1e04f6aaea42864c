"""Latent attention's kernels around their tiles' edges: the product per head of few rows with the rotated parts beside it, the
preparation with the row in registers, the single rows' queries and the merge of the keys' parts, each against float64."""
import pytest
import torch

import kernel_refs as refs

pytestmark = pytest.mark.gpu


@pytest.fixture(scope='module')
def ops():
    from qil_amd import ops
    ops.library.load()
    return ops


def rand(*shape, dtype=torch.float32, scale=1.0, seed=0):
    g = torch.Generator().manual_seed(seed + sum(shape))
    return (torch.randn(*shape, generator=g) * scale).to(dtype).cuda()


def near_sum(got, want, terms, dtype=torch.float32):
    """A float32 sum of ``terms`` products of N(0, 1) values: within 2^-24 sqrt(terms) of each of its ``terms`` partial sums (an
    ample 4e-7 terms^0.5 of the size sqrt(terms)), then one rounding to ``dtype``."""
    torch.testing.assert_close(got.double(), want, atol=4e-7 * terms, rtol=2.0 ** -8 if dtype == torch.bfloat16 else 1e-6)


# rows around the block's 8 and the kernel's last, k around its steps (32, 64 a load; 256, 512 a turn) and of odd length, outputs
# that do not fill a block, few and many blocks (32 or 64 outputs)
@pytest.mark.parametrize('n', [1, 8, 9, 32, 33, 255])
@pytest.mark.parametrize('heads,k,o', [(1, 1, 8), (2, 33, 24), (3, 130, 72), (16, 512, 128), (16, 128, 512), (2, 1025, 40)])
@pytest.mark.parametrize('kind', ['float32', 'bfloat16', 'gated'])
def test_products_per_head(ops, n, heads, k, o, kind):
    dtype = torch.float32 if kind == 'float32' else torch.bfloat16
    x, w = rand(n, heads * (k + 3)), rand(heads, k, o, dtype=dtype, seed=1)       # (inputs behind a head's k are not read)
    gate = rand(n, heads * o, seed=2).to(dtype) if kind == 'gated' else None
    want = torch.einsum('nhk,hko->nho', x.double().view(n, heads, -1)[..., :k], w.double()).reshape(n, -1)
    if gate is not None:
        want *= torch.sigmoid(gate.double())
    near_sum(ops.head_product(x, w, heads=heads, out_dtype=dtype, gate=gate), want, k, dtype)


@pytest.mark.parametrize('n', [1, 9, 32, 33, 256])
@pytest.mark.parametrize('heads,dim,rot,rank', [(1, 12, 2, 8), (5, 33, 6, 40), (16, 128, 64, 512), (3, 64, 130, 20)])
@pytest.mark.parametrize('dtype', [torch.float32, torch.bfloat16])
def test_queries_in_the_latents_space(ops, n, heads, dim, rot, rank, dtype):
    """The turned parts: an angle of up to 3,000 times a float32 frequency is off by 3,000 * 2^-24, two terms of size 4."""
    if n == 256 and dtype == torch.bfloat16:
        pytest.skip('the batched product of the GPU BLAS rounds its result to bfloat16')
    q, k_up = rand(n, heads * (dim + rot), dtype=dtype), rand(heads, dim, rank, dtype=dtype, seed=1)
    freq = torch.tensor([500.0 ** (-2 * i / rot) for i in range(rot // 2)], dtype=torch.float32).cuda()
    positions = (torch.arange(n, dtype=torch.int32) * 37 % 3000).cuda()
    got = ops.latent_query(q, k_up, heads=heads, dim=dim, rot=rot, rank=rank, frequencies=freq, positions=positions)
    got, x = got.view(n, heads, rank + rot), q.double().view(n, heads, -1)
    near_sum(got[..., :rank], torch.einsum('nhk,hko->nho', x[..., :dim], k_up.double()), dim)
    angle = (positions.double()[:, None] * freq.double())[:, None]
    u, v = x[..., dim:dim + rot // 2], x[..., dim + rot // 2:]
    want = torch.cat([u * angle.cos() - v * angle.sin(), v * angle.cos() + u * angle.sin()], -1)
    torch.testing.assert_close(got[..., rank:].double(), want, atol=8 * 3000 * 2.0 ** -24, rtol=1e-5)


# quads a thread: 1, 2 and 4 turns and the last that fit (256 threads take 1,024 quads), sizes beyond them and sizes that are no
# multiple of four (the kernel that reads element by element); rows on both sides of 64
@pytest.mark.parametrize('n', [1, 64, 65])
@pytest.mark.parametrize('q_rank,rank,rot,gates', [(4, 4, 4, 0), (1536, 512, 64, 0), (1536, 512, 64, 16), (2044, 2048, 8, 3),
                                                   (4096, 4096, 4, 0), (8196, 4, 4, 0), (30, 20, 6, 5), (256, 768, 4, 4)])
@pytest.mark.parametrize('kind', ['float32', 'bfloat16', 'partials'])
def test_preparation_of_latents(ops, n, q_rank, rank, rot, gates, kind):
    dtype, total = torch.float32 if kind == 'float32' else torch.bfloat16, q_rank + rank + rot + gates
    pad = -total % 4                                                     # rows of whole quads, as a stacked product has them
    down = rand(5, n, total + pad) if kind == 'partials' else rand(1, n, total + pad, dtype=dtype)
    value = down.double().sum(0)[:, :total]
    operand = ops.columns(ops.Partials(down) if kind == 'partials' else down[0], 0, total)
    wq, wc = 1 + 0.2 * rand(q_rank, seed=1), 1 + 0.2 * rand(rank, seed=2)
    freq = torch.tensor([300.0 ** (-2 * i / rot) for i in range(rot // 2)], dtype=torch.float32).cuda()
    positions = (torch.arange(n, dtype=torch.int32) * 41 % 2000).cuda()
    slots = (torch.arange(n, dtype=torch.int32) * 3).cuda()
    latent, rope = (torch.full((3 * n, 1, size), 7.0, dtype=dtype, device='cuda') for size in (rank, rot))
    copies = tuple(torch.full((n + 5, size), 7.0, dtype=dtype, device='cuda') for size in (rank, rot))
    got = ops.latent_prepare(operand, q_rank=q_rank, rank=rank, rot=rot, q_weight=wq, c_weight=wc, eps=1e-5, frequencies=freq,
                             positions=positions, slots=slots, latent=latent, rope=rope, dtype=dtype, gates=gates, copies=copies)
    got, gate = got if gates else (got, None)

    def norm(x, weight):
        return x / torch.sqrt(x.square().mean(-1, keepdim=True) + 1e-5) * weight.double()

    close = dict(atol=1e-5, rtol=2e-5) if dtype == torch.float32 else dict(atol=1e-4, rtol=2.0 ** -8)
    angle = positions.double()[:, None] * freq.double()
    u, v = value[:, q_rank + rank:][:, :rot // 2], value[:, q_rank + rank + rot // 2:][:, :rot // 2]
    turned = torch.cat([u * angle.cos() - v * angle.sin(), v * angle.cos() + u * angle.sin()], -1)
    c = norm(value[:, q_rank:q_rank + rank], wc)
    torch.testing.assert_close(got.double(), norm(value[:, :q_rank], wq), **close)
    torch.testing.assert_close(latent[slots.long(), 0].double(), c, **close)
    torch.testing.assert_close(rope[slots.long(), 0].double(), turned, atol=2e-3, rtol=close['rtol'])
    assert torch.equal(copies[0][:n], latent[slots.long(), 0]) and torch.equal(copies[1][:n], rope[slots.long(), 0])
    assert not copies[0][n:].any() and not copies[1][n:].any()
    others = torch.ones(3 * n, dtype=torch.bool)
    others[slots.long().cpu()] = False
    assert (latent[others.cuda()] == 7).all() and (rope[others.cuda()] == 7).all()
    if gates:
        torch.testing.assert_close(gate.double(), torch.sigmoid(value[:, -gates:]), atol=1e-6, rtol=1e-5)


# single rows of different lengths, keys in parts of their own or the plan's; heads that do not fill a block's 16 columns, sizes
# that are the template's (512 + 64) and smaller ones, a merge of one element group a part and of several
@pytest.mark.parametrize('heads,rank,rot', [(16, 512, 64), (5, 512, 64), (17, 512, 64), (3, 16, 8), (16, 208, 24), (4, 128, 8), (2, 496, 128)])
@pytest.mark.parametrize('key_parts', [None, (32, 1), (64, 40), (4096, 1)])
@pytest.mark.parametrize('window', [None, 70])
def test_single_rows_over_latents(ops, monkeypatch, heads, rank, rot, key_parts, window):
    """bfloat16 queries, probabilities and latents: eight bits each, an average over many keys."""
    monkeypatch.setattr(ops, 'LATENT_KEY_PARTS', key_parts)
    lengths, page = [1, 31, 32, 33, 64, 65, 700, 1283], 16
    n, pages = len(lengths), -(-max(lengths) // page)
    latent, rope = rand(n * pages, page, rank, dtype=torch.bfloat16), rand(n * pages, page, rot, dtype=torch.bfloat16, seed=1)
    tables = torch.randperm(n * pages, generator=torch.Generator().manual_seed(5)).to(torch.int32).view(n, pages)
    q = rand(n, heads * (rank + rot), seed=2)
    positions = torch.tensor(lengths, dtype=torch.int32) - 1
    cu, sink, gate = torch.arange(n + 1, dtype=torch.int32), rand(heads, seed=3), torch.rand(n, heads).cuda()
    plain = dict(page_size=page, scale=(rank + rot) ** -0.5, heads=heads, rank=rank, rot=rot, window=window)
    want = refs.latent_attention(q.cpu().to(torch.bfloat16).float(), latent=latent.cpu(), rope=rope.cpu(), block_tables=tables,
                                 row_seq=cu[:n], positions=positions, sink=sink.cpu(), gate=gate.cpu(), **plain)
    got = ops.latent_attention(q, latent=latent, rope=rope, block_tables=tables.cuda(), row_seq=cu[:n].cuda(),
                               positions=positions.cuda(), sink=sink, gate=gate, cu_seqlens=cu.cuda(),
                               seq_starts=positions.cuda(), n_seqs=n, max_query=1, max_context=max(lengths), **plain)
    torch.testing.assert_close(got.cpu(), want, atol=1e-2, rtol=1e-2)


# sizes that fill the template of 512 + 64 dims and sizes that end short of it, whose last dims are padding: what lies behind a
# query (the next head's, or nothing behind the last) and behind a key (its first dims stand in) must not reach a score
@pytest.mark.parametrize('heads,rank,rot', [(3, 512, 40), (16, 512, 48), (5, 512, 56), (5, 512, 64), (2, 496, 72)])
@pytest.mark.parametrize('rows', [(1, 1, 1, 1), (41, 1, 67, 3)])
@pytest.mark.parametrize('key_parts', [None, (64, 1), (32, 4)])
def test_dims_behind_a_row_stay_out_of_the_scores(ops, monkeypatch, heads, rank, rot, rows, key_parts):
    """Queries whose heads differ a hundredfold, so that a neighbour's dims would outweigh every score.  bfloat16 queries,
    probabilities and latents: eight bits each."""
    monkeypatch.setattr(ops, 'LATENT_KEY_PARTS', key_parts)
    starts, page = [50, 0, 31, 64], 16
    n, n_seqs, most = sum(rows), len(rows), max(a + b for a, b in zip(starts, rows))
    pages = -(-most // page)
    latent, rope = rand(n_seqs * pages, page, rank, dtype=torch.bfloat16), rand(n_seqs * pages, page, rot, dtype=torch.bfloat16, seed=1)
    tables = torch.randperm(n_seqs * pages, generator=torch.Generator().manual_seed(5)).to(torch.int32).view(n_seqs, pages)
    size = torch.tensor([1.0, 100.0]).repeat(heads)[:heads].repeat_interleave(rank + rot).cuda()
    q = rand(n, heads * (rank + rot), seed=2) * size
    positions = torch.tensor([a + i for a, b in zip(starts, rows) for i in range(b)], dtype=torch.int32)
    row_seq = torch.tensor([s for s, b in enumerate(rows) for _ in range(b)], dtype=torch.int32)
    cu = torch.tensor([sum(rows[:s]) for s in range(n_seqs + 1)], dtype=torch.int32)
    plain = dict(page_size=page, scale=(rank + rot) ** -0.5, heads=heads, rank=rank, rot=rot)
    want = refs.latent_attention(q.cpu().to(torch.bfloat16).float(), latent=latent.cpu(), rope=rope.cpu(), block_tables=tables,
                                 row_seq=row_seq, positions=positions, sink=None, **plain)
    got = ops.latent_attention(q, latent=latent, rope=rope, block_tables=tables.cuda(), row_seq=row_seq.cuda(),
                               positions=positions.cuda(), sink=None, cu_seqlens=cu.cuda(),
                               seq_starts=torch.tensor(starts, dtype=torch.int32).cuda(), n_seqs=n_seqs, max_query=max(rows),
                               max_context=most, **plain)
    small = slice(None, None, 2)                             # (the large heads' softmax hangs on a score's last bits)
    got, want = (v.view(n, heads, rank)[:, small] for v in (got.cpu(), want))
    torch.testing.assert_close(got, want, atol=1e-2, rtol=1e-2)


# on both sides of where the few-row product per head ends with a short k: by blocks (24 k - 768 of 64 outputs for eight rows) and rows
@pytest.mark.parametrize('n,heads,k,o', [(33, 2, 16, 64), (40, 4, 64, 64), (96, 16, 64, 256), (104, 16, 64, 256), (32, 16, 32, 256), (33, 3, 33, 24),
                                         (225, 16, 96, 256), (255, 2, 127, 64), (255, 2, 128, 64)])
def test_products_per_head_where_their_form_changes(ops, n, heads, k, o):
    x, w = rand(n, heads * k), rand(heads, k, o, dtype=torch.bfloat16, seed=1)
    want = torch.einsum('nhk,hko->nho', x.double().view(n, heads, k), w.double()).reshape(n, -1)
    near_sum(ops.head_product(x, w, heads=heads, out_dtype=torch.bfloat16), want, k, torch.bfloat16)
