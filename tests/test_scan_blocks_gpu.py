"""The recurrences in blocks of 64 tokens on the matrix cores, around their tiles' edges, against the token-by-token reference."""
import pytest
import torch

import kernel_refs as refs

pytestmark = pytest.mark.gpu


@pytest.fixture(scope='module')
def ops():
    from qil_amd import ops
    ops.library.load()
    return ops


# Heads' sizes: the kernels' three dims, one to four and six column tiles of 64 (four, two or one a block).  Lengths: a block of
# one token, whole blocks, halves of a block (32), one more and one less; two sequences, the second begun elsewhere.
@pytest.mark.parametrize('dtype', [torch.float32, torch.bfloat16])
@pytest.mark.parametrize('mode', ['decay', 'mlstm'])
@pytest.mark.parametrize('dim, vdim', [(64, 64), (128, 256), (256, 128), (64, 192), (128, 384)])
@pytest.mark.parametrize('counts', [(32, 1), (33, 64), (129, 95)])
@pytest.mark.parametrize('shift', [0, 1])
def test_blocks_of_tokens_on_the_matrix_cores(ops, dtype, mode, dim, vdim, counts, shift):
    """``shift`` 1 puts every row's values on odd columns: pairs are not aligned, the general kernels take the step."""
    heads, n, rot = 2, sum(counts), dim // 2
    g = torch.Generator().manual_seed(dim + vdim + n)
    proj = torch.randn(n, 2 * heads * dim + heads * vdim + 2 * shift, generator=g).to(dtype)
    where = dict(heads=heads, dim=dim, vdim=vdim, q_offset=0, k_offset=heads * dim, v_offset=2 * heads * dim + shift)
    slot = refs.state_scan_slot(heads=heads, dim=dim, vdim=vdim, mode=mode)
    state = torch.randn(3, slot, generator=g)
    index = dict(cu_seqlens=torch.tensor([0, counts[0], n], dtype=torch.int32), seq_starts=torch.tensor([0, 70], dtype=torch.int32),
                 seq_slots=torch.tensor([2, 0], dtype=torch.int32))
    extra = dict(frequencies=torch.tensor([50.0 ** (-2 * i / rot) for i in range(rot // 2)]), rot=rot, q_scale=0.9, k_scale=dim ** -0.5)
    if mode == 'mlstm':
        tiles, mats = -(-vdim // 16), heads * dim * vdim
        tops = state[:, mats + heads * dim:].view(3, heads, tiles + 1)
        tops[:] = tops[:, :, :1].clone()
        extra.update(gates=torch.randn(n, 2 * heads, generator=g) * 3, gate_bias=torch.randn(2 * heads, generator=g), cap=6.0)
    else:
        extra.update(decay=torch.tensor([0.9, 0.999]))
    on = lambda values: {k: v.cuda() if isinstance(v, torch.Tensor) else v for k, v in values.items()}
    got_state, want_state = state.cuda(), state.clone()
    want = refs.state_scan(proj, mode=mode, state=want_state, n_seqs=2, **where, **index, **extra)
    got = ops.state_scan(proj.cuda(), mode=mode, state=got_state, n_seqs=2, max_query=max(counts), **where, **on(index), **on(extra))
    # every result is a float32 sum of at most 256 (state rows) + 129 (keys) terms, made in another order: 2^-24 sqrt(385) = 1.2e-6
    # of the largest partial sums on average, ten times that for the worst of 1e5 elements; the reference's own walk, which rounds
    # the state once a token, is as far off
    for a, b in ((got[0], want[0]), (got[1], want[1]), (got_state[[0, 2]], want_state[[0, 2]])):
        if b is not None:
            torch.testing.assert_close(a.cpu(), b, atol=2.4e-5 * max(1.0, b.abs().max().item()), rtol=2.4e-5)
    assert torch.equal(got_state[1].cpu(), state[1])


# one, two and four pieces a lane, whole and not, a head's size and an offset that four elements do not divide (general kernel)
@pytest.mark.parametrize('dtype', [torch.float32, torch.bfloat16])
@pytest.mark.parametrize('vdim', [4, 252, 256, 260, 512, 1020, 1024, 1028, 130])
@pytest.mark.parametrize('offset', [0, 8, 2])
def test_head_norms_and_gates_of_every_width(ops, dtype, vdim, offset):
    n, heads = 5, 3                                              # 15 heads: the last block of four waves is not full
    g = torch.Generator().manual_seed(vdim)
    o = torch.randn(n, heads * vdim, generator=g) * 5
    source = torch.randn(n, offset + heads * vdim + 4, generator=g).to(dtype)
    weight, below = 1 + 0.3 * torch.randn(heads * vdim, generator=g), torch.rand(n, heads, generator=g) + 0.1
    for gate, w, b in (('sigmoid', weight, below), ('silu', None, None)):
        got = ops.head_norm_gate(o.cuda(), source.cuda(), gate_offset=offset, heads=heads, vdim=vdim, eps=1e-5, gate=gate, out_dtype=dtype,
                                 weight=None if w is None else w.cuda(), denominators=None if b is None else b.cuda())
        v = o.double().view(n, heads, vdim) / (1 if b is None else b.double()[..., None])
        v = (v / (v.square().mean(-1, keepdim=True) + 1e-5).sqrt()).reshape(n, -1) * (1 if w is None else w.double())
        z = source[:, offset:offset + heads * vdim].double()
        want = v * torch.sigmoid(z) * (z if gate == 'silu' else 1)
        # a sum of vdim squares and a handful of roundings in float32, then one to the type
        torch.testing.assert_close(got.double().cpu(), want, atol=1e-6, rtol=2e-6 if dtype == torch.float32 else 2.0 ** -8)


# one row group's last row and beyond (16 groups), whole and odd sizes of a head, one and several blocks of 64 columns; sequences that
# begin, continue and share nothing; a state that holds NaN where a sequence begins
@pytest.mark.parametrize('dtype', [torch.float32, torch.bfloat16])
@pytest.mark.parametrize('mode', ['decay', 'channel'])
@pytest.mark.parametrize('dim, vdim, rot', [(1, 64, 0), (17, 64, 16), (64, 128, 64), (128, 256, 128), (130, 64, 2), (256, 192, 128)])
def test_one_token_a_sequence(ops, dtype, mode, dim, vdim, rot):
    heads, n = 3, 5
    g = torch.Generator().manual_seed(dim + vdim)
    pad = -(heads * dim * 2) % 4                                  # the values' columns begin at a multiple of four elements
    proj = torch.randn(n, 2 * heads * dim + pad + heads * vdim + (-(2 * heads * dim + pad + heads * vdim)) % 4, generator=g).to(dtype)
    where = dict(heads=heads, dim=dim, vdim=vdim, q_offset=0, k_offset=heads * dim, v_offset=2 * heads * dim + pad)
    state = torch.randn(7, heads * dim * vdim, generator=g)
    state[3] = float('nan')                                      # the slot of a sequence that begins
    index = dict(cu_seqlens=torch.arange(n + 1, dtype=torch.int32), seq_starts=torch.tensor([5, 0, 1000, 31, 7], dtype=torch.int32),
                 seq_slots=torch.tensor([6, 3, 0, 1, 4], dtype=torch.int32))
    extra = dict(frequencies=torch.tensor([50.0 ** (-2 * i / max(rot, 2)) for i in range(rot // 2)]) if rot else None, rot=rot,
                 q_scale=0.9, k_scale=dim ** -0.5)
    extra.update(dict(decay=torch.tensor([0.9, 0.999, 0.5])) if mode == 'decay' else dict(gates=torch.randn(n, heads * dim, generator=g), cap=4.0))
    on = lambda values: {k: v.cuda() if isinstance(v, torch.Tensor) else v for k, v in values.items()}
    got_state, want_state = state.cuda(), state.clone()
    takes = ops.library.load().qil_state_token_takes
    moved = proj.cuda()
    assert takes(moved.data_ptr(), got_state.data_ptr(), int(dtype == torch.bfloat16), proj.shape[1], where['v_offset'], dim, vdim, rot,
                 ops.SCAN_MODES[mode])
    want, _ = refs.state_scan(proj, mode=mode, state=want_state, n_seqs=n, **where, **index, **extra)
    got, below = ops.state_scan(moved, mode=mode, state=got_state, n_seqs=n, max_query=1, **where, **on(index), **on(extra))
    assert below is None
    # a state element is one product and one sum, a result a float32 sum of ``dim`` products; positions of 1,000 turn by angles that
    # float32 holds to 6e-5
    for a, b in ((got.cpu(), want), (got_state[index['seq_slots'].long()].cpu(), want_state[index['seq_slots'].long()])):
        torch.testing.assert_close(a, b, atol=1e-4 * max(1.0, b.abs().max().item()), rtol=2e-5)
    assert torch.equal(got_state[[2, 5]].cpu(), state[[2, 5]])


# on both sides of where a wave takes a head: heads of 76 and 80 elements, and 1,534 and 1,536 heads of 768
@pytest.mark.parametrize('n,heads,vdim', [(5, 3, 76), (5, 3, 80), (767, 2, 768), (768, 2, 768), (3, 2, 1024), (600, 4, 64)])
def test_head_norms_where_their_form_changes(ops, n, heads, vdim):
    g = torch.Generator().manual_seed(vdim)
    o, source = torch.randn(n, heads * vdim, generator=g).cuda(), torch.randn(n, 8 + heads * vdim, generator=g).bfloat16().cuda()
    weight = (1 + 0.2 * torch.randn(heads * vdim, generator=g)).cuda()
    got = ops.head_norm_gate(o, source, gate_offset=8, heads=heads, vdim=vdim, weight=weight, eps=1e-5, gate='silu', out_dtype=torch.bfloat16)
    x, z = o.double().view(n, heads, vdim), source[:, 8:].double()
    want = (x / (x.square().mean(-1, keepdim=True) + 1e-5).sqrt()).view(n, -1) * weight.double() * z * torch.sigmoid(z)
    torch.testing.assert_close(got.double(), want, atol=1e-6, rtol=2.0 ** -8 + 1e-5)      # float32, then one rounding to bfloat16
