"""The recurrence with a step size per head in blocks of 128 tokens, which pass through LDS 64 at a time: sequences that end at, one
before and one after a half and a block, heads that fill no tile, and values that are no numbers in a neighbour."""
import pytest
import torch

import kernel_refs as refs
from qil_amd import ops
from test_dogozen_kernels_gpu import ints

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('raw', ['bfloat16', 'float32', 'three splits'])
@pytest.mark.parametrize('dim,vdim', [(128, 64), (8, 8), (72, 72), (256, 136)])
def test_sequences_that_end_at_halves_and_blocks(dim, vdim, raw):
    heads, groups, lengths = 2, 1, [63, 64, 65, 40, 127, 128, 129, 192, 193]
    g = torch.Generator().manual_seed(dim + vdim)
    n, inner = sum(lengths), heads * vdim
    cu = [sum(lengths[:i]) for i in range(len(lengths) + 1)]
    u = (torch.randn(n, inner + 2 * dim, generator=g) / dim ** 0.25).to(torch.bfloat16)
    u[cu[3]:cu[4]] = float('nan')                          # a neighbour that holds no numbers
    steps = torch.randn(3 if raw == 'three splits' else 1, n, heads, generator=g)
    steps = ops.Partials(steps) if raw == 'three splits' else steps[0].to(getattr(torch, raw))
    bias, rates = torch.randn(heads, generator=g), -torch.exp(torch.randn(heads, generator=g) - 2)
    state = torch.randn(len(lengths), heads * dim * vdim, generator=g)
    starts = [0 if i % 2 else 5 for i in range(len(lengths))]
    columns = dict(mode='step', heads=heads, dim=dim, vdim=vdim, groups=groups, v_offset=0, k_offset=inner, q_offset=inner + dim)
    index = dict(cu_seqlens=ints(cu), seq_starts=ints(starts), seq_slots=ints(range(len(lengths))))
    want_state, got_state = state.clone(), state.cuda()
    want, _ = refs.state_scan(u, gates=steps, gate_bias=bias, decay=rates, state=want_state, n_seqs=len(lengths), **index, **columns)
    on_gpu = ops.Partials(steps.tensor.cuda()) if raw == 'three splits' else steps.cuda()
    got, _ = ops.state_scan(u.cuda(), gates=on_gpu, gate_bias=bias.cuda(), decay=rates.cuda(), state=got_state,
                            n_seqs=len(lengths), max_query=max(lengths), **{k: v.cuda() for k, v in index.items()}, **columns)
    for i in range(len(lengths)):
        if i == 3:
            continue
        rows = slice(cu[i], cu[i + 1])
        scale = max(1.0, want[rows].abs().max().item())    # float32 sums in another order, up to dim + 193 terms
        torch.testing.assert_close(got[rows].cpu(), want[rows], atol=2e-5 * scale, rtol=2e-5)
        torch.testing.assert_close(got_state[i].cpu(), want_state[i], atol=2e-5 * scale, rtol=2e-5)
