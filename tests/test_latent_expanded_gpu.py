"""Latent attention of whole prompts over expanded keys and values."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope='module')
def ops():
    from qil_amd import ops
    ops.library.load()
    return ops


# sequences of one row, ending and beginning inside tiles of 64 keys and blocks of 128 rows, alone and side by side
@pytest.mark.parametrize('lengths', [[1], [64, 64], [63, 1, 65, 129], [300, 7, 211], [1000]])
@pytest.mark.parametrize('heads,sinks,gated', [(16, True, False), (3, False, True)])
def test_expanded_attention(ops, lengths, heads, sinks, gated):
    """Against float64.  A neighbour's rows may hold anything: the rows of the last sequence are NaN for all the others, and
    their results are compared with those of a step without it.  Values of size one under weights that sum to one, rounded
    to bfloat16 as the weights are: 2^-8 each."""
    n, padded = sum(lengths), ops.expanded_rows(sum(lengths))
    g = torch.Generator().manual_seed(n + heads)
    rand = lambda *shape: torch.randn(*shape, generator=g).to(torch.bfloat16).cuda()
    q, k, kr, vt = rand(n, heads * 192), rand(padded, heads * 128), rand(padded, 64), rand(heads * 128, padded)
    k[n:], kr[n:], vt[:, n:] = 0, 0, 0
    sink = torch.randn(heads, generator=g).cuda() if sinks else None
    gate = torch.rand(n, heads, generator=g).cuda() if gated else None
    frequencies = (10000.0 ** (-torch.arange(32) / 32.0)).to(torch.float32).cuda()
    ends = torch.tensor([0] + lengths).cumsum(0)
    scale = 192 ** -0.5
    run = lambda q, k, kr, vt: ops.latent_expanded(q, k, kr, vt, heads=heads, cu_seqlens=ends.to(torch.int32).cuda(), frequencies=frequencies,
                                                   sink=sink, gate=gate, scale=scale, n_seqs=len(lengths), max_query=max(lengths))
    got = run(q, k, kr, vt)
    want = torch.empty(n, heads, 128, dtype=torch.float64, device='cuda')
    for a, b in zip(ends[:-1].tolist(), ends[1:].tolist()):
        t = b - a
        angle = torch.arange(t, device='cuda', dtype=torch.float32)[:, None] * frequencies
        cos, sin = angle.double().cos()[:, None], angle.double().sin()[:, None]
        mine = q[a:b].double().view(t, heads, 192)
        u, v = mine[..., 128:160], mine[..., 160:]
        turned = torch.cat([u * cos - v * sin, v * cos + u * sin], -1).to(torch.bfloat16).double()       # as the kernel rounds it
        keys, values = k[a:b].double().view(t, heads, 128), vt[:, a:b].double().view(heads, 128, t)
        for h in range(heads):
            s = (mine[:, h, :128] @ keys[:, h].t() + turned[:, h] @ kr[a:b].double().t()) * scale
            s = s.masked_fill(torch.ones(t, t, dtype=torch.bool, device='cuda').triu(1), float('-inf'))
            if sinks:
                s = torch.cat([s, sink[h].double().expand(t, 1)], 1)
            want[a:b, h] = torch.softmax(s, -1)[:, :t] @ values[h].t()
    if gated:
        want = want * gate.double()[..., None]
    torch.testing.assert_close(got.double().view(n, heads, 128), want, atol=2.0 ** -6, rtol=2.0 ** -7)
    if len(lengths) > 1:
        first = int(ends[-2])
        q, k, kr, vt = (x.clone() for x in (q, k, kr, vt))
        q[first:], k[first:], kr[first:], vt[:, first:] = (float('nan'),) * 4
        assert torch.equal(run(q, k, kr, vt)[:first], got[:first])


def test_the_engine_takes_whole_prompts_to_it(ops, monkeypatch):
    """One step of two whole prompts with and without the expanded path: the caches hold the same bits, and logits that differ
    by bfloat16's roundings only; the second step, behind cached tokens, does not take it."""
    from qil_amd import Qwen3, ModelRunner
    latent = dict(heads=4, dim=128, rot_dim=64, vdim=128, kv_rank=128, q_rank=96, rot=dict(base=10000.0, dims=64), scale=192 ** -0.5)
    config = dict(architecture='Fubapel', vocab=301, width=256, loop=dict(start=0, stop=0, times=1), norm=dict(eps=1e-5), residual_mult=1.0,
                  layers=[dict(type='latent_attention', mlp=dict(kind='dense', ff=512, limit=7.0), mixer=latent)] * 2)
    model = Qwen3.from_config(config, seed=3, dtype=torch.bfloat16, device='cuda:0')
    calls, real = [], ops.latent_expanded
    monkeypatch.setattr(ops, 'latent_expanded', lambda *a, **kw: calls.append(1) or real(*a, **kw))
    tokens = torch.randint(0, 301, (700,), generator=torch.Generator().manual_seed(1)).tolist()

    def steps():
        runner = ModelRunner(model, num_pages=128, max_requests=2)
        runner.admit(0), runner.admit(1)
        first = runner.step([(0, tuple(tokens[:411]), (0, 410)), (1, tuple(tokens[411:]), (288,))])
        counted = len(calls)
        second = runner.step([(0, tuple(tokens[:600]), (599,))])
        assert len(calls) == counted
        return first, second, [group['tensors']['latent'][0].clone() for group in runner.cache.kv_groups]

    first, second, caches = steps()
    assert len(calls) == 2
    monkeypatch.setattr(ops, 'EXPAND_FEWEST_ROWS', 1 << 30)
    plain_first, plain_second, plain_caches = steps()
    assert len(calls) == 2
    used = lambda c: c.view(-1, 128)[:704].view(torch.int16)
    assert all(torch.equal(used(a)[:411], used(b)[:411]) for a, b in zip(caches, plain_caches))
    for a, b in ((first, plain_first), (second, plain_second)):
        assert (a - b).norm() < 0.02 * b.norm()


@pytest.mark.parametrize('change,kept', [({}, True), (dict(gate='head'), True), (dict(dtype=torch.float32), False), (dict(window=64), False),
                                         (dict(gate='element'), False), (dict(dim=64), False), (dict(rot_dim=32), False), (dict(vdim=64), False)])
def test_only_layers_that_may_expand_keep_the_value_weight_twice(ops, change, kept):
    from qil_amd.parts.latent_attention import LatentAttention
    from qil_amd.parts.rotary import RotaryFrequencies
    sizes = dict(width=256, heads=4, dim=128, rot_dim=64, vdim=128, kv_rank=128, q_rank=96, scale=192 ** -0.5, eps=1e-5,
                 dtype=torch.bfloat16) | change
    layer = LatentAttention(position=RotaryFrequencies(rot_dim=sizes['rot_dim'], base=10000.0, device='cuda'), **sizes)
    layer.p = {name: torch.zeros(spec.shape, dtype=sizes['dtype'], device='cuda') for name, spec in layer.param_specs().items()}
    layer.finalize()
    assert (layer.v_rows is not None) == kept
