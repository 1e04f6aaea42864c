"""The step function against the plain whole-sequence implementation, under every way of cutting.

Each test runs three ways: on the CPU with the kernels' plain references substituted (this proves
batches, block tables, slots, row selection and page reuse, not the kernels), and on the GPU with
the HIP kernels in float32 and in bfloat16 (marked ``gpu``).  The cache is filled with NaN first,
so a read of a slot that was never written, or of another request's page, shows.
"""
import random

import pytest
import torch

import plain_qwen3 as plain
from qil_amd.engine import ModelRunner, StepEntry
from qil_amd.weights import load_model

CONFIGS = {'A': (plain.TINY_A, 0, 4), 'B': (plain.TINY_B, 1, 8), 'C': (plain.TINY_C, 2, 3), 'D': (plain.TINY_D, 3, 16),
           'E': (plain.TINY_E, 4, 8)}


def poison(runner):
    for group in runner.cache.kv_groups:
        group['k'].fill_(float('nan'))
        group['v'].fill_(float('nan'))


def tokens_for(config, length, seed):
    r = random.Random(seed)
    return [r.randrange(config['vocab_size']) for _ in range(length)]


# float32: summation orders differ from the CPU's, nothing else.  bfloat16: a few roundings to 8
# bits of logits of size ~1 (the plain implementation with the reference's bfloat16 roundings is
# itself 0.005-0.008 away from float32 on these models).
TOLERANCE = {torch.float32: dict(atol=5e-6, rtol=5e-5), torch.bfloat16: dict(atol=0.015, rtol=0.015)}
BACKENDS = [pytest.param(('cpu', torch.float32), id='cpu-refs'),
            pytest.param(('cuda', torch.float32), id='gpu-f32', marks=pytest.mark.gpu),
            pytest.param(('cuda', torch.bfloat16), id='gpu-bf16', marks=pytest.mark.gpu)]


class Case:
    def __init__(self, config, weights, model, page_size, dtype):
        self.config, self.weights, self.model, self.page_size, self.dtype = config, weights, model, page_size, dtype

    def __iter__(self):
        return iter((self.config, self.weights, self.model, self.page_size))

    def close(self, actual, expected):
        actual = actual.to('cpu')
        assert torch.isfinite(actual).all()
        error = (actual - expected).abs().max().item()
        print(f'max abs error {error:.3e} ({self.dtype})')
        torch.testing.assert_close(actual, expected, **TOLERANCE[self.dtype])


@pytest.fixture(params=BACKENDS)
def backend(request):
    device, dtype = request.param
    if device == 'cpu':
        request.getfixturevalue('cpu_kernels')
    return device, dtype


@pytest.fixture(params=sorted(CONFIGS))
def case(request, model_folder, backend):
    device, dtype = backend
    config, seed, page_size = CONFIGS[request.param]
    folder, weights = model_folder(config, seed)
    model = load_model(folder, dtype=dtype, device=device)
    return Case(config, weights, model, page_size, dtype)


def test_whole_prompt_matches_plain(case):
    config, weights, model, page_size = case
    runner = ModelRunner(model, num_pages=16, page_size=page_size)
    poison(runner)
    tokens = tokens_for(config, 23, 5)
    assert runner.admit('a')
    logits = runner.step([StepEntry('a', tuple(tokens), tuple(range(len(tokens))))])
    case.close(logits, plain.logits(tokens, weights, config))
    runner.release('a')
    runner.cache.check()
    assert runner.cache.free_pages == [16]


@pytest.mark.parametrize('cuts', [[11], [1] * 11, [2, 4, 1, 4], [7, 2, 2]])
def test_portions_match_whole(case, cuts):
    config, weights, model, page_size = case
    runner = ModelRunner(model, num_pages=8, page_size=page_size)
    poison(runner)
    tokens = tokens_for(config, sum(cuts), 9)
    runner.admit(0)
    got, at = [], 0
    for size in cuts:
        got.append(runner.step([StepEntry(0, tuple(tokens[at:at + size]), tuple(range(size)))]))
        at += size
    case.close(torch.cat(got), plain.logits(tokens, weights, config))


def test_mixed_batch_with_page_reuse(case):
    """Up to four live requests, portions beside single tokens, so few pages that they are reused."""
    config, weights, model, page_size = case
    lengths = [19, 7, 26, 12, 9, 15]
    prompts = {i: tokens_for(config, n, 100 + i) for i, n in enumerate(lengths)}
    expected = {i: plain.logits(p, weights, config) for i, p in prompts.items()}
    pages = sum(-(-n // page_size) for n in sorted(lengths)[-4:])
    runner = ModelRunner(model, num_pages=pages, page_size=page_size, max_requests=4)
    poison(runner)
    r = random.Random(3)
    waiting, live, done, used_pages = list(prompts), {}, {}, []
    while waiting or live:
        while waiting and len(live) < 4:
            need = -(-len(prompts[waiting[0]]) // page_size)
            held = sum(-(-len(prompts[i]) // page_size) for i in live)
            if held + need > pages:
                break
            i = waiting.pop(0)
            assert runner.admit(i)
            live[i] = 0
        order = list(live)
        r.shuffle(order)
        entries = []
        for i in order:
            left = len(prompts[i]) - live[i]
            size = 1 if live[i] >= len(prompts[i]) - 3 else min(left, r.choice([2, 3, 5, 8]))
            entries.append(StepEntry(i, tuple(prompts[i][live[i]:live[i] + size]), tuple(range(size))))
        logits = runner.step(entries)
        at = 0
        for entry in entries:
            size = len(entry.tokens)
            done.setdefault(entry.request, []).append(logits[at:at + size])
            at += size
            live[entry.request] += size
            if live[entry.request] == len(prompts[entry.request]):
                used_pages += runner.cache.table(0, entry.request)
                runner.release(entry.request)
                del live[entry.request]
        runner.cache.check()
    assert len(used_pages) > len(set(used_pages)), 'the test must reuse pages'
    for i in prompts:
        case.close(torch.cat(done[i]), expected[i])
    assert runner.cache.free_pages == [pages]


def test_selected_rows_and_nothing_wanted(case):
    config, weights, model, page_size = case
    runner = ModelRunner(model, num_pages=8, page_size=page_size)
    tokens = tokens_for(config, 9, 1)
    runner.admit('x')
    assert runner.step([StepEntry('x', tuple(tokens[:4]), ())]) is None
    logits = runner.step([StepEntry('x', tuple(tokens[4:]), (4, 0))])
    expected = plain.logits(tokens, weights, config)
    case.close(logits, expected[[8, 4]])


def test_requests_with_several_tokens_come_first_and_logits_keep_the_callers_order(case):
    """A step of single tokens and portions in turns: inside, the sequences of several rows are put first (the tile
    kernel gets blocks for them alone), the logits come back in the order of the caller's entries and wants."""
    config, weights, model, page_size = case
    runner = ModelRunner(model, num_pages=64, page_size=page_size)
    poison(runner)
    lengths = {'a': 7, 'b': 12, 'c': 5, 'd': 9, 'e': 3}
    tokens = {r: tokens_for(config, n, seed) for seed, (r, n) in enumerate(lengths.items())}
    expected = {r: plain.logits(t, weights, config) for r, t in tokens.items()}
    for r in lengths:
        runner.admit(r)
    # a, c and e have all but their last token behind them; b and d bring portions
    runner.step([StepEntry(r, tuple(tokens[r][:-1]), ()) for r in 'ace'])
    runner.step([StepEntry('b', tuple(tokens['b'][:4]), ()), StepEntry('d', tuple(tokens['d'][:2]), ())])
    entries = [StepEntry('a', tuple(tokens['a'][-1:]), (0,)), StepEntry('b', tuple(tokens['b'][4:]), (7, 0, 3)),
               StepEntry('c', tuple(tokens['c'][-1:]), ()), StepEntry('d', tuple(tokens['d'][2:]), (6,)),
               StepEntry('e', tuple(tokens['e'][-1:]), (0,))]
    described, ctx = runner.prepare(entries)
    assert [e.request for e in described] == ['b', 'd', 'a', 'c', 'e'] == ctx.requests and ctx.tile_seqs == 2
    assert ctx.single_rows.tolist() == [15, 16, 17] and ctx.logit_rows.tolist() == [15, 7, 0, 3, 14, 17]
    logits = runner.step(entries)
    want = torch.stack([expected['a'][6], expected['b'][11], expected['b'][4], expected['b'][7], expected['d'][8],
                        expected['e'][2]])
    case.close(logits, want)
    assert all(runner.computed(r) == n for r, n in lengths.items())


def test_longest_context_of_the_portions(case):
    """Not that of the rows alone beside them; a graph's description is for any context of its bucket, or for the portions' that it
    is made for."""
    config, weights, model, page_size = case
    runner = ModelRunner(model, num_pages=64, page_size=page_size)
    tokens = {r: tokens_for(config, n, seed) for seed, (r, n) in enumerate({'long': 24, 'b': 11, 'c': 7}.items())}
    for r in tokens:
        runner.admit(r)
    runner.step([StepEntry('long', tuple(tokens['long'][:-1]), ()), StepEntry('b', tuple(tokens['b'][:5]), ())])
    entries = [StepEntry('long', tuple(tokens['long'][-1:]), (0,)), StepEntry('b', tuple(tokens['b'][5:]), ()), StepEntry('c', tuple(tokens['c']), ())]
    described, pieces, facts = runner._describe(entries)
    flat = torch.from_numpy(pieces.flat()).to(model.device)
    context = lambda bucket, portions=None: runner._context(described, pieces, facts, flat, max_context=bucket, tile_context=portions)
    assert (context(None).max_context, context(None).tile_context) == (24, 11)
    assert (context(32).max_context, context(32).tile_context) == (32, None)
    assert (context(32, 7).max_context, context(32, 7).tile_context) == (32, 7)


def test_step_validation(case):
    config, weights, model, page_size = case
    runner = ModelRunner(model, num_pages=2, page_size=page_size)
    runner.admit('a')
    for bad in ([], [StepEntry('a', (), ())], [StepEntry('zz', (1,), ())], [StepEntry('a', (config['vocab_size'],), ())],
                [StepEntry('a', (True,), ())], [StepEntry('a', (1,), (1,))],
                [StepEntry('a', (1,), ()), StepEntry('a', (2,), ())]):
        with pytest.raises(ValueError):
            runner.step(bad)
    from qil_amd.cache import CacheFull
    with pytest.raises(CacheFull):
        runner.step([StepEntry('a', tuple([1] * (2 * page_size + 1)), ())])
    runner.cache.check()


def test_prefill_then_last_32_one_by_one(case):
    config, weights, model, page_size = case
    tokens = tokens_for(config, 75, 21)
    runner = ModelRunner(model, num_pages=-(-75 // page_size), page_size=page_size)
    poison(runner)
    runner.admit('r')
    head = len(tokens) - 32
    got = [runner.step([StepEntry('r', tuple(tokens[:head]), tuple(range(head)))])]
    for t in tokens[head:]:
        got.append(runner.step([StepEntry('r', (t,), (0,))]))
    case.close(torch.cat(got), plain.logits(tokens, weights, config))


def test_first_tokens_of_a_sequence(case):
    config, weights, model, page_size = case
    tokens = tokens_for(config, 3, 33)
    runner = ModelRunner(model, num_pages=2, page_size=page_size)
    poison(runner)
    runner.admit('r')
    got = [runner.step([StepEntry('r', (t,), (0,))]) for t in tokens]
    case.close(torch.cat(got), plain.logits(tokens, weights, config))


def test_long_decoding_crosses_attention_splits(case):
    """Single tokens up to a context longer than one attention split (256 keys)."""
    config, weights, model, page_size = case
    tokens = tokens_for(config, 300, 44)
    runner = ModelRunner(model, num_pages=-(-300 // page_size), page_size=page_size)
    poison(runner)
    runner.admit('r')
    got = [runner.step([StepEntry('r', tuple(tokens[:200]), (199,))])]
    for t in tokens[200:]:
        got.append(runner.step([StepEntry('r', (t,), (0,))]))
    case.close(torch.cat(got), plain.logits(tokens, weights, config)[199:])


def test_which_steps_a_decode_graph_takes(model_folder, cpu_kernels):
    from qil_amd.engine.graphs import DecodeGraphs
    folder, _ = model_folder(plain.TINY_A, 0)
    runner = ModelRunner(load_model(folder, dtype=torch.float32, device='cpu'), num_pages=4, page_size=4)
    graphs = DecodeGraphs(runner)
    assert graphs.takes([StepEntry('a', (1,), (0,)), ('b', [2], [0])])
    assert not graphs.takes([('a', [1])])                       # nothing wanted (the third member may be missing)
    assert not graphs.takes([StepEntry('a', (1, 2), (1,))]) and not graphs.takes([StepEntry('a', (1,), ())])
    assert not graphs.takes([])


def test_which_portions_share_a_graph(model_folder, cpu_kernels, monkeypatch):
    """Beside a decoding row: the portions of a prompt that comes in in several, its first one too, one graph of their sizes,
    captured at their second coming; a whole prompt and another one's last portion of as many tokens one each, planned for the
    prompt's tokens and for any context; every logit against the plain model.  (A graph here is its step, launched again.)"""
    from qil_amd.engine import graphs as graph_module
    planned = []

    class Launched:
        def __init__(self, runner, entries, pieces, facts, bucket, sampler=None, tile_context=None):
            self.runner, self.meta = runner, torch.from_numpy(pieces.flat()).clone()
            self.context = runner._context(entries, pieces, facts, self.meta, max_context=bucket, tile_context=tile_context)
            self.tables = [view.block_tables for view in runner.views], [view.slots for view in runner.views]
            planned.append((tuple(len(e.tokens) for e in entries), tile_context))

        def load(self, pieces):
            self.meta.copy_(torch.from_numpy(pieces.flat()))

        def run(self):
            for view, table, slots in zip(self.runner.views, *self.tables):
                view.block_tables, view.slots = table, slots
            return self.runner.model.forward(self.context, self.runner.views)

    monkeypatch.setattr(graph_module, '_Graph', Launched)
    config = plain.TINY_A
    folder, weights = model_folder(config, 3)
    runner = ModelRunner(load_model(folder, dtype=torch.float32, device='cpu'), num_pages=40, page_size=4)
    poison(runner)
    runner.graphs = graph_module.DecodeGraphs(runner)
    runner.graphs.takes = lambda entries: False
    row, prompt = tokens_for(config, 60, 5), tokens_for(config, 40, 6)
    want_row, want = plain.logits(row, weights, config), plain.logits(prompt, weights, config)
    runner.admit('row')
    runner.step([StepEntry('row', tuple(row[:30]), ())])
    fed, captures = 30, []

    def beside(request, start, count, wanted):
        nonlocal fed
        places = (count - 1,) if wanted else ()
        logits = runner.step([StepEntry(request, tuple(prompt[start:start + count]), places), StepEntry('row', (row[fed],), (0,))])
        rows = [want[start + count - 1]] * wanted + [want_row[fed]]
        torch.testing.assert_close(logits, torch.stack(rows), **TOLERANCE[torch.float32])
        fed += 1
        captures.append(runner.graphs.mixed_captures)

    for request in 'ab':                                    # three portions of 8 and a last one of 8 that wants logits
        runner.admit(request)
        for start in (0, 8, 16):
            beside(request, start, 8, False)
        beside(request, 24, 8, True)
        runner.release(request)
    assert captures == [0, 1, 1, 1, 1, 1, 1, 2] and planned == [((8, 1), None)] * 2
    for request in 'cde':                                   # whole prompts of as many tokens as those last portions
        runner.admit(request)
        beside(request, 0, 8, True)
        runner.release(request)
    assert captures[8:] == [2, 3, 3] and planned[2:] == [((8, 1), 8)] and runner.graphs.mixed_replays == 8
    runner.cache.check()


@pytest.mark.gpu
@pytest.mark.parametrize('dtype', [torch.float32, torch.bfloat16])
def test_graph_replays_equal_eager_launches(model_folder, dtype):
    """Decode steps replayed from a captured HIP graph give bit for bit what eager launches give,
    on every replay, with eager work (a prompt portion of another request) between replays."""
    config, seed, page_size = CONFIGS['B']
    folder, weights = model_folder(config, seed)
    model = load_model(folder, dtype=dtype, device='cuda')
    runners = [ModelRunner(model, num_pages=24, page_size=page_size, graphs=flag) for flag in (True, False)]
    prompts = {r: tokens_for(config, n, 60 + n) for r, n in (('a', 21), ('b', 9), ('c', 40))}
    outputs = [[], []]
    for which, runner in enumerate(runners):
        poison(runner)
        for r in 'ab':
            runner.admit(r)
            runner.step([StepEntry(r, tuple(prompts[r][:5]), ())])
        runner.admit('c')
        fed = {'a': 5, 'b': 5, 'c': 0}
        for turn in range(8):
            batch = [StepEntry(r, (prompts[r][fed[r]],), (0,)) for r in ('b', 'a') if fed[r] < len(prompts[r])]
            outputs[which].append(runner.step(batch))
            for entry in batch:
                fed[entry.request] += 1
            runner.step([StepEntry('c', tuple(prompts['c'][fed['c']:fed['c'] + 3]), ())])     # eager work in between
            fed['c'] += 3
            torch.cuda.synchronize()
    assert runners[0].graphs.replays >= 8 and runners[0].graphs.captures <= 3
    for with_graph, eager in zip(*outputs):
        torch.testing.assert_close(with_graph, eager, atol=0, rtol=0)
    expected = plain.logits(prompts['a'], weights, config)
    got = torch.cat([step[1:2] if step.shape[0] == 2 else step[0:1] for step in outputs[0]])[:8].cpu()
    torch.testing.assert_close(got, expected[5:13], **TOLERANCE[dtype])


@pytest.mark.gpu
@pytest.mark.parametrize('dtype', [torch.float32, torch.bfloat16])
def test_steps_with_portions_replay_a_graph_of_their_shape(model_folder, dtype):
    """A shape of step that comes again (a portion of five tokens beside two decoded tokens, the requests in
    another order every step) runs launch by launch the first time, is captured the second time and replayed
    from then on, with other work between the replays; every step's logits are those of a runner without graphs
    up to the order of sums in attention (the graph cuts the context by its bucket), and the plain model's."""
    config, seed, page_size = CONFIGS['B']
    folder, weights = model_folder(config, seed)
    model = load_model(folder, dtype=dtype, device='cuda')
    prompts = {r: tokens_for(config, n, 70 + n) for r, n in (('p', 60), ('a', 30), ('b', 30), ('other', 25))}
    outputs = []
    for flag in (True, False):
        runner = ModelRunner(model, num_pages=40, page_size=page_size, graphs=flag)
        poison(runner)
        fed = {}
        for r, head in (('p', 4), ('a', 9), ('b', 13), ('other', 2)):
            runner.admit(r)
            runner.step([StepEntry(r, tuple(prompts[r][:head]), ())])
            fed[r] = head
        got = {r: [] for r in 'pab'}
        for turn in range(9):
            order = ['p', 'a', 'b'] if turn % 3 == 0 else ['a', 'p', 'b'] if turn % 3 == 1 else ['b', 'a', 'p']
            entries = [StepEntry(r, tuple(prompts[r][fed[r]:fed[r] + (5 if r == 'p' else 1)]), (4, 0) if r == 'p' else (0,))
                       for r in order]
            logits = runner.step(entries)
            at = 0
            for entry in entries:
                for w in entry.want:
                    got[entry.request].append((fed[entry.request] + w, logits[at].cpu()))
                    at += 1
                fed[entry.request] += len(entry.tokens)
            runner.step([StepEntry('other', tuple(prompts['other'][fed['other']:fed['other'] + 2]), ())])   # other work in between
            fed['other'] += 2
            torch.cuda.synchronize()
        if flag:
            assert runner.graphs.mixed_captures == 2 and runner.graphs.mixed_replays >= 14, \
                (runner.graphs.mixed_captures, runner.graphs.mixed_replays)      # the step's shape and the other work's
        runner.cache.check()
        outputs.append(got)
    for r in 'pab':
        expected = plain.logits(prompts[r], weights, config)
        for (place, with_graph), (same_place, eager) in zip(outputs[0][r], outputs[1][r]):
            assert place == same_place
            torch.testing.assert_close(with_graph, eager, **TOLERANCE[dtype])
            torch.testing.assert_close(with_graph, expected[place], **TOLERANCE[dtype])


HEAD_SIZES = [16, 32, 48, 64, 80, 96, 112, 128, 160, 192, 256]
# every even size is allowed (qil/config.py:29-30); those that are no multiple of 8 are padded by the attention part
EVEN_HEAD_SIZES = [2, 6, 20, 72, 100, 10, 36, 250]


def random_configuration(r, head_sizes=HEAD_SIZES):
    """Every size and option drawn at random: head sizes in steps of 16 up to 256 (or of ``head_sizes``), one to eight
    kv heads with groups of one to sixteen, widths and vocabularies that are no powers of two, biases, tied or own
    head."""
    kv, group = r.choice([1, 1, 2, 2, 3, 4, 5, 8]), r.choice([1, 2, 3, 4, 5, 6, 7, 8, 16])
    return dict(architectures=['Qwen3ForCausalLM'], model_type='qwen3', vocab_size=r.randrange(50, 3000),
                hidden_size=r.choice([2, 4, 8]) * r.randrange(9, 160),
                intermediate_size=r.choice([2, 8, 16]) * r.randrange(5, 90), num_hidden_layers=r.randrange(1, 4),
                num_attention_heads=kv * group, num_key_value_heads=kv,
                head_dim=r.choice(head_sizes), max_position_embeddings=2048,
                rms_norm_eps=r.choice([1e-6, 1e-5, 3e-4]), rope_theta=r.choice([1e4, 5e5, 1e6]),
                attention_bias=r.random() < 0.3, tie_word_embeddings=r.random() < 0.5, hidden_act='silu',
                eos_token_id=None)


@pytest.mark.gpu
@pytest.mark.parametrize('dtype', [torch.float32, torch.bfloat16])
@pytest.mark.parametrize('seed', range(27))
def test_random_configurations_in_mixed_batches(model_folder, seed, dtype):
    """Configurations drawn at random, six short prompts and one of hundreds of tokens in portions of 1 to 130
    tokens, up to four live, pages reused, the pool full of NaN.  The logits of these models are not all of
    size 1 (widths up to 1,272), so the error is measured against the largest logit of the request.  Seeds 12 to 19
    have head sizes of 2, 6, 10, 20, 36, 72, 100 and 250 elements, one after the other; seeds from 20 on groups of
    17, 24, 32 and 20 query heads a kv head (more than a matrix-core tile of the decode kernel holds), then 16, 32 and
    12 kv heads."""
    r = random.Random(seed)
    config = random_configuration(r, [EVEN_HEAD_SIZES[seed - 12]] if 12 <= seed < 20 else HEAD_SIZES)
    if seed >= 20:
        kv, group = [(1, 17), (1, 24), (1, 32), (2, 20), (16, 1), (32, 1), (12, 2)][seed - 20]
        config.update(num_attention_heads=kv * group, num_key_value_heads=kv, head_dim=r.choice([32, 64, 128]))
    page_size = r.choice([3, 4, 8, 16, 16, 32])
    folder, weights = model_folder(config, seed)
    model = load_model(folder, dtype=dtype, device='cuda')
    lengths = [r.randrange(1, 90) for _ in range(6)] + [r.randrange(200, 700)]
    prompts = {i: tokens_for(config, n, 1000 * seed + i) for i, n in enumerate(lengths)}
    pages = sum(-(-n // page_size) for n in sorted(lengths)[-4:]) + 1
    runner = ModelRunner(model, num_pages=pages, page_size=page_size, max_requests=4)
    poison(runner)
    waiting, live, done = list(prompts), {}, {}
    while waiting or live:
        while waiting and len(live) < 4:
            need = -(-len(prompts[waiting[0]]) // page_size)
            if sum(-(-len(prompts[i]) // page_size) for i in live) + need > pages:
                break
            i = waiting.pop(0)
            assert runner.admit(i)
            live[i] = 0
        order = list(live)
        r.shuffle(order)
        entries = []
        for i in order:
            left = len(prompts[i]) - live[i]
            size = 1 if left <= 3 or r.random() < 0.3 else min(left, r.choice([2, 3, 5, 8, 17, 40, 130]))
            entries.append(StepEntry(i, tuple(prompts[i][live[i]:live[i] + size]), tuple(range(size))))
        logits = runner.step(entries).cpu()
        at = 0
        for entry in entries:
            size = len(entry.tokens)
            done.setdefault(entry.request, []).append(logits[at:at + size])
            at += size
            live[entry.request] += size
            if live[entry.request] == len(prompts[entry.request]):
                runner.release(entry.request)
                del live[entry.request]
        runner.cache.check()
    assert runner.cache.free_pages == [pages]
    for i in prompts:
        got, want = torch.cat(done[i]), plain.logits(prompts[i], weights, config)
        assert torch.isfinite(got).all()
        largest = max(1.0, want.abs().max().item())
        assert (got - want).abs().max().item() <= TOLERANCE[dtype]['atol'] * largest, (config, page_size, i)


@pytest.mark.parametrize('backend', BACKENDS, indirect=True)
def test_schedule_with_a_repeated_layer_and_a_shared_cache(model_folder, backend):
    """The run order is data: layer 0 runs twice (each run with a cache of its own) and the last entry
    reads layer 1's cache instead of writing one.  Chunked steps equal the plain whole-sequence run."""
    from qil_amd.parts import ScheduleEntry
    from qil_amd.registry import read_model_config
    from qil_amd.weights import load_weights
    device, dtype = backend
    config, seed, page_size = CONFIGS['B']
    folder, weights = model_folder(config, seed)
    entry, typed = read_model_config(folder)
    model = entry.build(typed, dtype=dtype, device=device)
    model.schedule = [ScheduleEntry(0), ScheduleEntry(1), ScheduleEntry(0), ScheduleEntry(2), ScheduleEntry(1, cache_of=1)]
    load_weights(model, folder)
    order = [(0, None), (1, None), (0, None), (2, None), (1, 1)]
    tokens = tokens_for(config, 41, 17)
    hidden = plain.scheduled_hidden_states(tokens, weights, config, order)
    expected = plain.linear(plain.rms_norm(hidden, weights['model.norm.weight'], config['rms_norm_eps']),
                            plain.head_weight(weights, config))
    runner = ModelRunner(model, num_pages=8, page_size=page_size)
    poison(runner)
    assert runner.cache.kv_groups[0]['k'].shape[0] == 4           # four owning entries, one reader
    runner.admit('r')
    got, at = [], 0
    for size in (9, 2, 17, 1, 1, 11):
        got.append(runner.step([StepEntry('r', tuple(tokens[at:at + size]), tuple(range(size)))]))
        at += size
    Case(config, weights, model, page_size, dtype).close(torch.cat(got), expected)
