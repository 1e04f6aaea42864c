"""Captured steps: decode batches that share a graph by rows rounded up (inert rows fill the rest), and a mixer
that adds into a state of its own under graphs (a new graph warms up on inert inputs, so the step it was made for
runs once)."""
import random
from dataclasses import dataclass

import pytest
import torch

import plain_qwen3 as plain

pytestmark = pytest.mark.gpu

TOLERANCE = {torch.float32: dict(atol=5e-6, rtol=5e-5), torch.bfloat16: dict(atol=0.015, rtol=0.015)}


def random_tokens(config, length, seed):
    r = random.Random(seed)
    return [r.randrange(config['vocab_size']) for _ in range(length)]


def test_row_buckets():
    from qil_amd.engine.graphs import row_bucket
    assert [row_bucket(n) for n in (1, 2, 3, 4, 5, 8, 9, 13, 16, 17, 32, 33, 63, 64, 65)] == [1, 2, 4, 4, 8, 8, 12, 16, 16, 20, 32, 40, 64, 64, 72]


@pytest.mark.parametrize('dtype', [torch.float32, torch.bfloat16])
def test_a_shrinking_decode_batch_shares_graphs(model_folder, dtype):
    """Seven requests decode together and end one after the other: the batch goes from 7 rows to 1 and replays
    four graphs (8, 4, 2 and 1 rows), not seven.  The pool is full of NaN, the spare page too; every logit against
    the plain model and against a runner that launches its kernels one by one."""
    from qil_amd.engine import ModelRunner, StepEntry
    from qil_amd.weights import load_model
    config = plain.TINY_B
    folder, weights = model_folder(config, 8)
    model = load_model(folder, dtype=dtype, device='cuda')
    lengths = [21, 24, 13, 30, 17, 26, 34]
    heads = [9, 5, 4, 12, 2, 6, 3]
    sequences = {r: random_tokens(config, n, 20 + r) for r, n in enumerate(lengths)}
    expected = {r: plain.logits(t, weights, config) for r, t in sequences.items()}
    outputs = []
    for with_graphs in (True, False):
        runner = ModelRunner(model, num_pages=7 * 5, page_size=8, max_requests=7, graphs=with_graphs)
        for group in runner.cache.kv_groups:
            group['k'].fill_(float('nan')), group['v'].fill_(float('nan'))
        fed, rows = {}, []
        for r in sequences:
            runner.admit(r)
        runner.step([StepEntry(r, tuple(sequences[r][:heads[r]]), ()) for r in sequences])
        fed = dict(enumerate(heads))
        live, sizes = list(sequences), []
        while live:
            order = list(live) if len(rows) % 2 else live[::-1]
            sizes.append(len(order))
            logits = runner.step([StepEntry(r, (sequences[r][fed[r]],), (0,)) for r in order]).cpu()
            assert logits.shape[0] == len(order)
            for i, r in enumerate(order):
                rows.append((r, fed[r], logits[i]))
                fed[r] += 1
                if fed[r] == len(sequences[r]):
                    runner.release(r)
                    live.remove(r)
        assert set(sizes) == {1, 2, 3, 4, 5, 6, 7}
        if with_graphs:
            assert runner.graphs.captures == 4 and runner.graphs.replays == len(sizes), runner.graphs.captures
        runner.cache.check()
        assert runner.cache.free_pages == [7 * 5]
        outputs.append(rows)
    for (r, place, replayed), (r2, place2, launched) in zip(*outputs):
        assert (r, place) == (r2, place2) and torch.isfinite(replayed).all()
        torch.testing.assert_close(replayed, launched, **TOLERANCE[dtype], msg=lambda m: f'{r} at {place} against launches: {m}')
        torch.testing.assert_close(replayed, expected[r][place], **TOLERANCE[dtype], msg=lambda m: f'{r} at {place}: {m}')


def test_serving_loop_with_a_batch_that_shrinks(model_folder):
    """Through ``Engine`` with the draw inside the graph: six requests of different lengths; the tokens are the plain
    greedy choice and the loop captured a graph per row bucket, not per batch size."""
    from qil_amd import Engine
    from qil_amd.weights import load_model
    config = plain.TINY_A
    folder, weights = model_folder(config, 9)
    model = load_model(folder, dtype=torch.float32, device='cuda')
    prompts = [random_tokens(config, 3 + 2 * i, 60 + i) for i in range(6)]
    engine = Engine(model, num_pages=64, page_size=4, token_budget=64, prefill_chunk=16, max_active=6)
    ids = [engine.submit(p, max_new_tokens=4 + 3 * i, ignore_eos=True) for i, p in enumerate(prompts)]
    while not engine.idle:
        engine.step()
    for i, (request, prompt) in enumerate(zip(ids, prompts)):
        assert engine.result(request)['token_ids'] == plain.greedy(prompt, 4 + 3 * i, weights, config)
    stats = engine.stats()
    assert stats['graph_captures'] <= 4 and stats['graph_replays'] >= 15, stats
    engine.cache.check()
    assert engine.cache.free_pages == [64]


def test_a_mixer_that_adds_into_its_state_runs_under_graphs(tmp_path):
    """A running mean of a request's inputs kept in a state slot, written with device tensors alone: the mixer declares
    itself safe for graphs although running a step twice would add its inputs twice.  Decode steps and recurring
    portions replay graphs; their logits equal those of a runner that launches every kernel, whole prompts equal
    portions, and a request that takes over a slot starts from nothing."""
    from qil_amd import ops
    from qil_amd.engine import ModelRunner, StepEntry
    from qil_amd.parts import (Mixer, ParamSpec, StateNeed, RMSNorm, GatedMLP, PreNormBlock, Embedding, LMHead,
                               CausalLM, ScheduleEntry)
    from qil_amd.registry import register_architecture
    from qil_amd.weights import write_random_model, load_model

    class RunningMean(Mixer):
        graph_safe = True

        def __init__(self, width, dtype):
            super().__init__()
            self.width, self.dtype = width, dtype

        def param_specs(self):
            return {'mix.weight': ParamSpec((self.width, self.width))}

        def cache_need(self):
            return StateNeed((self.width,), 'float32')

        def forward(self, h, ctx, cache):
            rows, slots = ctx.row_seq.long(), ctx.seq_slots.long()
            n = h.shape[0]
            same = rows[:, None] == rows[None, :]
            earlier = torch.ones((n, n), dtype=torch.bool, device=h.device).tril()
            prefix = (same & earlier).float() @ h.float()                      # sums within the step
            past = torch.where((ctx.seq_starts == 0)[:, None], torch.zeros((), device=h.device), cache.state[slots])
            sums = prefix + past[rows]
            cache.state.index_copy_(0, slots, sums[ctx.cu_seqlens[1:].long() - 1])
            return ops.linear((sums / (ctx.positions + 1)[:, None]).to(self.dtype), self.p['mix.weight'], None)

    @dataclass(frozen=True)
    class ToyConfig:
        vocab_size: int
        hidden_size: int
        intermediate_size: int
        num_hidden_layers: int
        rms_norm_eps: float = 1e-6
        max_position_embeddings: int = 256

        @classmethod
        def from_dict(cls, data):
            return cls(**{k: data[k] for k in cls.__dataclass_fields__ if k in data})

        def to_dict(self):
            return dict(self.__dict__, architectures=['ToyRunningMeanLM'], model_type='toy_running_mean')

    def build(config, *, dtype, device):
        embedding = Embedding(config.vocab_size, config.hidden_size)
        blocks = [PreNormBlock(mixer_norm=RMSNorm(config.hidden_size, config.rms_norm_eps),
                               mixer=RunningMean(config.hidden_size, dtype),
                               ffn_norm=RMSNorm(config.hidden_size, config.rms_norm_eps),
                               ffn=GatedMLP(width=config.hidden_size, intermediate=config.intermediate_size, dtype=dtype),
                               dtype=dtype) for _ in range(config.num_hidden_layers)]
        final_norm, head = RMSNorm(config.hidden_size, config.rms_norm_eps), LMHead(config.vocab_size, config.hidden_size)
        names = {'embed.weight': (embedding, 'weight'), 'norm.weight': (final_norm, 'weight'), 'head.weight': (head, 'weight')}
        for i, block in enumerate(blocks):
            for prefix, part in block.parts().items():
                for local in part.param_specs():
                    names[f'layers.{i}.{prefix}.{local}'] = (part, local)
        return CausalLM(config=config, embedding=embedding, blocks=blocks,
                        schedule=[ScheduleEntry(i) for i in range(len(blocks))], final_norm=final_norm, head=head,
                        names=names, dtype=dtype, device=device)

    register_architecture('ToyRunningMeanLM', model_type='toy_running_mean', config_class=ToyConfig, build=build,
                          replace=True)
    data = dict(architectures=['ToyRunningMeanLM'], model_type='toy_running_mean', vocab_size=120, hidden_size=48,
                intermediate_size=80, num_hidden_layers=2)
    folder = write_random_model(tmp_path / 'toy', data, seed=4)
    model = load_model(folder, dtype=torch.float32, device='cuda')
    sequences = {name: random_tokens(data, n, 30 + i) for i, (name, n) in enumerate((('a', 40), ('b', 27), ('c', 33), ('d', 36)))}

    def run(with_graphs, portions):
        runner = ModelRunner(model, num_pages=1, page_size=16, max_requests=3, graphs=with_graphs)
        runner.cache.state_groups[0]['state'].fill_(float('nan'))            # nobody may read what nobody wrote
        got = {name: [] for name in sequences}
        fed = {name: 0 for name in sequences}
        live = ['a', 'b', 'd']                                                 # three rows: a graph of four, one inert
        for name in live:
            runner.admit(name)
        while live:
            entries = []
            for name in list(live):
                left = len(sequences[name]) - fed[name]
                size = min(left, portions.get(name, 1)) if left > 12 else 1     # portions first, then token by token
                entries.append(StepEntry(name, tuple(sequences[name][fed[name]:fed[name] + size]), tuple(range(size))))
            logits = runner.step(entries)
            at = 0
            for entry in entries:
                size = len(entry.tokens)
                got[entry.request].append(logits[at:at + size].cpu())
                at += size
                fed[entry.request] += size
                if fed[entry.request] == len(sequences[entry.request]):
                    runner.release(entry.request)
                    live.remove(entry.request)
                    if entry.request == 'b':                                   # c takes over b's slot and its state
                        runner.admit('c')
                        live.append('c')
        graphs = runner.graphs
        return {name: torch.cat(rows) for name, rows in got.items()}, graphs

    whole, _ = run(False, {'a': 100, 'b': 100, 'c': 100, 'd': 100})
    eager, none = run(False, {'a': 4, 'b': 4, 'c': 4, 'd': 4})
    replayed, graphs = run(True, {'a': 4, 'b': 4, 'c': 4, 'd': 4})
    assert none is None and graphs.safe() and graphs.replays >= 10 and graphs.mixed_replays >= 2, \
        (graphs.replays, graphs.mixed_replays)
    for name in sequences:
        assert torch.isfinite(replayed[name]).all()
        torch.testing.assert_close(replayed[name], eager[name], atol=1e-5, rtol=1e-4)
        torch.testing.assert_close(replayed[name], whole[name], atol=1e-5, rtol=1e-4)
    # the state matters: the last logits of a request differ from those of its last token alone
    alone = ModelRunner(model, num_pages=1, page_size=16, max_requests=2, graphs=False)
    alone.admit('z')
    last = alone.step([StepEntry('z', tuple(sequences['a'][-1:]), (0,))]).cpu()
    assert not torch.allclose(last[0], whole['a'][-1], atol=1e-3)


def test_a_recurring_shape_gives_the_same_bits_launched_and_replayed(model_folder):
    """The first time a step's shape comes it is launched kernel by kernel, the second time captured and replayed,
    from then on replayed.  The same tokens at the same positions three times over (other requests, other pages):
    float32 logits equal bit for bit, because the first run is laid out and planned as the graph is."""
    from qil_amd.engine import ModelRunner, StepEntry
    from qil_amd.weights import load_model
    config = plain.TINY_B
    folder, weights = model_folder(config, 10)
    model = load_model(folder, dtype=torch.float32, device='cuda')
    long, short = random_tokens(config, 300, 1), random_tokens(config, 40, 2)
    runner = ModelRunner(model, num_pages=48, page_size=8, max_requests=2)
    for group in runner.cache.kv_groups:
        group['k'].fill_(float('nan')), group['v'].fill_(float('nan'))
    seen = []
    for occurrence in range(3):
        p, q = ('p', occurrence), ('q', occurrence)
        runner.admit(p), runner.admit(q)
        first = runner.step([StepEntry(q, tuple(short[:33]), (32,)), StepEntry(p, tuple(long[:250]), (0, 249))])
        second = runner.step([StepEntry(p, tuple(long[250:255]), (0, 4)), StepEntry(q, (short[33],), (0,))])
        seen.append((first.cpu(), second.cpu()))
        runner.release(p), runner.release(q)
    assert runner.graphs.mixed_captures == 2 and runner.graphs.mixed_replays == 4
    expected_long, expected_short = plain.logits(long[:255], weights, config), plain.logits(short[:34], weights, config)
    torch.testing.assert_close(seen[0][0], torch.stack((expected_short[32], expected_long[0], expected_long[249])), **TOLERANCE[torch.float32])
    torch.testing.assert_close(seen[0][1], torch.stack((expected_long[250], expected_long[254], expected_short[33])), **TOLERANCE[torch.float32])
    for first, second in seen[1:]:
        assert torch.equal(first, seen[0][0]) and torch.equal(second, seen[0][1])


# heads of 32 (the general kernel), and of 128 behind a context bucket of 2,048
LONG_HEADS = dict(plain.TINY_B, head_dim=128, num_attention_heads=4, max_position_embeddings=4096)


@pytest.mark.parametrize('dtype', [torch.float32, torch.bfloat16])
@pytest.mark.parametrize('config', [plain.TINY_B, LONG_HEADS], ids=['heads-of-32', 'heads-of-128'])
def test_whole_prompts_have_graphs_of_their_own(model_folder, monkeypatch, config, dtype):
    """Two prompts of 40 and 23 tokens whole beside a decoding row of 300, and portions of as many tokens of longer prompts, from
    their start (without a wanted place), right behind their first token and deep in them: the same sizes and bucket, two
    plans of the portions' attention.  Three times over, so launched, captured and replayed; every logit against the plain model."""
    from qil_amd import ops
    from qil_amd.engine import ModelRunner, StepEntry
    from qil_amd.weights import load_model
    folder, weights = model_folder(config, 13)
    model = load_model(folder, dtype=dtype, device='cuda')
    row, prompts = random_tokens(config, 318, 5), [random_tokens(config, 400, 6), random_tokens(config, 400, 7)]
    want_row, want = plain.logits(row, weights, config), [plain.logits(tokens, weights, config) for tokens in prompts]
    runner = ModelRunner(model, num_pages=200, page_size=8, max_requests=3)
    for group in runner.cache.kv_groups:
        group['k'].fill_(float('nan')), group['v'].fill_(float('nan'))
    plans, plan = [], ops.portion_key_parts

    def recorded(*arguments, **forms):
        result = plan(*arguments, **forms)
        plans.append((arguments[10], result))               # what the portions are known to reach, what is made of it
        return result

    runner.admit('row')
    runner.step([StepEntry('row', tuple(row[:300]), ())])
    monkeypatch.setattr(ops, 'portion_key_parts', recorded)
    fed, seen = 300, {True: set(), False: set()}
    for occurrence in range(3):
        for start, wanted in ((0, True), (0, False), (1, True), (24, True), (300, True)):
            for name, tokens in zip('ab', prompts):
                runner.admit(name)
                if start:
                    runner.step([StepEntry(name, tuple(tokens[:start]), ())])
            plans.clear()
            entries = [StepEntry(name, tuple(tokens[start:start + count]), (0, count - 1) if wanted else ())
                       for name, tokens, count in zip('ab', prompts, (40, 23))]
            logits = runner.step([StepEntry('row', (row[fed],), (0,))] + entries[::-1]).cpu()
            rows = [want_row[fed]] + ([want[1][start], want[1][start + 22], want[0][start], want[0][start + 39]] if wanted else [])
            torch.testing.assert_close(logits, torch.stack(rows), **TOLERANCE[dtype])
            seen[start == 0 and wanted].update(plans)
            runner.release('a'), runner.release('b')
            fed += 1
    shapes = [key for key in runner.graphs.mixed if key[0] == (40, 23, 1)]
    assert sorted(shapes, key=str) == sorted([((40, 23, 1), (2, 2, 1), longest_of(config), 40), ((40, 23, 1), (2, 2, 1), longest_of(config), None),
                                              ((40, 23, 1), (0, 0, 1), longest_of(config), None)], key=str)
    assert runner.graphs.mixed_replays >= 2 * 3, runner.graphs.mixed_replays
    (told, whole), = seen[True]
    (not_told, other), = seen[False]
    assert (told, not_told) == (40, None) and other[1] > 1
    general = dtype == torch.bfloat16 and config['head_dim'] == 32
    assert whole == (other if general else (0, 1))


def longest_of(config):
    return min(2048, config['max_position_embeddings'])


def test_more_recurring_shapes_than_the_store_holds(model_folder, monkeypatch):
    """Three shapes of mixed steps in turns with room for two graphs: the first two are captured at their second
    coming and replayed from then on; the third is launched kernel by kernel until it has come four times, then takes
    the place of the least recently replayed one.  A capture costs about two launched steps, so a store that took in
    every shape at its second coming would capture at every step here and never replay.  Every logit against the
    plain model."""
    from qil_amd.engine import ModelRunner, StepEntry
    from qil_amd.engine import graphs as graph_module
    from qil_amd.weights import load_model
    monkeypatch.setattr(graph_module, 'MAX_MIXED_GRAPHS', 2)
    config = plain.TINY_A
    folder, weights = model_folder(config, 11)
    model = load_model(folder, dtype=torch.float32, device='cuda')
    tokens = random_tokens(config, 400, 4)
    expected = plain.logits(tokens, weights, config)
    runner = ModelRunner(model, num_pages=120, page_size=4, max_requests=1)
    runner.admit('r')
    fed, captures = 0, []
    for turn in range(7):
        for size in (2, 3, 5):
            logits = runner.step([StepEntry('r', tuple(tokens[fed:fed + size]), (0, size - 1))]).cpu()
            torch.testing.assert_close(logits, expected[[fed, fed + size - 1]], **TOLERANCE[torch.float32])
            fed += size
        captures.append(runner.graphs.mixed_captures)
    # turn 0: nothing; turn 1: the shapes of 2 and 3 tokens; the shape of 5 at its fourth coming (turn 3); the one it
    # pushed out not before it has come four times again
    assert captures[:4] == [0, 2, 2, 3] and captures[-1] <= 4, captures
    assert runner.graphs.mixed_replays >= 11, runner.graphs.mixed_replays


def test_more_decode_batch_sizes_than_the_store_holds(model_folder, monkeypatch):
    """Decode batches of 1, 2 and 3 requests in turns with room for two graphs: the third size is launched kernel by
    kernel until it has come three times, then takes the place of the least recently replayed graph.  Every logit
    against the plain model, whichever way the step ran."""
    from qil_amd.engine import ModelRunner, StepEntry
    from qil_amd.engine import graphs as graph_module
    from qil_amd.weights import load_model
    monkeypatch.setattr(graph_module, 'MAX_GRAPHS', 2)
    config = plain.TINY_B
    folder, weights = model_folder(config, 12)
    model = load_model(folder, dtype=torch.float32, device='cuda')
    sequences = {r: random_tokens(config, 60, 40 + r) for r in range(3)}
    expected = {r: plain.logits(t, weights, config) for r, t in sequences.items()}
    runner = ModelRunner(model, num_pages=24, page_size=8, max_requests=3)
    for group in runner.cache.kv_groups:
        group['k'].fill_(float('nan')), group['v'].fill_(float('nan'))
    fed = {}
    for r in sequences:
        runner.admit(r)
        runner.step([StepEntry(r, tuple(sequences[r][:5]), ())])
        fed[r] = 5
    history = []
    for turn in range(8):
        for members in ((0,), (1, 2), (0, 1, 2)):             # graphs of 1, 2 and 4 rows
            logits = runner.step([StepEntry(r, (sequences[r][fed[r]],), (0,)) for r in members]).cpu()
            for i, r in enumerate(members):
                torch.testing.assert_close(logits[i], expected[r][fed[r]], **TOLERANCE[torch.float32])
                fed[r] += 1
        history.append((runner.graphs.captures, runner.graphs.replays))
    # turn 0: two captures, the third size launched; it is captured at its third coming (turn 2) and pushes the
    # graph of one row out, which comes back at its third coming after that
    assert [c for c, _ in history[:3]] == [2, 2, 3], history
    assert history[-1][0] <= 6 and history[-1][1] >= 14, history
    runner.cache.check()
