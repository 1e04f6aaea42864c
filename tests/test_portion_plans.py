"""How paged attention shares out the keys of prompt portions that run beside rows alone: what it asks of the kernels, recorded
(no GPU needed: the rules are host code, and nothing is launched)."""
import ctypes

import pytest
import torch

from qil_amd import ops

BFLOAT16, FLOAT32 = torch.bfloat16, torch.float32


class Recorder:
    """The kernel library's rules as they are; what would launch a kernel is written down instead."""

    def __init__(self, lib):
        self.lib, self.calls = lib, {}

    def __getattr__(self, name):
        if name.endswith(('_takes', '_workspace', '_key_parts', '_tile_parts', '_waves', '_code')):
            return getattr(self.lib, name)

        def launch(*arguments):
            self.calls.setdefault(name, []).append(arguments)
            return 0
        return launch


@pytest.fixture
def recorded(monkeypatch):
    """paged_attention of portions ((rows, start) each) beside rows alone (their contexts): the recorder behind it."""
    try:
        lib = ops.library.load()
    except ops.library.KernelLibraryError as error:
        pytest.skip(f'kernel library not available here: {error}')

    def run(portions, alone, *, heads=16, kv_heads=8, d=128, dtype=BFLOAT16, page=16, told=True, first=True, **masks):
        recorder = Recorder(lib)
        monkeypatch.setattr(ops.library, 'load', lambda: recorder)
        monkeypatch.setattr(ops, '_require', lambda *a, **k: None)
        monkeypatch.setattr(ops, '_stream', lambda: None)
        monkeypatch.setattr(ops, '_decode_shares', lambda *a: (64, 1, 0, None))
        seqs = list(portions) + [(1, c - 1) for c in alone]
        ints = lambda values: torch.tensor(values, dtype=torch.int32)
        cu = [sum(n for n, _ in seqs[:i]) for i in range(len(seqs) + 1)]
        longest = max(n + s for n, s in seqs)
        cache = torch.empty((1, kv_heads, page, d), dtype=dtype)
        positions = [s + j for n, s in seqs for j in range(n)]
        ops.paged_attention(
            torch.empty((cu[-1], heads * d), dtype=dtype), heads=heads, kv_heads=kv_heads, head_dim=d, k_cache=cache,
            v_cache=cache.transpose(2, 3).contiguous(), page_size=page,
            block_tables=torch.zeros((len(seqs), -(-longest // page)), dtype=torch.int32),
            row_seq=ints([i for i, (n, _) in enumerate(seqs) for _ in range(n)]), positions=ints(positions), cu_seqlens=ints(cu),
            seq_starts=ints([s for _, s in seqs]), single_rows=ints(cu[len(portions):-1]), n_seqs=len(seqs),
            max_query=max(n for n, _ in seqs), max_context=longest, scale=1.0, window=masks.pop('window', None),
            tile_seqs=len(portions) if first else None, tile_context=max(n + s for n, s in portions) if told else None, **masks)
        recorder.positions = positions
        return recorder
    return run


# positions in the argument lists of the kernels' entries
MERGE_ROWS, MERGE_PART, MERGE_PARTS = 4, 8, 9


@pytest.mark.parametrize('portions,alone', [([(64, 960)], [16384]), ([(128, 0)], [8192, 20]), ([(1024, 0)], [40000]), ([(300, 1200), (40, 0)], [2048]),
                                            ([(64, 960)], [])])
@pytest.mark.parametrize('told', [False, True])
@pytest.mark.parametrize('first', [False, True])
@pytest.mark.parametrize('sizes', [dict(), dict(heads=32), dict(heads=8, kv_heads=2, d=64), dict(d=96), dict(d=256), dict(dtype=FLOAT32),
                                   dict(softcap=30.0), dict(slopes=torch.zeros(16)), dict(window=700), dict(sinks=torch.zeros(16))])
def test_every_row_that_is_merged_has_all_its_parts(recorded, portions, alone, told, first, sizes):
    """The merge goes by a row's position alone: where it takes the rows alone as well (``tile_seqs`` not given), the parts have to
    reach as far as they do."""
    if 'slopes' in sizes or 'sinks' in sizes:
        sizes = dict(sizes, **{name: value[:sizes.get('heads', 16)] for name, value in sizes.items() if name in ('slopes', 'sinks')})
    got = recorded(portions, alone, told=told, first=first, **sizes)
    for call in got.calls.get('qil_attn_merge', []):
        rows, part, parts = call[MERGE_ROWS], call[MERGE_PART], call[MERGE_PARTS]
        if parts > 1 and call[2] is None:                   # no row index: the step's first rows
            assert rows in (sum(n for n, _ in portions), len(got.positions))
            assert max(got.positions[:rows]) // part < parts, (part, parts)


def plan_of(recorder):
    """(keys a part, parts) of the portions' kernel."""
    if 'qil_attn_tile_bf16_parts' in recorder.calls:
        return recorder.calls['qil_attn_tile_bf16_parts'][0][-3:-1]
    if 'qil_attn_tile_in_parts' in recorder.calls:
        return recorder.calls['qil_attn_tile_in_parts'][0][-5:-3]
    assert 'qil_attn_tile' in recorder.calls
    return 0, 1


PORTIONS = [[(16, 0)], [(64, 0)], [(128, 0)], [(300, 0)], [(400, 0), (100, 0)], [(512, 0)], [(700, 0)], [(1000, 0)], [(64, 150)], [(64, 500)],
            [(128, 900)], [(300, 1200)], [(600, 1000)], [(128, 3000)]]


@pytest.mark.parametrize('sizes', [dict(dtype=FLOAT32), dict(heads=8, d=256, dtype=FLOAT32), dict(heads=14, kv_heads=2, d=64, dtype=FLOAT32), dict(kv_heads=4, softcap=30.0),
                                   dict(kv_heads=4, slopes=torch.zeros(16)), dict(kv_heads=4, d=96), dict(d=256), dict(page=24)])
def test_kernels_with_parts_of_other_sizes_keep_the_steps_plan(recorded, sizes):
    """... unless all keys of the portions lie in its first part, which the general kernel for bfloat16 cuts all the same."""
    for portions in PORTIONS:
        for context in (1100, 2048, 6144, 16384):
            longest = max(n + s for n, s in portions)
            if longest >= context:
                continue
            part, parts = plan_of(recorded(portions, [context], told=False, **sizes))
            general = sizes.get('dtype', BFLOAT16) == BFLOAT16 and (sizes.get('d') == 96 or 'page' in sizes)
            want = (0, 1) if longest <= part and not general else (part, parts)
            assert plan_of(recorded(portions, [context], **sizes)) == want, (portions, context)


@pytest.mark.parametrize('sizes', [dict(), dict(heads=32), dict(heads=64), dict(kv_heads=4, d=64), dict(heads=14, kv_heads=2, d=64), dict(window=700),
                                   dict(sinks=torch.zeros(16))])
def test_portions_on_the_kernels_for_heads_of_64_and_128(recorded, sizes):
    """In one piece where the step's first part holds all their keys; planned for their own context where they bring most of it
    themselves or it is long enough to be cut, and the merge keeps to them; else as the step."""
    for portions in PORTIONS:
        for context in (1100, 2048, 6144, 16384):
            longest, rows = max(n + s for n, s in portions), max(n for n, _ in portions)
            if longest >= context:
                continue
            step = plan_of(recorded(portions, [context], told=False, **sizes))
            own = plan_of(recorded(portions, [], told=False, **sizes))
            got = plan_of(recorded(portions, [context], **sizes))
            if step[1] > 1 and longest <= step[0]:
                assert got == (0, 1)
            elif step[1] > 1 and (longest == rows or longest >= 1024):
                assert got == own
            else:
                assert got == step
            behind = plan_of(recorded(portions, [context], first=False, **sizes))
            assert behind == (got if got == (0, 1) and step[0] >= longest else step)


def test_a_kept_first_range_stays_in_one_part(recorded):
    for told in (False, True):
        assert plan_of(recorded([(128, 900)], [6144], kv_heads=4, window=512, keep_first=64, told=told)) == (0, 1)
