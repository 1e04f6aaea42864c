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
