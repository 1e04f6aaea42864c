"""Each HIP kernel alone against its plain reference, at sizes other than the tiny models'."""
import pytest
import torch

import kernel_refs as refs
import plain_qwen3 as plain

pytestmark = pytest.mark.gpu

DTYPES = [torch.float32, torch.bfloat16]
TOL = {torch.float32: dict(atol=2e-6, rtol=2e-5), torch.bfloat16: dict(atol=0.008, rtol=0.008)}


@pytest.fixture(scope='module')
def ops():
    from qil_amd import ops
    ops.library.load()
    return ops


def rand(*shape, dtype=torch.float32, scale=1.0, seed=0):
    g = torch.Generator().manual_seed(seed + sum(shape))
    return (torch.randn(*shape, generator=g) * scale).to(dtype).cuda()


def check(actual, expected, dtype, scale=1.0):
    assert torch.isfinite(actual.float()).all()
    tol = {k: v * (scale if k == 'atol' else 1) for k, v in TOL[dtype].items()}
    torch.testing.assert_close(actual.float().cpu(), expected.float().cpu(), **tol)


@pytest.mark.parametrize('dtype', DTYPES)
@pytest.mark.parametrize('vocab,width', [(301, 72), (1000, 1024), (50, 4100)])
def test_embed(ops, dtype, vocab, width):
    table = rand(vocab, width, dtype=dtype)
    tokens = torch.tensor([0, vocab - 1, 7, 7, vocab // 2], dtype=torch.int32).cuda()
    out = ops.embed(tokens, table)
    assert out.dtype == torch.float32
    torch.testing.assert_close(out, table[tokens.long()].float(), atol=0, rtol=0)


@pytest.mark.parametrize('dtype', DTYPES)
@pytest.mark.parametrize('rows,width', [(1, 72), (5, 1000), (3, 4096), (2, 5120)])
def test_add_rmsnorm(ops, dtype, rows, width):
    stream, delta = rand(rows, width, scale=3.0), rand(rows, width, dtype=dtype, seed=1)
    weight = (1 + 0.3 * rand(width, seed=2)).contiguous()
    for eps in (1e-6, 1e-2):
        want_stream = stream.clone()
        want = refs.add_rmsnorm(want_stream, delta, weight, eps, dtype)
        got_stream = stream.clone()
        got = ops.add_rmsnorm(got_stream, delta, weight, eps, dtype)
        torch.testing.assert_close(got_stream, want_stream, atol=0, rtol=0)
        check(got, want, dtype, scale=4)
        check(ops.add_rmsnorm(got_stream.clone(), None, weight, eps, dtype),
              refs.add_rmsnorm(want_stream.clone(), None, weight, eps, dtype), dtype, scale=4)
    # a library routine pins the formula: float32, no delta
    if dtype == torch.float32:
        expected = torch.nn.functional.rms_norm(stream, (width,), weight, 1e-6)
        check(ops.add_rmsnorm(stream.clone(), None, weight, 1e-6, dtype), expected, dtype, scale=4)
    rows_index = torch.tensor([rows - 1, 0], dtype=torch.int32).cuda()
    before = stream.clone()
    got = ops.rows_rmsnorm(stream, delta, rows_index, weight, 1e-5, dtype)
    torch.testing.assert_close(stream, before, atol=0, rtol=0)
    check(got, refs.rows_rmsnorm(stream, delta, rows_index, weight, 1e-5, dtype), dtype, scale=4)


@pytest.mark.parametrize('dtype', DTYPES)
@pytest.mark.parametrize('rows,width,splits', [(3, 72, 1), (8, 4096, 4), (5, 1000, 2), (2, 6000, 3)])
def test_add_rmsnorm_of_partial_sums(ops, dtype, rows, width, splits):
    """The delta as float32 partial sums of a K-split product: added in split order."""
    stream = rand(rows, width, scale=3.0)
    parts = rand(splits, rows, width, seed=5)
    weight = (1 + 0.3 * rand(width, seed=2)).contiguous()
    want_stream = stream.clone()
    for i in range(splits):                       # the kernel's order: stream + p0 + p1 + ...
        want_stream += parts[i]
    want = refs.add_rmsnorm(want_stream.clone(), None, weight, 1e-6, dtype)
    got_stream = stream.clone()
    got = ops.add_rmsnorm(got_stream, ops.Partials(parts), weight, 1e-6, dtype)
    torch.testing.assert_close(got_stream, want_stream, atol=1e-6, rtol=1e-6)
    check(got, want, dtype, scale=4)
    index = torch.tensor([rows - 1], dtype=torch.int32).cuda()
    check(ops.rows_rmsnorm(stream, ops.Partials(parts), index, weight, 1e-6, dtype), want[rows - 1:], dtype, scale=4)


def test_rmsnorm_rounds_before_the_weight(ops):
    """bfloat16: the normalised value is rounded, then multiplied by the weight (qil/model.py:22-23)."""
    width = 64
    stream = rand(1, width, scale=2.0)
    weight = torch.full((width,), 1.00390625 + 2 ** -10).cuda()      # not a bfloat16 number
    got = ops.add_rmsnorm(stream.clone(), None, weight, 1e-6, torch.bfloat16).float()
    n = stream * torch.rsqrt(stream.square().mean(-1, keepdim=True) + 1e-6)
    rounded_first = (n.bfloat16().float() * weight).bfloat16().float()
    torch.testing.assert_close(got, rounded_first, atol=0, rtol=0)


SHAPES = [(1, 301, 72), (5, 384, 96), (17, 200, 136), (70, 130, 52), (130, 257, 1030), (8, 4096, 4096),
          (64, 1000, 2048), (33, 96, 224), (300, 192, 96)]


@pytest.mark.parametrize('m,n,k', SHAPES)
@pytest.mark.parametrize('bias', [False, True])
def test_linear_float32(ops, m, n, k, bias):
    x, w = rand(m, k), rand(n, k, seed=1, scale=k ** -0.5)
    b = rand(n, seed=2) if bias else None
    want = (x.double() @ w.double().t() + (b.double() if bias else 0)).float()
    check(ops.linear(x, w, b), want, torch.float32, scale=4)


@pytest.mark.parametrize('k', [192, 256, 320, 384, 448, 512, 576, 1024, 4096])
@pytest.mark.parametrize('m', [1, 8, 9, 16])
def test_linear_float32_whole_lines(ops, m, k):
    """The float32 product of up to 16 rows that reads W in whole cache lines: every number of stages from 3
    on (the last three to five run apart from the inner ones), rows of W past the end of a wave's sixteen and
    of a block's 128, whole and split over K; and a row's result does not depend on the rows beside it."""
    n = 130 if k != 1024 else 2100
    x, w = rand(m, k), rand(n, k, seed=1, scale=k ** -0.5)
    want = x.double() @ w.double().t()
    assert ops.library.load().qil_gemm_f32_splits(m, n, k) >= 1
    check(ops.linear(x, w, None), want, torch.float32, scale=4)
    got = ops.linear(x, w, None, partials=True)
    check(got.sum() if isinstance(got, ops.Partials) else got, want, torch.float32, scale=4)
    # the last row beside other rows (the same number of them, so the same kernel and the same split over K): bit for
    # bit the same sums
    parts = got.tensor if isinstance(got, ops.Partials) else got[None]
    others = rand(m, k, seed=7) * 3
    others[m - 1] = x[m - 1]
    again = ops.linear(others, w, None, partials=True)
    again = again.tensor if isinstance(again, ops.Partials) else again[None]
    assert again.shape == parts.shape
    torch.testing.assert_close(again[:, m - 1], parts[:, m - 1], atol=0, rtol=0)
    if m > 1:
        assert not torch.equal(again[:, 0], parts[:, 0])


@pytest.mark.parametrize('m,n,k', [(8, 24576, 4096), (1, 24576, 4096), (5, 43557, 192), (3, 41000, 320), (8, 50000, 384),
                                   (2, 45000, 448), (7, 43000, 512)])
def test_linear_float32_whole_lines_in_blocks_of_16_waves(ops, m, n, k):
    """The same kernel in blocks of 16 waves (256 columns), which the plan picks for up to 8 rows where only such blocks
    fill the chip in one round: every number of stages from 3 on, columns past the end of a wave's sixteen and of the
    block's 256, whole and split over K; against float64, and a row's sums do not depend on the rows beside it."""
    lib = ops.library.load()
    splits = lib.qil_gemm_f32_splits(m, n, k)
    assert lib.qil_gemm_f32_waves(m, n, k, splits) == 16 and lib.qil_gemm_f32_waves(16, n, k, lib.qil_gemm_f32_splits(16, n, k)) != 16
    x, w = rand(m, k), rand(n, k, seed=1, scale=k ** -0.5)
    want = x.double() @ w.double().t()
    got = ops.linear(x, w, None, partials=True)
    parts = got.tensor if isinstance(got, ops.Partials) else got[None]
    assert parts.shape == (splits, m, n) and torch.isfinite(parts).all()
    check(parts.sum(0), want, torch.float32, scale=4)
    if splits == 1:
        check(ops.linear(x, w, None), want, torch.float32, scale=4)
    others = rand(m, k, seed=7) * 3
    others[m - 1] = x[m - 1]
    again = ops.linear(others, w, None, partials=True)
    again = again.tensor if isinstance(again, ops.Partials) else again[None]
    torch.testing.assert_close(again[:, m - 1], parts[:, m - 1], atol=0, rtol=0)


@pytest.mark.parametrize('k', [192, 256, 320, 384, 448, 512, 576, 640, 704, 1024, 4096])
@pytest.mark.parametrize('m', [17, 32, 33, 48, 64])
def test_linear_float32_whole_lines_of_17_to_64_rows(ops, m, k):
    """The float32 product of 17 to 64 rows with A passing through LDS a stage at a time: every number of stages from
    3 on (the first stages in an unrolled loop of three, the last ones apart), two or four row tiles, rows of W past the
    end of a wave's sixteen and of a block's 128, whole and split over K; a row's result does not depend on how many
    rows come after it."""
    n = 130 if k != 1024 else 2100
    x, w = rand(m, k), rand(n, k, seed=1, scale=k ** -0.5)
    want = x.double() @ w.double().t()
    check(ops.linear(x, w, None), want, torch.float32, scale=4)
    got = ops.linear(x, w, None, partials=True)
    check(got.sum() if isinstance(got, ops.Partials) else got, want, torch.float32, scale=4)
    fewer = ops.linear(x[:17].contiguous(), w, None, partials=True)
    tensor = lambda r: r.tensor if isinstance(r, ops.Partials) else r[None]
    assert tensor(fewer).shape[0] == tensor(got).shape[0]
    torch.testing.assert_close(tensor(fewer), tensor(got)[:, :17], atol=0, rtol=0)


@pytest.mark.parametrize('m,n,k', [(3, 1024, 4096), (16, 300, 2048), (20, 4096, 4096), (64, 1024, 3072), (33, 130, 516),
                                   (48, 2000, 100), (65, 512, 1024), (128, 4096, 1024), (160, 6144, 4096)])
def test_linear_float32_partial_sums(ops, m, n, k):
    """Up to 64 rows the float32 product streams W through the float32 matrix-core instruction and may come
    back split over K; with more rows it is one tensor unless the tiled matrix-core kernel splits K to fill the chip."""
    x, w = rand(m, k), rand(n, k, seed=1, scale=k ** -0.5)
    got = ops.linear(x, w, None, partials=True)
    want = x.double() @ w.double().t()
    if isinstance(got, ops.Partials):
        assert got.splits == ops.library.load().qil_gemm_f32_splits(m, n, k) > 1 and got.shape == (m, n)
        check(got.sum(), want, torch.float32, scale=4)
    else:
        assert m > 64 or ops.library.load().qil_gemm_f32_splits(m, n, k) == 1
        check(got, want, torch.float32, scale=4)
    if k >= 2048 and n <= 4096 and m <= 64:
        assert isinstance(got, ops.Partials), 'a product with few columns and a long K should be split'


@pytest.mark.parametrize('m', [65, 127, 128, 129, 255, 256, 257, 700])
@pytest.mark.parametrize('n,k', [(128, 64), (130, 96), (97, 4096), (1000, 224), (6144, 1024)])
def test_linear_float32_of_many_rows_on_the_matrix_cores(ops, m, n, k):
    """The float32 product of more than 64 rows with K in whole stages of 32: v_mfma_f32_32x32x2_f32 on tiles loaded
    straight into LDS, 128 rows a block up to 128 rows and 256 beyond.  Row and column counts that end inside a
    block's tile, inside a wave's tile and inside a group of four columns; 2 stages (the fewest) to 128; with and
    without bias; K whole and in every number of splits it takes up to 8; against float64.  A row's result is the
    same in another place of another batch, bit for bit."""
    lib = ops.library.load()
    x, w, b = rand(m, k), rand(n, k, seed=1, scale=k ** -0.5), rand(n, seed=2)
    want = x.double() @ w.double().t()
    assert lib.qil_gemm_f32_mfma_takes(m, n, k, 1) and not lib.qil_gemm_f32_mfma_takes(m, n, k + 16, 1)
    raw = torch.cuda.current_stream().cuda_stream
    # a sum of 4,096 float32 products made one after the other is further from float64 than one of 1,024 (measured
    # on these numbers: 9.6e-6 at most here, 1.07e-5 by the vector units' kernel at K = 4,100, which adds the same way)
    scale = 4 if k < 4096 else 8
    def product(rows, bias, splits=1):
        out = torch.full((splits, rows.shape[0], n), float('nan'), device='cuda')
        status = lib.qil_gemm_f32_mfma(rows.data_ptr(), w.data_ptr(), bias.data_ptr() if bias is not None else None,
                                       out.data_ptr(), rows.shape[0], n, k, splits, raw)
        return status, out
    status, whole = product(x, None)
    assert status == 0
    check(whole[0], want, torch.float32, scale=scale)
    check(product(x, b)[1][0], want + b.double(), torch.float32, scale=scale)
    moved = torch.cat([x[m - 60:], x[:3]]).contiguous()
    torch.testing.assert_close(product(moved, None)[1][0, :60], whole[0, m - 60:], atol=0, rtol=0)
    for splits in range(2, 9):
        takes = (k // 32) % splits == 0 and k // 32 // splits >= 2
        assert bool(lib.qil_gemm_f32_mfma_takes(m, n, k, splits)) == takes
        status, parts = product(x, None, splits)
        assert status == (0 if takes else -1)
        if takes:
            assert torch.isfinite(parts).all()
            check(parts.double().sum(0), want, torch.float32, scale=scale)
            assert product(x, b, splits)[0] == -1                                # a bias goes with one split
    planned = lib.qil_gemm_f32_mfma_splits(m, n, k)
    assert planned >= 1 and lib.qil_gemm_f32_mfma_takes(m, n, k, planned)
    check(ops.linear(x, w, b), want + b.double(), torch.float32, scale=scale)    # the op, whichever kernel it picks
    got = ops.linear(x, w, None, partials=True)
    check(got.sum() if isinstance(got, ops.Partials) else got, want, torch.float32, scale=scale)


@pytest.mark.parametrize('m,n,k', SHAPES)
@pytest.mark.parametrize('out_dtype', [torch.bfloat16, torch.float32])
@pytest.mark.parametrize('bias', [False, True])
def test_linear_bfloat16(ops, m, n, k, out_dtype, bias):
    x, w = rand(m, k, dtype=torch.bfloat16), rand(n, k, dtype=torch.bfloat16, seed=1, scale=k ** -0.5)
    b = rand(n, seed=2) if bias else None
    want = x.double() @ w.double().t() + (b.double() if bias else 0)
    got = ops.linear(x, w, b, out_dtype=out_dtype)
    assert got.dtype == out_dtype
    if out_dtype == torch.float32:           # exact products, float32 sums: only the order differs
        check(got, want, torch.float32, scale=8)
    else:
        check(got, want, torch.bfloat16, scale=2)


@pytest.mark.parametrize('m,n,k', [(1, 4096, 4096), (8, 6144, 4096), (8, 4096, 12288), (64, 1024, 3072), (16, 130, 52),
                                   (3, 96, 224), (40, 200, 1030), (24, 6144, 4096), (32, 300, 1024), (17, 48, 384),
                                   (64, 6144, 4096), (48, 4096, 4096), (33, 2100, 1024), (70, 256, 512)])
def test_linear_partial_sums(ops, m, n, k):
    """Few rows, bfloat16: the product may come back split over K; the parts add up to it."""
    x, w = rand(m, k, dtype=torch.bfloat16), rand(n, k, dtype=torch.bfloat16, seed=1, scale=k ** -0.5)
    got = ops.linear(x, w, None, partials=True)
    if not isinstance(got, ops.Partials):                  # many rows, or a K that is not split: one bfloat16 result
        whole = k % 128 or k < 384 or ops.library.load().qil_gemm_bf16_splits(m, n, k) == 1
        assert m > ops.STREAM_GEMM_MOST_ROWS or (m > ops.STREAM_GEMM_MAX_ROWS and whole)
        check(got, x.double() @ w.double().t(), torch.bfloat16, scale=2)
        return
    assert isinstance(got, ops.Partials) and got.shape == (m, n)
    check(got.sum(), x.double() @ w.double().t(), torch.float32, scale=8)
    if k >= 4096 and n <= 8192:
        assert got.splits > 1, 'a product with few columns and a long K should be split'


@pytest.mark.parametrize('k', [384, 512, 640, 768, 896, 1024, 1152, 1280, 1408, 2432])
@pytest.mark.parametrize('m', [17, 32, 33, 64, 65, 96, 97, 128, 129, 160, 161, 192])
def test_linear_17_to_192_rows(ops, m, k):
    """The kernel that passes A through LDS in stages, at every number of stages from 3 on (the first and the
    last stages run apart from the inner ones), at both numbers of row tiles, with rows of W past the end
    of a wave's and of a block's sixteen, whole and split over K."""
    n = 130 if k != 1024 else 2100
    x, w = rand(m, k, dtype=torch.bfloat16), rand(n, k, dtype=torch.bfloat16, seed=1, scale=k ** -0.5)
    want = x.double() @ w.double().t()
    assert ops.library.load().qil_gemm_bf16_streams(m, n, k, 0) == 1
    check(ops.linear(x, w, None, out_dtype=torch.float32), want, torch.float32, scale=8)
    check(ops.linear(x, w, None), want, torch.bfloat16, scale=2)
    got = ops.linear(x, w, None, partials=True)
    if isinstance(got, ops.Partials):
        assert got.splits > 1
        check(got.sum(), want, torch.float32, scale=8)
    else:
        check(got, want, torch.bfloat16, scale=2)
    # a row's result does not depend on the rows beside it
    alone = ops.linear(x[m - 17:].contiguous(), w, None, out_dtype=torch.float32)
    torch.testing.assert_close(alone, ops.linear(x, w, None, out_dtype=torch.float32)[m - 17:], atol=0, rtol=0)


def test_linear_rows_do_not_depend_on_the_batch(ops):
    """A row's result is the same alone, among 7 and among 16 (one kernel, one order of the sums): bit for bit.
    Among 40 another kernel adds the same exact products in another order: equal up to float32 rounding."""
    x, w = rand(40, 512, dtype=torch.bfloat16), rand(300, 512, dtype=torch.bfloat16, seed=1, scale=0.05)
    few = ops.linear(x[:16].contiguous(), w, None, out_dtype=torch.float32)
    torch.testing.assert_close(ops.linear(x[3:4].contiguous(), w, None, out_dtype=torch.float32), few[3:4], atol=0, rtol=0)
    torch.testing.assert_close(ops.linear(x[:7].contiguous(), w, None, out_dtype=torch.float32), few[:7], atol=0, rtol=0)
    whole = ops.linear(x, w, None, out_dtype=torch.float32)
    torch.testing.assert_close(ops.linear(x[17:40].contiguous(), w, None, out_dtype=torch.float32), whole[17:], atol=0, rtol=0)
    check(whole[:16], few.double(), torch.float32, scale=8)


@pytest.mark.parametrize('m,n,k', [(8, 4096, 12288), (1, 4096, 12288), (16, 1024, 3072), (3, 2560, 9728), (8, 5120, 25600),
                                   (9, 5120, 17408), (4, 64, 384), (8, 4096, 4096)])
def test_linear_adds_into_the_stream(ops, monkeypatch, m, n, k):
    """The product whose epilogue adds the complete sums into the float32 residual stream and leaves the rows' sums of
    squares in pieces of 16 columns, against float64."""
    lib = ops.library.load()
    x = rand(m, k, dtype=torch.bfloat16)
    w = rand(n, k, dtype=torch.bfloat16, seed=3, scale=k ** -0.5)
    before = rand(m, n, scale=2.0, seed=7)
    expected = before.double() + x.double() @ w.double().t()
    stream = before.clone()
    assert lib.qil_gemm_bf16_add_takes(m, n, k)
    monkeypatch.setattr(ops, 'ADD_GEMM_FEW_ROWS', 0)                              # whatever the sizes: the adding kernel
    added = ops.linear(x, w, None, partials=True, add_to=stream)
    assert isinstance(added, ops.Added) and added.squares.shape == (n // 16, m)
    torch.testing.assert_close(stream.double().cpu(), expected.cpu(), atol=2e-4, rtol=1e-4)
    pieces = stream.double().square().reshape(m, n // 16, 16).sum(-1).t()
    torch.testing.assert_close(added.squares.double().cpu(), pieces.cpu(), atol=1e-5, rtol=1e-5)
    raw = torch.cuda.current_stream().cuda_stream
    for groups, ksplit in ((1, 8), (2, 4), (1, 2), (3, 1), (8, 1)):
        if k % (128 * ksplit) or k // (128 * ksplit) < 3:
            continue
        stream = before.clone()
        assert lib.qil_gemm_bf16_add(x.data_ptr(), w.data_ptr(), stream.data_ptr(), None, m, n, k, groups, ksplit, raw) == 0
        torch.testing.assert_close(stream.double().cpu(), expected.cpu(), atol=2e-4, rtol=1e-4)
    # what the kernel does not take comes back as a result to be added by the caller
    tall = rand(40, k, dtype=torch.bfloat16)
    stream = rand(40, n, seed=9)
    kept = stream.clone()
    assert not isinstance(ops.linear(tall, w, None, partials=True, add_to=stream), ops.Added)
    torch.testing.assert_close(stream, kept, atol=0, rtol=0)


@pytest.mark.parametrize('m,n,k', [(1, 6144, 4096), (8, 6144, 4096), (16, 6144, 4096), (3, 4096, 1024), (8, 10240, 5120),
                                   (5, 6144, 2560), (2, 48, 384), (7, 272, 1152)])
def test_linear_of_a_normed_stream(ops, monkeypatch, m, n, k):
    """The product that makes the RMSNorm of the residual stream while it stages its operand, from the sums of squares
    that the adding product left, against the norm kernel followed by the product of partial sums: the same
    normalised bfloat16 values (up to one rounding of the statistics), the same sums."""
    stream = rand(m, k, scale=3.0)
    weight = (1 + 0.3 * rand(k, seed=2)).contiguous()
    w = rand(n, k, dtype=torch.bfloat16, seed=3, scale=k ** -0.5)
    # the stream as an adding product leaves it: complete, with its squares in pieces
    half = rand(m, 384, dtype=torch.bfloat16, seed=11)
    monkeypatch.setattr(ops, 'ADD_GEMM_FEW_ROWS', 0)
    added = ops.linear(half, rand(k, 384, dtype=torch.bfloat16, seed=12, scale=0.05), None, partials=True, add_to=stream)
    assert isinstance(added, ops.Added)
    kept = stream.clone()
    lazy = ops.Normed(stream, weight, 1e-6, torch.bfloat16, added)
    got = ops.linear(lazy, w, None, partials=True)
    assert isinstance(got, ops.Partials)
    torch.testing.assert_close(stream, kept, atol=0, rtol=0)                      # the stream is read only
    normalised = ops.add_rmsnorm(stream.clone(), None, weight, 1e-6, torch.bfloat16)
    torch.testing.assert_close(lazy.materialize(), normalised, atol=0, rtol=0)
    want = ops.linear(normalised, w, None, partials=True)
    assert isinstance(want, ops.Partials) and want.splits == got.splits
    # a sum of squares in another order may move the statistics by one rounding, and a normalised value with it
    torch.testing.assert_close(got.tensor, want.tensor, atol=2e-3, rtol=1e-3)
    expected = normalised.double() @ w.double().t()
    torch.testing.assert_close(got.sum().double().cpu(), expected.cpu(), atol=2e-3, rtol=1e-3)
    # with a bias the norm kernel runs first: the same values
    biased = ops.linear(ops.Normed(stream, weight, 1e-6, torch.bfloat16, added), w, rand(n, seed=5), partials=True)
    torch.testing.assert_close(biased.double().cpu(), (expected + rand(n, seed=5).double()).cpu(), atol=0.03, rtol=0.02)


@pytest.mark.parametrize('dtype', DTYPES)
def test_silu_mul(ops, dtype):
    for inner in (136, 132, 131):                          # eight, four and one element a thread
        gate_up = rand(7, 2 * inner, dtype=dtype, scale=3.0)
        want = torch.nn.functional.silu(gate_up[:, :inner].double()) * gate_up[:, inner:].double()
        check(ops.silu_mul(gate_up), want, dtype, scale=8)
        parts = rand(3, 7, 2 * inner, scale=2.0, seed=9)
        total = parts[0] + parts[1] + parts[2]
        want = torch.nn.functional.silu(total[:, :inner].double()) * total[:, inner:].double()
        check(ops.silu_mul(ops.Partials(parts), dtype), want, dtype, scale=8)


@pytest.mark.parametrize('m,inner,k', [(1, 12288, 4096), (8, 3072, 1024), (5, 48, 384), (8, 208, 2048), (3, 16, 128),
                                       (8, 1040, 256), (7, 136, 100), (12, 256, 1024), (40, 64, 256)])
@pytest.mark.parametrize('dtype', DTYPES)
def test_gated_linear(ops, m, inner, k, dtype):
    """silu(x gate^T) * (x up^T): the fused few-row kernel where it takes the sizes (rows <= 16, inner % 16 == 0,
    K % 128 == 0), the product followed by the activation elsewhere; both against float64."""
    x = rand(m, k, dtype=dtype)
    w = rand(2 * inner, k, dtype=dtype, seed=1, scale=2.0 * k ** -0.5)
    y = x.double() @ w.double().t()
    want = torch.nn.functional.silu(y[:, :inner]) * y[:, inner:]
    def close(got):
        if dtype == torch.float32:          # float32 sums of K products: their rounding goes with the size of the sums, as
            assert torch.isfinite(got).all()                # in the products' own tests, not with the result's
            torch.testing.assert_close(got.double().cpu(), want.cpu(), atol=2e-6 * want.abs().max().item(), rtol=2e-5)
        else:
            check(got, want, dtype, scale=8)
    got = ops.gated_linear(x, w)
    assert got.dtype == dtype and got.shape == (m, inner)
    close(got)
    if inner % 16 == 0:                                   # the same with the rows in turns of 16
        turns = ops.interleave_gate_up(w[:inner].contiguous(), w[inner:].contiguous())
        assert torch.equal(turns[:16], w[:16]) and torch.equal(turns[16:32], w[inner:inner + 16])
        close(ops.gated_linear(x, turns, interleaved=True))
        y_turns = (x.double() @ turns.double().t()).to(dtype)
        check(ops.silu_mul(y_turns, interleaved=True), ops.silu_mul((x.double() @ w.double().t()).to(dtype)), dtype, scale=0)


@pytest.mark.parametrize('m', [1, 31, 33, 65, 96, 128, 129, 160, 161, 200, 256, 257, 300, 512, 513, 777, 1024])
@pytest.mark.parametrize('n,k', [(4096, 4096), (6144, 1024), (96, 256), (160, 4160), (24576, 512), (32, 320)])
def test_products_of_up_to_256_rows_loaded_straight_into_lds(ops, m, n, k):
    """The kernel for 65 to 256 rows (it takes fewer too, and up to 1,024 in equal blocks of rows): 32 x 32 x 16
    products, W and A loaded straight into LDS, a wave of its own for A, K split over blocks.  Every plan it makes (2
    to 4 multiplying waves, 1 to 16 splits) and forced splits, partial sums and direct results in both types, against
    float64; and through the op."""
    lib = ops.library.load()
    x = rand(m, k, dtype=torch.bfloat16)
    w = rand(n, k, dtype=torch.bfloat16, seed=1, scale=2.0 * k ** -0.5)
    want = x.double() @ w.double().t()
    raw = torch.cuda.current_stream().cuda_stream
    planned = lib.qil_gemm_bf16_mid_splits(m, n, k)
    assert 1 <= planned <= 16 and (k // 64) % planned == 0 and k // 64 // planned >= 4
    for splits in sorted({planned, 1, 2, 5, 16}):
        stages = k // 64
        takes = stages % splits == 0 and stages // splits >= 4
        out = torch.full((splits, m, n), float('nan'), dtype=torch.float32, device='cuda')
        status = lib.qil_gemm_bf16_mid(x.data_ptr(), w.data_ptr(), out.data_ptr(), m, n, k, 0, splits, raw)
        assert status == (0 if takes else -1), (splits, status)
        if takes:
            assert torch.isfinite(out).all()
            torch.testing.assert_close(out.double().sum(0).cpu(), want.cpu(), atol=3e-6 * want.abs().max().item(), rtol=1e-4)
    direct = torch.full((m, n), float('nan'), dtype=torch.bfloat16, device='cuda')
    assert lib.qil_gemm_bf16_mid(x.data_ptr(), w.data_ptr(), direct.data_ptr(), m, n, k, 1, 1, raw) == 0
    check(direct, want, torch.bfloat16, scale=8)
    assert lib.qil_gemm_bf16_mid(x.data_ptr(), w.data_ptr(), direct.data_ptr(), m, n, k, 1, 2, raw) == -1   # partial sums are float32
    got = ops.linear(x, w, None, partials=True)
    if isinstance(got, ops.Partials):
        torch.testing.assert_close(got.sum().double().cpu(), want.cpu(), atol=3e-6 * want.abs().max().item(), rtol=1e-4)
    else:
        check(got, want, torch.bfloat16, scale=8)
    check(ops.linear(x, w), want, torch.bfloat16, scale=8)


def test_products_of_up_to_256_rows_refuse_other_sizes(ops):
    lib = ops.library.load()
    assert lib.qil_gemm_bf16_mid_splits(1025, 4096, 4096) == 0                   # rows
    # beyond 256 rows the op sends it only the products that the library is slow at
    assert lib.qil_gemm_bf16_mid_rows_takes(512, 4096, 12288) and lib.qil_gemm_bf16_mid_rows_takes(300, 6144, 4096)
    assert not lib.qil_gemm_bf16_mid_rows_takes(300, 24576, 4096) and not lib.qil_gemm_bf16_mid_rows_takes(256, 4096, 4096)
    assert not lib.qil_gemm_bf16_mid_rows_takes(512, 6144, 4096) and not lib.qil_gemm_bf16_mid_rows_takes(513, 1024, 3072)
    assert not lib.qil_gemm_bf16_mid_rows_takes(300, 4100, 4096)
    assert lib.qil_gemm_bf16_mid_splits(128, 4100, 4096) == 0                    # columns in whole waves
    assert lib.qil_gemm_bf16_mid_splits(128, 4096, 4000) == 0                    # K in whole stages
    assert lib.qil_gemm_bf16_mid_splits(128, 4096, 192) == 0                     # four stages at least
    x = rand(128, 192, dtype=torch.bfloat16)
    w = rand(64, 192, dtype=torch.bfloat16, seed=1)
    check(ops.linear(x, w), x.double() @ w.double().t(), torch.bfloat16, scale=8)   # the op finds another way


@pytest.mark.parametrize('m,n,k,bias', [(700, 4096, 4096, False), (2112, 6144, 1024, False), (1025, 1024, 3072, True),
                                        (300, 24576, 512, False)])
def test_large_products_without_the_gpu_blas(ops, monkeypatch, m, n, k, bias):
    """``OWN_LARGE_PRODUCTS``: bfloat16 products of many rows on this library's own kernels (from 512 rows on blocks of
    256 x 256, below that the 32 x 32 tile kernel, 1,024 rows at a time); no call of torch.mm, the same bits every
    time, against float64.  A size the kernels do not take still goes to the BLAS."""
    x = rand(m, k, dtype=torch.bfloat16)
    w = rand(n, k, dtype=torch.bfloat16, seed=1, scale=2.0 * k ** -0.5)
    b = rand(n, seed=2) if bias else None
    want = x.double() @ w.double().t() + (b.double() if bias else 0)
    with_blas = ops.linear(x, w, b)
    monkeypatch.setattr(ops, 'OWN_LARGE_PRODUCTS', True)
    calls = []
    real_mm = torch.mm
    monkeypatch.setattr(torch, 'mm', lambda *a, **kw: calls.append(a[0].shape) or real_mm(*a, **kw))
    got = ops.linear(x, w, b)
    assert not calls and got.dtype == torch.bfloat16 and got.shape == (m, n)
    check(got, want, torch.bfloat16, scale=8)
    check(with_blas, want, torch.bfloat16, scale=8)
    for _ in range(3):
        assert torch.equal(ops.linear(x, w, b), got)
    odd = rand(m, 200, dtype=torch.bfloat16)                     # K in no whole stages: the kernel does not take it
    ops.linear(odd, rand(64, 200, dtype=torch.bfloat16, seed=3))
    assert len(calls) == 1


@pytest.mark.parametrize('m,n,k', [(2048, 4096, 4096), (2048, 6144, 1024), (300, 96, 192), (257, 1056, 448), (1000, 4128, 1024),
                                   (33, 64, 128), (513, 160, 448), (129, 288, 320), (1, 32, 128)])
def test_products_in_blocks_of_256_columns(ops, m, n, k):
    """The kernel for products of many rows alone, through its C interface: blocks of 128 x 128 (with two splits of the
    first size of 256 x 256), rows, columns and stages that fill no block, tile or ring; bfloat16 and float32 results
    against float64; partial sums of 2 splits of K, which add up to the float32 result; the same bits every time."""
    lib = ops.library.load()
    x = rand(m, k, dtype=torch.bfloat16)
    w = rand(n, k, dtype=torch.bfloat16, seed=1, scale=2.0 * k ** -0.5)
    want = x.double() @ w.double().t()
    stream = torch.cuda.current_stream().cuda_stream

    def product(dtype, splits=1):
        out = torch.full((splits, m, n) if splits > 1 else (m, n), 7.0, dtype=dtype, device='cuda')
        assert lib.qil_gemm_bf16_wide_takes(m, n, k, splits)
        status = lib.qil_gemm_bf16_wide(x.data_ptr(), w.data_ptr(), out.data_ptr(), m, n, k, 0 if dtype == torch.float32 else 1,
                                        splits, stream)
        assert status == 0
        return out

    got = product(torch.bfloat16)
    check(got, want, torch.bfloat16, scale=8)
    exact = product(torch.float32)
    largest = want.abs().max().item()
    torch.testing.assert_close(exact, want.float(), atol=2e-6 * largest, rtol=2e-5)
    assert torch.equal(got, exact.bfloat16())                    # one rounding, of the float32 sum
    for _ in range(2):
        assert torch.equal(product(torch.bfloat16), got)
    if k % 128 == 0 and k // 128 >= 2:
        halves = product(torch.float32, splits=2)
        torch.testing.assert_close(halves.sum(0), exact, atol=2e-6 * largest, rtol=2e-5)
        only_first = x[:, :k // 2].double() @ w[:, :k // 2].double().t()
        torch.testing.assert_close(halves[0], only_first.float(), atol=2e-6 * largest, rtol=2e-5)


@pytest.mark.parametrize('m,inner,k', [(2048, 3072, 1024), (2048, 1024, 512), (700, 1520, 448), (513, 48, 128), (1, 16, 128)])
@pytest.mark.parametrize('dtype', DTYPES)
def test_gated_products_in_blocks_of_256_columns(ops, monkeypatch, m, inner, k, dtype):
    """The same kernel with the gate's epilogue (gate and up rows in turns of 16, silu(gate) * up written once), alone
    and through ``gated_linear`` under ``OWN_LARGE_PRODUCTS``, where neither torch.mm nor the activation kernel runs;
    blocks of 128 x 128, results in bfloat16 and float32, against float64."""
    lib = ops.library.load()
    x = rand(m, k, dtype=torch.bfloat16)
    stacked = rand(2 * inner, k, dtype=torch.bfloat16, seed=1, scale=2.0 * k ** -0.5)
    y = x.double() @ stacked.double().t()
    want = torch.nn.functional.silu(y[:, :inner]) * y[:, inner:]
    w = ops.interleave_gate_up(stacked[:inner].contiguous(), stacked[inner:].contiguous())
    assert lib.qil_gemm_bf16_wide_gated_takes(m, inner, k)
    out = torch.full((m, inner), 7.0, dtype=dtype, device='cuda')
    assert lib.qil_gemm_bf16_wide_gated(x.data_ptr(), w.data_ptr(), out.data_ptr(), m, inner, k, 0 if dtype == torch.float32 else 1,
                                        torch.cuda.current_stream().cuda_stream) == 0
    largest = max(1.0, want.abs().max().item())
    if dtype == torch.float32:
        torch.testing.assert_close(out, want.float(), atol=2e-6 * largest, rtol=2e-5)
    else:
        check(out, want, torch.bfloat16, scale=largest)
    if m >= 512:
        monkeypatch.setattr(ops, 'OWN_LARGE_PRODUCTS', True)
        calls = []
        real_mm, real_silu = torch.mm, ops.silu_mul
        monkeypatch.setattr(torch, 'mm', lambda *a, **kw: calls.append('mm') or real_mm(*a, **kw))
        monkeypatch.setattr(ops, 'silu_mul', lambda *a, **kw: calls.append('silu') or real_silu(*a, **kw))
        through = ops.gated_linear(x, w, out_dtype=dtype, interleaved=True)
        assert not calls and torch.equal(through, out)


def test_products_in_blocks_of_256_columns_refuse_other_sizes(ops):
    lib = ops.library.load()
    assert lib.qil_gemm_bf16_wide_takes(2048, 4096, 4096, 1)
    assert not lib.qil_gemm_bf16_wide_takes(2048, 4100, 4096, 1)                 # columns in whole tiles of 32
    assert not lib.qil_gemm_bf16_wide_takes(2048, 4096, 4080, 1)                 # K in whole pairs of stages
    assert not lib.qil_gemm_bf16_wide_takes(2048, 4096, 4064, 1)
    assert not lib.qil_gemm_bf16_wide_takes(2048, 4096, 96, 1)                   # four stages at least
    assert not lib.qil_gemm_bf16_wide_takes(2048, 4096, 4096, 3)                 # splits of whole pairs of stages
    assert not lib.qil_gemm_bf16_wide_takes(2048, 4096, 256, 4)                  # four stages a split
    assert not lib.qil_gemm_bf16_wide_takes(1 << 20, 4096, 4096, 1)              # operands below 4 GB
    x = rand(64, 96, dtype=torch.bfloat16)
    out = torch.zeros((64, 64), dtype=torch.bfloat16, device='cuda')
    assert lib.qil_gemm_bf16_wide(x.data_ptr(), x.data_ptr(), out.data_ptr(), 64, 64, 96, 1, 1,
                                  torch.cuda.current_stream().cuda_stream) == -1
    x = rand(64, 256, dtype=torch.bfloat16)
    assert lib.qil_gemm_bf16_wide_takes(64, 64, 256, 2)
    assert lib.qil_gemm_bf16_wide(x.data_ptr(), x.data_ptr(), out.data_ptr(), 64, 64, 256, 1, 2,   # bfloat16 partial sums: no
                                  torch.cuda.current_stream().cuda_stream) == -1


@pytest.mark.parametrize('m', [17, 32, 33, 64, 65, 100, 160, 256])
@pytest.mark.parametrize('inner,k', [(12288, 4096), (6144, 256), (9216, 320)])
def test_gated_linear_of_17_to_256_rows_on_32_x_32_tiles(ops, m, inner, k):
    """The same kernel with the gate's epilogue: a wave's 32 columns are 16 gates and their 16 ups (rows in turns of
    16), one split, the result written once; the op uses it from 17 rows on.  Against float64 and against the
    product followed by the activation."""
    lib = ops.library.load()
    x = rand(m, k, dtype=torch.bfloat16)
    stacked = rand(2 * inner, k, dtype=torch.bfloat16, seed=1, scale=2.0 * k ** -0.5)
    y = x.double() @ stacked.double().t()
    want = torch.nn.functional.silu(y[:, :inner]) * y[:, inner:]
    w = ops.interleave_gate_up(stacked[:inner].contiguous(), stacked[inner:].contiguous())
    assert lib.qil_gemm_bf16_mid_gated_takes(m, inner, k)
    assert not lib.qil_gemm_bf16_mid_gated_takes(m, 1024, k)                     # too few columns for one split
    raw = torch.cuda.current_stream().cuda_stream
    for code, dtype in ((1, torch.bfloat16), (0, torch.float32)):
        out = torch.full((m, inner), float('nan'), dtype=dtype, device='cuda')
        assert lib.qil_gemm_bf16_mid_gated(x.data_ptr(), w.data_ptr(), out.data_ptr(), m, inner, k, code, raw) == 0
        if dtype == torch.float32:
            assert torch.isfinite(out).all()
            torch.testing.assert_close(out.double().cpu(), want.cpu(), atol=2e-6 * want.abs().max().item(), rtol=1e-4)
        else:
            check(out, want, dtype, scale=8)
    got = ops.gated_linear(x, w, interleaved=True)
    assert got.dtype == torch.bfloat16 and got.shape == (m, inner)
    check(got, want, torch.bfloat16, scale=8)
    unfused = ops.silu_mul(ops.linear(x, w, None, partials=True), torch.bfloat16, interleaved=True)
    check(unfused, want, torch.bfloat16, scale=8)


@pytest.mark.parametrize('m', [17, 32, 33, 64, 65, 96, 100, 128, 129, 160, 161, 192])
@pytest.mark.parametrize('inner,k', [(12288, 4096), (8192, 1024), (8208, 384), (80, 512)])
def test_gated_linear_of_17_to_192_rows(ops, m, inner, k):
    """The gate's epilogue in the kernel that passes A through LDS in stages: a block owns 64 result columns, four
    waves make the gate products and four the up products.  The op prefers the 32 x 32 tile kernel where that takes
    the sizes, so this one is called directly, small results forced through it.  Against float64, and against the
    product followed by the activation."""
    lib = ops.library.load()
    x = rand(m, k, dtype=torch.bfloat16)
    stacked = rand(2 * inner, k, dtype=torch.bfloat16, seed=1, scale=2.0 * k ** -0.5)
    y = x.double() @ stacked.double().t()
    want = torch.nn.functional.silu(y[:, :inner]) * y[:, inner:]
    w = ops.interleave_gate_up(stacked[:inner].contiguous(), stacked[inner:].contiguous())
    assert bool(lib.qil_gemm_bf16_gated_takes(m, inner, k, 1)) == (inner >= 8192 and m <= 64)
    assert not lib.qil_gemm_bf16_gated_takes(m, inner, k, 0)                     # stacked rows: the two kernels
    raw = torch.cuda.current_stream().cuda_stream
    assert lib.qil_gemm_bf16_gated(x.data_ptr(), stacked.data_ptr(), x.data_ptr(), m, inner, k, 1, 1, 0, 0, raw) == -1
    for code, dtype in ((1, torch.bfloat16), (0, torch.float32)):
        out = torch.full((m, inner), float('nan'), dtype=dtype, device='cuda')
        status = lib.qil_gemm_bf16_gated(x.data_ptr(), w.data_ptr(), out.data_ptr(), m, inner, k, code, 1, 0, 1, raw)
        if m > 64:
            assert status == -1                                                   # the op's fallback is the faster way
            continue
        assert status == 0
        if dtype == torch.float32:                           # float32 sums of K products: their rounding goes with their size
            assert torch.isfinite(out).all()
            torch.testing.assert_close(out.double().cpu(), want.cpu(), atol=2e-6 * want.abs().max().item(), rtol=1e-4)
        else:
            check(out, want, dtype, scale=8)
    got = ops.gated_linear(x, w, interleaved=True)
    assert got.dtype == torch.bfloat16 and got.shape == (m, inner)
    check(got, want, torch.bfloat16, scale=8)
    unfused = ops.silu_mul(ops.linear(x, w, None, partials=True), torch.bfloat16, interleaved=True)
    torch.testing.assert_close(got.float(), unfused.float(), atol=0.05, rtol=0.02)
    check(ops.gated_linear(x, stacked), want, torch.bfloat16, scale=8)


def test_gated_linear_block_shapes(ops):
    """Every block shape of the fused kernel (pairs a block x waves a pair) gives the same sums up to their order."""
    from qil_amd.ops import library
    lib = library.load()
    m, inner, k = 8, 400, 2048
    x = rand(m, k, dtype=torch.bfloat16)
    w = rand(2 * inner, k, dtype=torch.bfloat16, seed=1, scale=2.0 * k ** -0.5)
    y = x.double() @ w.double().t()
    want = torch.nn.functional.silu(y[:, :inner]) * y[:, inner:]
    turns = ops.interleave_gate_up(w[:inner].contiguous(), w[inner:].contiguous())
    stream = torch.cuda.current_stream().cuda_stream
    for pairs, ksplit in ((1, 1), (3, 4), (12, 1), (1, 8), (2, 2), (5, 2), (6, 2)):
        out = torch.full((m, inner), float('nan'), dtype=torch.float32, device='cuda')
        assert lib.qil_gemm_bf16_gated(x.data_ptr(), w.data_ptr(), out.data_ptr(), m, inner, k, 0, pairs, ksplit, 0, stream) == 0
        check(out, want, torch.float32, scale=8)
        out.fill_(float('nan'))
        assert lib.qil_gemm_bf16_gated(x.data_ptr(), turns.data_ptr(), out.data_ptr(), m, inner, k, 0, pairs, ksplit, 1, stream) == 0
        check(out, want, torch.float32, scale=8)


class Rot:
    def __init__(self, head_dim, theta, positions, rot_dim=None):
        rot_dim = rot_dim or head_dim
        angles = plain.rotary_angles(torch.arange(positions), rot_dim, theta)
        self.cos, self.sin, self.rot_dim = angles.cos().cuda(), angles.sin().cuda(), rot_dim


@pytest.mark.parametrize('dtype', DTYPES)
@pytest.mark.parametrize('heads,kv_heads,d,rot,page_size', [(4, 2, 16, 16, 4), (5, 1, 48, 48, 3), (32, 8, 128, 128, 16),
                                                            (6, 2, 64, 32, 7), (2, 2, 256, 256, 16)])
def test_qk_norm_rope_store(ops, dtype, heads, kv_heads, d, rot, page_size):
    n, pages = 9, 6
    qkv = rand(n, (heads + 2 * kv_heads) * d, dtype=dtype)
    qw, kw = 1 + 0.2 * rand(d, seed=3), 1 + 0.2 * rand(d, seed=4)
    rotation = Rot(d, 10000.0, 600, rot)
    positions = torch.tensor([0, 1, 2, 17, 18, 19, 500, 3, 599], dtype=torch.int32).cuda()
    slots = torch.randperm(pages * page_size)[:n].to(torch.int32).cuda()
    caches = [torch.full((pages, kv_heads, page_size, d) if i % 2 == 0 else (pages, kv_heads, d, page_size), float('nan'),
                         dtype=dtype).cuda() for i in range(4)]
    args = dict(heads=heads, kv_heads=kv_heads, head_dim=d, q_weight=qw, k_weight=kw, eps=1e-5, rotation=rotation,
                positions=positions, slots=slots, page_size=page_size, dtype=dtype)
    want = refs.qk_norm_rope_store(qkv.clone(), k_cache=caches[0], v_cache=caches[1], **args)
    got = ops.qk_norm_rope_store(qkv.clone(), k_cache=caches[2], v_cache=caches[3], **args)
    check(got, want, dtype, scale=4)
    for mine, theirs in ((caches[2], caches[0]), (caches[3], caches[1])):
        written = ~torch.isnan(theirs.float())
        assert (written == ~torch.isnan(mine.float())).all(), 'other slots were written'
        check(mine[written], theirs[written], dtype, scale=4)
    # a reader of another entry's cache stores nothing and still shapes q
    untouched = [c.clone() for c in caches[2:]]
    again = ops.qk_norm_rope_store(qkv.clone(), k_cache=caches[2], v_cache=caches[3], **{**args, 'slots': None})
    torch.testing.assert_close(again, got, atol=0, rtol=0)
    for before, after in zip(untouched, caches[2:]):
        assert torch.equal(torch.nan_to_num(before.float()), torch.nan_to_num(after.float()))
    # the same from float32 partial sums
    halves = torch.stack((qkv.float() * 0.25, qkv.float() * 0.75)).contiguous()
    fresh = [torch.full_like(c, float('nan')) for c in caches[2:]]
    split = ops.qk_norm_rope_store(ops.Partials(halves), k_cache=fresh[0], v_cache=fresh[1], **args)
    check(split, want, dtype, scale=4)
    written = ~torch.isnan(caches[0].float())
    check(fresh[0][written], caches[0][written], dtype, scale=4)


def test_rotation_pairs_and_signs(ops):
    """Unit vector at index 0 at position p -> cos p at index 0 and sin p at index d/2: rules out
    interleaved pairing and a wrong sign (qil/model.py:42-46).  No norms, float32."""
    d, p = 16, 3
    qkv = torch.zeros(1, 3 * d).cuda()
    qkv[0, 0] = 1.0
    rotation = Rot(d, 1.0, 8)              # theta 1: every frequency is 1, angle = position
    cache = torch.zeros(1, 1, 4, d).cuda()
    v_cache = torch.zeros(1, 1, d, 4).cuda()
    q = ops.qk_norm_rope_store(qkv, heads=1, kv_heads=1, head_dim=d, q_weight=None, k_weight=None, eps=0.0,
                               rotation=rotation, positions=torch.tensor([p], dtype=torch.int32).cuda(),
                               slots=torch.tensor([2], dtype=torch.int32).cuda(), k_cache=cache, v_cache=v_cache,
                               page_size=4, dtype=torch.float32)
    expected = torch.zeros(d)
    expected[0], expected[d // 2] = torch.cos(torch.tensor(3.0)), torch.sin(torch.tensor(3.0))
    torch.testing.assert_close(q[0].cpu(), expected, atol=1e-6, rtol=0)


def build_cache(lengths, page_size, kv_heads, d, dtype, seed=37):
    """NaN-filled pool, interleaved page allocation, random histories (tests/qil/test_paged_attention.py:10-31)."""
    torch.manual_seed(seed)
    pages = sum(-(-n // page_size) for n in lengths) + 2
    k_cache = torch.full((pages, kv_heads, page_size, d), float('nan'), dtype=dtype)
    v_cache = torch.full((pages, kv_heads, d, page_size), float('nan'), dtype=dtype)    # transposed pages
    free, tables = list(range(pages)), [[] for _ in lengths]
    for end in range(1, max(lengths) + page_size, page_size):
        for i, n in enumerate(lengths):
            while len(tables[i]) < -(-min(end, n) // page_size):
                tables[i].append(free.pop(0))
    histories = []
    for i, n in enumerate(lengths):
        k, v = torch.randn(n, kv_heads, d).to(dtype), torch.randn(n, kv_heads, d).to(dtype)
        j = torch.arange(n)
        page = torch.tensor(tables[i])[j // page_size]
        k_cache[page, :, j % page_size] = k
        v_cache[page, :, :, j % page_size] = v
        histories.append((k, v))
    width = max(len(t) for t in tables)
    table = torch.tensor([t + [0] * (width - len(t)) for t in tables], dtype=torch.int32)
    return k_cache.cuda(), v_cache.cuda(), table.cuda(), histories


ATT_TOL = {torch.float32: dict(atol=2e-6, rtol=2e-5), torch.bfloat16: dict(atol=0.008, rtol=0.008)}


@pytest.mark.parametrize('dtype', DTYPES)
@pytest.mark.parametrize('lengths,page_size,d,heads,kv_heads', [      # tests/qil/test_paged_attention.py:90-97
    ([1], 16, 128, 16, 8),
    ([1, 15, 16, 17], 16, 128, 16, 8),
    ([65, 3, 511, 257], 3, 40, 6, 2),
    ([1025, 1, 256, 513], 16, 128, 16, 8),
    ([31, 512], 16, 64, 4, 4),
    ([3, 257], 7, 256, 8, 1),
    ([300, 2], 4, 48, 5, 1),
    ([700], 16, 128, 64, 8),
    ([33, 200], 16, 80, 8, 2),                                  # head sizes in steps of 16
    ([129], 8, 96, 6, 3),
    ([64, 7], 16, 112, 4, 1),
    ([40, 300], 16, 32, 4, 2),
    ([19, 130], 8, 160, 4, 2),
])
def test_decode_rows_against_float64(ops, dtype, lengths, page_size, d, heads, kv_heads):
    k_cache, v_cache, table, histories = build_cache(lengths, page_size, kv_heads, d, dtype)
    rows = len(lengths)
    qkv = rand(rows, heads * d, dtype=dtype)
    positions = torch.tensor([n - 1 for n in lengths], dtype=torch.int32).cuda()
    row_seq = torch.arange(rows, dtype=torch.int32).cuda()
    args = dict(heads=heads, kv_heads=kv_heads, head_dim=d, k_cache=k_cache, v_cache=v_cache, page_size=page_size,
                block_tables=table, row_seq=row_seq, positions=positions, cu_seqlens=None, seq_starts=None, single_rows=None,
                n_seqs=rows, max_query=1, max_context=max(lengths), scale=d ** -0.5, window=None)
    got = ops.paged_attention(qkv, **args)
    expected = []
    for row, (k, v) in enumerate(histories):             # float64, explicit GQA map (:35-40)
        q = qkv[row].reshape(heads, d).double().cpu()
        kh = k.double().repeat_interleave(heads // kv_heads, dim=1).transpose(0, 1)
        vh = v.double().repeat_interleave(heads // kv_heads, dim=1).transpose(0, 1)
        score = (q[:, None, :] * kh).sum(-1) * d ** -0.5
        expected.append((score.softmax(-1)[..., None] * vh).sum(1).reshape(-1))
    expected = torch.stack(expected)
    assert torch.isfinite(got.float()).all()
    torch.testing.assert_close(got.double().cpu(), expected, **ATT_TOL[dtype])
    if rows > 1:                                         # another owner's pages cannot matter (:106-111)
        j = torch.arange(lengths[1])
        page = table[1].long()[j // page_size]
        k_cache[page, :, j % page_size] = 999.0
        v_cache[page, :, :, j % page_size] = -999.0
        torch.testing.assert_close(ops.paged_attention(qkv, **args)[0], got[0], atol=0, rtol=0)


def test_decode_rows_with_parts_that_fill_the_rounds(ops):
    """33 rows of 8 kv heads are more blocks than CUs: the matrix-core decode kernel then cuts the contexts into four
    parts; against float64, with contexts that end in every part."""
    dtype, page_size, d, heads, kv_heads = torch.bfloat16, 16, 128, 16, 8
    lengths = [2048 - 61 * i for i in range(33)]
    assert ops._decode_parts(len(lengths), kv_heads, max(lengths)) == (512, 4)
    k_cache, v_cache, table, histories = build_cache(lengths, page_size, kv_heads, d, dtype)
    rows = len(lengths)
    qkv = rand(rows, heads * d, dtype=dtype)
    args = dict(heads=heads, kv_heads=kv_heads, head_dim=d, k_cache=k_cache, v_cache=v_cache, page_size=page_size,
                block_tables=table, row_seq=torch.arange(rows, dtype=torch.int32).cuda(),
                positions=torch.tensor([n - 1 for n in lengths], dtype=torch.int32).cuda(), cu_seqlens=None,
                seq_starts=None, single_rows=None, n_seqs=rows, max_query=1, max_context=max(lengths), scale=d ** -0.5,
                window=None)
    got = ops.paged_attention(qkv, **args)
    expected = []
    for row, (k, v) in enumerate(histories):
        q = qkv[row].reshape(heads, d).double().cpu()
        kh = k.double().repeat_interleave(heads // kv_heads, dim=1).transpose(0, 1)
        vh = v.double().repeat_interleave(heads // kv_heads, dim=1).transpose(0, 1)
        score = (q[:, None, :] * kh).sum(-1) * d ** -0.5
        expected.append((score.softmax(-1)[..., None] * vh).sum(1).reshape(-1))
    torch.testing.assert_close(got.double().cpu(), torch.stack(expected), **ATT_TOL[dtype])


@pytest.mark.parametrize('lengths,window,d,heads,kv_heads,out_features', [
    ([2100, 1, 700, 1290, 64, 2047, 300, 1500], None, 128, 32, 8, 4096),
    ([900, 2100, 33], 500, 128, 32, 4, 300),
    ([5000], None, 128, 32, 8, 1024),
    ([600, 700], None, 64, 8, 2, 300),                      # too short a K for the fused path: merged first
])
def test_linear_merges_unmerged_attention(ops, lengths, window, d, heads, kv_heads, out_features):
    """The output projection takes attention results whose context parts are not merged yet and merges
    them while it stages its operand: bit for bit what the merge kernel followed by the product gives."""
    dtype, page_size = torch.bfloat16, 16
    k_cache, v_cache, table, _ = build_cache(lengths, page_size, kv_heads, d, dtype)
    rows = len(lengths)
    q = rand(rows, heads * d, dtype=dtype)
    positions = torch.tensor([n - 1 for n in lengths], dtype=torch.int32).cuda()
    args = dict(heads=heads, kv_heads=kv_heads, head_dim=d, k_cache=k_cache, v_cache=v_cache, page_size=page_size,
                block_tables=table, row_seq=torch.arange(rows, dtype=torch.int32).cuda(), positions=positions,
                cu_seqlens=None, seq_starts=None, single_rows=None, n_seqs=rows, max_query=1, max_context=max(lengths),
                scale=d ** -0.5, window=window)
    w = rand(out_features, heads * d, dtype=dtype, seed=3, scale=(heads * d) ** -0.5)
    merged = ops.paged_attention(q, **args)
    assert isinstance(merged, torch.Tensor)
    want = ops.linear(merged, w, None, partials=True)
    lazy = ops.paged_attention(q, unmerged=True, **args)
    assert isinstance(lazy, ops.Unmerged), 'several context parts and only single rows: nothing to merge yet'
    got = ops.linear(lazy, w, None, partials=True)
    assert isinstance(got, ops.Partials) and isinstance(want, ops.Partials)
    torch.testing.assert_close(got.tensor, want.tensor, atol=0, rtol=0)
    torch.testing.assert_close(lazy.merge(), merged, atol=0, rtol=0)
    biased = ops.linear(ops.paged_attention(q, unmerged=True, **args), w, rand(out_features, seed=5))     # no fused path: merges first
    check(biased, merged.double() @ w.double().t() + rand(out_features, seed=5).double(), dtype, scale=2)


@pytest.mark.parametrize('lengths,window,d,heads,kv_heads,out_features,page_size', [
    ([2100, 1, 700, 1290, 64, 2047, 300, 1500], None, 128, 16, 8, 1024, 16),      # Qwen3-0.6B sizes, 8 rows
    ([900, 2100, 33], 500, 128, 32, 4, 300, 16),                                # a window; columns that fill no block
    ([700], None, 64, 5, 5, 77, 8),                                            # one row, one head a kv head
    ([3000, 5, 1200, 64, 65, 800, 90, 2300, 400, 17, 1000, 2000, 1, 300, 600, 1900], None, 40, 8, 2, 200, 16),   # 16 rows, d = 40
    ([600, 700], None, 40, 3, 1, 50, 4),                                       # K no whole stage: merged first
    ([600] * 17, None, 64, 4, 2, 64, 16),                                      # 17 rows: merged by the attention
])
def test_linear_float32_merges_unmerged_attention(ops, lengths, window, d, heads, kv_heads, out_features, page_size):
    """The float32 output projection of up to 16 rows merges the row kernel's context parts while it stages its
    operand: bit for bit what the merge kernel followed by the product gives."""
    dtype = torch.float32
    k_cache, v_cache, table, _ = build_cache(lengths, page_size, kv_heads, d, dtype)
    rows = len(lengths)
    q = rand(rows, heads * d, dtype=dtype)
    positions = torch.tensor([n - 1 for n in lengths], dtype=torch.int32).cuda()
    args = dict(heads=heads, kv_heads=kv_heads, head_dim=d, k_cache=k_cache, v_cache=v_cache, page_size=page_size,
                block_tables=table, row_seq=torch.arange(rows, dtype=torch.int32).cuda(), positions=positions,
                cu_seqlens=None, seq_starts=None, single_rows=None, n_seqs=rows, max_query=1, max_context=max(lengths),
                scale=d ** -0.5, window=window)
    w = rand(out_features, heads * d, dtype=dtype, seed=3, scale=(heads * d) ** -0.5)
    merged = ops.paged_attention(q, **args)
    assert isinstance(merged, torch.Tensor)
    want = ops.linear(merged, w, None, partials=True)
    lazy = ops.paged_attention(q, unmerged=True, **args)
    if rows > 16:
        assert isinstance(lazy, torch.Tensor)
        torch.testing.assert_close(lazy, merged, atol=0, rtol=0)
        return
    assert isinstance(lazy, ops.Unmerged), 'several context parts and only single rows: nothing to merge yet'
    got = ops.linear(lazy, w, None, partials=True)
    fused = bool(ops.library.load().qil_gemm_f32_unmerged_takes(rows, out_features, heads, d, got.splits if isinstance(got, ops.Partials) else 1))
    assert fused == ((heads * d) % 64 == 0 and heads * d >= 192)
    as_tensor = lambda r: r.tensor if isinstance(r, ops.Partials) else r[None]
    torch.testing.assert_close(as_tensor(got), as_tensor(want), atol=0, rtol=0)
    torch.testing.assert_close(lazy.merge(), merged, atol=0, rtol=0)
    check(as_tensor(got).sum(0), merged.double() @ w.double().t(), dtype, scale=2)
    biased = ops.linear(ops.paged_attention(q, unmerged=True, **args), w, rand(out_features, seed=5))     # no fused path: merges first
    check(biased, merged.double() @ w.double().t() + rand(out_features, seed=5).double(), dtype, scale=2)


@pytest.mark.parametrize('rows,width,inner,interleaved', [
    (1, 1024, 3072, True), (8, 1024, 3072, True), (16, 320, 192, True), (5, 200, 256, False), (3, 64, 448, True),
    (2, 48, 100, False),                                      # K no whole stage: the activation kernel runs
    (17, 128, 256, True),                                     # too many rows: the activation kernel runs
])
def test_linear_float32_makes_the_gated_activation(ops, rows, width, inner, interleaved):
    """A float32 down product of up to 16 rows takes the gate and up products' partial sums and makes silu(gate) * up
    while it stages its operand: bit for bit what the activation kernel followed by the product gives."""
    x = rand(rows, width)
    gate, up = rand(inner, width, seed=1, scale=width ** -0.5), rand(inner, width, seed=2, scale=width ** -0.5)
    both = ops.interleave_gate_up(gate, up) if interleaved else torch.cat([gate, up]).contiguous()
    down = rand(width + 8, inner, seed=3, scale=inner ** -0.5)
    hidden = ops.gated_linear(x, both, torch.float32, interleaved=interleaved)
    assert isinstance(hidden, torch.Tensor)
    check(hidden, torch.nn.functional.silu(x.double() @ gate.double().t()) * (x.double() @ up.double().t()), torch.float32, scale=2)
    want = ops.linear(hidden, down, None, partials=True)
    lazy = ops.gated_linear(x, both, torch.float32, interleaved=interleaved, lazy=True)
    if rows > 16:
        assert isinstance(lazy, torch.Tensor)
        torch.testing.assert_close(lazy, hidden, atol=0, rtol=0)
        return
    assert isinstance(lazy, ops.Gated)
    torch.testing.assert_close(lazy.materialize(), hidden, atol=0, rtol=0)
    got = ops.linear(lazy, down, None, partials=True)
    as_tensor = lambda r: r.tensor if isinstance(r, ops.Partials) else r[None]
    torch.testing.assert_close(as_tensor(got), as_tensor(want), atol=0, rtol=0)
    check(as_tensor(got).sum(0), hidden.double() @ down.double().t(), torch.float32, scale=2)
    whole = ops.linear(ops.gated_linear(x, both, torch.float32, interleaved=interleaved, lazy=True), down)   # a tensor is asked for
    assert isinstance(whole, torch.Tensor)
    check(whole, hidden.double() @ down.double().t(), torch.float32, scale=2)


@pytest.mark.parametrize('lengths,page_size,d,heads,kv_heads,window,norm,rot,splits', [
    ([2100, 1, 700, 1290, 64, 2047, 300, 33], 16, 128, 32, 8, None, True, 128, 8),     # the benchmark's sizes
    ([1, 2, 31, 32, 33, 64, 65, 96], 8, 64, 6, 2, None, True, 64, 3),                  # every edge of a 32-key step and of a page
    ([257, 512, 513], 32, 128, 8, 1, 100, False, 64, 1),                               # no norm, half of the head rotated, a window
    ([40, 1000], 16, 64, 16, 1, None, True, 0, 2),                                     # 16 heads a kv head, no rotation
    ([5000], 16, 128, 5, 5, None, True, 32, 5),                                        # one head a kv head, many parts
    ([37 * i % 900 + 1 for i in range(30)], 16, 128, 16, 8, None, True, 128, 4),       # thirty rows
])
def test_decode_attention_fused_is_the_two_kernels(ops, lengths, page_size, d, heads, kv_heads, window, norm, rot, splits):
    """Queries, new key and new value made inside the attention kernel from the q/k/v product's partial sums:
    the attention result and the pages are bit for bit what qk_norm_rope_store followed by paged_attention
    leave (the last token of every history is the step's new token)."""
    dtype = torch.bfloat16
    rows = len(lengths)
    total = heads + 2 * kv_heads
    k_cache, v_cache, table, _ = build_cache(lengths, page_size, kv_heads, d, dtype)
    positions = torch.tensor([n - 1 for n in lengths], dtype=torch.int32).cuda()
    row_seq = torch.arange(rows, dtype=torch.int32).cuda()
    slots = (table[row_seq.long(), (positions // page_size).long()] * page_size + positions % page_size).to(torch.int32)
    qkv = ops.Partials(rand(splits, rows, total * d, scale=0.7, seed=21))
    q_w = (1 + 0.1 * rand(d, seed=22)) if norm else None
    k_w = (1 + 0.1 * rand(d, seed=23)) if norm else None
    rotation = Rot(d, 10000.0, max(lengths), rot) if rot else None
    sizes = dict(heads=heads, kv_heads=kv_heads, head_dim=d)
    assert ops.decode_attention_takes(qkv, page_size=page_size, rotation=rotation, dtype=dtype, **sizes)
    k_two, v_two = k_cache.clone(), v_cache.clone()
    q = ops.qk_norm_rope_store(qkv, q_weight=q_w, k_weight=k_w, eps=1e-6, rotation=rotation, positions=positions,
                               slots=slots, k_cache=k_two, v_cache=v_two, page_size=page_size, dtype=dtype, **sizes)
    want = ops.paged_attention(q, k_cache=k_two, v_cache=v_two, page_size=page_size, block_tables=table, row_seq=row_seq,
                               positions=positions, cu_seqlens=None, seq_starts=None, single_rows=None, n_seqs=rows,
                               max_query=1, max_context=max(lengths), scale=d ** -0.5, window=window, **sizes)
    k_one, v_one = k_cache.clone(), v_cache.clone()
    got = ops.decode_attention(qkv, q_weight=q_w, k_weight=k_w, eps=1e-6, rotation=rotation, positions=positions,
                               writes=True, k_cache=k_one, v_cache=v_one, page_size=page_size, block_tables=table,
                               row_seq=row_seq, max_context=max(lengths), scale=d ** -0.5, window=window, **sizes)
    assert torch.isfinite(got.float()).all()
    torch.testing.assert_close(got, want, atol=0, rtol=0)
    same = lambda a, b: torch.equal(a.view(torch.int16), b.view(torch.int16))          # NaN-filled pages: compare the bits
    assert same(k_one, k_two) and same(v_one, v_two), 'the pages differ'
    # a reader of another layer's cache: nothing is written, the new token's key and value are read from the pages
    k_read, v_read = k_two.clone(), v_two.clone()
    read = ops.decode_attention(qkv, q_weight=q_w, k_weight=k_w, eps=1e-6, rotation=rotation, positions=positions,
                                writes=False, k_cache=k_read, v_cache=v_read, page_size=page_size, block_tables=table,
                                row_seq=row_seq, max_context=max(lengths), scale=d ** -0.5, window=window, **sizes)
    torch.testing.assert_close(read, want, atol=0, rtol=0)
    assert same(k_read, k_two) and same(v_read, v_two)


def mixed_attention_case(ops, dtype, lengths, chunks, page_size, d, heads, kv_heads, window, scale=0.3, table_width=None):
    """Sequences of `lengths` cached tokens whose last `chunks[i]` positions are this step's rows.  `table_width`:
    the block tables get so many columns (a pool for contexts far longer than these)."""
    k_cache, v_cache, table, histories = build_cache(lengths, page_size, kv_heads, d, dtype)
    if table_width is not None:
        wide = torch.zeros((table.shape[0], table_width), dtype=torch.int32, device=table.device)
        wide[:, :table.shape[1]] = table
        table = wide
    starts = [n - c for n, c in zip(lengths, chunks)]
    positions = [p for s, c in zip(starts, chunks) for p in range(s, s + c)]
    row_seq = [i for i, c in enumerate(chunks) for _ in range(c)]
    cu = [0]
    for c in chunks:
        cu.append(cu[-1] + c)
    single = [cu[i] for i, c in enumerate(chunks) if c == 1]
    n = cu[-1]
    dev = lambda values: torch.tensor(values, dtype=torch.int32).cuda()
    qkv = rand(n, heads * d, dtype=dtype)
    got = ops.paged_attention(qkv, heads=heads, kv_heads=kv_heads, head_dim=d, k_cache=k_cache, v_cache=v_cache,
                              page_size=page_size, block_tables=table, row_seq=dev(row_seq), positions=dev(positions),
                              cu_seqlens=dev(cu), seq_starts=dev(starts), single_rows=dev(single) if max(chunks) > 1 else None,
                              n_seqs=len(lengths), max_query=max(chunks), max_context=max(lengths), scale=scale,
                              window=window)
    q = qkv.reshape(n, heads, d).double().cpu()
    expected = torch.cat([
        plain.attention(q[cu[i]:cu[i + 1]], histories[i][0].double(), histories[i][1].double(),
                        torch.arange(starts[i], lengths[i]), scale, window)
        for i in range(len(lengths))]).reshape(n, heads * d)
    assert torch.isfinite(got.float()).all()
    torch.testing.assert_close(got.double().cpu(), expected, **ATT_TOL[dtype])


@pytest.mark.parametrize('dtype', DTYPES)
@pytest.mark.parametrize('window', [None, 5, 64, 300])
def test_prompt_rows_and_window(ops, dtype, window):
    """Rows of a portion at positions 290..339 of a 340-token request beside a decoded row of another."""
    mixed_attention_case(ops, dtype, [340, 77], [50, 1], 8, 32, 6, 2, window)


@pytest.mark.parametrize('dtype', DTYPES)
@pytest.mark.parametrize('lengths,chunks,page_size,d,heads,kv_heads', [
    ([70, 70, 5, 33], [70, 2, 5, 17], 16, 128, 16, 8),          # whole prompt, two-token portion, short, middle
    ([129, 64, 1000, 16], [129, 1, 3, 16], 16, 128, 32, 8),     # g = 4; a portion deep in a long context
    ([257, 100], [200, 31], 3, 40, 6, 2),                       # page size 3, head size 40, g = 3
    ([90, 45], [90, 45], 7, 256, 8, 1),                         # head size 256, one kv head (g = 8)
    ([300, 19], [151, 19], 4, 48, 5, 1),                        # g = 5
    ([66, 40, 20], [35, 40, 2], 8, 16, 4, 4),                   # g = 1, head size 16
    ([513], [513], 16, 64, 4, 2),                               # g = 2
    ([2048], [2048], 16, 128, 8, 2),
    ([150, 40], [150, 13], 16, 80, 8, 2),                       # head sizes in steps of 16
    ([200], [77], 8, 96, 6, 3),
    ([90, 30], [45, 30], 16, 112, 4, 1),
    ([100], [100], 16, 32, 4, 2),
    ([70, 20], [70, 9], 8, 160, 4, 2),
])
def test_prompt_portions_against_float64(ops, dtype, lengths, chunks, page_size, d, heads, kv_heads):
    mixed_attention_case(ops, dtype, lengths, chunks, page_size, d, heads, kv_heads, None, scale=d ** -0.5)


@pytest.mark.parametrize('lengths,chunks,page_size,d,heads,kv_heads,window', [
    ([700, 90, 33], [100, 1, 33], 8, 128, 16, 4, None),
    ([513, 64], [513, 2], 16, 64, 4, 2, None),
    ([600, 64], [77, 17], 8, 128, 10, 2, 100),
])
def test_block_tables_wider_than_the_fast_prompt_kernels_keep(ops, lengths, chunks, page_size, d, heads, kv_heads, window):
    """The bfloat16 prompt kernels of head sizes 64 and 128 keep a sequence's block table in LDS, up to 4,096 entries
    (32,768 tokens at pages of 8); a wider table goes to the general tile kernel.  Tables of 4,100 columns here, with
    short contexts in them (the table's width, not the context, decides), against float64."""
    lib = ops.library.load()
    assert lib.qil_attn_tile_bf16_takes(d, page_size, 4096) and not lib.qil_attn_tile_bf16_takes(d, page_size, 4100)
    mixed_attention_case(ops, torch.bfloat16, lengths, chunks, page_size, d, heads, kv_heads, window, scale=d ** -0.5,
                         table_width=4100)


@pytest.mark.parametrize('growth', [0.02, 0.11, 1.5])
@pytest.mark.parametrize('waves', [4, 16])
def test_prompt_attention_with_scores_that_grow_along_the_keys(ops, growth, waves):
    """The kernel for head size 128 keeps a row's reference exponent until a score exceeds it by 2^8.  Keys whose
    scores grow by `growth` (in the exponent, to base 2) from one key to the next move it never within a tile's
    reach, every few tiles, or at every tile: probabilities up to 2^8 and rescaled sums, against float64."""
    page_size, d, heads, kv_heads, n, rows = 16, 128, 8, 2, 1200, 330
    k_cache, v_cache, table, histories = build_cache([n], page_size, kv_heads, d, torch.bfloat16)
    torch.manual_seed(5)
    direction = torch.nn.functional.normalize(torch.randn(kv_heads, d), dim=-1)
    j = torch.arange(n, dtype=torch.float32)
    k = (0.05 * torch.randn(n, kv_heads, d) + j[:, None, None] * 0.01 * direction).to(torch.bfloat16)
    page = table[0].cpu()[(j.long() // page_size)].long()
    k_cache[page.cuda(), :, (j.long() % page_size).cuda()] = k.cuda()
    histories[0] = (k, histories[0][1])
    scale = 1.0
    # a query along the direction: score of key j = j * 0.01 * |q|, so |q| = growth / (0.01 * log2(e))
    g = heads // kv_heads
    q = torch.stack([direction[h // g] * (growth / (0.01 * 1.4426950408889634)) for h in range(heads)])
    qkv = (q[None] + 0.02 * torch.randn(rows, heads, d)).to(torch.bfloat16).reshape(rows, heads * d).cuda()
    start = n - rows
    dev = lambda values: torch.tensor(values, dtype=torch.int32).cuda()
    lib = ops.library.load()
    lib.qil_attn_tile_waves(waves)
    try:
        got = ops.paged_attention(qkv, heads=heads, kv_heads=kv_heads, head_dim=d, k_cache=k_cache, v_cache=v_cache,
                                  page_size=page_size, block_tables=table, row_seq=dev([0] * rows),
                                  positions=dev(list(range(start, n))), cu_seqlens=dev([0, rows]), seq_starts=dev([start]),
                                  single_rows=dev([]), n_seqs=1, max_query=rows, max_context=n, scale=scale, window=None)
    finally:
        lib.qil_attn_tile_waves(0)
    expected = plain.attention(qkv.reshape(rows, heads, d).double().cpu(), k.double(), histories[0][1].double(),
                               torch.arange(start, n), scale).reshape(rows, heads * d)
    assert torch.isfinite(got.float()).all()
    torch.testing.assert_close(got.double().cpu(), expected, **ATT_TOL[torch.bfloat16])


@pytest.mark.parametrize('lengths,chunks,heads,kv_heads,window', [
    ([700, 90, 33], [700, 31, 33], 16, 4, None),                # g = 4: 32 rows of 4 heads a group
    ([513, 200], [300, 200], 8, 4, None),                       # g = 2: 64 rows of 2 heads
    ([400], [400], 4, 4, None),                                 # g = 1: 128 rows of one head
    ([600, 64], [600, 17], 10, 2, None),                        # g = 5: two chunks of heads
])
def test_prompt_attention_in_two_groups_of_waves(ops, lengths, chunks, heads, kv_heads, window):
    """Short prompts of head size 128 run in blocks of 8 waves, two groups that halve a block's keys; forced here on
    longer ones and on several sequences, against float64."""
    lib = ops.library.load()
    lib.qil_attn_tile_waves(16)
    try:
        mixed_attention_case(ops, torch.bfloat16, lengths, chunks, 16, 128, heads, kv_heads, window, scale=128 ** -0.5)
    finally:
        lib.qil_attn_tile_waves(0)


@pytest.mark.parametrize('lengths,chunks,d,heads,kv_heads,window,split', [
    ([700, 90, 33], [100, 1, 33], 128, 16, 4, None, (64, 2)),    # parts of one tile; a whole short prompt beside it
    ([513, 200, 64], [70, 200, 1], 128, 8, 4, None, (128, 2)),   # a part's edge inside a portion's rows (512 | 513)
    ([640], [129], 64, 4, 2, None, (192, 2)),                    # head size 64; a portion that starts on an edge
    ([600, 64], [77, 17], 128, 10, 2, 100, (64, 3)),             # a window: the first parts hold nothing for a row
    ([900], [2], 128, 8, 8, 300, (256, 2)),                      # two rows, g = 1
    ([1030, 300], [130, 2], 64, 6, 2, 64, (64, 4)),              # g = 3, a window of one part's size
])
def test_prompt_portion_with_keys_in_parts(ops, monkeypatch, lengths, chunks, d, heads, kv_heads, window, split):
    """A portion deep in a long context has its keys cut into parts that are merged afterwards; forced on short
    contexts here, with edges of parts at and inside the portion's rows, against float64."""
    monkeypatch.setattr(ops, 'TILE_KEY_PARTS', split)
    mixed_attention_case(ops, torch.bfloat16, lengths, chunks, 16, d, heads, kv_heads, window, scale=d ** -0.5)


@pytest.mark.parametrize('dtype,lengths,chunks,page_size,d,heads,kv_heads,window,split', [
    (torch.float32, [700, 90, 33], [100, 1, 33], 16, 128, 16, 4, None, (64, 2)),    # parts of two float32 tiles
    (torch.float32, [513, 200, 64], [70, 200, 1], 16, 128, 16, 8, None, (128, 2)),  # a part's edge inside a portion's rows
    (torch.float32, [640], [129], 8, 64, 4, 2, None, (192, 2)),                     # a portion that starts on an edge
    (torch.float32, [600, 64], [77, 17], 4, 40, 10, 2, 100, (64, 3)),               # d = 40, g = 5, a window
    (torch.float32, [900], [2], 16, 256, 2, 2, 300, (256, 2)),                      # two rows, g = 1, d = 256
    (torch.bfloat16, [1030, 300], [130, 2], 16, 96, 6, 2, 64, (64, 4)),             # bfloat16 of a head size without a kernel of its own
    (torch.bfloat16, [700, 40], [300, 40], 3, 128, 8, 4, None, (128, 2)),           # ... or of pages of 3 keys
])
def test_prompt_portion_with_keys_in_parts_on_the_general_kernel(ops, monkeypatch, dtype, lengths, chunks, page_size, d,
                                                                 heads, kv_heads, window, split):
    """The float32 path, and bfloat16 sizes without a kernel of their own, cut a portion's keys into parts on the
    general tile kernel; forced on short contexts here, against float64."""
    monkeypatch.setattr(ops, 'TILE_KEY_PARTS', split)
    mixed_attention_case(ops, dtype, lengths, chunks, page_size, d, heads, kv_heads, window, scale=d ** -0.5)


@pytest.mark.parametrize('dtype,d,page_size', [(torch.float32, 128, 16), (torch.float32, 64, 16), (torch.bfloat16, 96, 16)])
@pytest.mark.parametrize('lengths,chunks,heads,kv_heads,window', [
    ([2048], [128], 16, 8, None),
    ([3000] + [900] * 6, [128] + [1] * 6, 8, 2, None),          # one portion beside decoded rows
    ([2500], [130], 8, 2, 1100),
])
def test_general_tile_kernel_deep_in_a_long_context(ops, dtype, d, page_size, lengths, chunks, heads, kv_heads, window):
    """The sizes at which the general kernel's split is chosen by itself."""
    lib = ops.library.load()
    table_stride = -(-max(lengths) // page_size)
    part, parts = ops.tile_key_parts(lib, dtype, sum(c > 1 for c in chunks), max(chunks), heads, kv_heads, d, page_size,
                                     table_stride, max(lengths))
    assert parts > 1 and part % 64 == 0 and part * parts >= max(lengths)
    mixed_attention_case(ops, dtype, lengths, chunks, page_size, d, heads, kv_heads, window, scale=d ** -0.5)


@pytest.mark.parametrize('lengths,chunks,heads,kv_heads,window', [
    ([2048], [128], 32, 8, None),
    ([4000, 3000, 1500], [64, 1, 2], 16, 8, None),
    ([5000], [130], 8, 2, 1100),
    ([3000] + [900] * 12, [128] + [1] * 12, 32, 8, None),       # one portion beside a dozen decoded rows
])
def test_prompt_portion_deep_in_a_long_context(ops, lengths, chunks, heads, kv_heads, window):
    """The sizes at which the split is chosen by itself (sequences of one row do not count as work)."""
    lib = ops.library.load()
    table_stride = -(-max(lengths) // 16)
    part, parts = ops.tile_key_parts(lib, torch.bfloat16, sum(c > 1 for c in chunks), max(chunks), heads, kv_heads, 128,
                                     16, table_stride, max(lengths))
    assert parts > 1 and part % 64 == 0 and part * parts >= max(lengths)
    mixed_attention_case(ops, torch.bfloat16, lengths, chunks, 16, 128, heads, kv_heads, window, scale=128 ** -0.5)


def test_one_far_key_among_hundreds(ops):
    """Scale one early key so its score dominates: the output must be that key's value, from the
    right page and the right kv head (h // g, not h % kv_heads)."""
    page_size, d, heads, kv_heads, n = 16, 64, 8, 2, 900
    k_cache, v_cache, table, histories = build_cache([n], page_size, kv_heads, d, torch.float32)
    target = 37
    q = rand(1, heads * d)
    for h in range(heads):
        kvh = h // (heads // kv_heads)
        direction = histories[0][0][target, kvh] / histories[0][0][target, kvh].norm()
        q[0, h * d:(h + 1) * d] = 200.0 * direction.cuda()
    got = ops.paged_attention(q, heads=heads, kv_heads=kv_heads, head_dim=d, k_cache=k_cache, v_cache=v_cache,
                              page_size=page_size, block_tables=table, positions=torch.tensor([n - 1], dtype=torch.int32).cuda(),
                              row_seq=torch.zeros(1, dtype=torch.int32).cuda(), cu_seqlens=None, seq_starts=None, single_rows=None,
                              n_seqs=1, max_query=1, max_context=n, scale=1.0, window=None)
    for h in range(heads):
        kvh = h // (heads // kv_heads)
        torch.testing.assert_close(got[0, h * d:(h + 1) * d].cpu(), histories[0][1][target, kvh], atol=1e-4, rtol=1e-4)


def pointed_queries(histories, row_seq, targets, heads, kv_heads, d, dtype):
    """Queries whose every head points, 200 long, along the key `targets[r]` of its kv head in row r's history:
    that key's score then stands out by hundreds, the softmax is one-hot and the output is that key's value."""
    q = torch.zeros(len(targets), heads, d)
    for r, (s, target) in enumerate(zip(row_seq, targets)):
        for h in range(heads):
            key = histories[s][0][target, h // (heads // kv_heads)].float()
            q[r, h] = 200.0 * key / key.norm()
    return q.reshape(len(targets), heads * d).to(dtype).cuda()


def values_of(histories, row_seq, targets, heads, kv_heads):
    return torch.stack([histories[s][1][t].float().repeat_interleave(heads // kv_heads, 0).reshape(-1)
                        for s, t in zip(row_seq, targets)])


def test_decode_kernel_finds_one_key_at_the_edges_of_its_parts(ops):
    """bfloat16 matrix-core decode kernel, context in nine parts of 256 keys: a key at 0, at the ends of a 32-key
    step, at the last place of a part, at the first of the next, and the newest key, each dominant for one row."""
    page_size, d, heads, kv_heads, n = 16, 128, 8, 2, 2100
    targets = [0, 31, 32, 255, 256, 1023, 1024, 2047, 2048, n - 1]
    rows = len(targets)
    k_cache, v_cache, table, histories = build_cache([n] * rows, page_size, kv_heads, d, torch.bfloat16)
    part, parts = ops._decode_parts(rows, kv_heads, n)
    assert part == 256 and parts == 9 and ops.library.load().qil_attn_decode_takes(heads, kv_heads, d, page_size)
    row_seq = list(range(rows))
    q = pointed_queries(histories, row_seq, targets, heads, kv_heads, d, torch.bfloat16)
    args = dict(heads=heads, kv_heads=kv_heads, head_dim=d, k_cache=k_cache, v_cache=v_cache, page_size=page_size,
                block_tables=table, positions=torch.full((rows,), n - 1, dtype=torch.int32).cuda(),
                row_seq=torch.arange(rows, dtype=torch.int32).cuda(), cu_seqlens=None, seq_starts=None, single_rows=None,
                n_seqs=rows, max_query=1, max_context=n, scale=1.0, window=None)
    want = values_of(histories, row_seq, targets, heads, kv_heads)
    torch.testing.assert_close(ops.paged_attention(q, **args).float().cpu(), want, atol=1e-6, rtol=0)
    lazy = ops.paged_attention(q, unmerged=True, **args)                      # merged by the output projection's kernel
    assert isinstance(lazy, ops.Unmerged)
    torch.testing.assert_close(lazy.merge().float().cpu(), want, atol=1e-6, rtol=0)


def test_fused_decode_kernel_finds_one_key_also_the_one_in_registers(ops):
    """The decode kernel that makes its own queries (no norm and no rotation here, so the queries can be aimed):
    dominant keys at the edges of parts and steps in the pages, and the step's own new key, which the kernel
    holds in registers and writes into the pages."""
    page_size, d, heads, kv_heads, n = 16, 128, 8, 2, 1500
    targets = [0, 255, 256, 511, 512, 1471, 1472, n - 2, n - 1, n - 1]
    rows, total = len(targets), heads + 2 * kv_heads
    k_cache, v_cache, table, histories = build_cache([n] * rows, page_size, kv_heads, d, torch.bfloat16)
    row_seq = list(range(rows))
    q = pointed_queries(histories, row_seq, targets, heads, kv_heads, d, torch.float32)
    new_k = torch.stack([h[0][n - 1].float().reshape(-1) for h in histories]).cuda()        # the newest token's key and value
    new_v = torch.stack([h[1][n - 1].float().reshape(-1) for h in histories]).cuda()
    whole = torch.cat([q, new_k, new_v], dim=1)
    qkv = ops.Partials(torch.stack([0.25 * whole, 0.75 * whole]).contiguous())                # two partial sums of it
    positions = torch.full((rows,), n - 1, dtype=torch.int32).cuda()
    j = n - 1
    k_cache[table[:, j // page_size].long(), :, j % page_size] = float('nan')                 # the pages do not hold it yet
    v_cache[table[:, j // page_size].long(), :, :, j % page_size] = float('nan')
    sizes = dict(heads=heads, kv_heads=kv_heads, head_dim=d)
    assert ops.decode_attention_takes(qkv, page_size=page_size, rotation=None, dtype=torch.bfloat16, **sizes)
    assert ops._decode_parts(rows, kv_heads, n)[1] > 1
    got = ops.decode_attention(qkv, q_weight=None, k_weight=None, eps=0.0, rotation=None, positions=positions, writes=True,
                               k_cache=k_cache, v_cache=v_cache, page_size=page_size, block_tables=table,
                               row_seq=torch.arange(rows, dtype=torch.int32).cuda(), max_context=n, scale=1.0, window=None,
                               **sizes)
    torch.testing.assert_close(got.float().cpu(), values_of(histories, row_seq, targets, heads, kv_heads), atol=1e-6, rtol=0)
    written = k_cache[table[:, j // page_size].long(), :, j % page_size].float().cpu()
    torch.testing.assert_close(written, torch.stack([h[0][j].float() for h in histories]), atol=0, rtol=0)


@pytest.mark.parametrize('length,chunk,split', [(700, 100, (64, 2)), (300, 300, None), (2048, 128, None)])
def test_prompt_kernels_find_one_key_at_the_edges_of_tiles_and_parts(ops, monkeypatch, length, chunk, split):
    """bfloat16 prompt attention (32 x 32 tiles; keys in one piece or in parts that are merged): every row aims at
    one key, in turn the first, the ends of 32- and 64-key tiles, its own key and the one before it."""
    page_size, d, heads, kv_heads = 16, 128, 4, 2
    if split is not None:
        monkeypatch.setattr(ops, 'TILE_KEY_PARTS', split)
    k_cache, v_cache, table, histories = build_cache([length], page_size, kv_heads, d, torch.bfloat16)
    start = length - chunk
    fixed = [0, 31, 32, 63, 64, 127, 128, 191, 192]
    targets = []
    for i in range(chunk):
        position = start + i
        choices = [t for t in fixed + [start - 1, start] if 0 <= t <= position] + [position, max(position - 1, 0)]
        targets.append(choices[i % len(choices)])
    row_seq = [0] * chunk
    q = pointed_queries(histories, row_seq, targets, heads, kv_heads, d, torch.bfloat16)
    dev = lambda values: torch.tensor(values, dtype=torch.int32).cuda()
    if split is None and length > 1000:
        parts = ops.tile_key_parts(ops.library.load(), torch.bfloat16, 1, chunk, heads, kv_heads, d, page_size,
                                   table.shape[1], length)[1]
        assert parts > 1, 'a portion deep in a context: the split is chosen by itself'
    got = ops.paged_attention(q, heads=heads, kv_heads=kv_heads, head_dim=d, k_cache=k_cache, v_cache=v_cache,
                              page_size=page_size, block_tables=table, row_seq=dev(row_seq),
                              positions=dev(list(range(start, length))), cu_seqlens=dev([0, chunk]), seq_starts=dev([start]),
                              single_rows=dev([]), n_seqs=1, max_query=chunk, max_context=length, scale=1.0, window=None)
    torch.testing.assert_close(got.float().cpu(), values_of(histories, row_seq, targets, heads, kv_heads), atol=1e-6, rtol=0)


@pytest.mark.parametrize('dtype,d,page_size', [(torch.float32, 128, 16), (torch.float32, 40, 4), (torch.bfloat16, 96, 16)])
@pytest.mark.parametrize('length,chunk,split', [(700, 100, (64, 2)), (300, 300, None), (2048, 128, None)])
def test_general_tile_kernel_finds_one_key_at_the_edges_of_tiles_and_parts(ops, monkeypatch, dtype, d, page_size, length,
                                                                         chunk, split):
    """The general tile kernel (float32; bfloat16 sizes without a kernel of their own), keys in one piece or in
    parts that are merged: every row aims at one key, in turn the first, the ends of 32- and 64-key tiles and of
    the parts, its own key and the one before it."""
    heads, kv_heads = 4, 2
    if split is not None:
        monkeypatch.setattr(ops, 'TILE_KEY_PARTS', split)
    k_cache, v_cache, table, histories = build_cache([length], page_size, kv_heads, d, dtype)
    start = length - chunk
    fixed = [0, 31, 32, 63, 64, 127, 128, 191, 192, 255, 256]
    targets = []
    for i in range(chunk):
        position = start + i
        choices = [t for t in fixed + [start - 1, start] if 0 <= t <= position] + [position, max(position - 1, 0)]
        targets.append(choices[i % len(choices)])
    row_seq = [0] * chunk
    q = pointed_queries(histories, row_seq, targets, heads, kv_heads, d, dtype)
    dev = lambda values: torch.tensor(values, dtype=torch.int32).cuda()
    if split is None and length > 1000:
        part, parts = ops.tile_key_parts(ops.library.load(), dtype, 1, chunk, heads, kv_heads, d, page_size,
                                         table.shape[1], length)
        assert parts > 1 and part in (128, 192, 256), 'a portion deep in a context: the split is chosen by itself'
    got = ops.paged_attention(q, heads=heads, kv_heads=kv_heads, head_dim=d, k_cache=k_cache, v_cache=v_cache,
                              page_size=page_size, block_tables=table, row_seq=dev(row_seq),
                              positions=dev(list(range(start, length))), cu_seqlens=dev([0, chunk]), seq_starts=dev([start]),
                              single_rows=dev([]), n_seqs=1, max_query=chunk, max_context=length, scale=1.0, window=None)
    torch.testing.assert_close(got.float().cpu(), values_of(histories, row_seq, targets, heads, kv_heads), atol=1e-6, rtol=0)


def test_sampling(ops):
    vocab = 151936
    logits = rand(5, vocab, scale=2.0)
    logits[0, 70000] = logits[0, 123] = 50.0             # tie: lowest index wins (qil/engine.py:100)
    logits[3] = logits[2]                                # the same logits, seed and temperature: only the counter differs
    temperatures = torch.tensor([0.0, 0.0, 0.8, 0.8, 1.7]).cuda()
    seeds = torch.tensor([0, 0, 11, 11, -5], dtype=torch.int32).cuda()
    counters = torch.tensor([0, 0, 3, 4, 9], dtype=torch.int32).cuda()
    tokens, finite = ops.sample(logits, temperatures, seeds, counters)
    assert finite.tolist() == [1] * 5
    assert tokens[0].item() == 123 and tokens[1].item() == logits[1].argmax().item()
    scores = refs.sample_scores(logits.cpu(), temperatures.cpu(), seeds.cpu(), counters.cpu())
    for row in range(2, 5):                               # the drawn token is the reference's, or within float noise of it
        assert scores[row, tokens[row].item()] >= scores[row].max() - 1e-4
    assert tokens[2].item() != tokens[3].item()          # different counters draw independently (the two best scores of each row lie 0.5 apart)
    assert scores[2].argmax().item() != scores[3].argmax().item()
    again, _ = ops.sample(logits, temperatures, seeds, counters)
    assert again.tolist() == tokens.tolist()
    logits[3, 5] = float('nan')
    logits[1, 9] = float('inf')
    _, finite = ops.sample(logits, temperatures, seeds, counters)
    assert finite.tolist() == [1, 0, 1, 0, 1]


def test_sampling_frequencies(ops):
    """Many draws with different counters follow softmax(logits / T)."""
    vocab, draws, t = 7, 4000, 0.7
    row = torch.tensor([0.1, 1.2, -0.5, 2.0, 0.0, 1.9, -3.0])
    logits = row.repeat(draws, 1).cuda()
    tokens, _ = ops.sample(logits, torch.full((draws,), t).cuda(), torch.full((draws,), 42, dtype=torch.int32).cuda(),
                           torch.arange(draws, dtype=torch.int32).cuda())
    observed = torch.bincount(tokens.cpu().long(), minlength=vocab).float() / draws
    expected = torch.softmax(row / t, dim=0)
    assert (observed - expected).abs().max() < 4 * (expected * (1 - expected) / draws).sqrt().max() + 1e-3


def test_sizes_the_kernels_refuse(ops):
    with pytest.raises(ValueError):
        ops.check_attention_geometry(heads=4, kv_heads=2, head_dim=264, dtype=torch.bfloat16)
    with pytest.raises(ValueError):
        ops.check_attention_geometry(heads=5, kv_heads=2, head_dim=32, dtype=torch.bfloat16)
    with pytest.raises(ValueError):
        ops.check_attention_geometry(heads=4, kv_heads=2, head_dim=32, dtype=torch.float16)
    with pytest.raises(RuntimeError):
        ops.embed(torch.zeros(2, dtype=torch.int32), torch.zeros(4, 8))     # CPU tensors: no fallback


def test_device_info_is_what_the_plans_assume(ops, capfd):
    """The library asks the runtime for the compute units and the LDS of the GPU; on the MI355X the tests run on they
    are what the kernels' plans were made for, and the loader has nothing to warn about."""
    import ctypes
    from qil_amd.ops import library
    units, lds = ctypes.c_int(0), ctypes.c_int(0)
    assert library.load().qil_device_info(ctypes.byref(units), ctypes.byref(lds)) == 0
    assert units.value == library.PLANNED_COMPUTE_UNITS and lds.value >= library.PLANNED_LDS_BYTES, (units.value, lds.value)
    library._device_checked = False
    library.check_device()
    assert 'compute units' not in capfd.readouterr().err
