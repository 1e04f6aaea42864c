"""Products that add into the stream in groups of eight columns: few rows of few columns, against float64."""
import pytest
import torch

from test_kernels_gpu import rand

pytestmark = pytest.mark.gpu


@pytest.fixture(scope='module')
def ops():
    from qil_amd import ops
    ops.library.load()
    return ops


# one, odd and eight rows; the fewest and most columns that take groups of eight, the least K a wave can have and one stage more;
# one column group more than that, one row more, a K that eight waves cannot share: groups of sixteen
@pytest.mark.parametrize('m,n,k,narrow', [(1, 1024, 3072, True), (3, 512, 3072, True), (8, 2048, 6144, True), (5, 1040, 4096, True), (8, 528, 7168, True),
                                          (8, 2064, 3072, False), (9, 1024, 3072, False), (8, 1024, 3200, False), (8, 496, 3072, False),
                                          (8, 1024, 2048, False)])
def test_adds_in_groups_of_eight_columns(ops, m, n, k, narrow):
    lib = ops.library.load()
    assert lib.qil_gemm_bf16_add_takes(m, n, k)
    x, w = rand(m, k, dtype=torch.bfloat16), rand(n, k, dtype=torch.bfloat16, seed=3, scale=k ** -0.5)
    before = rand(m, n, scale=2.0, seed=7)
    stream = before.clone()
    added = ops.linear(x, w, None, partials=True, add_to=stream)
    columns = 8 if narrow else 16
    assert isinstance(added, ops.Added) and added.squares.shape == (n // columns, m)
    # a float32 sum of k products of unit variance: 1e-6 sqrt(log k) of it on average, and an addition to values of size two
    torch.testing.assert_close(stream.double(), before.double() + x.double() @ w.double().t(), atol=2e-5, rtol=1e-5)
    pieces = stream.double().square().reshape(m, n // columns, columns).sum(-1).t()
    torch.testing.assert_close(added.squares.double(), pieces, atol=1e-5, rtol=1e-5)
    # the product behind it takes the norm from as many pieces as there are
    weight, q = 1 + 0.1 * rand(n, seed=5), rand(256, n, dtype=torch.bfloat16, seed=6, scale=n ** -0.5)
    normed = ops.Normed(stream, weight, 1e-6, torch.bfloat16, added)
    got = ops.linear(normed, q, None, partials=True)
    want = ops.linear(ops.add_rmsnorm(stream, None, weight, 1e-6, torch.bfloat16), q, None, partials=True)
    value = lambda y: y.tensor.sum(0) if isinstance(y, ops.Partials) else y.float()
    torch.testing.assert_close(value(got), value(want), atol=2.0 ** -6, rtol=2.0 ** -7)


@pytest.mark.parametrize('m,n,k', [(1, 1024, 3072), (8, 2048, 6144), (9, 1024, 3072)])
def test_adds_by_the_older_entry_leave_pieces_of_sixteen(ops, m, n, k):
    """qil_gemm_bf16_add writes N / 16 pieces a row whatever the sizes, and nothing behind them."""
    lib = ops.library.load()
    x, w = rand(m, k, dtype=torch.bfloat16), rand(n, k, dtype=torch.bfloat16, seed=3, scale=k ** -0.5)
    stream, squares = rand(m, n, scale=2.0, seed=7), torch.full((n // 8, m), 7.0, device='cuda')
    want = stream.double() + x.double() @ w.double().t()
    assert lib.qil_gemm_bf16_add(x.data_ptr(), w.data_ptr(), stream.data_ptr(), squares.data_ptr(), m, n, k, 0, 0, ops._stream()) == 0
    # as above: a float32 sum of k products of unit variance, added to values of size two
    torch.testing.assert_close(stream.double(), want, atol=2e-5, rtol=1e-5)
    pieces = stream.double().square().reshape(m, n // 16, 16).sum(-1).t()
    torch.testing.assert_close(squares[:n // 16].double(), pieces, atol=1e-5, rtol=1e-5)
    assert (squares[n // 16:] == 7).all()
