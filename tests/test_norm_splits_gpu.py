"""The norm that adds a product's partial sums, at the widths and numbers of splits where its form changes, against float64."""
import pytest
import torch

from test_kernels_gpu import rand

pytestmark = pytest.mark.gpu


@pytest.fixture(scope='module')
def ops():
    from qil_amd import ops
    ops.library.load()
    return ops


# the last width of every block size, one vector less and one more; every number of splits asked for at once, one less and one more
@pytest.mark.parametrize('width', [4, 252, 256, 260, 1024, 1028, 1152, 2048, 2052, 2560, 4096, 4100, 5120, 8192])
@pytest.mark.parametrize('splits', [1, 2, 3, 4, 5, 8, 9, 15, 16, 17])
def test_sums_and_norms(ops, width, splits):
    n, eps = 3, 1e-6
    stream, weight = rand(n, width, seed=1), 1 + 0.1 * rand(width, seed=2)
    parts = ops.Partials(rand(splits, n, width, scale=splits ** -0.5, seed=3))
    total = stream.double() + parts.tensor.double().sum(0)
    want = total / (total.square().mean(1, keepdim=True) + eps).sqrt() * weight.double()
    # a float32 sum of `splits` + 1 values of size one: splits 2^-24 of the largest partial sum, ample in 4e-7 splits^0.5 + 4e-7
    near = dict(atol=4e-7 * (1 + splits ** 0.5) * 4, rtol=1e-6)
    rows = torch.tensor([2, 0], dtype=torch.int32).cuda()
    before = stream.clone()
    picked = ops.rows_rmsnorm(stream, parts, rows, weight, eps, torch.float32)
    assert torch.equal(stream, before)
    torch.testing.assert_close(picked.double(), want[[2, 0]], **near)
    got = ops.add_rmsnorm(stream, parts, weight, eps, torch.float32)
    torch.testing.assert_close(got.double(), want, **near)
    torch.testing.assert_close(stream.double(), total, **near)
    half = ops.add_rmsnorm(before, parts, weight, eps, torch.bfloat16)
    torch.testing.assert_close(half.double(), want, atol=1e-6, rtol=2.0 ** -7)       # two roundings to bfloat16
