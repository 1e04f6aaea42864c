"""Products of more than 256 rows on this library's kernel: the block shapes that sizes choose, at their edges."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope='module')
def ops():
    from qil_amd import ops
    ops.library.load()
    return ops


def rand(*shape, dtype=torch.float32, scale=1.0, seed=0):
    g = torch.Generator().manual_seed(seed + sum(shape))
    return (torch.randn(*shape, generator=g) * scale).to(dtype).cuda()


# blocks of 128 x 128 with two blocks a CU; 128 x 128 alone on its CU with the longer ring, in one split and in
# several, with fewer stages than the ring holds, with rows and columns that fill no block
@pytest.mark.parametrize('m,n,k', [(1025, 6112, 1024), (700, 6144, 448), (643, 4096, 1024), (257, 1056, 128), (600, 992, 2048),
                                   (1000, 1024, 3072), (513, 2048, 192), (300, 4128, 576)])
def test_products_that_stay_off_the_blas(ops, monkeypatch, m, n, k):
    """``linear`` without and with partial sums and ``gated_linear``, against float64; no library product.

    A float32 sum of k products is off by at most about sqrt(k) 2^-24 of its terms' size; 3e-6 of the largest result
    covers k = 3072.  The bfloat16 result is one rounding of it: 2^-8 of itself."""
    lib = ops.library.load()
    monkeypatch.setattr(torch, 'mm', lambda *a, **kw: pytest.fail('a library product'))
    x, w = rand(m, k, dtype=torch.bfloat16), rand(n, k, dtype=torch.bfloat16, seed=1, scale=2.0 * k ** -0.5)
    want = x.double() @ w.double().t()
    largest = want.abs().max().item()
    if lib.qil_gemm_bf16_wide_splits(m, n, k, 0):
        got = ops.linear(x, w)
        assert got.dtype == torch.bfloat16
        torch.testing.assert_close(got.double(), want, atol=3e-6 * largest, rtol=2.0 ** -8)
    assert lib.qil_gemm_bf16_wide_splits(m, n, k, 1)
    got = ops.linear(x, w, partials=True)
    if isinstance(got, ops.Partials):
        torch.testing.assert_close(got.sum().double(), want, atol=3e-6 * largest, rtol=2e-5)
    else:
        torch.testing.assert_close(got.double(), want, atol=3e-6 * largest, rtol=2.0 ** -8)
    inner = n // 2
    if not lib.qil_gemm_bf16_wide_gated_wanted(m, inner, k):
        return
    both = ops.interleave_gate_up(w[:inner].contiguous(), w[inner:].contiguous())
    gated = ops.gated_linear(x, both, interleaved=True)
    want = torch.nn.functional.silu(want[:, :inner]) * want[:, inner:]
    torch.testing.assert_close(gated.double(), want, atol=3e-5 * want.abs().max().item(), rtol=2.0 ** -8)


def test_where_the_blas_takes_over(ops):
    lib = ops.library.load()
    for m, n, k in ((2048, 6144, 4096), (700, 4096, 12288), (4096, 6144, 1024), (600, 1000, 1024), (600, 1024, 1000)):
        assert lib.qil_gemm_bf16_wide_splits(m, n, k, 1) == 0
    assert not lib.qil_gemm_bf16_wide_gated_wanted(2048, 3072, 1024) and not lib.qil_gemm_bf16_wide_gated_wanted(256, 3072, 1024)


# (shape, splits): 0 blocks of 256 x 256, 1 of 128 x 128 with two a CU, 2 of 128 x 128 with the long ring.  Rows and columns that
# fill no block, K of fewer stages than a ring (5 or 9), of a number that ends anywhere in it, and long
@pytest.mark.parametrize('m,n,k,splits,shape', [(1400, 8224, 448, 1, 0), (2000, 4128, 1024, 1, 0), (700, 8224, 1024, 2, 0), (513, 8224, 128, 1, 1),
                                                (700, 6112, 192, 1, 1), (1000, 4128, 1024, 1, 1), (257, 6112, 1024, 2, 1), (257, 1056, 128, 1, 2),
                                                (700, 992, 1088, 1, 2), (300, 2080, 1024, 2, 2), (260, 96, 4096, 8, 2)])
def test_every_block_shape(ops, m, n, k, splits, shape):
    """The kernel alone, plain in bfloat16 and float32 and with the gate's epilogue in both, or its partial sums, against float64;
    bounds as in ``test_products_that_stay_off_the_blas`` (the gate multiplies two such sums: ten times the float32 bound)."""
    lib = ops.library.load()
    stream = torch.cuda.current_stream().cuda_stream
    assert lib.qil_gemm_bf16_wide_shape(m, n, k, splits) == shape
    x, w = rand(m, k, dtype=torch.bfloat16), rand(n, k, dtype=torch.bfloat16, seed=1, scale=2.0 * k ** -0.5)
    pieces = torch.stack([x[:, a:a + k // splits].double() @ w[:, a:a + k // splits].double().t() for a in range(0, k, k // splits)])
    largest = pieces.abs().max().item()
    if splits > 1:
        got = torch.full((splits, m, n), 7.0, device='cuda')
        assert lib.qil_gemm_bf16_wide(x.data_ptr(), w.data_ptr(), got.data_ptr(), m, n, k, 0, splits, stream) == 0
        torch.testing.assert_close(got.double(), pieces, atol=3e-6 * largest, rtol=2e-5)
        return
    want, inner = pieces[0], n // 2
    both = ops.interleave_gate_up(w[:inner].contiguous(), w[inner:].contiguous())
    gated = torch.nn.functional.silu(want[:, :inner]) * want[:, inner:]
    for dtype, code, close in ((torch.float32, 0, 2e-5), (torch.bfloat16, 1, 2.0 ** -8)):
        got = torch.full((m, n), 7.0, dtype=dtype, device='cuda')
        assert lib.qil_gemm_bf16_wide(x.data_ptr(), w.data_ptr(), got.data_ptr(), m, n, k, code, 1, stream) == 0
        torch.testing.assert_close(got.double(), want, atol=3e-6 * largest, rtol=close)
        got = torch.full((m, inner), 7.0, dtype=dtype, device='cuda')
        assert lib.qil_gemm_bf16_wide_gated(x.data_ptr(), both.data_ptr(), got.data_ptr(), m, inner, k, code, stream) == 0
        torch.testing.assert_close(got.double(), gated, atol=3e-5 * gated.abs().max().item(), rtol=close)
