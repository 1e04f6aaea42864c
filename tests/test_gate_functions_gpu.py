"""Gated products with every gate function in their epilogue, in each kernel that has one, against float64."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope='module')
def ops():
    from qil_amd import ops
    ops.library.load()
    return ops


def rand(*shape, seed, scale=1.0, dtype=torch.bfloat16):
    g = torch.Generator().manual_seed(seed)
    return (torch.randn(*shape, generator=g) * scale).to(dtype).cuda()


def gate(g, u, activation, limit, alpha):
    if activation == 'clamped_swish':
        g, u = g.clamp(max=limit), u.clamp(-limit, limit)
        return g * torch.sigmoid(alpha * g) * (u + 1)
    return torch.relu(g) * u if activation == 'relu' else g * torch.sigmoid(g) * u


# one, eight and sixteen rows (the few-row kernel), 17 and 64 (16 x 16 stages; 32 x 32 tiles where there are columns enough), 65 and
# 256 (tiles), 300 and 600 (blocks of 128), each with as many columns as the kernel asks for
@pytest.mark.parametrize('activation,limit,alpha', [('silu', 0.0, 1.0), ('clamped_swish', 1.5, 1.702), ('relu', 0.0, 1.0)])
@pytest.mark.parametrize('m,inner,k,kernel', [(1, 48, 256, 'few'), (8, 6144, 512, 'few'), (16, 1040, 1024, 'few'), (17, 8192, 384, 'chunks'),
                                              (64, 8208, 512, 'chunks'), (65, 12288, 256, 'mid'), (256, 12304, 256, 'mid'), (300, 1536, 512, 'wide'),
                                              (600, 3072, 256, 'wide')])
def test_every_gate_function_inside_the_product(ops, activation, limit, alpha, m, inner, k, kernel):
    lib = ops.library.load()
    takes = {'few': lambda: lib.qil_gemm_bf16_gated_takes(m, inner, k, 1), 'chunks': lambda: lib.qil_gemm_bf16_gated_takes(m, inner, k, 1),
             'mid': lambda: lib.qil_gemm_bf16_mid_gated_takes(m, inner, k), 'wide': lambda: lib.qil_gemm_bf16_wide_gated_takes(m, inner, k)}
    assert takes[kernel]()
    x, w = rand(m, k, seed=m), rand(2 * inner, k, seed=inner, scale=2 * k ** -0.5)
    both = ops.interleave_gate_up(w[:inner].contiguous(), w[inner:].contiguous())
    out = torch.full((m, inner), float('nan'), dtype=torch.bfloat16, device='cuda')
    args = (x.data_ptr(), both.data_ptr(), out.data_ptr(), m, inner, k, 1)
    act = (ops.GATE_FUNCTIONS[activation], limit, alpha, torch.cuda.current_stream().cuda_stream)
    if kernel in ('few', 'chunks'):
        assert lib.qil_gemm_bf16_gated_act(*args, 0, 0, 1, *act) == 0
    else:
        assert (lib.qil_gemm_bf16_mid_gated_act if kernel == 'mid' else lib.qil_gemm_bf16_wide_gated_act)(*args, *act) == 0
    g, u = (x.double() @ w[:inner].double().t(), x.double() @ w[inner:].double().t())
    want = gate(g, u, activation, limit, alpha)
    # gate and up of size two: float32 sums of k products within 1e-6 k^0.5, an activation of slope up to about |g| + |u| <= 16, then
    # one rounding to bfloat16
    near = dict(atol=5e-4, rtol=2.0 ** -8)
    torch.testing.assert_close(out.double(), want, **near)
    through = ops.gated_linear(x, both, interleaved=True, activation=activation, limit=limit, alpha=alpha)
    separate = ops.gated_act(ops.Partials(torch.cat([g, u], 1).float()[None]), torch.bfloat16, activation=activation, limit=limit, alpha=alpha) \
        if kernel != 'wide' else None                            # (a wide product may be the library's, rounded before its activation)
    if separate is not None:
        torch.testing.assert_close(through.double(), separate.double(), atol=1e-3, rtol=2.0 ** -7)
    # operands that do not begin at multiples of 16 bytes are taken as before
    if m == 8 and activation != 'silu':
        shifted = torch.empty(m * k + 1, dtype=torch.bfloat16, device='cuda')[1:].view(m, k).copy_(x)
        torch.testing.assert_close(ops.gated_linear(shifted, both, interleaved=True, activation=activation, limit=limit, alpha=alpha).double(),
                                   want, atol=5e-4, rtol=2.0 ** -7)


def test_gate_functions_that_do_not_exist(ops):
    lib, x = ops.library.load(), rand(8, 256, seed=1)
    w, out = rand(96, 256, seed=2), rand(8, 48, seed=3)
    raw = torch.cuda.current_stream().cuda_stream
    for act in (-1, 3, 16):
        assert lib.qil_gemm_bf16_gated_act(x.data_ptr(), w.data_ptr(), out.data_ptr(), 8, 48, 256, 1, 0, 0, 1, act, 0.0, 1.0, raw) == -1


def test_silu_looks_at_no_numbers(ops):
    x, w = rand(3, 256, seed=1), rand(512, 256, seed=3, scale=0.06)
    for interleaved in (False, True):
        got = ops.gated_linear(x, w, interleaved=interleaved, limit=None, alpha=None)
        assert torch.equal(got, ops.gated_linear(x, w, interleaved=interleaved))
