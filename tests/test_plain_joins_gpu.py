"""The residual join of plain bfloat16 products: the kernel with the row in registers at its narrowest and widest rows, and calls
just outside of what it takes, which the general kernel serves."""
import pytest
import torch

import kernel_refs as refs
from qil_amd import ops
from test_dogozen_kernels_gpu import close

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('two', [True, False])
@pytest.mark.parametrize('n,width,offset', [(3, 512, 16), (1, 1024, 0), (130, 2048, 8), (2, 8192, 16),      # in registers
                                            (3, 520, 16), (2, 8704, 16), (5, 512, 4), (5, 512, 3)])         # the general kernel
def test_join_of_plain_products(n, width, offset, two):
    g = torch.Generator().manual_seed(n * width + offset)
    value = lambda columns: torch.randn(n, columns, generator=g).to(torch.bfloat16)
    left, right, ffn, gates = value(width), value(width + 8), value(width), value(2 * width + 24)
    bias, stream, weight = torch.randn(2 * width, generator=g), torch.randn(n, width, generator=g), torch.rand(width, generator=g) + 0.5

    def joined(put):
        mixed = ops.Weighted(put(left), ops.columns(put(right), 8, width), 0.7, -1.3) if two else put(left)
        return ops.Joined(mixed, put(ffn), ops.columns(put(gates), offset, 2 * width), put(bias), None, None)
    want_stream, got_stream = stream.clone(), stream.cuda()
    want = refs.residual_join(want_stream, joined(lambda t: t), weight, 1e-5, torch.bfloat16)
    got = ops.residual_join(got_stream, joined(lambda t: t.cuda()), weight.cuda(), 1e-5, torch.bfloat16)
    torch.testing.assert_close(got_stream.cpu(), want_stream, atol=2e-5, rtol=2e-5)        # the stream is float32 in both
    close(got, want, torch.bfloat16, 2.0)
