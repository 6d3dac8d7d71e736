"""The decode linears of at most 16 tokens at the edges of their K steps: one to eight steps a wave, chunks beyond them,
and both sides of the limit of the one-launch form, against the fp64 oracle; one launch and two give the same bits."""
import pytest
import torch

from cosmos_rl_amd import ops
from oracle import fp8_oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("K", [128, 384, 640, 1024, 1152, 3968, 4096, 4224, 4864, 8192, 8320, 12416])
@pytest.mark.parametrize("M,N", [(1, 16), (2, 48), (4, 272), (16, 32)])
def test_k_steps(dev, M, N, K):
    g = torch.Generator().manual_seed(M * 100003 + K)
    x = (torch.randn(M, K, generator=g) * 2).to(torch.bfloat16)
    qw, sw = O.quant_rowwise((torch.randn(N, K, generator=g) * 0.05).to(torch.bfloat16))
    ref = O.fp8_linear_rowwise(x, qw, sw, accum=torch.float64)
    w = qw.to(dev).view(torch.float8_e4m3fn).t()
    out = ops.fp8_linear(x.to(dev), w, sw.to(dev), out_dtype=torch.float32)
    assert O.rel_frobenius(out.cpu(), ref) <= 1e-4  # the matrix pipe sums a K step with less than fp32 precision: 2e-5
    qx, sx = O.quant_rowwise(x)
    two = ops.scaled_mm(qx.to(dev).view(torch.float8_e4m3fn), w, sx.to(dev), sw.to(dev).t(), out_dtype=torch.float32)
    assert torch.equal(out, two)
