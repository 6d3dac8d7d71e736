"""The token quantiser of the FP8 linear: few rows take a workgroup a row, more rows the weights' kernels.  Either way the linear has the
bits of the weights' quantiser in front of the scaled product."""
import pytest
import torch

from cosmos_rl_amd import ops
from oracle import fp8_oracle as O

pytestmark = pytest.mark.gpu


# rows on either side of the line (1280 up to 4096 columns, 256 beyond), one to four vectors a thread, the last of them partly filled
@pytest.mark.parametrize("K,rows", [(512, (5, 33)), (528, (5, 1280, 1281)), (1040, (7, 100)), (2064, (1280, 1281)), (4096, (64,)), (4112, (5, 256, 257)), (8208, (17, 256, 257)),
                                    (16400, (256,)), (18944, (33, 257)), (32768, (9,)), (32784, (9,))])
def test_linear_has_the_bits_of_the_two_steps(dev, K, rows):
    q, s = ops.quant_rowwise(O.make_weight((32, K), seed=3).to(dev))
    for M in rows:
        x = O.make_activation(M, K, seed=M, chan_outlier_frac=0.005, outlier_mul=30.0).to(dev)
        x[0], x[1, 0], x[2, K - 1], x[3, 5] = 0.0, float("inf"), float("nan"), -3e38
        wide = torch.zeros(M, K + 8, dtype=torch.bfloat16, device=dev)
        wide[:, :K] = x
        qx, sx = ops.quant_rowwise(x)
        want = ops.scaled_mm(qx, q.t(), sx, s, out_dtype=torch.float32)
        for y in (x, wide[:, :K]):
            got = ops.fp8_linear(y, q.t(), s, out_dtype=torch.float32)
            assert torch.equal(got.isnan(), want.isnan()) and torch.equal(got.nan_to_num(7.0), want.nan_to_num(7.0)), M
