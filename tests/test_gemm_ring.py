"""The ring GEMM (middle of the range of token counts) at the edges of its tiles, K steps and slices, through the entry points
that take memory for partial sums, against the dequantised product in float64."""
import pytest
import torch

from cosmos_rl_amd import _lib, ops

pytestmark = pytest.mark.gpu

# rows around a tile's 64 and 128, columns that end inside a wave's share, one K step and a few (the ring is 5 to 10 deep), odd
# and even numbers of steps, a last step of 32 .. 112; long K with few columns: slices
SHAPES = [(5, 16, 128), (17, 48, 384), (63, 144, 640), (64, 128, 1152), (65, 272, 896), (127, 80, 256), (128, 1040, 2304), (129, 256, 1280),
          (200, 400, 12800), (33, 208, 18944), (300, 4624, 512), (7, 4096, 4224)]
TAILS = [(70, 304, 160), (100, 80, 2880), (16, 400, 2208), (260, 272, 7264)]


def _out(M, N, dev, dtype):
    return torch.full((M + 1, N + 8), 7.0, dtype=dtype, device=dev)


def _check(out, want, M, N, dtype, slack):
    """fp32 sums within 1e-4 of the exact ones (the matrix pipe sums a K step with less than fp32 precision; measured 2e-5), bf16
    within 1e-3 of their bf16; nothing beyond M and N"""
    got = out[:M, :N].double().cpu()
    ref = want if dtype == torch.float32 else want.float().to(torch.bfloat16).double()
    assert float((got - ref).norm() / ref.norm()) <= (1e-4 if dtype == torch.float32 else 1e-3) + slack
    assert bool((out[M:] == 7.0).all()) and bool((out[:, N:] == 7.0).all())


def _partial(kind, M, N, K, dev):
    need = _lib.load().cfp8_gemm_partial_bytes(kind, M, N, K)
    return torch.empty(max(need, 256), dtype=torch.uint8, device=dev), need


def _stream():
    return torch.cuda.current_stream().cuda_stream


@pytest.mark.parametrize("M,N,K", SHAPES + TAILS)
def test_mxfp4(dev, M, N, K):
    from oracle import mxfp4_oracle as MX
    g = torch.Generator().manual_seed(M + N + K)
    x = torch.randn(M, K, generator=g).to(torch.bfloat16)
    q, s = ops.quant_rowwise(x.to(dev))
    w, ws = ops.quant_mxfp4((torch.randn(N, K, generator=g) * 0.05).to(torch.bfloat16).to(dev))
    want = MX.gemm(q.cpu(), s.cpu().reshape(-1), w.cpu(), ws.cpu()).double()
    part, need = _partial(_lib.DISPATCH_MXFP4, M, N, K, dev)
    for dtype in (torch.float32, torch.bfloat16):
        for have in {0, need // 2, need}:
            out = _out(M, N, dev, dtype)
            _lib.check(_lib.load().cfp8_gemm_mxfp4_split(q.data_ptr(), K, s.data_ptr(), w.data_ptr(), K // 2, ws.data_ptr(), K // 32, out.data_ptr(),
                                                         N + 8, ops._out_code(dtype), M, N, K, part.data_ptr(), have, _stream()))
            _check(out, want, M, N, dtype, 0.0)
