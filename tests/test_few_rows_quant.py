"""The token quantiser of the FP8 linear: few rows take a workgroup a row, more rows the weights' kernels.  Either way the linear has the
bits of the weights' quantiser in front of the scaled product."""
import pytest
import torch

from cosmos_rl_amd import _lib, ops
from oracle import fp8_oracle as O

pytestmark = pytest.mark.gpu


# rows on either side of the line (768 up to 1024 columns, 1200 from 2064 to 2552, 1280 up to 4096, 256 beyond), one to four vectors a thread, the last of them partly filled
@pytest.mark.parametrize("K,rows", [(512, (5, 33)), (528, (5, 768, 769)), (1040, (7, 1280, 1281)), (2064, (1200, 1201)), (2560, (1280, 1281)), (4096, (64,)), (4112, (5, 256, 257)), (8208, (17, 256, 257)),
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


# one launch for up to 4 tokens: 4, 8 or 16 weight rows a workgroup, by 1024 and 2048 rows and 256 and 2048 columns, beside the two steps
@pytest.mark.parametrize("N,K", [(16, 128), (64, 256), (64, 384), (16, 2176), (1008, 2048), (1024, 2176), (1024, 4096), (1040, 4096), (2048, 896), (2064, 2176), (896, 4864), (2048, 8192), (1040, 8192)])
@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32])
def test_one_launch_linear(dev, N, K, dt):
    w = O.make_weight((N, K), seed=4).to(dev)
    q, s = ops.quant_rowwise(w)
    spread = torch.zeros(N, K + 128, dtype=torch.uint8, device=dev)   # rows that do not follow each other
    spread[:, :K] = q.view(torch.uint8)
    apart = spread.view(torch.float8_e4m3fn)[:, :K]
    bias = torch.randn(N, device=dev).to(torch.bfloat16)
    for M in (1, 2, 3, 4) if K <= 4096 else (1,):
        x = O.make_activation(M, K, seed=M, chan_outlier_frac=0.005, outlier_mul=30.0).to(dev)
        qx, sx = ops.quant_rowwise(x)
        for weight in (q, apart):
            for b in (None, bias):
                assert torch.equal(ops.fp8_linear(x, weight.t(), s, bias=b, out_dtype=dt), ops.scaled_mm(qx, q.t(), sx, s, bias=b, out_dtype=dt)), M


# up to 16 tokens: 4, 8 or 16 weight rows a workgroup, one and several chunks of K; a column's bits do not depend on how many rows lie beside it
@pytest.mark.parametrize("K", [128, 384, 896, 2048, 2176, 4864, 8192])
@pytest.mark.parametrize("M", [1, 2, 5, 16])
def test_product_of_few_tokens(dev, M, K):
    q, s = ops.quant_rowwise(O.make_weight((4096, K), seed=6).to(dev))
    x = O.make_activation(M, K, seed=M)
    qx, sx = ops.quant_rowwise(x.to(dev))
    call = _lib.load().cfp8_scaled_mm_rowwise   # (the kernel for 16 tokens whatever the shape)

    def product(rows, dt):
        out = torch.zeros(M, rows, dtype=dt, device=dev)
        _lib.check(call(qx.data_ptr(), K, sx.data_ptr(), q.data_ptr(), K, s.data_ptr(), out.data_ptr(), rows, _lib.OUT_F32 if dt == torch.float32 else _lib.OUT_BF16,
                        M, rows, K, torch.cuda.current_stream().cuda_stream))
        return out
    for dt in (torch.bfloat16, torch.float32):
        whole = product(4096, dt)
        for rows in (16, 1008, 1024, 1040, 2048, 2064):
            assert torch.equal(product(rows, dt), whole[:, :rows])
    want = O.fp8_linear_rowwise(x, q.view(torch.uint8).cpu()[:1040], s.cpu()[:1040], accum=torch.float64)
    # (fp32 sums of K products against 64 bits)
    assert O.rel_frobenius(product(1040, torch.float32).cpu(), want) < 1e-3


# wide weights, one launch of streams: one K step, fewer and more than a wave has in flight, odd and even numbers of them, the longest; a last workgroup with waves beyond N
@pytest.mark.parametrize("N,K", [(12304, 2176), (16384, 128), (28688, 384), (18944, 640), (16400, 4096), (13312, 2048), (37888, 1152)])
def test_wide_linear_as_streams_has_the_bits_of_the_two_steps(dev, N, K):
    g = torch.Generator(device=dev).manual_seed(N + K)
    w = (torch.randn(N, K, generator=g, device=dev) * 0.05).to(torch.bfloat16)
    q, s = ops.quant_rowwise(w)
    mq, ms = ops.quant_mxfp4(w)
    bias = torch.randn(N, generator=g, device=dev).to(torch.bfloat16)
    for M in (1, 2, 3, 4):
        for kind, name in ((_lib.DISPATCH_LINEAR, "linear_stream"), (_lib.DISPATCH_LINEAR_MXFP4, "linear_mxfp4_stream")):
            assert _lib.gemm_dispatch_info(kind, M, N, K, cus=torch.cuda.get_device_properties(dev).multi_processor_count, flags=_lib.DISPATCH_SPLIT).startswith(name)
        x = torch.randn(M, K + 16, generator=g, device=dev).to(torch.bfloat16)[:, :K]   # a pitch of its own
        if M == 4:
            x[1, 3], x[2] = float("nan"), 0.0
        qx, sx = ops.quant_rowwise(x.contiguous())
        for dt in (torch.bfloat16, torch.float32):
            for b in (None, bias):
                got, want = ops.fp8_linear(x, q.t(), s, bias=b, out_dtype=dt), ops.scaled_mm(qx, q.t(), sx, s, bias=b, out_dtype=dt)
                assert torch.equal(got.isnan(), want.isnan()) and torch.equal(got.nan_to_num(7.0), want.nan_to_num(7.0)), M
            got, want = ops.linear_mxfp4(x, (mq, ms), dt), ops.gemm_mxfp4((qx, sx), (mq, ms), dt)
            assert torch.equal(got.isnan(), want.isnan()) and torch.equal(got.nan_to_num(7.0), want.nan_to_num(7.0)), M


def test_wide_linear_of_one_token_up_to_8192_columns(dev):
    g = torch.Generator(device=dev).manual_seed(5)
    q, s = ops.quant_rowwise((torch.randn(12800, 8192, generator=g, device=dev) * 0.05).to(torch.bfloat16))
    x = torch.randn(1, 8192, generator=g, device=dev).to(torch.bfloat16)
    qx, sx = ops.quant_rowwise(x)
    assert torch.equal(ops.fp8_linear(x, q.t(), s), ops.scaled_mm(qx, q.t(), sx, s, out_dtype=torch.bfloat16))


# weights and scales inside rows of their own pitch, whose other bytes are NaN in e4m3, the largest codes and NaN scales; the last row ends with its memory.  Odd numbers of K steps:
# MXFP4 weights are loaded by two, and an odd last one ends in the middle of a load (which bytes are read is a static_assert in gemm_ring_few.h)
@pytest.mark.parametrize("N,K", [(8224, 128), (8224, 384), (12304, 640), (12304, 3968), (8208, 4096)])
@pytest.mark.parametrize("M", [1, 4])
def test_wide_linear_of_weights_with_a_pitch(dev, M, N, K):
    took = _lib.gemm_dispatch_info(_lib.DISPATCH_LINEAR_MXFP4, M, N, K, cus=torch.cuda.get_device_properties(dev).multi_processor_count, flags=_lib.DISPATCH_SPLIT)
    assert took.startswith("linear_mxfp4_stream "), took
    g = torch.Generator(device=dev).manual_seed(N + K + M)
    x = torch.randn(M, K, generator=g, device=dev).to(torch.bfloat16)
    w = (torch.randn(N, K, generator=g, device=dev) * 0.05).to(torch.bfloat16)

    def pitched(t, more, filler):
        whole = torch.full((N, t.shape[1] + more), filler, dtype=torch.uint8, device=dev)
        whole[:, more:] = t.view(torch.uint8)
        return whole[:, more:]

    (q, s), (mq, ms) = ops.quant_rowwise(w), ops.quant_mxfp4(w)
    pq, pmq, pms = pitched(q, 48, 0x7F), pitched(mq, 64, 0x77), pitched(ms, 3, 0xFF)
    lib, st = _lib.load(), torch.cuda.current_stream().cuda_stream
    work = torch.empty(lib.cfp8_linear_workspace_bytes(M, K), dtype=torch.uint8, device=dev)
    for dt in (torch.bfloat16, torch.float32):
        out = torch.full((M, N + 8), 7.0, dtype=dt, device=dev)
        _lib.check(lib.cfp8_linear_mxfp4(x.data_ptr(), K, pmq.data_ptr(), pmq.stride(0), pms.data_ptr(), pms.stride(0), out.data_ptr(), N + 8, ops._out_code(dt), M, N, K, None, 0, st))
        assert torch.equal(out[:, :N], ops.linear_mxfp4(x, (mq, ms), dt)) and bool((out[:, N:] == 7.0).all())
        out.fill_(7.0)
        _lib.check(lib.cfp8_linear_rowwise_split(x.data_ptr(), K, pq.data_ptr(), pq.stride(0), s.data_ptr(), None, out.data_ptr(), N + 8, ops._out_code(dt), M, N, K,
                                                 work.data_ptr(), work.numel(), st))
        assert torch.equal(out[:, :N], ops.fp8_linear(x, q.t(), s, out_dtype=dt)) and bool((out[:, N:] == 7.0).all())
