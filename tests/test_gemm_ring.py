"""The ring GEMM (middle of the range of token counts) at the edges of its tiles, K steps and slices, through the entry points
that take memory for partial sums, against the dequantised product in float64."""
import pytest
import torch

from cosmos_rl_amd import _lib, ops

pytestmark = pytest.mark.gpu

# rows around a tile's 64 and 128, columns that end inside a wave's share, one K step and a few (the ring is 3 to 8 deep), odd
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


def _rowwise_want(q, s, w, sw, bias):
    want = (q.double() * s.double().reshape(-1, 1)) @ (w.double() * sw.double().reshape(-1, 1)).t()
    return (want if bias is None else want + bias.double()).cpu()


# the shapes above, the streamers of few tokens, and thousands of rows with remainders of tiles of 128
@pytest.mark.parametrize("M,N,K", SHAPES + TAILS + [(1, 400, 1152), (3, 272, 4864), (16, 144, 4224), (90, 10256, 128), (4000, 4112, 384), (4096 + 120, 4096 + 112, 512),
                                                    (4096 + 130, 4096 + 144, 384), (2100, 9216, 640), (8000, 4352, 512)])
@pytest.mark.parametrize("biased", [False, True])
def test_rowwise(dev, M, N, K, biased):
    g = torch.Generator(device=dev).manual_seed(M + N + K)
    x = torch.randn(M, K, generator=g, device=dev).to(torch.bfloat16)
    q, s = ops.quant_rowwise(x)
    w, sw = ops.quant_rowwise((torch.randn(N, K, generator=g, device=dev) * 0.05).to(torch.bfloat16))
    bias = torch.randn(N, generator=g, device=dev).to(torch.bfloat16) if biased else None
    want = _rowwise_want(q, s, w, sw, bias)
    part, need = _partial(_lib.DISPATCH_ROWWISE, M, N, K, dev)
    for dtype in (torch.float32, torch.bfloat16):
        for have in {0, need // 2, need}:
            out = _out(M, N, dev, dtype)
            _lib.check(_lib.load().cfp8_scaled_mm_rowwise_split(q.data_ptr(), K, s.data_ptr(), w.data_ptr(), K, sw.data_ptr(), ops._ptr(bias),
                                                                out.data_ptr(), N + 8, ops._out_code(dtype), M, N, K, part.data_ptr(), have, _stream()))
            # (a bf16 product is rounded before the bias is added and the sum again: 2^-9 of it more at most)
            _check(out, want, M, N, dtype, 2.0 ** -9 if biased and dtype == torch.bfloat16 else 0.0)
            y = ops.fp8_linear(x, w.t(), sw, bias=bias, out_dtype=dtype)
            if have == need:
                assert torch.equal(y, out[:M, :N])
                if biased:
                    assert torch.equal(y, ops.fp8_linear(x, w.t(), sw, out_dtype=dtype) + bias)


# the walking 256 x 256 tiles with edges.  Remainders of rows (1, 6, 64, 129) and of columns (16, 144) as quarter tiles and as a last
# row or column of whole ones, each alone and both, with a partial last round dealt out as quarter tiles and without: (M, N, K), whether
# there is one, whether a remainder is quarter tiles
EDGES = [((2310, 12288, 512), False, False), ((2304, 18960, 640), False, False), ((2310, 12304, 512), False, False), ((2310, 12432, 512), False, False),
         ((2177, 18960, 640), False, False), ((2048, 8208, 1152), False, True), ((2048, 8336, 1152), True, False), ((2177, 8192, 1152), True, False),
         ((2049, 8208, 1152), True, True), ((2177, 8208, 1152), True, True), ((1536, 12304, 1152), True, True), ((1600, 12432, 1792), True, True),
         ((2049, 9216, 2560), True, True), ((2048, 8192, 640), False, False), ((2304, 8192, 1152), True, False)]


# (full tiles without a bias take the walking form without edges)
@pytest.mark.parametrize("shape,tail,quarters,biased", [(*e, b) for b in (False, True) for e in EDGES if b or e[0][0] % 256 or e[0][1] % 256])
def test_rowwise_edges(dev, shape, tail, quarters, biased):
    M, N, K = shape
    cus = torch.cuda.get_device_properties(dev).multi_processor_count
    took = _lib.gemm_dispatch_info(_lib.DISPATCH_ROWWISE, M, N, K, cus=cus, flags=_lib.DISPATCH_SPLIT | (_lib.DISPATCH_BIAS if biased else 0))
    assert took.startswith("gemm_rowwise_edge") and ("tail=0" not in took) == tail and ("edges=0" not in took) == quarters, took
    g = torch.Generator(device=dev).manual_seed(M + N + K)
    q, s = ops.quant_rowwise(torch.randn(M, K, generator=g, device=dev).to(torch.bfloat16))
    w, sw = ops.quant_rowwise((torch.randn(N, K, generator=g, device=dev) * 0.05).to(torch.bfloat16))
    bias = torch.randn(N, generator=g, device=dev).to(torch.bfloat16) if biased else None
    want = _rowwise_want(q, s, w, sw, bias)
    for dtype in (torch.float32, torch.bfloat16):
        runs = []
        for _ in range(3):  # (a missing wait between a tile's stores and the next one's loads would show as a difference)
            out = _out(M, N, dev, dtype)
            _lib.check(_lib.load().cfp8_scaled_mm_rowwise_split(q.data_ptr(), K, s.data_ptr(), w.data_ptr(), K, sw.data_ptr(), ops._ptr(bias),
                                                                out.data_ptr(), N + 8, ops._out_code(dtype), M, N, K, None, 0, _stream()))
            runs.append(out)
        assert torch.equal(runs[0], runs[1]) and torch.equal(runs[0], runs[2])
        _check(runs[0], want, M, N, dtype, 2.0 ** -9 if biased and dtype == torch.bfloat16 else 0.0)
        # the bits of the other kernels, cut along N into calls that the entry point without partial sums takes, the bias added as torch does
        cut = (N // 256 + 1) // 2 * 256
        parts = []
        for n0, n1 in ((0, cut), (cut, N)):
            o = torch.empty(M, n1 - n0, dtype=dtype, device=dev)
            _lib.check(_lib.load().cfp8_scaled_mm_rowwise(q.data_ptr(), K, s.data_ptr(), w[n0:].data_ptr(), K, sw[n0:].data_ptr(), o.data_ptr(), n1 - n0,
                                                          ops._out_code(dtype), M, n1 - n0, K, _stream()))
            parts.append(o if bias is None else o + bias[n0:n1])
        same = M if M % 256 == 0 or M % 256 > 16 else M // 256 * 256  # (the kernel for up to 16 rows adds the sums of four waves)
        assert torch.equal(runs[0][:same, :N], torch.cat(parts, 1)[:same])


@pytest.mark.parametrize("M,N,K", [(2310, 12304, 512), (33, 272, 256), (5, 48, 128)])
def test_rowwise_without_a_bias_keeps_the_sign_of_zero(dev, M, N, K):
    """Products that the scales take below the smallest fp32 number keep their sign: no bias is not a bias of +0."""
    g = torch.Generator(device=dev).manual_seed(M)
    sign = torch.where(torch.rand(M, 1, generator=g, device=dev) < 0.5, -1.0, 1.0)
    a = (sign * torch.ones(M, K, device=dev)).to(torch.float8_e4m3fn)
    b = torch.ones(N, K, device=dev).to(torch.float8_e4m3fn)
    out = ops.scaled_mm(a, b.t(), torch.full((M, 1), 1e-30, device=dev), torch.full((1, N), 1e-30, device=dev), out_dtype=torch.float32)
    assert not bool(out.any()) and torch.equal(torch.signbit(out), (sign < 0).expand(M, N))


def test_rowwise_bias_of_another_kind(dev):
    """A bias that no epilogue takes (fp32) is added as torch adds it."""
    x = torch.randn(5, 256, device=dev).to(torch.bfloat16)
    w, sw = ops.quant_rowwise(torch.randn(48, 256, device=dev).to(torch.bfloat16))
    b = torch.randn(48, device=dev)
    assert torch.equal(ops.fp8_linear(x, w.t(), sw, bias=b), ops.fp8_linear(x, w.t(), sw) + b)


# the shapes above, scales of a slice that do not fit beside the ring's stages on 128 rows (63 steps and more), full tiles with
# and without rows behind them
@pytest.mark.parametrize("M,N,K", SHAPES + [(1, 2048, 7168), (24, 18432, 1152), (70, 4112, 8192), (1000, 1536, 1664), (1024 + 5, 24576, 384), (2048 + 130, 12288, 2048)])
@pytest.mark.parametrize("kn", [False, True])
def test_block(dev, M, N, K, kn):
    g = torch.Generator(device=dev).manual_seed(M + N + K)
    q, s = ops.groupwise_activation_quant(torch.randn(M, K, generator=g, device=dev).to(torch.bfloat16))
    w = (torch.randn(N, K, generator=g, device=dev) * 0.05).to(torch.float8_e4m3fn)
    sw = torch.rand(-(-N // 128), K // 128, generator=g, device=dev) + 0.5
    want = ((q.double() * s.double().repeat_interleave(128, 1)) @ (w.double() * sw.double().repeat_interleave(128, 0)[:N].repeat_interleave(128, 1)).t()).cpu()
    sb, strides = (sw.t().contiguous(), (1, sw.shape[0])) if kn else (sw, (K // 128, 1))
    part, need = _partial(_lib.DISPATCH_BLOCK, M, N, K, dev)
    for dtype in (torch.float32, torch.bfloat16):
        for have in {0, need // 2, need}:
            out = _out(M, N, dev, dtype)
            _lib.check(_lib.load().cfp8_gemm_block128_split(q.data_ptr(), K, s.data_ptr(), w.data_ptr(), K, sb.data_ptr(), *strides, out.data_ptr(), N + 8,
                                                            ops._out_code(dtype), M, N, K, part.data_ptr(), have, _stream()))
            _check(out, want, M, N, dtype, 0.0)


# the tiles of the ring kernel for every weight format, with slices of K and without, with weights loaded as a stream (one row of tiles, and
# what else ring_once names) and cacheably, some with a last step of 64: the smallest products with remainders of rows and columns that
# the choice takes there
FORMS = [("block", 64, 64, False, 67, 208, 384), ("block", 64, 64, False, 5, 208, 384), ("block", 64, 64, True, 67, 208, 2176), ("block", 64, 64, True, 49, 208, 2176),
         ("block", 64, 128, False, 67, 9232, 384), ("block", 64, 128, False, 5, 52304, 256), ("block", 64, 128, True, 67, 2832, 5248), ("block", 128, 128, False, 138, 10960, 384),
         ("block", 128, 128, True, 67, 5648, 7296), ("mxfp4", 64, 64, False, 131, 208, 384), ("mxfp4", 64, 64, False, 19, 208, 640), ("mxfp4", 64, 64, True, 150, 208, 2432),
         ("mxfp4", 64, 64, True, 70, 208, 3584), ("mxfp4", 64, 64, True, 65, 80, 3520), ("mxfp4", 64, 128, False, 131, 9232, 384), ("mxfp4", 64, 128, False, 5, 208, 384),
         ("mxfp4", 64, 128, True, 131, 2064, 7296), ("mxfp4", 64, 128, True, 66, 208, 1792), ("mxfp4", 64, 128, True, 65, 80, 1728), ("mxfp4", 128, 64, False, 131, 5648, 384),
         ("mxfp4", 128, 64, False, 67, 9232, 640), ("mxfp4", 128, 64, False, 131, 5648, 448), ("mxfp4", 128, 64, False, 67, 9232, 448), ("mxfp4", 128, 64, True, 131, 1808, 5248),
         ("mxfp4", 128, 64, True, 67, 2832, 2944), ("mxfp4", 128, 128, False, 131, 11792, 384), ("mxfp4", 128, 128, False, 82, 16848, 256),
         ("mxfp4", 128, 128, False, 81, 16976, 320), ("mxfp4", 128, 128, True, 131, 2832, 7296), ("mxfp4", 128, 128, True, 67, 5648, 7296),
         ("mxfp4", 128, 128, True, 131, 2832, 7360), ("mxfp4", 128, 128, True, 67, 5648, 5312), ("rowwise", 64, 64, False, 67, 208, 384), ("rowwise", 64, 64, False, 34, 8656, 256),
         ("rowwise", 64, 64, False, 5, 80, 320), ("rowwise", 64, 64, True, 67, 208, 2176), ("rowwise", 64, 64, True, 51, 208, 2560), ("rowwise", 64, 64, True, 54, 80, 1728),
         ("rowwise", 64, 128, False, 131, 9232, 384), ("rowwise", 64, 128, False, 5, 58704, 256), ("rowwise", 64, 128, True, 131, 1808, 5248),
         ("rowwise", 64, 128, True, 131, 1808, 5312), ("rowwise", 64, 128, True, 17, 8912, 10624), ("rowwise", 64, 128, True, 17, 8704, 8896),
         ("rowwise", 128, 64, False, 131, 5648, 384), ("rowwise", 128, 64, False, 67, 9232, 384), ("rowwise", 128, 64, True, 1500, 208, 5248),
         ("rowwise", 128, 64, True, 67, 2832, 3712), ("rowwise", 128, 64, True, 1031, 208, 7360), ("rowwise", 128, 64, True, 67, 2832, 3776),
         ("rowwise", 128, 128, False, 515, 3600, 640), ("rowwise", 128, 128, False, 131, 11792, 704), ("rowwise", 128, 128, False, 67, 29072, 512),
         ("rowwise", 128, 128, False, 65, 25424, 704), ("rowwise", 128, 128, True, 131, 2832, 9344), ("rowwise", 128, 128, True, 67, 9232, 5248)]
# where the choice takes the form for few rows: tiles of 16 rows, strips of 16 weight rows a workgroup
FEW_FORMS = [("block", 1, 4, True, 5, 208, 2176), ("block", 1, 5, False, 5, 18448, 384), ("block", 1, 8, True, 5, 5648, 2432),
             ("block", 5, 5, False, 67, 18448, 384), ("mxfp4", 1, 4, True, 5, 208, 9344), ("mxfp4", 2, 8, True, 19, 208, 2176),
             ("mxfp4", 5, 5, False, 67, 18448, 384), ("rowwise", 1, 4, False, 5, 14864, 384), ("rowwise", 1, 4, True, 5, 208, 7296),
             ("rowwise", 1, 6, False, 5, 23568, 384), ("rowwise", 1, 8, True, 5, 5648, 7296), ("rowwise", 1, 8, True, 5, 5648, 3776),
             ("rowwise", 5, 6, False, 67, 23568, 640), ("rowwise", 5, 5, False, 67, 18448, 448)]


@pytest.mark.parametrize("kernel,mode,bm,bn,sliced,M,N,K", [("gemm_ring", *f) for f in FORMS] + [("gemm_ring_few", *f) for f in FEW_FORMS])
def test_every_form(dev, kernel, mode, bm, bn, sliced, M, N, K):
    from oracle import mxfp4_oracle as MX
    kind = {"rowwise": _lib.DISPATCH_ROWWISE, "block": _lib.DISPATCH_BLOCK, "mxfp4": _lib.DISPATCH_MXFP4}[mode]
    cus = torch.cuda.get_device_properties(dev).multi_processor_count
    took = _lib.gemm_dispatch_info(kind, M, N, K, cus=cus, flags=_lib.DISPATCH_SPLIT).split("; ")
    assert took[0].startswith(f"{kernel}<{mode},{bm},{bn}>") and ("slices=1 " not in took[0]) == sliced and len(took) == 1 + sliced, took
    g = torch.Generator(device=dev).manual_seed(M + N + K)
    x = torch.randn(M, K, generator=g, device=dev).to(torch.bfloat16)
    w = torch.randn(N, K, generator=g, device=dev) * 0.05
    if mode == "rowwise":
        a, b = ops.quant_rowwise(x), ops.quant_rowwise(w.to(torch.bfloat16))
        want = _rowwise_want(*a, *b, None)
        run = lambda dtype: ops.scaled_mm(a[0], b[0].t(), a[1], b[1].reshape(1, N), out_dtype=dtype)
    elif mode == "block":
        a = ops.groupwise_activation_quant(x)
        b = w.to(torch.float8_e4m3fn), torch.rand(-(-N // 128), K // 128, generator=g, device=dev) + 0.5
        want = ((a[0].double() * a[1].double().repeat_interleave(128, 1)) @
                (b[0].double() * b[1].double().repeat_interleave(128, 0)[:N].repeat_interleave(128, 1)).t()).cpu()
        run = lambda dtype: ops.gemm_fp8_fp8_bf16_nt(a, b, torch.empty(M, N, device=dev, dtype=dtype))
    else:
        a, b = ops.quant_rowwise(x), ops.quant_mxfp4(w.to(torch.bfloat16))
        want = MX.gemm(a[0].cpu(), a[1].cpu().reshape(-1), b[0].cpu(), b[1].cpu()).double()
        run = lambda dtype: ops.gemm_mxfp4(a, b, dtype)
    for dtype in (torch.float32, torch.bfloat16):
        ref = want if dtype == torch.float32 else want.float().to(torch.bfloat16).double()
        got = run(dtype).double().cpu()
        assert float((got - ref).norm() / ref.norm()) <= (1e-4 if dtype == torch.float32 else 1e-3)
        assert float((got - ref).abs().max()) <= (1e-3 if dtype == torch.float32 else 2.0 ** -7) * float(ref.abs().max())


def test_a_bias_that_torch_follows(dev):
    """the epilogue adds a bias only where nothing else would see the addition"""
    x = torch.randn(33, 256, device=dev).to(torch.bfloat16)
    q, s = ops.scaled_fp8_quant((torch.randn(384, 256, device=dev) * 0.05).to(torch.bfloat16), use_per_token_if_dynamic=True)
    bias = torch.randn(384, device=dev).to(torch.bfloat16)
    want = ops.fp8_linear(x, q.t(), s, bias=bias)
    learnt = torch.nn.Parameter(bias.clone())
    got = ops.fp8_linear(x, q.t(), s, bias=learnt)
    got.sum().backward()
    assert torch.equal(got.detach(), want) and bool((learnt.grad == 33).all())
    with torch.autograd.forward_ad.dual_level():
        dual = torch.autograd.forward_ad.make_dual(bias, torch.ones_like(bias))
        tangent = torch.autograd.forward_ad.unpack_dual(ops.fp8_linear(x, q.t(), s, bias=dual)).tangent
    assert tangent is not None and bool((tangent == 1).all())
    many = torch.func.vmap(lambda b: ops.fp8_linear(x, q.t(), s, bias=b))(torch.stack([bias, bias + 1]))
    assert torch.equal(many[0], want)
    with pytest.raises(RuntimeError):
        ops.fp8_linear(x, q.t(), s, bias=bias.cpu())


# few rows, a strip of 16 weight rows a wave: row tiles of 16 up to the last (16, one; 128, eight; 208, thirteen in the shallower ring, 255 and 256, sixteen), 3 to 12 waves, a last
# workgroup with waves beyond N, strips on both sides of a 128-block's edge, one K step, fewer than the ring is deep, a last step of 16 and of 64
FEW = [("rowwise", 3, 16, 8208, 128), ("rowwise", 3, 17, 12288, 400), ("rowwise", 4, 32, 16384, 704), ("rowwise", 5, 33, 18944, 384), ("rowwise", 7, 80, 28560, 1792), ("rowwise", 10, 81, 37888, 256),
       ("rowwise", 9, 128, 32784, 128), ("rowwise", 12, 129, 49152, 144), ("rowwise", 10, 208, 37904, 640), ("rowwise", 9, 209, 36864, 448), ("rowwise", 9, 256, 33024, 512),
       ("mxfp4", 3, 5, 8208, 128), ("mxfp4", 3, 17, 12288, 416), ("mxfp4", 4, 32, 16384, 640), ("mxfp4", 3, 4, 8448, 4256), ("mxfp4", 5, 33, 18944, 256), ("mxfp4", 5, 113, 16400, 3232), ("mxfp4", 7, 96, 24592, 2592), ("mxfp4", 9, 128, 32784, 352),
       ("mxfp4", 10, 129, 37888, 128), ("mxfp4", 9, 144, 32784, 352), ("mxfp4", 12, 200, 49152, 480), ("mxfp4", 10, 208, 37904, 512), ("mxfp4", 9, 209, 32784, 416), ("mxfp4", 10, 240, 37904, 256), ("mxfp4", 11, 225, 41008, 2176), ("mxfp4", 9, 255, 33040, 288),
       ("block", 3, 1, 12288, 128), ("block", 3, 32, 8208, 1024), ("block", 4, 7, 16256, 640), ("block", 5, 33, 18432, 256), ("block", 5, 65, 16400, 384), ("block", 6, 128, 24464, 1536), ("block", 7, 112, 28544, 1408)]


@pytest.mark.parametrize("mode,strips,M,N,K", FEW)
def test_strips_of_few_rows(dev, mode, strips, M, N, K):
    from oracle import mxfp4_oracle as MX
    kind = {"rowwise": _lib.DISPATCH_ROWWISE, "block": _lib.DISPATCH_BLOCK, "mxfp4": _lib.DISPATCH_MXFP4}[mode]
    took = _lib.gemm_dispatch_info(kind, M, N, K, cus=torch.cuda.get_device_properties(dev).multi_processor_count, flags=_lib.DISPATCH_SPLIT)
    assert took.startswith(f"gemm_ring_few<{mode},{-(-M // 16)},{strips}>{' ktail' if K % 128 else ''} slices=1 grid={-(-N // (16 * strips))} block={64 * strips} "), took
    g = torch.Generator(device=dev).manual_seed(M + N + K)
    x, w = torch.randn(M, K, generator=g, device=dev), torch.randn(N, K, generator=g, device=dev) * 0.05
    x[0, ::7] = float("inf") if M > 1 else 1.0  # (rows do not reach each other)
    if mode == "rowwise":
        a, b = ops.quant_rowwise(x.to(torch.bfloat16)), ops.quant_rowwise(w.to(torch.bfloat16))
        want = _rowwise_want(*a, *b, None)
        run = lambda dtype: ops.scaled_mm(a[0], b[0].t(), a[1], b[1].reshape(1, N), out_dtype=dtype)
    elif mode == "mxfp4":
        a, b = ops.quant_rowwise(x.to(torch.bfloat16)), ops.quant_mxfp4(w.to(torch.bfloat16))
        want = MX.gemm(a[0].cpu(), a[1].cpu().reshape(-1), b[0].cpu(), b[1].cpu()).double()
        run = lambda dtype: ops.gemm_mxfp4(a, b, dtype)
    else:
        a = ops.groupwise_activation_quant(x.to(torch.bfloat16))
        b = w.to(torch.float8_e4m3fn), torch.rand(-(-N // 128), K // 128, generator=g, device=dev) + 0.5
        want = ((a[0].double() * a[1].double().repeat_interleave(128, 1)) @
                (b[0].double() * b[1].double().repeat_interleave(128, 0)[:N].repeat_interleave(128, 1)).t()).cpu()
        run = lambda dtype: ops.gemm_fp8_fp8_bf16_nt(a, b, torch.full((M, N), 7.0, device=dev, dtype=dtype))
    for dtype in (torch.float32, torch.bfloat16):
        got = run(dtype)
        assert all(torch.equal(got.nan_to_num(3.0), run(dtype).nan_to_num(3.0)) for _ in range(2))
        first = 1 if M > 1 else 0
        _check(torch.nn.functional.pad(got[first:], (0, 8, 0, 1), value=7.0), want[first:], M - first, N, dtype, 0.0)


# the same with a bias, all of K a workgroup and in slices, and operands inside rows of their own pitch, whose other bytes are NaN in e4m3 and the largest codes and scales; the last row ends with its memory
STRIPS_PITCHED = [("rowwise", 3, 17, 8208, 400), ("rowwise", 5, 33, 18944, 384), ("rowwise", 7, 80, 28560, 1808), ("rowwise", 10, 81, 37888, 256), ("rowwise", 9, 209, 36864, 448), ("rowwise", 4, 24, 2880, 2880),
                  ("mxfp4", 3, 5, 8208, 160), ("mxfp4", 5, 33, 18944, 384), ("mxfp4", 9, 144, 32784, 352), ("mxfp4", 4, 26, 3200, 2784), ("block", 5, 33, 16400, 384), ("block", 4, 9, 3840, 2176)]


@pytest.mark.parametrize("mode,strips,M,N,K", STRIPS_PITCHED)
def test_strips_of_few_rows_with_pitches_and_a_bias(dev, mode, strips, M, N, K):
    kind = {"rowwise": _lib.DISPATCH_ROWWISE, "block": _lib.DISPATCH_BLOCK, "mxfp4": _lib.DISPATCH_MXFP4}[mode]
    took = _lib.gemm_dispatch_info(kind, M, N, K, cus=torch.cuda.get_device_properties(dev).multi_processor_count, flags=_lib.DISPATCH_SPLIT)
    assert took.startswith(f"gemm_ring_few<{mode},{-(-M // 16)},{strips}>"), took
    g = torch.Generator(device=dev).manual_seed(M + N + K)
    x = torch.randn(M, K, generator=g, device=dev).to(torch.bfloat16)
    w = torch.randn(N, K, generator=g, device=dev) * 0.05
    bias = torch.randn(N, generator=g, device=dev).to(torch.bfloat16)

    def pitched(t, more, filler):
        whole = torch.full((t.shape[0], t.shape[1] + more), filler, dtype=torch.uint8, device=dev)
        whole[:, more:] = t.view(torch.uint8)
        return whole[:, more:]

    lib, (part, need) = _lib.load(), _partial(kind, M, N, K, dev)
    if mode == "block":
        (q, s), b = ops.groupwise_activation_quant(x), (w.to(torch.float8_e4m3fn), torch.rand(-(-N // 128), K // 128, generator=g, device=dev) + 0.5)
        plain = lambda dtype: ops.gemm_fp8_fp8_bf16_nt((q, s), b, torch.empty(M, N, device=dev, dtype=dtype))
    elif mode == "mxfp4":
        (q, s), b = ops.quant_rowwise(x), ops.quant_mxfp4(w.to(torch.bfloat16))
        plain = lambda dtype: ops.gemm_mxfp4((q, s), b, dtype)
        scales = pitched(b[1], 3, 0xFF)
    else:
        (q, s), b = ops.quant_rowwise(x), ops.quant_rowwise(w.to(torch.bfloat16))
        plain = lambda dtype: ops.scaled_mm(q, b[0].t(), s, b[1].reshape(1, N), out_dtype=dtype)
    pq, pw = pitched(q, 32, 0x7F), pitched(b[0], 64 if mode == "mxfp4" else 48, 0x77 if mode == "mxfp4" else 0x7F)
    for dtype in (torch.float32, torch.bfloat16):
        for add in (None, bias) if mode == "rowwise" else (None,):
            out = _out(M, N, dev, dtype)
            tail = (out.data_ptr(), N + 8, ops._out_code(dtype), M, N, K, part.data_ptr(), need, _stream())
            if mode == "block":
                rc = lib.cfp8_gemm_block128_split(pq.data_ptr(), pq.stride(0), s.data_ptr(), pw.data_ptr(), pw.stride(0), b[1].data_ptr(), K // 128, 1, *tail)
            elif mode == "mxfp4":
                rc = lib.cfp8_gemm_mxfp4_split(pq.data_ptr(), pq.stride(0), s.data_ptr(), pw.data_ptr(), pw.stride(0), scales.data_ptr(), scales.stride(0), *tail)
            else:
                rc = lib.cfp8_scaled_mm_rowwise_split(pq.data_ptr(), pq.stride(0), s.data_ptr(), pw.data_ptr(), pw.stride(0), b[1].data_ptr(), ops._ptr(add), *tail)
            _lib.check(rc)
            want = plain(dtype)
            assert torch.equal(out[:M, :N], want if add is None else want + add)
            assert bool((out[M:] == 7.0).all()) and bool((out[:, N:] == 7.0).all())
