"""The operators' native host path (csrc/torch_calls.cpp) beside the same steps in Python: what it takes gives the same tensors, what
it does not take it leaves alone, and an argument that the library refuses is refused in the same words."""
import pytest
import torch

from cosmos_rl_amd import _lib, ops
from oracle import fp8_oracle as O

pytestmark = pytest.mark.gpu


def _both(call, monkeypatch):
    """The call by the native path (which must have taken it: `took`) and step by step."""
    took = []
    for name in ("_linear_call", "_mxfp4_call"):
        native = ops._native({"_linear_call": "fp8_linear", "_mxfp4_call": "linear_mxfp4"}[name])

        def counted(*args, native=native):
            out = native(*args)
            took.append(out is not None)
            return out
        monkeypatch.setattr(ops, name, counted)
    one = call()
    monkeypatch.setattr(ops, "_linear_call", lambda *args: None)
    monkeypatch.setattr(ops, "_mxfp4_call", lambda *args: None)
    return one, call(), took[0]


def _same(a, b):
    assert a.shape == b.shape and a.stride() == b.stride() and a.dtype == b.dtype and not a.requires_grad and torch.equal(a, b)


def _operands(dev, M, N, K):
    x = O.make_activation(M, K, seed=1).to(dev)
    q, s = ops.quant_rowwise(O.make_weight((N, K), seed=2).to(dev))
    return x, q.t(), s, torch.randn(N, device=dev).to(torch.bfloat16)


@pytest.mark.parametrize("M,N,K", [(1, 16, 128), (1, 1152, 896), (3, 512, 4096), (33, 3584, 2304), (130, 1024, 272)])
@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32])
def test_linear(dev, M, N, K, dt, monkeypatch):
    x, w, s, b = _operands(dev, M, N, K)
    wide = torch.zeros(M, K + 64, device=dev, dtype=torch.bfloat16)
    wide[:, :K] = x
    params = (torch.nn.Parameter(w, requires_grad=False), torch.nn.Parameter(s, requires_grad=False))
    for call in (lambda: ops.fp8_linear(x, w, s, out_dtype=dt), lambda: ops.fp8_linear(x, w, s, bias=b, out_dtype=dt),
                 lambda: ops.fp8_linear(wide[:, :K], *params, out_dtype=dt), lambda: ops.fp8_linear(x.requires_grad_(), w, s.reshape(-1), out_dtype=dt)):
        one, two, took = _both(call, monkeypatch)
        assert took
        _same(one, two)


def test_linear_left_to_the_steps(dev, monkeypatch):
    M, N, K = 5, 256, 512
    x, w, s, b = _operands(dev, M, N, K)

    class Sub(torch.Tensor):
        pass

    class Seen(torch.overrides.TorchFunctionMode):
        calls = 0

        def __torch_function__(self, func, types, args=(), kwargs=None):
            Seen.calls += 1
            return func(*args, **(kwargs or {}))

    def seen():
        with Seen():
            return ops.fp8_linear(x, w, s)

    for call in (lambda: ops.fp8_linear(x.reshape(1, M, K), w, s), lambda: ops.fp8_linear(x.t().contiguous().t(), w, s), lambda: ops.fp8_linear(x, w, s.double()),
                 lambda: ops.fp8_linear(x, w, s, bias=b.float()), lambda: ops.fp8_linear(x, w, s, bias=torch.nn.Parameter(b)),
                 lambda: ops.fp8_linear(x.as_subclass(Sub), w, s).as_subclass(torch.Tensor), lambda: ops.fp8_linear(x[:0], w, s), lambda: ops.fp8_linear(x, w, s[:1]), seen):
        one, two, took = _both(call, monkeypatch)
        assert not took
        assert one.shape == two.shape and torch.equal(one, two) and one.requires_grad == two.requires_grad
    assert Seen.calls


@pytest.mark.filterwarnings("ignore")
def test_watched_and_wrapped_calls_are_left_to_the_steps(dev, monkeypatch):
    """A dispatch mode sees the calls, tracing and torch.func's wrappers end as they do step by step (with an error where a wrapped tensor has
    no memory); tokens with a tangent give the plain result either way."""
    from torch.utils._python_dispatch import TorchDispatchMode
    M, N, K = 5, 256, 512
    x, w, s, _ = _operands(dev, M, N, K)
    weight = ops.quant_mxfp4(O.make_weight((N, K), seed=2).to(dev))
    want = {"linear": ops.fp8_linear(x, w, s), "mxfp4": ops.linear_mxfp4(x, weight)}

    class Seen(TorchDispatchMode):
        calls = 0

        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            Seen.calls += 1
            return func(*args, **(kwargs or {}))

    def watched(op):
        with Seen():
            return op(x)

    def dual(op):
        with torch.autograd.forward_ad.dual_level():
            out = op(torch.autograd.forward_ad.make_dual(x, torch.ones_like(x)))
            assert torch.autograd.forward_ad.unpack_dual(out).tangent is None
            return out

    def ended(call):
        try:
            return call()
        except Exception as e:
            return type(e)

    for name, op in (("linear", lambda x: ops.fp8_linear(x, w, s)), ("mxfp4", lambda x: ops.linear_mxfp4(x, weight))):
        before = Seen.calls
        one, two, took = _both(lambda: watched(op), monkeypatch)
        assert not took and Seen.calls > before and torch.equal(one, want[name]) and torch.equal(two, want[name])
        one, two, took = _both(lambda: dual(op), monkeypatch)
        assert took and torch.equal(one, want[name]) and torch.equal(two, want[name])
        for call in (lambda: torch.func.vmap(op)(torch.stack([x, x])), lambda: torch.func.jvp(op, (x,), (x,)), lambda: torch.func.vjp(op, x),
                     lambda: torch.jit.trace(op, (x,), check_trace=False) and None):
            one, two, took = _both(lambda: ended(call), monkeypatch)
            assert not took and (one is two or type(one) is type(two))


def test_mxfp4(dev, monkeypatch):
    for M, N, K, dt in ((1, 64, 128, None), (4, 256, 2880, torch.float32), (40, 512, 1024, None)):
        x, weight = O.make_activation(M, K, seed=1).to(dev), ops.quant_mxfp4(O.make_weight((N, K), seed=2).to(dev))
        one, two, took = _both(lambda: ops.linear_mxfp4(x, weight, out_dtype=dt), monkeypatch)
        assert took
        _same(one, two)
        one, two, took = _both(lambda: ops.linear_mxfp4(x[None], weight, out_dtype=dt), monkeypatch)
        assert not took and torch.equal(one, two)


def test_refusals(dev, monkeypatch):
    x, w, s, b = _operands(dev, 5, 256, 512)
    pitched = torch.zeros(5, 515, device=dev, dtype=torch.bfloat16)[:, :512]   # rows that are not 16-byte aligned
    for call in (lambda: ops.fp8_linear(pitched, w, s), lambda: ops.fp8_linear(x.half(), w, s), lambda: ops.fp8_linear(x, w, s, out_dtype=torch.float16),
                 lambda: ops.fp8_linear(x.cpu(), w, s), lambda: ops.fp8_linear(x, w.t(), s), lambda: ops.fp8_linear(x, w, s[:-1]),
                 lambda: ops.fp8_linear(x, torch.zeros(256, 512, device=dev, dtype=torch.bfloat16).t(), s)):
        said = []
        for native in (ops._native("fp8_linear"), lambda *args: None):
            monkeypatch.setattr(ops, "_linear_call", native)
            with pytest.raises((ValueError, RuntimeError)) as e:
                call()
            said.append((type(e.value), str(e.value)))
        assert said[0] == said[1]


def test_current_stream(dev):
    """The call is on the stream that is current, as in Python."""
    x, w, s, _ = _operands(dev, 8, 512, 1024)
    want = ops.fp8_linear(x, w, s)
    stream = torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(stream):
        y = torch.zeros_like(x)
        torch.cuda._sleep(20_000_000)
        y.copy_(x)
        out = ops.fp8_linear(y, w, s)   # on another stream than the copy it would read zeros
    stream.synchronize()
    assert torch.equal(out, want)
    assert _lib.CALLS_PATH.exists()
