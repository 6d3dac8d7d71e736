"""The work that users of the FP8 path have it do, as cases that can be timed and compared.

Six kinds, each through the package's public entry points:

  linear  the four FP8 linears of one decoder layer (qkv with its bias, o, gate_up, down) in a rollout engine:
          ``Fp8LinearMethod.apply`` on bf16 activations, from one token of decode to a prefill of thousands
  moe     one MoE layer's experts on routed tokens: ``grouped_experts_forward`` with ``DSGroupGEMM``
  block   a block-scaled linear: the 1x128 activation quantiser and ``gemm_fp8_fp8_bf16_nt``
  mxfp4   the gate_up and down linears of a layer with MXFP4 weights: ``linear_mxfp4``
  sync    the weights of a few layers quantised row by row into the engine: ``QuantizedWeightReceiver.flush_completions``
  cast    the weights of a few layers cast tensorwise by a trainer that owns the GPU: ``quant_tensorwise_multi``

Sizes are those of the decoder layers that the package's benchmark and tests run, and generic ones around them.
"""
import os
import sys

import torch

for _p in (os.path.join(os.getcwd(), "cosmos-rl_amd"),):
    if _p not in sys.path:
        sys.path.insert(0, _p)

from cosmos_rl_amd import ops  # noqa: E402
from cosmos_rl_amd.policy.kernel.group_gemms import DSGroupGEMM  # noqa: E402
from cosmos_rl_amd.policy.kernel.moe.moe import grouped_experts_forward  # noqa: E402
from cosmos_rl_amd.rollout.vllm_rollout.monkey_patch_for_fp8 import Fp8LinearMethod  # noqa: E402
from cosmos_rl_amd.rollout.vllm_rollout.vllm_rollout import FP8RolloutMixin  # noqa: E402
from cosmos_rl_amd.rollout.worker.rollout_control import QuantizedWeightReceiver  # noqa: E402

DEV = "cuda"
SMALL = {"hidden": 896, "kv": 128, "inter": 4864}      # Qwen2.5-0.5B: the smallest policy that is trained in earnest
LARGE = {"hidden": 3584, "kv": 512, "inter": 18944}    # Qwen2.5-7B


def listed():
    return [
        # one sequence decoding on the small policy: launches and host time are all of it
        dict(name="linear_small_1", kind="linear", tokens=1, **SMALL),
        # a decode batch of a rollout engine, not a power of two: weights are streamed
        dict(name="linear_33", kind="linear", tokens=33, **LARGE),
        # one prompt, or a chunk of prefill beside decodes: a count of tokens that no tile divides
        dict(name="linear_1111", kind="linear", tokens=1111, **LARGE),
        # a full prefill batch
        dict(name="linear_8192", kind="linear", tokens=8192, **LARGE),
        # experts of Qwen3-30B-A3B: a decode batch that touches most experts with about one row each ...
        dict(name="moe_16", kind="moe", tokens=16, experts=128, topk=8, hidden=2048, inter=768),
        # ... a chunk of prefill, some fifty rows an expert ...
        dict(name="moe_777", kind="moe", tokens=777, experts=128, topk=8, hidden=2048, inter=768),
        # ... and the training or prefill batch of the benchmark
        dict(name="moe_8192", kind="moe", tokens=8192, experts=128, topk=8, hidden=2048, inter=768),
        # block-scaled weights of DeepSeek-V3's dense MLP: a decode batch and a training batch
        dict(name="block_24", kind="block", tokens=24, rows=18432, cols=7168),
        dict(name="block_4096", kind="block", tokens=4096, rows=18432, cols=7168),
        # MXFP4 weights, a large decode batch or a short prompt
        dict(name="mxfp4_200", kind="mxfp4", tokens=200, **LARGE),
        # one flush group of a weight sync: four layers received, quantised into the engine's parameters
        dict(name="sync_4", kind="sync", layers=4, **LARGE),
        # eight layers of policy weights cast by the trainer, every projection a tensor of its own
        dict(name="cast_8", kind="cast", layers=8, **LARGE),
    ]


def _log(rng, lo, hi):
    """A whole number from lo to hi, its logarithm spread evenly."""
    return min(hi, max(lo, int(round(lo * (hi / lo) ** rng.random()))))


def draw(rng):
    kind = rng.choice(["linear", "linear", "moe", "moe", "block", "mxfp4", "sync", "cast"])
    # hidden sizes of decoder layers are multiples of 128 as a rule; 2880 is GPT-OSS's
    hidden = 2880 if rng.random() < 0.15 else 128 * rng.randint(7, 28)
    layer = {"hidden": hidden, "kv": 128 * rng.randint(1, 8), "inter": 128 * rng.randint(38, 148)}
    if kind == "linear":
        return dict(kind=kind, tokens=_log(rng, 1, 8192), **layer)
    if kind == "moe":
        return dict(kind=kind, tokens=_log(rng, 1, 8192), experts=rng.choice([32, 64, 128]), topk=rng.randint(4, 8),
                    hidden=128 * rng.randint(8, 28), inter=128 * rng.randint(4, 12))
    if kind == "block":
        return dict(kind=kind, tokens=_log(rng, 1, 4096), rows=128 * rng.randint(12, 144), cols=128 * rng.randint(12, 56))
    if kind == "mxfp4":
        return dict(kind=kind, tokens=_log(rng, 1, 4096), **layer)
    return dict(kind=kind, layers=rng.randint(1, 8), **layer)


# ---- inputs -----------------------------------------------------------------
def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _weight(g, *shape):
    return torch.randn(*shape, generator=g, device=DEV, dtype=torch.bfloat16) * 0.02


def _activation(g, tokens, cols):
    """N(0, 1) with 0.5 % of the channels thirty times as large, as activations in front of a linear have them."""
    x = torch.randn(tokens, cols, generator=g, device=DEV, dtype=torch.bfloat16)
    hot = torch.rand(cols, generator=g, device=DEV) < 0.005
    return torch.where(hot, x * 30, x)


def _linear_shapes(c):
    """[out, in] of qkv, o, gate_up, down: the engine's fused parameters."""
    h, i = c["hidden"], c["inter"]
    return [(h + 2 * c["kv"], h), (h, h), (2 * i, h), (h, i)]


def _split_shapes(c):
    """[out, in] of the policy's own parameters of a layer: q, k, v, o, gate, up, down."""
    h, i, kv = c["hidden"], c["inter"], c["kv"]
    return [(h, h), (kv, h), (kv, h), (h, h), (i, h), (i, h), (h, i)]


class _Names:
    """Weight names as the engine has them: nothing to map."""

    @staticmethod
    def get_unsplited_weight_name(name):
        return name

    @staticmethod
    def rollout_map_local_key_to_hf_key(name):
        return name


class _Engine(FP8RolloutMixin):
    """A rollout whose model is a dict of parameters."""

    def __init__(self, params):
        self._model_param_map = params
        self._engine_initialized = True


def _prepare_linear(c, g):
    layers = []
    for n, (rows, cols) in enumerate(_linear_shapes(c)):
        layer = torch.nn.Module()
        layer.weight = torch.nn.Parameter(_weight(g, rows, cols), requires_grad=False)
        layer.quant_method = Fp8LinearMethod()
        layer.quant_method.process_weights_after_loading(layer)
        bias = torch.randn(rows, generator=g, device=DEV, dtype=torch.bfloat16) if n == 0 else None
        layers.append((layer, _activation(g, c["tokens"], cols), bias))
    return {"layers": layers}


def _prepare_moe(c, g):
    E, H, I, T, K = c["experts"], c["hidden"], c["inter"], c["tokens"], c["topk"]
    strategy, module = DSGroupGEMM(torch.nn.SiLU(), fuse_gate_up=True), torch.nn.Module()
    for name, rows, cols in (("gate_proj", I, H), ("up_proj", I, H), ("down_proj", H, I)):
        w = strategy.arrange_expert_weights(list(_weight(g, E, rows, cols)), name, module)
        module.register_parameter(f"{name}_weight", torch.nn.Parameter(w, requires_grad=False))
    scores, indices = torch.rand(T, E, generator=g, device=DEV).topk(K, dim=1)
    mask = torch.rand(T, generator=g, device=DEV) < 0.98   # the batch's padding tokens go to no expert
    mask[0] = True
    return {"strategy": strategy, "module": module, "experts": E, "x": torch.randn(T, H, generator=g, device=DEV, dtype=torch.bfloat16),
            "mask": mask, "indices": indices, "weights": torch.softmax(scores, dim=1).to(torch.bfloat16)}


def _prepare_block(c, g):
    weight = ops.per_block_cast_to_fp8(_weight(g, c["rows"], c["cols"]))
    return {"weight": weight, "x": torch.randn(c["tokens"], c["cols"], generator=g, device=DEV, dtype=torch.bfloat16)}


def _prepare_mxfp4(c, g):
    layers = []
    for rows, cols in _linear_shapes(c)[2:]:
        layers.append((ops.quant_mxfp4(_weight(g, rows, cols)), _activation(g, c["tokens"], cols)))
    return {"layers": layers}


def _prepare_sync(c, g):
    received, params, fp8 = {}, {}, {}
    for n in range(c["layers"]):
        for name, (rows, cols) in zip(("qkv_proj", "o_proj", "gate_up_proj", "down_proj"), _linear_shapes(c)):
            key = f"model.layers.{n}.{name}.weight"
            received[key] = torch.nn.Parameter(_weight(g, rows, cols), requires_grad=False)
            fp8[key] = torch.zeros(rows, cols, device=DEV, dtype=torch.uint8).view(torch.float8_e4m3fn).t()
            params[key] = fp8[key]
            params[key.replace(".weight", ".weight_scale")] = torch.zeros(rows, 1, device=DEV)
    return {"receiver": QuantizedWeightReceiver(_Engine(params), _Names, received, fp8), "groups": [[k] for k in received], "params": params}


def _prepare_cast(c, g):
    return {"weights": [_weight(g, rows, cols) for _ in range(c["layers"]) for rows, cols in _split_shapes(c)]}


def prepare(case, seed):
    state = globals()["_prepare_" + case["kind"]](case, _gen(seed))
    state["kind"] = case["kind"]
    return state


# ---- one pass ---------------------------------------------------------------
def _run_linear(s):
    return [layer.quant_method.apply(layer, x, bias) for layer, x, bias in s["layers"]]


def _run_moe(s):
    return grouped_experts_forward(s["x"], s["mask"], s["weights"], s["indices"], s["strategy"], s["module"], s["experts"])


def _run_block(s):
    x = ops.groupwise_activation_quant(s["x"])
    out = torch.empty(s["x"].shape[0], s["weight"][0].shape[0], device=DEV, dtype=torch.bfloat16)
    return ops.gemm_fp8_fp8_bf16_nt(x, s["weight"], out)


def _run_mxfp4(s):
    return [ops.linear_mxfp4(x, weight) for weight, x in s["layers"]]


def _run_sync(s):
    s["receiver"].flush_completions(s["groups"])
    return s["params"]


def _run_cast(s):
    with ops.gpu_is_mine():
        return ops.quant_tensorwise_multi(s["weights"])


def run(state):
    return globals()["_run_" + state["kind"]](state)


# ---- what a pass cannot do without ------------------------------------------
def work(case):
    kind, T = case["kind"], case.get("tokens", 0)
    if kind == "linear":
        shapes = _linear_shapes(case)
        return {"bytes": sum(n * k + 4 * n + 2 * T * (n + k) for n, k in shapes), "flops": sum(2 * T * n * k for n, k in shapes)}
    if kind == "mxfp4":
        shapes = _linear_shapes(case)[2:]
        return {"bytes": sum(n * k / 2 + n * k / 32 + 2 * T * (n + k) for n, k in shapes), "flops": sum(2 * T * n * k for n, k in shapes)}
    if kind == "moe":
        E, H, I, K = case["experts"], case["hidden"], case["inter"], case["topk"]
        touched = E * (1 - (1 - K / E) ** T)  # experts that uniform routing gives at least one token
        return {"bytes": touched * 3 * H * I + 4 * T * H + 10 * T * K, "flops": 6 * T * K * H * I}
    if kind == "block":
        n, k = case["rows"], case["cols"]
        return {"bytes": n * k + n * k / 4096 + 2 * T * (n + k), "flops": 2 * T * n * k}
    # quantisers: two bytes in, one out an element; rowwise scales besides
    if kind == "sync":
        return {"bytes": case["layers"] * sum(3 * n * k + 4 * n for n, k in _linear_shapes(case)), "flops": 0}
    return {"bytes": case["layers"] * sum(3 * n * k for n, k in _split_shapes(case)), "flops": 0}


def tolerance(case):
    # quantised weights are defined to the bit
    if case["kind"] in ("sync", "cast"):
        return "exact"
    # Four times the measured distance between a path's bf16 results and the same computed with 64-bit sums from the
    # same quantised operands: sums alone move a result by one bf16 rounding now and then (4e-4 in norm); the bias of
    # qkv is added to a rounded or an unrounded product (2.7e-3); between the experts' two products an fp8 rounding of
    # the hidden activation can move as well (3.3e-3).
    return {"rel": {"linear": 1.1e-2, "moe": 1.3e-2, "block": 1.7e-3, "mxfp4": 1.7e-3}[case["kind"]]}
