"""The one-call MoE experts (cfp8_moe_experts, what grouped_experts_forward runs for the FP8 strategy) against the chain of
the separate entry points, each of which has its own test against the oracle.  Every form of it has the chain's bits."""
import pytest
import torch

from cosmos_rl_amd import _lib, ops

pytestmark = pytest.mark.gpu


def _module(dev, E, H, I, seed):
    from cosmos_rl_amd.policy.kernel.group_gemms import DSGroupGEMM
    g = torch.Generator(device=dev).manual_seed(seed)
    strategy, module = DSGroupGEMM(torch.nn.SiLU(), fuse_gate_up=True), torch.nn.Module()
    for name, rows, cols in (("gate_proj", I, H), ("up_proj", I, H), ("down_proj", H, I)):
        w = (torch.randn(E, rows, cols, generator=g, device=dev) * 0.05).to(torch.bfloat16)
        module.register_parameter(f"{name}_weight", torch.nn.Parameter(strategy.arrange_expert_weights(list(w), name, module), requires_grad=False))
    return strategy, module


def _chain(x, mask, w, idx, strategy, module, E):
    from cosmos_rl_amd.policy.kernel.moe.moe import combine_expert_outputs, route_tokens
    r = route_tokens(idx, mask, E)
    return combine_expert_outputs(strategy.execute_from_tokens(x, r.row_tokens, r.m_sizes, r.m_offsets, module, row_map=r.row_map), r, w)


@pytest.mark.parametrize("T,E,topk,H,I", [(1, 8, 2, 256, 128), (5, 4, 4, 128, 256), (1, 129, 8, 4096, 1536), (33, 70, 7, 3584, 896), (90, 3, 3, 640, 1408), (40, 16, 8, 384, 128), (700, 7, 3, 1024, 768), (3300, 7, 2, 1152, 1024),
                                          (200, 3, 1, 4224, 640), (130, 6, 2, 512, 1664),
                                              (777, 64, 8, 1024, 896)])
@pytest.mark.parametrize("masked", [False, True])
def test_one_call_experts(dev, T, E, topk, H, I, masked):
    from cosmos_rl_amd.policy.kernel.moe.moe import grouped_experts_forward
    strategy, module = _module(dev, E, H, I, T)
    g = torch.Generator(device=dev).manual_seed(T + 1)
    x = torch.randn(T, H, generator=g, device=dev).to(torch.bfloat16)
    idx = torch.rand(T, E, generator=g, device=dev).topk(topk, dim=1).indices
    w = torch.rand(T, topk, generator=g, device=dev)
    mask = (torch.rand(T, generator=g, device=dev) < 0.7) if masked else None
    for wt, it in ((torch.bfloat16, torch.int64), (torch.float32, torch.int32)):
        junk = torch.full((64 << 20,), 0x7F, dtype=torch.uint8, device=dev)   # what the workspace holds before is no number
        del junk
        y = grouped_experts_forward(x, mask, w.to(wt), idx.to(it), strategy, module, E)
        want = _chain(x, mask, w.to(torch.bfloat16), idx, strategy, module, E)
        assert torch.equal(y.view(torch.int16), want.view(torch.int16))
    if masked:
        assert not bool(y[~mask].any())


# the form on tiles of 64 rows: experts of no, few, 64, 65 and many rows, one to 31 steps of K, more experts than a wave has lanes;
# the form for decode batches with experts of several tiles of 16 rows, 5 to 32 steps of K (a multiple of 16, and not)
@pytest.mark.parametrize("T,E,topk,H,I", [(64, 1, 1, 384, 256), (65, 2, 1, 128, 128), (130, 3, 2, 3968, 128), (700, 66, 8, 256, 3968), (1500, 200, 8, 640, 384),
                                          (1600, 1, 1, 256, 128),
                                          (48, 40, 8, 4096, 256), (60, 50, 8, 2688, 1536), (300, 256, 8, 640, 128)])
def test_one_call_experts_uneven(dev, T, E, topk, H, I):
    from cosmos_rl_amd.policy.kernel.moe.moe import grouped_experts_forward
    strategy, module = _module(dev, E, H, I, T)
    g = torch.Generator(device=dev).manual_seed(T + 2)
    x = torch.randn(T, H, generator=g, device=dev).to(torch.bfloat16)
    like = torch.rand(T, E, generator=g, device=dev) + 0.6 * torch.rand(E, generator=g, device=dev)   # some experts are liked better
    idx = like.topk(topk, dim=1).indices
    w = torch.rand(T, topk, generator=g, device=dev).to(torch.bfloat16)
    mask = torch.rand(T, generator=g, device=dev) < 0.9
    y = grouped_experts_forward(x, mask, w, idx, strategy, module, E)
    want = _chain(x, mask, w, idx, strategy, module, E)
    assert torch.equal(y.view(torch.int16), want.view(torch.int16))
    assert not bool(y[~mask].any())


# experts of many rows, of which the products learn on the device how many there are: far fewer tiles of rows than the bound, fewer and
# more than CUs, none at all; 2 to 33 steps of K in either product, of which 4 to 32 take the kernel made for them, hidden sizes that are
# no multiple of its 256 columns among them; weights that are loaded as a stream; experts of at most 64 rows in a tile of 128, also
# where only gate_up is that kernel's
@pytest.mark.parametrize("T,E,topk,H,I,keep", [(9000, 16, 8, 1024, 768, 0.3), (9000, 16, 8, 512, 640, 0.6), (6000, 20, 6, 1024, 1024, 0.1), (6000, 9, 6, 256, 768, 0.0),
                                               (2000, 5, 3, 896, 768, 0.9), (5000, 12, 4, 1152, 512, 0.8), (5000, 12, 4, 1280, 640, 0.8),
                                               (5000, 12, 4, 2176, 384, 0.8), (5001, 13, 4, 2048, 384, 0.8), (5000, 31, 4, 4096, 128, 1.0), (1200, 28, 4, 1024, 4224, 1.0), (3000, 6, 4, 4096, 512, 0.9), (1500, 3, 2, 4224, 256, 0.9),
                                               (9000, 9, 6, 640, 512, 0.9), (2000, 5, 2, 640, 4096, 0.9), (2000, 4, 2, 512, 4224, 0.9),
                                               (700, 64, 8, 2048, 1024, 0.9), (3200, 64, 1, 768, 512, 0.9)])
def test_one_call_experts_many_rows(dev, T, E, topk, H, I, keep):
    from cosmos_rl_amd.policy.kernel.moe.moe import grouped_experts_forward
    strategy, module = _module(dev, E, H, I, T)
    g = torch.Generator(device=dev).manual_seed(T + 3)
    x = torch.randn(T, H, generator=g, device=dev).to(torch.bfloat16)
    idx = torch.rand(T, E, generator=g, device=dev).topk(topk, dim=1).indices
    w = torch.rand(T, topk, generator=g, device=dev).to(torch.bfloat16)
    mask = torch.rand(T, generator=g, device=dev) < keep
    junk = torch.full((256 << 20,), 0x7F, dtype=torch.uint8, device=dev)   # what the workspace holds before is no number
    del junk
    y = grouped_experts_forward(x, mask, w, idx, strategy, module, E)
    want = _chain(x, mask, w, idx, strategy, module, E)
    assert torch.equal(y.view(torch.int16), want.view(torch.int16))
    assert not bool(y[~mask].any())


# infinities and NaN, from a token and from a weight, and products beyond bf16: they stay in their rows, on tiles of which a half is padding as well
@pytest.mark.parametrize("T,E,topk,H,I", [(700, 16, 4, 640, 512), (300, 5, 2, 1024, 768), (300, 5, 2, 1024, 384)])
def test_one_call_experts_of_values_that_are_no_numbers(dev, T, E, topk, H, I):
    from cosmos_rl_amd.policy.kernel.moe.moe import grouped_experts_forward
    strategy, module = _module(dev, E, H, I, T)
    g = torch.Generator(device=dev).manual_seed(T + 5)
    x = torch.randn(T, H, generator=g, device=dev).to(torch.bfloat16)
    x[1, 3], x[2, 5], x[3, 7], x[4], x[5] = float("inf"), float("nan"), float("-inf"), 3e38, 0.0
    module.get_parameter("down_proj_scales").data[E - 1, 0, 0] = float("inf")
    idx = torch.rand(T, E, generator=g, device=dev).topk(topk, dim=1).indices
    w = torch.rand(T, topk, generator=g, device=dev).to(torch.bfloat16)
    mask = torch.rand(T, generator=g, device=dev) < 0.9
    mask[:6] = True
    y = grouped_experts_forward(x, mask, w, idx, strategy, module, E)
    want = _chain(x, mask, w, idx, strategy, module, E)
    assert torch.equal(y.isnan(), want.isnan()) and torch.equal(y.nan_to_num(7.0), want.nan_to_num(7.0))
    plain = (idx != E - 1).all(1)
    plain[1:5] = False
    assert bool(y[2].isnan().all()) and bool(y[plain].isfinite().all()) and not bool(y[~mask].any())


# the tokens are quantised by workgroups behind the routing's, 256 groups each, four in turn a thread: in the one launch up to 1024 pairs, in the
# second of two beyond; rows of tokens that do not follow each other
@pytest.mark.parametrize("T,topk,H", [(1, 1, 128), (3, 8, 128), (51, 4, 640), (52, 4, 640), (128, 8, 640), (129, 8, 640), (1025, 1, 128), (410, 3, 1280), (1639, 2, 640), (4096, 1, 1024), (4097, 1, 1024), (3641, 2, 1152)])
def test_one_call_experts_quantised_beside_the_routing(dev, T, topk, H):
    from cosmos_rl_amd.policy.kernel.moe.moe import grouped_experts_forward
    E = 8
    strategy, module = _module(dev, E, H, 128, T)
    g = torch.Generator(device=dev).manual_seed(T + 4)
    x = torch.randn(T, H + 8, generator=g, device=dev).to(torch.bfloat16)[:, :H]
    idx = torch.rand(T, E, generator=g, device=dev).topk(topk, dim=1).indices
    w = torch.rand(T, topk, generator=g, device=dev).to(torch.bfloat16)
    mask = torch.rand(T, generator=g, device=dev) < 0.8
    y = grouped_experts_forward(x, mask, w, idx, strategy, module, E)
    want = _chain(x.contiguous(), mask, w, idx, strategy, module, E)
    assert torch.equal(y.view(torch.int16), want.view(torch.int16))


def test_one_call_experts_refuses_a_small_workspace(dev):
    t = torch.zeros(256, 256, device=dev, dtype=torch.bfloat16)
    need = _lib.load().cfp8_moe_experts_workspace_bytes(4, 2, 2, 256, 128)
    args = lambda n: _lib.load().cfp8_moe_experts(t.data_ptr(), 256, 4, 256, t.data_ptr(), 8, None, t.data_ptr(), 0, 2, 2, t.data_ptr(), t.data_ptr(),
                                                  t.data_ptr(), t.data_ptr(), 128, t.data_ptr(), 256, t.data_ptr(), n, None)
    assert need > 0 and args(need - 1) == _lib.EWORKSPACE


def test_one_call_experts_refuses_other_types(dev):
    """What the kernels would read as something else is refused before a launch."""
    E, T, H, I = 4, 6, 256, 128
    strategy, module = _module(dev, E, H, I, 5)
    x = torch.randn(T, H, device=dev).to(torch.bfloat16)
    idx = torch.rand(T, E, device=dev).topk(2, dim=1).indices
    w = torch.rand(T, 2, device=dev).to(torch.bfloat16)
    (gu, gus), dn, dns = strategy._interleaved(module), module.get_parameter("down_proj_fp8"), module.get_parameter("down_proj_scales")
    assert ops.moe_experts(x, None, w, idx, (gu, gus), (dn, dns)).shape == (T, H)
    wide = torch.randn(T, 2 * H, device=dev).to(torch.bfloat16)
    for bad in ((x.half(), (gu, gus), (dn, dns)), (x.float(), (gu, gus), (dn, dns)), (wide[:, ::2], (gu, gus), (dn, dns)), (x[None], (gu, gus), (dn, dns)),
                (x, (gu, gus.to(torch.bfloat16)), (dn, dns)), (x, (gu, gus), (dn, dns.double())), (x, (gu.view(torch.uint8), gus), (dn, dns)),
                (x, (gu, gus), (dn.to(torch.bfloat16), dns))):
        with pytest.raises(ValueError):
            ops.moe_experts(bad[0], None, w, idx, bad[1], bad[2])


def test_strategies_with_steps_of_their_own(dev):
    """A strategy derived from DSGroupGEMM that replaces one of its steps has that step called; one that adds to it keeps the
    one-call form.  An alignment that no layout has is refused on either way."""
    from cosmos_rl_amd.policy.kernel.group_gemms import DSGroupGEMM
    from cosmos_rl_amd.policy.kernel.moe.moe import grouped_experts_forward
    calls = []

    class Counted(DSGroupGEMM):
        def _run(self, *args, **kwargs):
            calls.append(1)
            return super()._run(*args, **kwargs)

    class Named(DSGroupGEMM):
        name = "experts"

    E, T, H, I = 4, 6, 256, 128
    strategy, module = _module(dev, E, H, I, 6)
    x = torch.randn(T, H, device=dev).to(torch.bfloat16)
    idx = torch.rand(T, E, device=dev).topk(2, dim=1).indices
    w = torch.rand(T, 2, device=dev).to(torch.bfloat16)
    want = grouped_experts_forward(x, None, w, idx, strategy, module, E)
    assert torch.equal(grouped_experts_forward(x, None, w, idx, Counted(torch.nn.SiLU(), fuse_gate_up=True), module, E), want) and calls == [1]
    named = Named(torch.nn.SiLU(), fuse_gate_up=True)
    assert torch.equal(named.forward_experts(x, None, w, idx, module, E), want)
    with pytest.raises(ValueError):
        grouped_experts_forward(x, None, w, idx, strategy, module, E, alignment=0)


def test_token_masks_of_other_forms(dev):
    from cosmos_rl_amd.policy.kernel.moe.moe import grouped_experts_forward, route_tokens
    E, T, H, I = 4, 6, 256, 128
    strategy, module = _module(dev, E, H, I, 3)
    g = torch.Generator(device=dev).manual_seed(4)
    x = torch.randn(T, H, generator=g, device=dev).to(torch.bfloat16)
    idx = torch.rand(T, E, generator=g, device=dev).topk(2, dim=1).indices
    w = torch.rand(T, 2, generator=g, device=dev).to(torch.bfloat16)
    want = grouped_experts_forward(x, None, w, idx, strategy, module, E)
    one = torch.ones(1, dtype=torch.bool, device=dev)
    for mask in (one, one[0], torch.ones(T, dtype=torch.int64, device=dev)):   # one value for all tokens, whole numbers
        assert torch.equal(grouped_experts_forward(x, mask, w, idx, strategy, module, E), want)
    for mask in (torch.ones(T, dtype=torch.bool), one.expand(T - 1)):          # on the host, too short: refused before a launch
        with pytest.raises((ValueError, RuntimeError)):
            grouped_experts_forward(x, mask, w, idx, strategy, module, E)
        with pytest.raises((ValueError, RuntimeError)):
            route_tokens(idx, mask, E)


# the forms of a decode batch and of a chunk of prefill, each with the shape that makes the choice: streams of strips with one K step in either product, more units of a wave than stages and fewer, experts of 16
# rows and more, as many tiles as workgroups have room for, 11 rows an expert of few weights; weights of which a strip a workgroup is read; down as streams behind tiles of 64 rows with one to six steps
# of K, 48 with seven or eight, 32 with 9 to 13, and by the ring kernel; tokens of which none is left
EXPERT_FORMS = [("few streams", 20, 64, 4, 4096, 128), ("few streams", 70, 130, 4, 128, 1536), ("few streams", 3, 128, 8, 2048, 768), ("few streams", 12, 4, 1, 4096, 1536),
                ("few streams", 33, 4, 1, 4096, 1536), ("few streams", 64, 40, 4, 3072, 640), ("few streams", 60, 256, 4, 512, 384), ("few streams", 33, 32, 8, 1152, 1408),
                ("few streams", 1, 9, 9, 4096, 1152), ("few streams", 130, 127, 8, 1664, 256), ("few streams", 48, 32, 8, 1024, 512), ("few strips", 1, 128, 8, 2048, 768),
                ("few strips", 30, 64, 4, 128, 1536), ("few strips", 90, 256, 4, 512, 384), ("few strips", 17, 3, 1, 4096, 1536), ("middle down=streams,64", 500, 70, 4, 3968, 128),
                ("middle down=streams,64", 300, 64, 6, 3968, 256), ("middle down=streams,64", 600, 127, 8, 2944, 384), ("middle down=streams,64", 400, 33, 3, 3584, 640),
                ("middle down=streams,64", 448, 128, 8, 2048, 768), ("middle down=streams,64", 450, 200, 8, 1536, 128), ("middle down=streams,48", 200, 64, 8, 1280, 896),
                ("middle down=streams,48", 250, 64, 8, 1024, 1024), ("middle down=streams,32", 160, 40, 5, 1152, 1152), ("middle down=streams,32", 150, 32, 4, 3584, 1536),
                ("middle down=streams,32", 170, 9, 1, 3968, 1664), ("middle down=ring", 40, 8, 4, 1024, 512), ("middle down=ring", 60, 4, 1, 3968, 3968)]


@pytest.mark.parametrize("form,T,E,topk,H,I", EXPERT_FORMS)
@pytest.mark.parametrize("kept", [1.0, 0.6, 0.0])
def test_one_call_experts_forms(dev, form, T, E, topk, H, I, kept):
    from cosmos_rl_amd.policy.kernel.moe.moe import grouped_experts_forward
    assert _lib.moe_experts_form(T, topk, E, H, I) == form
    strategy, module = _module(dev, E, H, I, T)
    g = torch.Generator(device=dev).manual_seed(T + 5)
    x = torch.randn(T, H, generator=g, device=dev).to(torch.bfloat16)
    like = torch.rand(T, E, generator=g, device=dev) + 0.9 * torch.rand(E, generator=g, device=dev)   # some experts are liked better
    idx, w = like.topk(topk, dim=1).indices, torch.rand(T, topk, generator=g, device=dev).to(torch.bfloat16)
    mask = torch.rand(T, generator=g, device=dev) < kept
    junk = torch.full((64 << 20,), 0x7F, dtype=torch.uint8, device=dev)   # what the workspace holds before is no number
    del junk
    y = grouped_experts_forward(x, mask, w, idx, strategy, module, E)
    want = _chain(x, mask, w, idx, strategy, module, E)
    assert torch.equal(y.view(torch.int16), want.view(torch.int16)) and not bool(y[~mask].any())
    assert torch.equal(grouped_experts_forward(x, mask, w, idx, strategy, module, E).view(torch.int16), want.view(torch.int16))
