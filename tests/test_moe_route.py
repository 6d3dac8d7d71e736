"""Expert-grouped row layout of routed tokens (cfp8_route_tokens) against a brute force over the pairs: integers, exact."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _by_loops(indices, mask, E, alignment, capacity, keep_empty):
    T, K = indices.shape
    groups = [[] for _ in range(E)]
    for t in range(T):
        for s in range(K):
            e = int(indices[t, s])
            if mask[t] and 0 <= e < E:
                groups[e].append((t, s))
    sizes = [max(len(g), alignment if keep_empty else 0) for g in groups]
    sizes = [-(-n // alignment) * alignment for n in sizes]
    row_tokens, row_experts, row_of, start = [-1] * capacity, [-1] * capacity, {}, 0
    for e, g in enumerate(groups):
        for i, (t, s) in enumerate(g):
            if start + i < capacity:
                row_tokens[start + i] = t
                row_of[(t, s)] = start + i
        for r in range(start, min(start + sizes[e], capacity)):
            row_experts[r] = e
        start += sizes[e]
    key = [[int(indices[t, s]) if mask[t] and 0 <= int(indices[t, s]) < E else E for s in range(K)] for t in range(T)]
    order = [sorted(range(K), key=lambda s: key[t][s]) for t in range(T)]
    row_map = [[row_of.get((t, s), -1) for s in order[t]] for t in range(T)]
    return row_tokens, row_experts, row_map, order, sizes


# one launch (up to 1024 pairs) and two on either side of the line, partial last workgroups, one expert, experts at and around
# powers of two and at the limit of the tables, repeated experts in a token, a capacity that cuts rows off
@pytest.mark.parametrize("T,K,E,alignment,distinct,short", [(1, 1, 1, 16, True, False), (3, 8, 128, 128, True, False), (128, 8, 64, 128, True, False), (205, 5, 64, 8, True, False), (90, 7, 40, 16, False, False), (512, 8, 128, 1, True, False),
                                                            (513, 8, 127, 128, True, False), (700, 6, 129, 16, False, False),
                                                            (2049, 3, 1024, 8, False, False), (1024, 4, 2, 64, False, True), (5000, 2, 33, 128, True, False)])
@pytest.mark.parametrize("keep_empty", [True, False])
def test_route_tokens(dev, T, K, E, alignment, distinct, short, keep_empty):
    from cosmos_rl_amd import _lib
    g = torch.Generator().manual_seed(T * 31 + E)
    indices = torch.rand(T, E, generator=g).topk(K, dim=1).indices if distinct else torch.randint(0, E, (T, K), generator=g)
    if T > 2:
        indices[T // 2, 0] = -1                    # an index no expert has
    mask = torch.rand(T, generator=g) < 0.9
    w = torch.rand(T, K, generator=g)
    capacity = T * K + E * alignment
    if short:
        capacity = T * K // 2
    want = _by_loops(indices, mask, E, alignment, capacity, keep_empty)
    lib = _lib.load()
    need = lib.cfp8_route_tokens_workspace_bytes(T, K, E)
    for it, wt in ((torch.int64, torch.bfloat16), (torch.int32, torch.float32)):
        ind, mk, wd = indices.to(it).to(dev), mask.to(dev), w.to(wt).to(dev)
        i32 = lambda *s: torch.full(s, 77, dtype=torch.int32, device=dev)
        rt, re, rm, ms, mo = i32(capacity), i32(capacity), i32(T, K), i32(E), i32(E)
        so = torch.full((T, K), 77, dtype=torch.int64, device=dev)
        sw = torch.zeros(T, K, dtype=torch.bfloat16, device=dev)
        ws = torch.empty(max(need, 1), dtype=torch.uint8, device=dev)
        _lib.check(lib.cfp8_route_tokens(ind.data_ptr(), ind.element_size(), mk.data_ptr(), T, K, E, alignment, _lib.ROUTE_KEEP_EMPTY if keep_empty else 0, capacity, rt.data_ptr(),
                                         re.data_ptr(), rm.data_ptr(), so.data_ptr(), wd.data_ptr(),
                                         _lib.IN_BF16 if wt == torch.bfloat16 else _lib.IN_F32, sw.data_ptr(), ms.data_ptr(), mo.data_ptr(),
                                         ws.data_ptr(), need, torch.cuda.current_stream().cuda_stream))
        for got, ref in ((rt, want[0]), (re, want[1]), (rm, want[2]), (so, want[3]), (ms, want[4])):
            assert got.cpu().tolist() == ref
        assert torch.equal(mo.cpu().long(), torch.tensor(want[4]).cumsum(0))
        assert torch.equal(sw.cpu(), torch.gather(w, 1, so.cpu()).to(torch.bfloat16))


@pytest.mark.parametrize("T,K,E,alignment,shift", [(16500, 8, 128, 128, 0.0), (33000, 8, 65, 16, 0.3), (131073, 1, 1000, 8, 0.0), (128, 8, 64, 16, 0.0)])
def test_route_tokens_many_pairs(dev, T, K, E, alignment, shift):
    """More pairs than 128 workgroups place in one round (131072), with partial last rounds: against a stable sort."""
    from cosmos_rl_amd.policy.kernel.moe.moe import route_tokens
    g = torch.Generator().manual_seed(T + E)
    indices = (torch.rand(T, E, generator=g) + shift * torch.rand(E, generator=g)).topk(K, dim=1).indices if E * T < 20e6 else torch.randint(0, E, (T, K), generator=g)
    mask = torch.rand(T, generator=g) < 0.9
    r = route_tokens(indices.to(dev), mask.to(dev), E, alignment)
    key = torch.where(mask[:, None], indices, E)
    order = torch.sort(key.reshape(-1), stable=True).indices
    counts = torch.bincount(key.reshape(-1), minlength=E + 1)[:E]
    sizes = ((counts.clamp_min(alignment) + alignment - 1) // alignment * alignment)
    ends, first = sizes.cumsum(0), counts.cumsum(0) - counts
    row_tokens, row_of = torch.full((r.row_tokens.numel(),), -1), torch.full((T * K,), -1)
    kept = order[:int(counts.sum())]
    e = key.reshape(-1)[kept]
    rows = (ends - sizes)[e] + torch.arange(kept.numel()) - first[e]
    row_tokens[rows], row_of[kept] = kept // K, rows
    slots = torch.sort(key, dim=1, stable=True).indices
    assert torch.equal(r.m_sizes.cpu().long(), sizes) and torch.equal(r.m_offsets.cpu().long(), ends)
    assert torch.equal(r.row_tokens.cpu().long(), row_tokens) and torch.equal(r.slot_order.cpu(), slots)
    assert torch.equal(r.row_map.cpu().long(), torch.gather(row_of.view(T, K), 1, slots))


def test_route_tokens_more_experts_than_the_tables_hold(dev):
    """The fallback gives what the kernel gives: 1024 experts by both, the fallback asked for by name."""
    from cosmos_rl_amd.policy.kernel.moe import moe
    g = torch.Generator().manual_seed(3)
    indices = torch.randint(0, 1024, (300, 4), generator=g)
    indices[7, 1], indices[8, 3], indices[299, 0] = -3, 1024, 5000        # indices no expert has
    indices = indices.to(dev)
    mask = (torch.rand(300, generator=g) < 0.8).to(dev)
    a = moe.route_tokens(indices, mask, 1024, 8)
    b = moe._route_tokens_by_sorting(indices, mask, 1024, 8, a.row_tokens.numel())
    for x, y in zip((a.row_tokens, a.row_map, a.slot_order, a.m_sizes, a.m_offsets), (b.row_tokens, b.row_map, b.slot_order, b.m_sizes, b.m_offsets)):
        assert torch.equal(x, y)
    assert moe.route_tokens(indices, mask, 1500, 8).m_sizes.numel() == 1500
