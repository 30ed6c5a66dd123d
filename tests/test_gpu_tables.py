"""The index tables the library forms on the device (chunk tables of packed input, routing tables of a
mixture-of-memories layer) against the tensor operations that form the same tables on the CPU: whole numbers, equal."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.int32, torch.int64])
@pytest.mark.parametrize("N,T,tail", [(1, 1, 0), (2, 64, 0), (7, 1000, 37), (255, 3000, 0), (257, 65536, 5), (4096, 20000, 0)])
def test_chunk_tables(cuda, N, T, tail, dtype):
    """Random offsets with empty sequences among them; ``tail`` rows behind the last sequence."""
    from linear_moe_amd._host import SeqPlan
    g = torch.Generator().manual_seed(N)
    cut = torch.sort(torch.randint(0, T - tail + 1, (N - 1,), generator=g)).values
    cu = torch.cat([torch.zeros(1, dtype=torch.int64), cut, torch.tensor([T - tail])]).to(dtype)
    ref = SeqPlan.__new__(SeqPlan)
    ref.seq_order = None
    ref._build_on_device(T, cu)
    strided = torch.stack([cu, cu], 1).to(cuda)[:, 0]
    for offs in (cu.to(cuda), strided):
        got = SeqPlan(1, T, offs, cuda)
        assert (got.N, got.NT) == (ref.N, ref.NT)
        for name in ("cu", "chunk_map", "seq_chunk0", "nt_dev", "seq_order"):
            x, y = getattr(got, name), getattr(ref, name)
            assert (x is None) == (y is None), name
            if x is not None:
                assert x.dtype == y.dtype and torch.equal(x.cpu(), y), name


@pytest.mark.parametrize("capacity", [None, 0.3])
@pytest.mark.parametrize("B,S,topk,E", [(1, 1, 1, 1), (3, 37, 2, 4), (2, 1024, 2, 8), (1, 2047, 1, 3), (2, 2049, 1, 64),
                                        (1, 5000, 4, 5), (40, 16, 2, 100), (2, 300, 1, 1024), (3, 3000, 2, 300)])
def test_routing_tables(cuda, B, S, topk, E, capacity):
    """Lengths around the segments of 512 (the last case: 2048) choices and the 64 lanes that rank them."""
    from linear_moe_amd.mom import _plan_by_sorting, mom_plan
    g = torch.Generator().manual_seed(B * S + E)
    sel = torch.topk(torch.rand(B, S, E, generator=g), topk, dim=-1).indices
    ref = _plan_by_sorting(sel.reshape(-1), B, S, topk, E, capacity)
    for s in (sel, sel.int()):
        got = mom_plan(s.to(cuda), E, capacity)
        assert got.T_total == ref.T_total and got.max_len == ref.max_len
        for name in ("src_token", "src_choice", "row_of", "cu_seqlens", "mem_offsets_dev", "max_len_dev"):
            x, y = getattr(got, name), getattr(ref, name)
            assert x.dtype == y.dtype and torch.equal(x.cpu(), y), name


@pytest.mark.parametrize("dtype", [torch.int32, torch.int64])
def test_routing_tables_of_views(cuda, dtype):
    """Choices that flatten to a view with a stride: one column of wider choices, one choice for all tokens."""
    from linear_moe_amd.mom import _plan_by_sorting, mom_plan
    B, S, E = 2, 300, 4
    sel = torch.topk(torch.rand(B, S, E, generator=torch.Generator().manual_seed(8)), 2, dim=-1).indices.to(dtype)
    wide = sel.to(cuda)
    for s, x in ((sel[:1, :, :1], wide[:1, :, :1]), (sel[..., 1:], wide[..., 1:]),
                 (sel[:1, :1, :1].expand(B, S, 1), wide[:1, :1, :1].expand(B, S, 1)),
                 (sel.transpose(0, 1), wide.transpose(0, 1))):
        b, t, k = s.shape
        ref, got = _plan_by_sorting(s.reshape(-1).long(), b, t, k, E, None), mom_plan(x, E)
        for name in ("src_token", "src_choice", "row_of", "cu_seqlens", "mem_offsets_dev", "max_len_dev"):
            assert torch.equal(getattr(got, name).cpu(), getattr(ref, name)), name


def test_memories_out_of_range_are_dropped(cuda):
    from linear_moe_amd.mom import mom_combine, mom_pack, mom_plan
    sel = torch.tensor([[[0, 9], [-1, 1], [1, 0]]]).to(cuda)
    plan = mom_plan(sel, 2)
    assert plan.row_of.tolist() == [[0, -1], [-1, 2], [3, 1]]
    assert plan.cu_seqlens.tolist() == [0, 2, 4] and plan.src_token.tolist() == [0, 2, 1, 2, -1, -1]
    x = torch.arange(24, dtype=torch.float32, device=cuda).view(1, 3, 8)
    y = mom_pack(x, plan).requires_grad_(True)
    assert (y[4:] == 0).all()
    w = torch.ones(1, 3, 2, device=cuda, requires_grad=True)
    mom_combine(y, plan, w).sum().backward()
    assert y.grad[:4].eq(1).all() and y.grad[4:].eq(0).all()
    assert torch.equal(w.grad.view(3, 2).ne(0).cpu(), torch.tensor([[True, False], [False, True], [True, True]]))


@pytest.mark.parametrize("capacity", [None, 0.2])
@pytest.mark.parametrize("B,S,topk,E", [(1, 63, 1, 16), (1, 65, 1, 17), (5, 511, 1, 2), (2, 513, 2, 16), (12, 512, 1, 16),
                                        (64, 16, 1, 16), (65, 16, 1, 16), (1, 16384, 1, 4), (1, 16385, 1, 4)])
def test_routing_tables_in_one_launch(cuda, B, S, topk, E, capacity):
    """On both sides of what one launch takes: 16 memories, 1024 counts, 16384 choices of 4 memories; some choices out of range."""
    from linear_moe_amd.mom import mom_plan
    sel = torch.topk(torch.rand(B, S, E, generator=torch.Generator().manual_seed(B + S + E)), topk, dim=-1).indices
    sel[:, ::7, -1] = E
    sel[:, ::11, 0] = -1
    # rows in order: by memory, batch row, time; the last max_len of every sequence
    flat = sel.reshape(B, S * topk)
    seqs = [[[b * S * topk + i for i in (flat[b] == e).nonzero()[:, 0].tolist()] for b in range(B)] for e in range(E)]
    longest = max(len(x) for row in seqs for x in row)
    keep = longest if capacity is None else min(longest, -int(-S * capacity // 1))
    kept = [x[len(x) - min(len(x), keep):] for row in seqs for x in row]
    choice = torch.tensor([c for x in kept for c in x], dtype=torch.int32)
    cu = torch.tensor([0] + [len(x) for x in kept]).cumsum(0)
    row_of = torch.full((B * S * topk,), -1, dtype=torch.int32)
    row_of[choice.long()] = torch.arange(len(choice), dtype=torch.int32)
    got = mom_plan(sel.to(cuda), E, capacity)
    n = len(choice)
    assert got.max_len == keep and torch.equal(got.cu_seqlens.cpu().long(), cu) and torch.equal(got.mem_offsets, cu[::B])
    assert torch.equal(got.row_of.cpu().view(-1), row_of)
    assert torch.equal(got.src_choice.cpu()[:n], choice) and torch.equal(got.src_token.cpu()[:n], choice // topk)
    assert (got.src_choice[n:] == -1).all() and (got.src_token[n:] == -1).all()
