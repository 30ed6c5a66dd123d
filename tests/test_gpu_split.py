"""Sequences cut along T for the sequential passes (few (sequence, head) pairs): outputs, final state and all
gradients against the token recurrence in float64, at the edges of the cut -- a last segment of one token, of whole
chunks, of a partial chunk; states in and out; packed sequences of very unequal length, some empty, some of one
segment."""
import pytest
import torch
import torch.nn.functional as F

from oracle import naive
from tests.util import TOL, gen, max_abs_rel, oracle_grads

pytestmark = pytest.mark.gpu


def is_cut(op, B, T, H, K, V, N=None, dtype=torch.bfloat16):
    """Whether the library cuts a call of these sizes (NT as the host layer counts it for offsets on the device)."""
    import ctypes as C
    from linear_moe_amd import _lib
    a = _lib.Args()
    a.dtype, a.B, a.T, a.H, a.K, a.V, a.N = _lib.LMOE_BF16 if dtype == torch.bfloat16 else _lib.LMOE_F32, B, T, H, K, V, N or B
    a.NT = B * ((T + 63) // 64) + (N if N else 0)
    a.cu_seqlens = 16 if N else None               # (only asked whether it is there)
    return _lib.load().lmoe_split_floats(C.byref(a), op, 1) > 0


def check(fn_ref, fn, ins, do, dht, cuda, dtype=torch.bfloat16):
    ref_o, ref_ht, ref = oracle_grads(fn_ref, ins, do, dht)
    dev = {n: x.to(cuda).requires_grad_(True) for n, x in ins.items()}
    o, ht = fn(**dev)
    grads = torch.autograd.grad([o, ht], list(dev.values()), [do.to(cuda), dht.to(cuda)])
    with torch.no_grad():                          # the forward-only instance
        of, hf = fn(**dev)
    torch.cuda.synchronize()
    tol = TOL[dtype]
    for x in (o, of):
        assert max_abs_rel(x.detach().cpu(), ref_o) < tol
    for x in (ht, hf):
        assert max_abs_rel(x.detach().cpu(), ref_ht) < tol
    for (n, r), x in zip(ref.items(), grads):
        assert max_abs_rel(x.cpu(), r) < tol, n


@pytest.mark.parametrize("B,T,H,K,V,lens", [
    (1, 2049, 2, 128, 128, None),                  # last chunk of one token
    (2, 2112, 1, 64, 64, None),                    # 33 whole chunks
    (1, 2400, 2, 64, 128, None),
    (1, 3000, 1, 128, 64, None),
    (1, 3000, 1, 128, 128, [3000]),
    (1, 10000, 1, 64, 128, [5000, 0, 5, 4995]),   # segments of two sequences, an empty one, one of a single segment
])
def test_gated_delta_rule_cut_along_t(cuda, B, T, H, K, V, lens):
    from linear_moe_amd import chunk_gated_delta_rule
    N = B if lens is None else len(lens)
    assert is_cut(2, B, T, H, K, V, None if lens is None else N)
    bf = lambda x: x.bfloat16()
    # slow decay (a state outlives several segments)
    ins = dict(q=bf(F.normalize(gen(7000, B, T, H, K), dim=-1)), k=bf(F.normalize(gen(7001, B, T, H, K), dim=-1)),
               v=bf(gen(7002, B, T, H, V)), g=-F.softplus(gen(7003, B, T, H)) * 0.003,
               beta=bf(torch.sigmoid(gen(7004, B, T, H))), h0=gen(7005, N, H, K, V) * 0.3)
    do, dht = bf(gen(7006, B, T, H, V)), gen(7007, N, H, K, V)
    cu = None if lens is None else torch.tensor([0] + lens).cumsum(0).to(torch.int32)
    cud = None if cu is None else cu.to(cuda)
    check(lambda q, k, v, g, beta, h0: naive.naive_recurrent_gated_delta_rule(q, k, v, g, beta, None, h0, True, cu, False),
          lambda q, k, v, g, beta, h0: chunk_gated_delta_rule(q, k, v, g, beta, None, h0, True, cud, False),
          ins, do, dht, cuda)


@pytest.mark.parametrize("lens,H", [([4096], 4), ([1472], 2), ([5000, 0, 1000, 1000], 2), ([2100, 1996], 4)])
def test_offsets_on_the_device_are_cut_as_those_on_the_host(cuda, lens, H):
    """Where cu_seqlens lies does not show: the same bits, outputs, states and every gradient."""
    from linear_moe_amd import chunk_gated_delta_rule
    T, N, D = sum(lens), len(lens), 128
    x = [F.normalize(gen(7400, 1, T, H, D), dim=-1).bfloat16(), F.normalize(gen(7401, 1, T, H, D), dim=-1).bfloat16(),
         gen(7402, 1, T, H, D).bfloat16(), -F.softplus(gen(7403, 1, T, H)) * 0.01, torch.sigmoid(gen(7404, 1, T, H)).bfloat16()]
    x = [t.to(cuda).requires_grad_(True) for t in x]
    h0 = gen(7405, N, H, D, D).to(cuda).requires_grad_(True)
    do, dht = gen(7406, 1, T, H, D).bfloat16().to(cuda), gen(7407, N, H, D, D).to(cuda)
    cu = torch.tensor([0] + lens).cumsum(0).to(torch.int32)
    outs = []
    for offs in (cu, cu.to(cuda)):
        o, ht = chunk_gated_delta_rule(*x, None, h0, True, offs, False)
        outs.append((o.detach(), ht.detach()) + torch.autograd.grad([o, ht], x + [h0], [do, dht]))
    torch.cuda.synchronize()
    for a, b in zip(*outs):
        assert torch.equal(a, b)


@pytest.mark.parametrize("dtype,B,T,H,K,V", [
    (torch.bfloat16, 1, 1281, 2, 128, 128),        # last chunk, and last segment, of one token
    (torch.bfloat16, 2, 1536, 1, 64, 64),          # whole chunks
    (torch.bfloat16, 1, 1500, 3, 64, 128),
    (torch.bfloat16, 2, 3000, 2, 128, 64),
    (torch.float32, 1, 321, 2, 64, 64),
    (torch.float32, 1, 512, 4, 64, 64),
    (torch.float32, 2, 1000, 1, 128, 128),
    (torch.float32, 1, 700, 3, 128, 64),
])
@pytest.mark.parametrize("gated", [True, False])
def test_simple_gla_cut_along_t(cuda, dtype, B, T, H, K, V, gated):
    from linear_moe_amd import chunk_simple_gla
    assert is_cut(0, B, T, H, K, V, dtype=dtype)
    ins = dict(q=gen(7100, B, T, H, K).to(dtype), k=(gen(7101, B, T, H, K) * K ** -0.5).to(dtype),
               v=gen(7102, B, T, H, V).to(dtype), h0=gen(7105, B, H, K, V) * 0.3)
    if gated:
        ins["g"] = -F.softplus(gen(7103, B, T, H)) * 0.003
    do, dht = gen(7106, B, T, H, V).to(dtype), gen(7107, B, H, K, V)
    check(lambda q, k, v, h0, g=None: naive.naive_recurrent_simple_gla(q, k, v, g, None, h0, True, None, False),
          lambda q, k, v, h0, g=None: chunk_simple_gla(q, k, v, g, None, h0, True, None, False),
          ins, do, dht, cuda, dtype)


@pytest.mark.parametrize("B,T,H,K,V", [
    (1, 2049, 2, 128, 128),                        # last chunk, and last segment, of one token
    (2, 2304, 1, 64, 64),                          # whole chunks
    (1, 2400, 2, 64, 128),
    (2, 3000, 2, 128, 64),
])
@pytest.mark.parametrize("head_first", [True, False])
def test_gla_cut_along_t(cuda, B, T, H, K, V, head_first):
    from linear_moe_amd import chunk_gla
    assert is_cut(1, B, T, H, K, V)
    tr = lambda x: x.transpose(1, 2) if head_first else x
    ins = dict(q=gen(7300, B, T, H, K).bfloat16(), k=(gen(7301, B, T, H, K) * K ** -0.5).bfloat16(),
               v=gen(7302, B, T, H, V).bfloat16(), g=F.logsigmoid(gen(7303, B, T, H, K)) * 0.01, h0=gen(7305, B, H, K, V) * 0.3)
    do, dht = gen(7306, B, T, H, V).bfloat16(), gen(7307, B, H, K, V)

    def ours(q, k, v, g, h0):
        o, ht = chunk_gla(tr(q), tr(k), tr(v), tr(g), None, h0, True, None, head_first)
        return tr(o), ht
    check(lambda q, k, v, g, h0: naive.naive_recurrent_gla(q, k, v, g, None, h0, True, None, False), ours, ins, do, dht, cuda)


@pytest.mark.parametrize("B,T,H,K,V", [(1, 1281, 2, 128, 128), (2, 1500, 1, 64, 64), (1, 2000, 2, 64, 128),
                                       (1, 1500, 2, 256, 64)])      # two key blocks: the divisor formed outside
def test_normalised_linear_attention_cut_along_t(cuda, B, T, H, K, V):
    """The normaliser's column goes through the cut beside the state, forward and backward."""
    from linear_moe_amd import chunk_linear_attn
    assert is_cut(0, B, T, H, min(K, 128), V)
    rows = lambda seed: torch.rand(B, H, T, K, generator=torch.Generator().manual_seed(seed)).bfloat16()
    ins = dict(q=rows(7200), k=rows(7201), v=gen(7202, B, H, T, V).bfloat16())
    do = gen(7206, B, H, T, V).bfloat16()
    leaves = {n: x.double().requires_grad_(True) for n, x in ins.items()}
    ref, _ = naive.naive_linear_attn(*leaves.values(), normalize=True)
    refs = torch.autograd.grad((ref * do.double()).sum(), list(leaves.values()))
    dev = {n: x.to(cuda).requires_grad_(True) for n, x in ins.items()}
    o, _ = chunk_linear_attn(*dev.values(), normalize=True)
    grads = torch.autograd.grad(o, list(dev.values()), do.to(cuda))
    torch.cuda.synchronize()
    for x, r in zip((o.detach(),) + grads, (ref.detach(),) + refs):
        assert max_abs_rel(x.cpu(), r) < TOL[torch.bfloat16]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_calls_without_heads_are_refused(cuda, dtype):
    """The rule of the cut sees a call before the op's checks do; the call still ends in the op's error."""
    from linear_moe_amd import chunk_gated_delta_rule, chunk_gla, chunk_simple_gla
    x, s = torch.empty(1, 3000, 0, 64, device=cuda, dtype=dtype), torch.empty(1, 3000, 0, device=cuda)
    for fn in (lambda: chunk_gated_delta_rule(x, x, x, s, s.to(dtype), head_first=False),
               lambda: chunk_simple_gla(x, x, x, s, head_first=False),
               lambda: chunk_gla(x, x, x, x.float(), head_first=False)):
        with pytest.raises(ValueError, match="dimension"):
            fn()


def lengths(op, B, T, H, K, V, N=None, dtype=torch.bfloat16):
    """Chunks per fine and per coarse segment."""
    import ctypes as C
    from linear_moe_amd import _lib
    a = _lib.Args()
    a.dtype, a.B, a.T, a.H, a.K, a.V, a.N = _lib.LMOE_BF16 if dtype == torch.bfloat16 else _lib.LMOE_F32, B, T, H, K, V, N or B
    a.NT = B * ((T + 63) // 64) + (N if N else 0)
    a.cu_seqlens = 16 if N else None               # (only asked whether it is there)
    fine, coarse = C.c_int32(), C.c_int32()
    assert _lib.load().lmoe_split_lengths(C.byref(a), op, C.byref(fine), C.byref(coarse)) == 0
    return fine.value, coarse.value


def check_part(fn_ref, fn, ins, do, dht, cuda, b, h, dtype=torch.bfloat16):
    """As check, the whole call against the oracle on batch row b and head h alone (rows and heads do not mix).
    Tensors [B, T, H, ...] and states [N, H, K, V]; b = None: packed input, all sequences."""
    cut = lambda x, state: (x if b is None else x[b:b + 1])[(slice(None),) * (1 if state else 2) + (slice(h, h + 1),)]
    ref_o, ref_ht, ref = oracle_grads(fn_ref, {n: cut(x, n == "h0") for n, x in ins.items()}, cut(do, False), cut(dht, True))
    dev = {n: x.to(cuda).requires_grad_(True) for n, x in ins.items()}
    o, ht = fn(**dev)
    grads = torch.autograd.grad([o, ht], list(dev.values()), [do.to(cuda), dht.to(cuda)])
    with torch.no_grad():
        of, hf = fn(**dev)
    torch.cuda.synchronize()
    for x, y in ((o, of), (ht, hf)):
        assert torch.equal(x.detach(), y)          # the forward-only instance is cut the same way
    assert max_abs_rel(cut(o.detach(), False).cpu(), ref_o) < TOL[dtype]
    assert max_abs_rel(cut(ht.detach(), True).cpu(), ref_ht) < TOL[dtype]
    for (n, r), x in zip(ref.items(), grads):
        assert max_abs_rel(cut(x, n == "h0").cpu(), r) < TOL[dtype], n


def delta_inputs(seed, B, T, H, K, V, N, gated=True):
    bf = lambda x: x.bfloat16()
    ins = dict(q=bf(F.normalize(gen(seed, B, T, H, K), dim=-1)), k=bf(F.normalize(gen(seed + 1, B, T, H, K), dim=-1)),
               v=bf(gen(seed + 2, B, T, H, V)), g=-F.softplus(gen(seed + 3, B, T, H)) * 0.003,
               beta=bf(torch.sigmoid(gen(seed + 4, B, T, H))), h0=gen(seed + 5, N, H, K, V) * 0.3)
    if not gated:
        del ins["g"]
    return ins, bf(gen(seed + 6, B, T, H, V)), gen(seed + 7, N, H, K, V)


@pytest.mark.parametrize("op,H,T,D,cut", [(0, 16, 1280, 128, False), (0, 32, 2048, 128, False), (0, 16, 2048, 128, True), (0, 16, 1280, 64, True),
                                          (2, 16, 1792, 128, False), (2, 16, 3008, 128, True), (2, 16, 2048, 64, True)])
def test_calls_that_narrow_slices_outrun_are_left_whole(cuda, op, H, T, D, cut):
    """On both sides of the line, dense and as one packed sequence; left whole, a call gives the bits that its rows have in a batch that fills the CUs."""
    from linear_moe_amd import chunk_gated_delta_rule, chunk_simple_gla
    assert (lengths(op, 1, T, H, D, D)[0] > 0) == cut
    if op == 2:
        assert (lengths(op, 1, T, H, D, D, 1)[0] > 0) == cut
    x = [F.normalize(gen(7600, 1, T, H, D), dim=-1).bfloat16(), F.normalize(gen(7601, 1, T, H, D), dim=-1).bfloat16(),
         gen(7602, 1, T, H, D).bfloat16(), -F.softplus(gen(7603, 1, T, H)) * 0.01, torch.sigmoid(gen(7604, 1, T, H)).bfloat16()]

    def run(n):
        d = [t.to(cuda).expand(n, *t.shape[1:]).contiguous().requires_grad_() for t in x[:5 if op == 2 else 4]]
        f = chunk_gated_delta_rule if op == 2 else chunk_simple_gla
        o, ht = f(*d, output_final_state=True, head_first=False)
        return [t[:1].detach() for t in (o, ht, *torch.autograd.grad(o, d, torch.ones_like(o)))]
    few, many = run(1), run(8)
    for a, b in zip(few, many):
        assert max_abs_rel(a, b) < TOL[torch.bfloat16]
        assert cut or torch.equal(a, b)


@pytest.mark.parametrize("B,T,H,K,V,lens,cut", [
    (1, 3001, 16, 128, 128, None, (3, 12)),        # four coarse segments, the last one of 11 chunks
    (1, 6000, 4, 64, 128, None, (3, 6)),           # the last one of two fine segments, the second of one chunk
    (1, 4096, 4, 128, 128, [2000, 2096], (2, 6)),
    (1, 6000, 4, 128, 128, [5300, 0, 700], (3, 9)),
    (1, 8000, 4, 64, 64, [64, 7935, 1], (3, 6)),
])
def test_gated_delta_rule_of_several_fine_segments(cuda, B, T, H, K, V, lens, cut):
    """Coarse segments of more than one fine segment: transitions alone in the last coarse segment, states handed on
    from every len3 / len1-th combination only, the first coarse segment left out of the backward's first step."""
    from linear_moe_amd import chunk_gated_delta_rule
    N = B if lens is None else len(lens)
    assert lengths(2, B, T, H, K, V, None if lens is None else N) == cut
    ins, do, dht = delta_inputs(7500, B, T, H, K, V, N)
    cu = None if lens is None else torch.tensor([0] + lens).cumsum(0).to(torch.int32)
    cud = None if cu is None else cu.to(cuda)
    check_part(lambda q, k, v, g, beta, h0: naive.naive_recurrent_gated_delta_rule(q, k, v, g, beta, None, h0, True, cu, False),
               lambda q, k, v, g, beta, h0: chunk_gated_delta_rule(q, k, v, g, beta, None, h0, True, cud, False),
               ins, do, dht, cuda, None if lens else B - 1, H - 1)


@pytest.mark.parametrize("gated", [True, False])
def test_delta_rule_cut_along_t_in_both_layouts(cuda, gated):
    """Head-first views of the tensors of a time-first call: the same bits; without a gate (chunk_delta_rule) too."""
    from linear_moe_amd import chunk_delta_rule, chunk_gated_delta_rule
    B, T, H, K, V = 1, 1601, 2, 128, 128
    assert lengths(2, B, T, H, K, V)[0] > 0
    ins, do, dht = delta_inputs(7600, B, T, H, K, V, B, gated)
    fn = chunk_gated_delta_rule if gated else chunk_delta_rule
    tr = lambda x: x.transpose(1, 2)
    order = ("q", "k", "v") + (("g",) if gated else ()) + ("beta",)

    def ours(head_first):
        def call(h0, **x):
            o, ht = fn(*(tr(x[n]) if head_first else x[n] for n in order), initial_state=h0, output_final_state=True,
                       head_first=head_first)
            return (tr(o) if head_first else o), ht
        return call
    check_part(lambda q, k, v, beta, h0, g=None: naive.naive_recurrent_gated_delta_rule(
        q, k, v, torch.zeros_like(beta) if g is None else g, beta, None, h0, True, None, False), ours(False), ins, do, dht, cuda, 0, 1)
    dev = {n: x.to(cuda).requires_grad_(True) for n, x in ins.items()}
    res = []
    for head_first in (False, True):
        o, ht = ours(head_first)(**dev)
        res.append((o.detach(), ht.detach()) + torch.autograd.grad([o, ht], list(dev.values()), [do.to(cuda), dht.to(cuda)]))
    for a, b in zip(*res):
        assert torch.equal(a, b)


@pytest.mark.parametrize("dtype,B,T,H,K,V,cut", [
    (torch.bfloat16, 2, 1500, 8, 128, 128, (3, 6)),
    (torch.bfloat16, 2, 2049, 8, 128, 128, (3, 9)),        # the last coarse segment of two fine ones, one token in the last chunk
    (torch.float32, 2, 1000, 8, 128, 128, (2, 8)),
    (torch.float32, 1, 1281, 8, 64, 64, (1, 3)),
])
@pytest.mark.parametrize("head_first", [True, False])
def test_simple_gla_of_several_fine_segments(cuda, dtype, B, T, H, K, V, cut, head_first):
    from linear_moe_amd import chunk_simple_gla
    assert lengths(0, B, T, H, K, V, dtype=dtype) == cut
    tr = lambda x: x.transpose(1, 2) if head_first else x
    ins = dict(q=gen(7700, B, T, H, K).to(dtype), k=(gen(7701, B, T, H, K) * K ** -0.5).to(dtype),
               v=gen(7702, B, T, H, V).to(dtype), g=-F.softplus(gen(7703, B, T, H)) * 0.003, h0=gen(7705, B, H, K, V) * 0.3)
    do, dht = gen(7706, B, T, H, V).to(dtype), gen(7707, B, H, K, V)

    def ours(q, k, v, g, h0):
        o, ht = chunk_simple_gla(tr(q), tr(k), tr(v), tr(g), None, h0, True, None, head_first)
        return tr(o), ht
    check_part(lambda q, k, v, g, h0: naive.naive_recurrent_simple_gla(q, k, v, g, None, h0, True, None, False), ours,
               ins, do, dht, cuda, B - 1, H - 1, dtype)


@pytest.mark.parametrize("B,T,H,K,V,cut", [(2, 3000, 8, 128, 128, (4, 12)), (2, 4000, 8, 64, 64, (4, 8))])
def test_gla_of_several_fine_segments(cuda, B, T, H, K, V, cut):
    from linear_moe_amd import chunk_gla
    assert lengths(1, B, T, H, K, V) == cut
    ins = dict(q=gen(7800, B, T, H, K).bfloat16(), k=(gen(7801, B, T, H, K) * K ** -0.5).bfloat16(),
               v=gen(7802, B, T, H, V).bfloat16(), g=F.logsigmoid(gen(7803, B, T, H, K)) * 0.01, h0=gen(7805, B, H, K, V) * 0.3)
    do, dht = gen(7806, B, T, H, V).bfloat16(), gen(7807, B, H, K, V)
    check_part(lambda q, k, v, g, h0: naive.naive_recurrent_gla(q, k, v, g, None, h0, True, None, False),
               lambda q, k, v, g, h0: chunk_gla(q, k, v, g, None, h0, True, None, False), ins, do, dht, cuda, B - 1, H - 1)


@pytest.mark.parametrize("D,T,B,H", [(128, 1601, 1, 2), (64, 2000, 2, 1)])
def test_mixer_core_cut_along_t(cuda, D, T, B, H):
    """v as a block of the projection, SiLU applied while the segments stage it: the bits of the op on silu(v)."""
    import linear_moe_amd as L
    assert lengths(2, B, T, H, D, D)[0] > 0
    qkv, do = gen(7900, T, B, H * 3 * D).bfloat16().to(cuda), gen(7903, B, T, H, D).bfloat16().to(cuda)
    g = -F.softplus(gen(7901, B, T, H)).to(cuda) * 0.003
    beta = torch.sigmoid(gen(7902, B, T, H)).bfloat16().to(cuda)
    res = []
    for core in (True, False):
        leaves = [t.clone().requires_grad_(True) for t in (qkv, g, beta)]
        if core:
            o = L.gdn_mixer_core(*leaves, H, D)
        else:
            q, k, v = L.gdn_qkv_prologue(leaves[0], H, D)
            o, _ = L.chunk_gated_delta_rule(q, k, v, leaves[1], leaves[2], head_first=False)
        res.append((o.detach(),) + torch.autograd.grad(o, leaves, do))
    torch.cuda.synchronize()
    (o1, dx1, dg1, db1), (o2, dx2, dg2, db2) = res
    assert torch.equal(o1, o2) and torch.equal(dg1, dg2) and torch.equal(db1, db2)
    d1, d2 = (x.view(T, B, H, 3 * D) for x in (dx1, dx2))
    assert torch.equal(d1[..., :2 * D], d2[..., :2 * D])
    assert max_abs_rel(d1[..., 2 * D:].float().cpu(), d2[..., 2 * D:].float().cpu()) < 1e-2   # dv: rounded once, not twice


def test_a_captured_packed_step_that_is_cut_follows_the_offsets_it_finds_at_replay(cuda):
    """The segments of packed sequences are found on the device: new offsets in the captured buffer (other lengths, a
    sequence of one chunk, an empty one, another number of chunks) give what an eager call on them gives."""
    from linear_moe_amd.gated_delta_rule import GDNCall
    T, H, D = 8000, 4, 128
    assert lengths(2, 1, T, H, D, D, 3) == (3, 12)
    x, do, dht = delta_inputs(8000, 1, T, H, D, D, 3)
    q, k, v, g, beta, h0 = (t.to(cuda) for t in x.values())
    do, dht = do.to(cuda), dht.to(cuda)
    offsets = [[0, 2600, 5300, 8000], [0, 1, 7000, 8000], [0, 8000, 8000, 8000], [0, 64, 128, 7990]]

    def step(call, cu):
        o, ht = call.forward(q, k, v, g, beta, None, h0, True, cu, False)
        return [o, ht] + [t for t in call.backward(do, dht) if t is not None]

    refs = [[t.clone() for t in step(GDNCall(keep=True), torch.tensor(c, dtype=torch.int32, device=cuda))] for c in offsets]
    cu = torch.tensor(offsets[0], dtype=torch.int32, device=cuda)
    call = GDNCall(keep=True)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        step(call, cu)
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        outs = step(call, cu)
    for i in (0, 1, 2, 3, 1, 0):
        cu.copy_(torch.tensor(offsets[i], dtype=torch.int32))
        for t in outs:
            t.zero_()
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        n = offsets[i][-1]                         # (rows behind the last sequence are nobody's)
        for j, (a, b) in enumerate(zip(outs, refs[i])):
            if a.shape[0] == 1:
                a, b = a[:, :n], b[:, :n]
            assert torch.equal(a, b), (i, j)


@pytest.mark.parametrize("gated", [True, False])
def test_error_of_the_cut_behind_a_drop_of_v(cuda, monkeypatch, gated):
    """A state that outlives many segments and a v that falls to a hundredth half way (the late chunks see what the early
    ones left): against float64 the cut call is as exact as the whole one.  Without a gate transitions and states are
    carried in two terms and the cut adds no rounding of its own: 1.05 for the scatter of two sums of as many roundings.
    Gated: the whole pass rounds the state for one product per chunk, the cut adds one product per fine segment with two
    rounded operands: with len1 >= 2 at most twice the variance, a factor sqrt(2) on the norm of the error."""
    from linear_moe_amd import chunk_delta_rule, chunk_gated_delta_rule
    from linear_moe_amd.gated_delta_rule import GDNCall
    T, H, D = 3001, 2, 128
    assert lengths(2, 1, T, H, D, D)[0] >= 2
    ins, _, _ = delta_inputs(8100, 1, T, H, D, D, 1, gated)
    ins["v"][:, T // 2:] *= 0.01
    d = {n: x.double() for n, x in ins.items()}
    g = d["g"] if gated else torch.zeros_like(d["beta"])
    ref, ref_ht = naive.naive_recurrent_gated_delta_rule(d["q"], d["k"], d["v"], g, d["beta"], None, d["h0"], True, None, False)
    x = [ins[n].to(cuda) for n in ("q", "k", "v") + (("g",) if gated else ()) + ("beta",)]
    h0, fn = ins["h0"].to(cuda), chunk_gated_delta_rule if gated else chunk_delta_rule

    def errors():
        with torch.no_grad():
            o, ht = fn(*x, initial_state=h0, output_final_state=True, head_first=False)
        diff = lambda a, r: (a.cpu().double() - r)
        n = T // 64 * 64
        per_chunk = lambda t: t[:, :n].reshape(n // 64, -1).norm(dim=1)
        return (per_chunk(diff(o, ref)) / per_chunk(ref)).max().item(), diff(o, ref).norm().item(), diff(ht, ref_ht).norm().item()

    cut = errors()
    monkeypatch.setattr(GDNCall, "_cut", lambda self, *a, **kw: setattr(self, "seg_ws", None))
    whole = errors()
    print(gated, "worst chunk, o, ht: cut", cut, "whole", whole)
    assert cut[0] < TOL[torch.bfloat16]
    bound = 2 ** 0.5 if gated else 1.05
    assert cut[1] < bound * whole[1] and cut[2] < bound * whole[2]


def by_chunks(B, T, H, K, V, final_state):
    """Whether a 4-byte call of chunk_simple_gla of three chunks and more runs chunk by chunk: it then asks for no workspace, while
    the pass is cut."""
    import ctypes as C
    from linear_moe_amd import _lib
    a = _lib.Args()
    a.dtype, a.B, a.T, a.H, a.K, a.V, a.N, a.NT = _lib.LMOE_F32, B, T, H, K, V, B, B * ((T + 63) // 64)
    assert _lib.load().lmoe_split_floats(C.byref(a), 0, 1) > 0
    a.o, a.ht = _lib.Tensor4(16, 0, 0, 0), 16 if final_state else None     # (only asked whether they are there)
    return _lib.load().lmoe_split_floats(C.byref(a), 0, 1) == 0


def test_which_4_byte_calls_run_chunk_by_chunk(cuda):
    for call, without, with_state in (((2, 500, 4, 64, 64), True, True), ((1, 512, 4, 128, 128), True, True), ((1, 511, 2, 128, 64), True, True),
                                      ((1, 512, 8, 128, 128), True, False), ((1, 513, 2, 64, 64), False, False)):
        assert (by_chunks(*call, False), by_chunks(*call, True)) == (without, with_state), call


@pytest.mark.parametrize("B,T,H,K,V", [
    (1, 1, 1, 64, 64), (2, 63, 3, 128, 64), (1, 64, 8, 64, 128), (1, 65, 2, 128, 128),      # one chunk, and one token more
    (2, 500, 4, 64, 64), (1, 512, 4, 128, 128), (1, 511, 2, 128, 64),      # seven waves with a chunk in front each, or eight
    (1, 512, 8, 128, 128),                                 # with a final state the pass
    (1, 513, 2, 64, 64), (32, 192, 4, 64, 64),             # beyond eight chunks, and more pairs than the CUs take: the pass
])
@pytest.mark.parametrize("gated", [False, True])
def test_simple_gla_4_byte_chunk_by_chunk(cuda, B, T, H, K, V, gated):
    """Short sequences in 4-byte elements: every chunk sums up the state it starts from.  With and without a final state, both
    layouts, a gate of 2-byte elements; the states saved for the backward are those of the chunks."""
    from linear_moe_amd import chunk_simple_gla
    ins = dict(q=gen(7500, B, T, H, K), k=gen(7501, B, T, H, K) * K ** -0.5, v=gen(7502, B, T, H, V), h0=gen(7505, B, H, K, V) * 0.3)
    if gated:                                               # (representable in either type)
        ins["g"] = (-F.softplus(gen(7503, B, T, H)) * 0.01).bfloat16().float()
    do, dht = gen(7506, B, T, H, V), gen(7507, B, H, K, V)
    check(lambda q, k, v, h0, g=None: naive.naive_recurrent_simple_gla(q, k, v, g, None, h0, True, None, False),
          lambda q, k, v, h0, g=None: chunk_simple_gla(q, k, v, g, None, h0, True, None, False),
          ins, do, dht, cuda, torch.float32)
    d = {n: x.to(cuda) for n, x in ins.items()}
    hf = {n: x.transpose(1, 2).contiguous() if n != "h0" else x for n, x in d.items()}
    o, _ = chunk_simple_gla(d["q"], d["k"], d["v"], d.get("g"), None, d["h0"], False, None, False)
    of, _ = chunk_simple_gla(hf["q"], hf["k"], hf["v"], hf.get("g"), None, hf["h0"])
    assert torch.equal(of.transpose(1, 2), o)
    ref, _ = naive.naive_recurrent_simple_gla(*(ins[n].double() if n in ins else None for n in ("q", "k", "v", "g")), None, ins["h0"].double(), False, None, False)
    assert max_abs_rel(o.cpu(), ref) < TOL[torch.float32]
    if gated:
        assert torch.equal(chunk_simple_gla(d["q"], d["k"], d["v"], d["g"].bfloat16(), None, d["h0"], False, None, False)[0], o)
