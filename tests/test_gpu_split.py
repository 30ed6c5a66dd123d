"""Sequences cut along T for the sequential passes (few (sequence, head) pairs, bfloat16): outputs, final state and all
gradients against the token recurrence in float64, at the edges of the cut -- a last segment of one token, of whole
chunks, of a partial chunk; states in and out; packed sequences of very unequal length, some empty, some of one
segment."""
import pytest
import torch
import torch.nn.functional as F

from oracle import naive
from tests.util import TOL, gen, max_abs_rel, oracle_grads

pytestmark = pytest.mark.gpu


def is_cut(op, B, T, H, K, V, N=None):
    """Whether the library cuts a call of these sizes (NT as the host layer counts it for offsets on the device)."""
    import ctypes as C
    from linear_moe_amd import _lib
    a = _lib.Args()
    a.dtype, a.B, a.T, a.H, a.K, a.V, a.N = _lib.LMOE_BF16, B, T, H, K, V, N or B
    a.NT = B * ((T + 63) // 64) + (N if N else 0)
    a.cu_seqlens = 16 if N else None               # (only asked whether it is there)
    return _lib.load().lmoe_split_floats(C.byref(a), op, 1) > 0


def check(fn_ref, fn, ins, do, dht, cuda):
    ref_o, ref_ht, ref = oracle_grads(fn_ref, ins, do, dht)
    dev = {n: x.to(cuda).requires_grad_(True) for n, x in ins.items()}
    o, ht = fn(**dev)
    grads = torch.autograd.grad([o, ht], list(dev.values()), [do.to(cuda), dht.to(cuda)])
    with torch.no_grad():                          # the forward-only instance
        of, hf = fn(**dev)
    torch.cuda.synchronize()
    tol = TOL[torch.bfloat16]
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
