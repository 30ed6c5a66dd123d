"""The launch path in native code (csrc/lmoe_native.cpp) against the same steps in Python: the same bits for every form
of a call that it takes, and None, i.e. the Python steps, for the forms it does not."""
import itertools

import pytest
import torch

pytestmark = pytest.mark.gpu


def _inputs(op, B, T, H, K, V, dtype, head_first, strided, gdt, cuda, seed=5):
    gen = torch.Generator(device=cuda).manual_seed(seed)
    rn = lambda *s: torch.randn(*s, generator=gen, device=cuda)

    def rows(D, dt=dtype):
        shape = (B, H, T, D) if head_first else (B, T, H, D)
        if not strided:
            return rn(*shape).to(dt)
        # a view with swapped axes of a wider buffer: aligned rows, strides of its own
        x = rn(B, shape[2], shape[1], D + 16).to(dt)
        return x.transpose(1, 2)[..., :D]
    norm = lambda x: x / x.float().norm(dim=-1, keepdim=True).to(x.dtype)
    tok = (B, H, T) if head_first else (B, T, H)
    q, k, v = norm(rows(K)), norm(rows(K)), rows(V)
    if strided:
        q = rows(K) * 0.1
    g = {0: lambda: -rn(*tok).abs().to(gdt) * 0.1, 1: lambda: (-rn(*q.shape).abs() * 0.05).to(gdt), 2: lambda: -rn(*tok).abs().to(gdt)}[op]()
    beta = torch.sigmoid(rn(*tok)).to(gdt) if op == 2 else None
    return dict(q=q, k=k, v=v, g=g, beta=beta)


def _call(op, keep):
    from linear_moe_amd.gated_delta_rule import GDNCall
    from linear_moe_amd.gla import GLACall
    from linear_moe_amd.simple_gla import SimpleGLACall
    return (SimpleGLACall, GLACall, GDNCall)[op](keep)


def _both(op, x, h0, ofs, cu, hf, do, dht, monkeypatch, **kw):
    """results of the two paths; ``kept`` forces the Python steps, the other one must not reach them"""
    import linear_moe_amd._host as host
    import linear_moe_amd.gated_delta_rule as gdr
    import linear_moe_amd.gla as gla
    import linear_moe_amd.simple_gla as sg
    args = [x["q"], x["k"], x["v"], x["g"]] + ([x["beta"]] if op == 2 else []) + [None, h0, ofs, cu, hf]
    out = []
    for keep in (True, False):
        c = _call(op, keep)
        with monkeypatch.context() as m:
            if not keep:
                for mod in (sg, gla, gdr):
                    m.setattr(mod, "base_args", None)          # (the Python steps would call it)
            o, ht = c.forward(*args, **kw)
            extra = (o,) if kw.get("norm_eps") is not None else ()
            out.append([o, ht, *c.backward(do, dht if ofs else None, *extra)])
    return out


FORMS = list(itertools.product((0, 1, 2), (torch.bfloat16, torch.float32), (True, False), (False, True)))


@pytest.mark.parametrize("op,dtype,head_first,strided", [f for f in FORMS if not (f[0] == 2 and f[1] == torch.float32)])
@pytest.mark.parametrize("T,with_state,gdt", [(1, True, torch.float32), (200, False, torch.bfloat16), (1900, True, torch.float32)])
def test_same_bits_as_the_python_steps(cuda, monkeypatch, op, dtype, head_first, strided, T, with_state, gdt):
    if op == 1 and dtype == torch.float32:
        gdt = torch.float32
    B, H, K, V = 2, 3, 64, 128
    x = _inputs(op, B, T, H, K, V, dtype, head_first, strided, gdt, cuda)
    h0 = torch.randn(B, H, K, V, device=cuda) if with_state else None
    do = torch.randn(x["v"].shape, device=cuda).to(dtype)
    dht = torch.randn(B, H, K, V, device=cuda)
    ref, got = _both(op, x, h0, with_state, None, head_first, do, dht, monkeypatch)
    for a, b in zip(ref, got):
        assert (a is None) == (b is None)
        if a is not None:
            assert a.dtype == b.dtype and a.shape == b.shape and a.stride() == b.stride() and torch.equal(a, b)


@pytest.mark.parametrize("op", [0, 1, 2])
@pytest.mark.parametrize("host_offsets", [True, False])
def test_same_bits_packed(cuda, monkeypatch, op, host_offsets):
    cu = torch.tensor([0, 70, 70, 71, 500], dtype=torch.int32)
    cu = cu if host_offsets else cu.to(cuda)
    x = _inputs(op, 1, 500, 2, 128, 128, torch.bfloat16, False, False, torch.float32, cuda)
    h0, dht = torch.randn(4, 2, 128, 128, device=cuda), torch.randn(4, 2, 128, 128, device=cuda)
    do = torch.randn_like(x["v"])
    ref, got = _both(op, x, h0, True, cu, False, do, dht, monkeypatch)
    assert all((a is None and b is None) or torch.equal(a, b) for a, b in zip(ref, got))


@pytest.mark.parametrize("T", [1, 1000])
def test_same_bits_normalized(cuda, monkeypatch, T):
    x = _inputs(0, 2, T, 2, 64, 64, torch.bfloat16, True, False, torch.float32, cuda)
    x["q"], x["k"], x["g"] = x["q"].abs(), x["k"].abs(), None
    do = torch.randn_like(x["v"])
    ref, got = _both(0, x, None, False, None, True, do, None, monkeypatch, norm_eps=1e-10)
    assert all((a is None and b is None) or torch.equal(a, b) for a, b in zip(ref, got))


def test_ungated_delta_rule_same_bits(cuda, monkeypatch):
    x = _inputs(2, 1, 2000, 2, 128, 64, torch.bfloat16, False, False, torch.bfloat16, cuda)
    x["g"] = None
    ref, got = _both(2, x, None, True, None, False, torch.randn_like(x["v"]), torch.randn(1, 2, 128, 64, device=cuda), monkeypatch)
    assert all((a is None and b is None) or torch.equal(a, b) for a, b in zip(ref, got))


@pytest.mark.parametrize("op", [0, 1, 2])
@pytest.mark.parametrize("head_first", [True, False])
def test_recurrent_same_bits(cuda, monkeypatch, op, head_first):
    import linear_moe_amd as L
    import linear_moe_amd.recurrent as rec
    x = _inputs(op, 3, 2, 2, 64, 128, torch.bfloat16, head_first, True, torch.float32, cuda)
    h0 = torch.randn(3, 2, 64, 128, device=cuda)
    f = (L.fused_recurrent_simple_gla, L.fused_recurrent_gla, L.fused_recurrent_gated_delta_rule)[op]
    args = [x["q"], x["k"], x["v"], x["g"]] + ([x["beta"]] if op == 2 else [])
    with monkeypatch.context() as m:
        m.setattr(rec, "base_args", None)
        got = f(*args, initial_state=h0, output_final_state=True, head_first=head_first)
    with monkeypatch.context() as m:
        m.setattr(rec, "native", lambda *a: None)
        ref = f(*args, initial_state=h0, output_final_state=True, head_first=head_first)
    assert torch.equal(ref[0], got[0]) and torch.equal(ref[1], got[1]) and ref[0].stride() == got[0].stride()


def test_other_calls_take_the_python_steps(cuda):
    """what the native path hands back: a subclass, a last dimension with a stride, misaligned rows, other types of gate
    or state; and what is refused stays refused, in the words of the Python steps"""
    import linear_moe_amd as L
    from linear_moe_amd._host import native
    x = _inputs(0, 2, 100, 2, 64, 64, torch.bfloat16, True, False, torch.float32, cuda)
    q, k, v, g = x["q"], x["k"], x["v"], x["g"]
    call = lambda q, k, v, g, h0=None: native("forward", "t", 0, q, k, v, g, None, h0, None, None, True, True, False, 0, 0.0, False)
    ref = L.chunk_simple_gla(q, k, v, g)[0]
    assert torch.equal(call(q, k, v, g)[0], ref)

    class Sub(torch.Tensor):
        pass

    wide = torch.zeros(2, 2, 100, 65, device=cuda, dtype=torch.bfloat16)
    wide[..., 1:] = q
    for other in ((q.as_subclass(Sub), k, v, g), (q.transpose(2, 3).contiguous().transpose(2, 3), k, v, g),
                  (wide[..., 1:], k, v, g), (q, k, v, g.half())):
        assert call(*other) is None
        assert (L.chunk_simple_gla(*other)[0].float() - ref.float()).abs().max() <= 1e-2 * ref.float().abs().max()
    h0 = torch.randn(2, 2, 64, 64, device=cuda)
    assert call(q, k, v, g, h0.bfloat16()) is None
    for bad, err in (((q, k[:, :, :50], v, g), ValueError), ((q, k.float(), v, g), ValueError), ((q, k, v, g[:, :, :50]), ValueError),
                     ((q, k.cpu(), v, g), RuntimeError)):
        assert call(*bad) is None
        with pytest.raises(err):
            L.chunk_simple_gla(*bad)
    with pytest.raises(ValueError):
        L.chunk_simple_gla(q, k, v, g, initial_state=h0[:1])


# What is saved for the backward, in the order it is handed to autograd (see the ops' ``call.saved``): the buffers of the
# forward pass behind q, k, v, gate(s); with norm_eps the output is the last one
SAVED = {"simple": ("q", "k", "v", "g", "hs"), "normalized": ("q", "k", "v", "hs", "den", "zs", "o"),
         "gla": ("q", "k", "v", "g", "hs", "amat", "qe", "ke", "gdec"),
         "gdn": ("q", "k", "v", "g", "beta", "h0", "hs", "tinv", "pmat", "gcum", "vnew"),
         "gdn_cut": ("q", "k", "v", "g", "beta", "h0", "hs", "tinv", "pmat", "gcum", "vnew", "seg_p")}


def _through_hooks(kind, cuda, change):
    """gradients of one call whose saved tensors come back as change(name, x)"""
    import linear_moe_amd as L
    op = 2 if kind.startswith("gdn") else 1 if kind == "gla" else 0
    B, T = (1, 4000) if kind == "gdn_cut" else (2, 200)
    x = _inputs(op, B, T, 2, 64, 64, torch.bfloat16, False, False, torch.float32, cuda)
    if kind == "normalized":
        x["q"], x["k"], x["g"] = x["q"].abs(), x["k"].abs(), None
    leaves = [t.requires_grad_() for t in x.values() if t is not None]
    names = SAVED[kind]
    count = [0]

    def pack(t):
        count[0] += 1
        return count[0] - 1, t

    with torch.autograd.graph.saved_tensors_hooks(pack, lambda p: change(names[p[0]], p[1])):
        if kind == "simple":
            o, _ = L.chunk_simple_gla(x["q"], x["k"], x["v"], x["g"], head_first=False)
        elif kind == "normalized":
            o, _ = L.chunk_linear_attn(x["q"], x["k"], x["v"], head_first=False)
        elif kind == "gla":
            o, _ = L.chunk_gla(x["q"], x["k"], x["v"], x["g"], head_first=False)
        else:
            h0 = torch.ones(B, 2, 64, 64, device=cuda, requires_grad=True)
            leaves.append(h0)
            o, _ = L.chunk_gated_delta_rule(x["q"], x["k"], x["v"], x["g"], x["beta"], initial_state=h0)
    assert count[0] == len(names), (count[0], names)
    do = torch.randn(o.shape, device=cuda, generator=torch.Generator(device=cuda).manual_seed(3)).to(o.dtype)
    return torch.autograd.grad(o, leaves, do)


def _misaligned(x):
    flat = torch.empty(x.numel() + 1, dtype=x.dtype, device=x.device)
    flat[1:] = x.reshape(-1)
    return flat[1:].view(x.shape)


@pytest.mark.parametrize("kind", list(SAVED))
def test_saved_tensors_that_come_back_changed(cuda, kind):
    """the kernels index the full extent of what was saved: another type, other strides or another place in memory of a buffer
    give the same gradients, a shorter buffer (or input) is refused before anything is launched"""
    ref = _through_hooks(kind, cuda, lambda n, x: x)
    buffers = [n for n in SAVED[kind] if n not in ("q", "k", "v", "g", "beta", "o")]
    changes = [lambda x: x.double() if x.dtype == torch.float32 else x.float(),
               lambda x: x.mT.contiguous().mT if x.dim() > 1 else x.double(), _misaligned]
    for name, f in itertools.product(buffers, changes):
        got = _through_hooks(kind, cuda, lambda n, x: f(x) if n == name else x)
        assert all(torch.equal(a, b) for a, b in zip(ref, got)), name
    for name in SAVED[kind]:
        for cut in (lambda x: x[:, :1] if x.dim() > 1 else x[:-4], lambda x: x[..., :-4], lambda x: x.cpu()):
            with pytest.raises((RuntimeError, ValueError)):
                _through_hooks(kind, cuda, lambda n, x: cut(x) if n == name else x)


def test_calls_handed_back_leave_no_error_behind(cuda):
    """a call that is not for the native path gives None, whatever stopped it and at whichever check"""
    from linear_moe_amd._host import native
    x = _inputs(2, 2, 100, 2, 64, 64, torch.bfloat16, False, False, torch.float32, cuda)
    f = lambda q, k, v, g, beta, scale=None, hf=False, eps=0.0: native("forward", "t", 2, q, k, v, g, beta, None, None, scale, False,
                                                                      hf, True, 0, eps, False)
    ok = (x["q"], x["k"], x["v"], x["g"], x["beta"])
    assert type(f(*ok)) is tuple
    assert f(*(t.float() for t in ok)) is None                                   # 4-byte delta rule
    assert f(*ok[:3], ok[3].half(), ok[4]) is None and f(*ok[:4], ok[4].double()) is None and f(*ok[:4], None) is None
    assert f(*ok, scale="x") is None and f(*ok, hf=torch.ones(2)) is None and f(*ok, eps="x") is None


@pytest.mark.parametrize("op", [0, 1, 2])
@pytest.mark.parametrize("head_first", [True, False])
@pytest.mark.parametrize("T", [200, 1900])
def test_backward_is_native_where_only_the_forward_was_not(cuda, monkeypatch, op, head_first, T):
    """a 2-byte gate of the other kind sends the forward to the Python steps, which convert it: the backward has nothing to
    convert any more and takes the native path, with the same bits"""
    import linear_moe_amd.gated_delta_rule as gdr
    import linear_moe_amd.gla as gla
    import linear_moe_amd.simple_gla as sg
    x = _inputs(op, 2, T, 2, 64, 64, torch.bfloat16, head_first, False, torch.float16, cuda)
    args = [x["q"], x["k"], x["v"], x["g"]] + ([x["beta"]] if op == 2 else []) + [None, None, False, None, head_first]
    do = torch.randn_like(x["v"])
    out = []
    for keep in (True, False):
        c = _call(op, keep)
        o, _ = c.forward(*args)
        with monkeypatch.context() as m:
            if not keep:
                for mod in (sg, gla, gdr):
                    m.setattr(mod, "base_args", None)
            out.append([o, *c.backward(do, None)])
    assert all((a is None and b is None) or torch.equal(a, b) for a, b in zip(*out))


def test_other_threads_run_while_a_call_allocates(cuda):
    """the interpreter's lock is not held over the allocations: a call on an empty cache spends most of its time in them, and
    another thread that only looks at the clock stands still for less than 0.4 of it (the middle of nine calls; 0.6 to 0.75 with
    the lock held)"""
    import sys
    import threading
    import time
    import linear_moe_amd as L
    x = _inputs(2, 4, 8192, 32, 128, 128, torch.bfloat16, False, False, torch.float32, cuda)
    x["q"].requires_grad_()
    interval, shares = sys.getswitchinterval(), []
    sys.setswitchinterval(1e-4)
    try:
        for _ in range(10):
            torch.cuda.synchronize()
            torch.cuda.empty_cache()
            worst, stop = [0.0], threading.Event()

            def watch():
                last = time.perf_counter()
                while not stop.is_set():
                    now = time.perf_counter()
                    worst[0] = max(worst[0], now - last)
                    last = now
            th = threading.Thread(target=watch)
            th.start()
            time.sleep(0.01)
            t = time.perf_counter()
            o = L.chunk_gated_delta_rule(**x)[0]
            t = time.perf_counter() - t
            stop.set()
            th.join()
            shares.append(worst[0] / t)
            del o
    finally:
        sys.setswitchinterval(interval)
    assert sorted(shares[1:])[4] < 0.4, shares


def _mods():
    import linear_moe_amd.gated_delta_rule as gdr
    import linear_moe_amd.gla as gla
    import linear_moe_amd.simple_gla as sg
    return sg, gla, gdr


@pytest.mark.parametrize("op", [0, 1, 2])
@pytest.mark.parametrize("form", ["dense", "head_first", "packed", "cut"])
@pytest.mark.parametrize("what", ["expanded do", "misaligned do", "bfloat16 dht", "strided dht"])
def test_backward_in_python_steps_behind_a_native_forward(cuda, monkeypatch, op, form, what):
    """the forward was native (no plan of a dense call, no dimensions kept); a gradient that has to be converted sends the backward
    to the Python steps, which give the bits of a call that took them throughout"""
    mod, hf = _mods()[op], form == "head_first"
    B, T, N = {"dense": (2, 200, 2), "head_first": (2, 200, 2), "packed": (1, 500, 4), "cut": (1, 4000, 1)}[form]
    cu = torch.tensor([0, 70, 70, 71, 500], dtype=torch.int32, device=cuda) if form == "packed" else None
    x = _inputs(op, B, T, 2, 64, 64, torch.bfloat16, hf, False, torch.float32, cuda)
    h0, dht = torch.randn(N, 2, 64, 64, device=cuda), torch.randn(N, 2, 64, 64, device=cuda)
    do = torch.randn_like(x["v"])
    if what == "expanded do":
        do = torch.ones((), device=cuda, dtype=torch.bfloat16).expand(x["v"].shape)
    elif what == "misaligned do":
        wide = torch.zeros(*do.shape[:3], 65, device=cuda, dtype=torch.bfloat16)
        wide[..., 1:] = do
        do = wide[..., 1:]
    else:
        dht = dht.bfloat16() if what == "bfloat16 dht" else dht.mT.contiguous().mT
    args = [x["q"], x["k"], x["v"], x["g"]] + ([x["beta"]] if op == 2 else []) + [None, h0, True, cu, hf]
    c = _call(op, True)
    ref = [*c.forward(*args), *c.backward(do, dht)]
    c = _call(op, False)
    with monkeypatch.context() as m:
        m.setattr(mod, "base_args", None)
        got = list(c.forward(*args))
    assert c.dims is None and (c.plan is None) == (cu is None) and (op != 2 or (c.saved[-1] is not None) == (form == "cut"))
    answers, native = [], mod.native
    with monkeypatch.context() as m:
        m.setattr(mod, "native", lambda *a: answers.append(native(*a)) or answers[-1])
        got += c.backward(do, dht)
    assert answers == [None]
    assert all((a is None and b is None) or torch.equal(a, b) for a, b in zip(ref, got))


def _wide_v(cuda, T):
    import linear_moe_amd as L
    x = _inputs(2, 2, T, 3, 128, 256, torch.bfloat16, False, True, torch.bfloat16, cuda)
    x["k"] = _inputs(2, 2, T, 3, 128, 64, torch.bfloat16, False, False, torch.float32, cuda)["k"]
    ls = [t.requires_grad_() for t in x.values()]
    o, ht = L.chunk_gated_delta_rule(*ls, output_final_state=True)
    return [o, ht], ls


def _mixer(cuda, T, D=64):
    import linear_moe_amd as L
    gen = torch.Generator(device=cuda).manual_seed(7)
    rn = lambda *s: torch.randn(*s, generator=gen, device=cuda)
    ls = [rn(T, 2, 3 * 3 * D).bfloat16(), -rn(2, T, 3).abs(), torch.sigmoid(rn(2, T, 3)).bfloat16()]
    ls = [t.requires_grad_() for t in ls]
    return [L.gdn_mixer_core(*ls, 3, D)], ls


def _with_den(cuda, T):
    from linear_moe_amd.simple_gla import chunk_simple_gla_with_den
    x = _inputs(0, 2, T, 3, 128, 64, torch.bfloat16, True, True, torch.float32, cuda)
    ls = [x["q"].abs(), x["k"].abs(), x["v"], torch.randn(2, 3, 128, 64, device=cuda, generator=torch.Generator(device=cuda).manual_seed(9))]
    ls = [t.detach().requires_grad_() for t in ls]
    o, den, ht = chunk_simple_gla_with_den(*ls[:3], None, ls[3], True)
    return [o, den, ht], ls


@pytest.mark.parametrize("form", [_wide_v, _mixer, lambda cuda, T: _mixer(cuda, T, 128), _with_den],
                         ids=["V=256", "mixer D=64", "mixer D=128", "den"])
@pytest.mark.parametrize("T", [1, 190, 4100])
def test_other_forms_same_bits(cuda, monkeypatch, form, T):
    """V = 256; silu(v), gradients written into the blocks of the projection's and the raw q, k of the mixer; den and its gradient"""
    out = []
    for python in (True, False):
        with monkeypatch.context() as m:
            for mod in _mods():
                m.setattr(mod, "native", lambda *a: None) if python else m.setattr(mod, "base_args", None)
            outs, ls = form(cuda, T)
            gen = torch.Generator(device=cuda).manual_seed(11)
            douts = [torch.randn(o.shape, generator=gen, device=cuda).to(o.dtype) for o in outs]
            out.append([*outs, *torch.autograd.grad(outs, ls, douts)])
    for a, b in zip(*out):
        assert a.dtype == b.dtype and a.shape == b.shape and torch.equal(a, b) and b.abs().max() > 0


# ---- the neighbours of the ops ----
def _neighbour_calls(cuda, B, T, H, D, dt):
    """name -> (function of the leaves, leaves): the steps of a mixer around the op and of a mixture of memories"""
    import linear_moe_amd as L
    gen = torch.Generator(device=cuda).manual_seed(11)
    rn = lambda *s: torch.randn(*s, generator=gen, device=cuda)
    sel = torch.randint(0, 4, (B, T, 2), generator=gen, device=cuda)
    plan = L.mom_plan(sel, 4)
    calls = {"gates": (L.gdn_gates, (rn(B, T, H).to(dt), rn(B, T, H).to(dt), rn(H), rn(H))),
             "swish": (L.swish_gate_relayout, (rn(B, T, H, D).to(dt), rn(T, B, H * D).to(dt))),
             "pack": (lambda x: L.mom_pack(x, plan), (rn(B, T, H * D).to(dt),)),
             "combine": (lambda y, w: L.mom_combine(y, plan, w), (rn(2 * B * T, H, D).to(dt), rn(B, T, 2).to(dt)))}
    if dt == torch.bfloat16:
        calls["mixer"] = (lambda x, g, beta: L.gdn_mixer_core(x, g, beta, H, D), (rn(T, B, H * 3 * D).to(dt), -rn(B, T, H).abs(), torch.sigmoid(rn(B, T, H)).to(dt)))
        calls["mixer, no gate of its own type"] = (calls["mixer"][0], (rn(T, B, H, 3 * D).to(dt), -rn(B, T, H).abs().to(dt), torch.sigmoid(rn(B, T, H))))
    return calls


def _no_native(m):
    import linear_moe_amd._host as host
    import linear_moe_amd.gates as gates
    import linear_moe_amd.layer_io as layer_io
    import linear_moe_amd.mom as mom
    for mod in (host, gates, layer_io, mom):
        m.setattr(mod, "native_call", lambda *a: None)


def _outputs(fn, leaves):
    leaves = [x.detach().requires_grad_(True) for x in leaves]
    outs = fn(*leaves)
    outs = outs if isinstance(outs, tuple) else (outs,)
    douts = [torch.randn(o.shape, generator=torch.Generator(device=o.device).manual_seed(3), device=o.device).to(o.dtype) for o in outs]
    return [o.detach() for o in outs] + list(torch.autograd.grad(outs, leaves, douts))


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("B,T,H,D", [(1, 1, 1, 64), (2, 130, 3, 128)])
def test_neighbours_same_bits(cuda, monkeypatch, B, T, H, D, dt):
    for name, (fn, leaves) in _neighbour_calls(cuda, B, T, H, D, dt).items():
        with monkeypatch.context() as m:
            _no_native(m)
            ref = _outputs(fn, leaves)
        with monkeypatch.context() as m:                   # (the Python steps would ask for it)
            import linear_moe_amd._lib as _lib
            m.setattr(_lib, "load", None)
            got = _outputs(fn, leaves)
        for a, b in zip(ref, got):
            assert a.dtype == b.dtype and a.shape == b.shape and a.stride() == b.stride() and torch.equal(a, b), name


def test_neighbours_in_other_forms(cuda, monkeypatch):
    """Strided leaves, wider parameters: what the native path hands back runs as it did."""
    B, T, H, D = 2, 70, 2, 64
    for name, (fn, leaves) in _neighbour_calls(cuda, B, T, H, D, torch.bfloat16).items():
        other = [x.transpose(-1, -2).contiguous().transpose(-1, -2) if x.dim() > 1 else x.double() for x in leaves]
        with monkeypatch.context() as m:
            _no_native(m)
            ref = _outputs(fn, other)
        for a, b in zip(ref, _outputs(fn, other)):
            assert a.dtype == b.dtype and torch.equal(a, b), name


@pytest.mark.parametrize("is64", [True, False])
@pytest.mark.parametrize("B,S,topk,E,capacity", [(1, 1, 1, 1, None), (2, 700, 2, 5, None), (3, 300, 2, 4, 0.4)])
def test_routing_tables_same_bits(cuda, monkeypatch, is64, B, S, topk, E, capacity):
    import linear_moe_amd as L
    from linear_moe_amd._host import SeqPlan
    sel = torch.randint(0, E, (B, S, topk), generator=torch.Generator().manual_seed(4)).to(torch.int64 if is64 else torch.int32).to(cuda)
    with monkeypatch.context() as m:
        _no_native(m)
        ref = L.mom_plan(sel, E, capacity)
        ref_seq = SeqPlan(1, max(ref.T_total, 1), ref.cu_seqlens, sel.device)
    got = L.mom_plan(sel, E, capacity)
    seq = SeqPlan(1, max(ref.T_total, 1), got.cu_seqlens, sel.device)
    assert (got.T_total, got.B, got.S, got.topk) == (ref.T_total, B, S, topk)
    for n in ("src_token", "src_choice", "row_of", "cu_seqlens", "max_len_dev", "mem_offsets_dev"):
        a, b = getattr(ref, n), getattr(got, n)
        assert a.dtype == b.dtype and a.shape == b.shape and torch.equal(a, b), n
    nt = int(ref_seq.nt_dev)
    assert (seq.N, seq.NT) == (ref_seq.N, ref_seq.NT) and torch.equal(seq.chunk_map[:nt], ref_seq.chunk_map[:nt])
    for n in ("cu", "seq_chunk0", "nt_dev", "seq_order"):
        a, b = getattr(ref_seq, n), getattr(seq, n)
        assert (a is None) == (b is None) and (a is None or torch.equal(a, b)), n


@pytest.mark.parametrize("name", ["gates", "swish", "combine", "mixer"])
def test_neighbours_refuse_or_convert_what_hooks_hand_back(cuda, name):
    """A saved tensor that comes back in another type, with other strides or at another place in memory is read as what was saved, or
    refused; one of another shape or device is refused."""
    fn, leaves = _neighbour_calls(cuda, 2, 70, 2, 64, torch.bfloat16)[name]
    ref, saved = _outputs(fn, leaves), []

    def through(change):
        count = [0]

        def pack(t):
            count[0] += 1
            return count[0] - 1, t
        with torch.autograd.graph.saved_tensors_hooks(pack, lambda p: change(*p)):
            return _outputs(fn, leaves)

    through(lambda i, t: saved.append(t) or t)
    same = [lambda x: x.clone(), lambda x: x.float() if x.dtype == torch.bfloat16 else x.double(),
            lambda x: x.mT.contiguous().mT if x.dim() > 1 else x.double(), _misaligned]
    other = [lambda x: x[:1] if x.shape[0] > 1 else x[:, :1], lambda x: x[..., :-8] if x.shape[-1] > 8 else x[..., :-1], lambda x: x.cpu()]
    converted = 0
    for i, f in itertools.product(range(len(saved)), same):
        try:
            got = through(lambda j, x: f(x) if i == j else x)
        except (RuntimeError, ValueError):
            continue
        converted += 1
        assert all(torch.equal(a, b) for a, b in zip(ref, got)), i
    assert converted >= (4 if name != "mixer" else 3) * len(saved)         # (q, k, v of another type than the call are refused)
    for i, f in itertools.product(range(len(saved)), other):
        with pytest.raises((RuntimeError, ValueError)):
            through(lambda j, x: f(x) if i == j else x)


def test_calls_without_a_node_are_still_functions_of_autograd_for_transforms(cuda):
    """Forward-only calls run without a node of the graph; what autograd refused it still refuses."""
    import linear_moe_amd as L
    from torch.autograd import forward_ad as fw
    q, k, v = (torch.randn(1, 2, 70, 64, device=cuda).bfloat16() for _ in range(3))
    ref = L.chunk_linear_attn(q, k, v, normalize=False)[0]
    assert ref.grad_fn is None
    with torch.no_grad():
        o = L.chunk_linear_attn(q.requires_grad_(), k, v, normalize=False)[0]
    assert torch.equal(o, ref) and not o.requires_grad
    o = L.chunk_linear_attn(q, k, v, normalize=False)[0]
    assert o.requires_grad and torch.equal(o, ref)
    q = q.detach()
    with fw.dual_level():
        with pytest.raises((RuntimeError, NotImplementedError)):
            L.chunk_simple_gla(fw.make_dual(q, q), k, v)
    with pytest.raises(RuntimeError):
        torch.func.vmap(lambda x: L.chunk_simple_gla(x, k, v)[0])(q.unsqueeze(0))
    with pytest.raises(RuntimeError):                      # (nothing of the call is mapped over)
        torch.func.vmap(lambda x: L.chunk_simple_gla(q, k, v)[0] + x)(torch.zeros(2, device=cuda))


@pytest.mark.filterwarnings("ignore")
@pytest.mark.parametrize("op", ["simple_gla", "linear_attn", "linear_attn normalized", "gla", "gated_delta_rule"])
def test_a_trace_replays_the_op_on_other_inputs(cuda, op):
    import linear_moe_amd as L
    f = {"simple_gla": lambda q, k, v: L.chunk_simple_gla(q, k, v, output_final_state=True),
         "linear_attn": lambda q, k, v: L.chunk_linear_attn(q, k, v, normalize=False, output_final_state=True),
         "linear_attn normalized": lambda q, k, v: L.chunk_linear_attn(q.abs(), k.abs(), v, output_final_state=True),
         "gla": lambda q, k, v: L.chunk_gla(q, k, v, -k.abs(), output_final_state=True),
         "gated_delta_rule": lambda q, k, v: L.chunk_gated_delta_rule(q, k, v, -q[..., 0].abs(), torch.sigmoid(k[..., 0]),
                                                                      output_final_state=True)}[op]
    gen = torch.Generator(device=cuda).manual_seed(2)
    x, y = ([0.1 * torch.randn(1, 130, 2, 64, device=cuda, generator=gen).bfloat16() for _ in range(3)] for _ in range(2))
    with torch.no_grad():
        traced = torch.jit.trace(f, x, check_trace=False)
        for a, b in zip(traced(*y), f(*y)):
            assert torch.equal(a, b)
