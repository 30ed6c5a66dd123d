"""What is timed when the speed of this package is asked for: the calls its users make, over the range they make
them in.  ``listed()`` are fixed cases, ``draw(rng)`` gives more of the same ranges, ``prepare`` makes what a program
holds before the call, ``run`` is one pass through the public entry points, ``work`` what that pass cannot do
without and ``tolerance`` how far another correct implementation at the same precision may be off."""
import math

import torch
import torch.nn.functional as F

import linear_moe_amd as L

CHUNK = 64


def listed():
    return [
        # a unit-test sized layer in float32 (the plumbing configuration of the reference's operators): launch-bound
        dict(name="linear_attn_fp32", kind="linear_attn_fp32", B=1, T=512, H=4, D=64),
        # one generated token of one sequence: nothing but latency
        dict(name="gdn_decode_1", kind="decode", op="gdn", B=1, H=16, D=128),
        # one generated token of a full serving batch: the states are read and written once
        dict(name="gla_decode_256", kind="decode", op="gla", B=256, H=16, D=128),
        # one prompt of odd length read in before generation: a single sequence on the whole card
        dict(name="gdn_prefill_1", kind="gdn_prefill", N=1, T=3001, H=16, D=128),
        # a batch of prompts with the retention / lightning-attention decay, final state kept for generation
        dict(name="retention_prefill", kind="retention_prefill", B=4, T=4096, H=16, D=128),
        # training step of basic linear attention with its normaliser (on by default), a length that is no multiple
        # of the chunk
        dict(name="linear_attn_train", kind="linear_attn_train", B=4, T=1000, H=16, K=128, V=128, normalize=True),
        # training step of gated linear attention, key heads half as wide as value heads
        dict(name="gla_train", kind="gla_train", B=8, T=2048, H=16, K=64, V=128),
        # training step of the gated delta rule, the headline of this package
        dict(name="gdn_train", kind="gdn_train", B=4, T=8192, H=16, D=128),
        # the same operator on one long sequence per card
        dict(name="gdn_train_long", kind="gdn_train", B=1, T=16384, H=16, D=128),
        # packed documents of log-normal lengths with states handed in and out (the largest case)
        dict(name="gdn_train_packed", kind="gdn_train_packed", N=16, T=65536, H=32, D=128),
        # the whole token mixer between its projections: gates, SiLU, L2 norms, operator, output gate
        dict(name="gdn_layer_train", kind="gdn_layer_train", B=2, T=2048, H=16, D=128),
        # mixture of memories: routing tables, packing, one operator call over all memories, combination
        dict(name="mom_train", kind="mom_train", B=2, T=2048, H=16, D=128, memories=4, topk=2),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _batch(rng, tokens, t_lo, t_hi, b_hi, heads):
    """B, T, H spread over their ranges with at most ``tokens`` (row, token, head) triples in all."""
    while True:
        c = dict(B=_log_int(rng, 1, b_hi), T=_log_int(rng, t_lo, t_hi), H=rng.choice(heads))
        if c["B"] * c["T"] * c["H"] <= tokens:
            return c


def draw(rng):
    kind = rng.choice(["linear_attn_fp32", "decode", "gdn_prefill", "retention_prefill", "linear_attn_train", "gla_train",
                       "gdn_train", "gdn_train_packed", "gdn_layer_train", "mom_train"])
    heads, dim = (4, 8, 16, 32), rng.choice((64, 128))
    if kind == "linear_attn_fp32":
        return dict(kind=kind, D=dim, **_batch(rng, 1 << 15, 64, 2048, 4, (2, 4, 8, 16)))
    if kind == "decode":
        return dict(kind=kind, op=rng.choice(("gdn", "gla", "simple_gla")), B=_log_int(rng, 1, 256), H=rng.choice(heads), D=dim)
    if kind == "gdn_prefill":
        while True:
            c = dict(kind=kind, N=_log_int(rng, 1, 16), T=_log_int(rng, 64, 32768), H=rng.choice(heads), D=dim)
            if c["T"] >= 8 * c["N"] and c["T"] * c["H"] <= 1 << 19:
                return c
    if kind == "retention_prefill":
        return dict(kind=kind, D=dim, **_batch(rng, 1 << 19, 64, 8192, 8, heads))
    if kind == "linear_attn_train":
        return dict(kind=kind, K=dim, V=rng.choice((64, 128)), normalize=rng.random() < 0.5,
                    **_batch(rng, 1 << 19, 128, 8192, 8, heads))
    if kind == "gla_train":
        return dict(kind=kind, K=dim, V=rng.choice((64, 128)), **_batch(rng, 1 << 19, 128, 8192, 8, heads))
    if kind == "gdn_train":
        return dict(kind=kind, D=dim, **_batch(rng, 1 << 19, 128, 16384, 8, heads))
    if kind == "gdn_train_packed":
        return dict(kind=kind, N=_log_int(rng, 2, 64), T=_log_int(rng, 1024, 49152), H=rng.choice((8, 16, 32)), D=dim)
    if kind == "gdn_layer_train":
        return dict(kind=kind, D=dim, **_batch(rng, 1 << 19, 128, 8192, 4, heads))
    return dict(kind=kind, D=dim, memories=rng.choice((4, 8)), topk=rng.choice((1, 2)),
                **_batch(rng, 1 << 18, 128, 8192, 4, (8, 16)))


class _Inputs:
    """Inputs on the GPU, from the seed alone."""

    def __init__(self, seed):
        self.g = torch.Generator(device="cuda").manual_seed(seed)

    def normal(self, *shape, dtype=torch.bfloat16, std=1.0):
        return (torch.randn(*shape, generator=self.g, device="cuda") * std).to(dtype)

    def uniform(self, *shape):
        return torch.rand(*shape, generator=self.g, device="cuda")

    def unit(self, *shape):
        return F.normalize(torch.randn(*shape, generator=self.g, device="cuda"), dim=-1).bfloat16()

    def beta(self, *shape):
        return torch.sigmoid(self.normal(*shape, dtype=torch.float32)).bfloat16()

    def decay(self, *shape):
        """Log-decays of the gated delta rule: -exp(A_log) softplus(x + dt_bias), one A_log and dt_bias per head."""
        a = 1 + 15 * self.uniform(shape[-1])
        return -a * F.softplus(self.normal(*shape, dtype=torch.float32) + self.normal(shape[-1], dtype=torch.float32, std=0.1))

    def channel_decay(self, *shape):
        """Per-channel log-decays of gated linear attention: logsigmoid(x) / 16."""
        return (F.logsigmoid(self.normal(*shape, dtype=torch.float32)) / 16).bfloat16()

    def offsets(self, N, T):
        """cu_seqlens of N sequences of log-normal lengths (at least one token each) that add up to T."""
        w = torch.exp(torch.randn(N, generator=self.g, device="cuda")).double().cpu()
        lens = 1 + (w / w.sum() * (T - N)).floor().long()
        lens[lens.argmax()] += T - lens.sum()
        cu = torch.zeros(N + 1, dtype=torch.int32)
        cu[1:] = lens.cumsum(0)
        return cu.cuda()


def prepare(case, seed):
    x, kind, H = _Inputs(seed), case["kind"], case["H"]
    s = dict(case=case)
    if kind == "linear_attn_fp32":
        B, T, D = case["B"], case["T"], case["D"]
        s["q"], s["k"], s["v"] = (x.normal(B, H, T, D, dtype=torch.float32) for _ in range(3))
    elif kind == "decode":
        B, D = case["B"], case["D"]
        # the delta rule is called time-first and normalises q, k itself, the other two head-first
        shape = (B, 1, H, D) if case["op"] == "gdn" else (B, H, 1, D)
        s["q"], s["k"], s["v"] = (x.normal(*shape) for _ in range(3))
        s["h"] = x.normal(B, H, D, D, dtype=torch.float32, std=0.1)
        if case["op"] == "gdn":
            s["g"], s["beta"] = x.decay(B, 1, H), x.beta(B, 1, H)
        elif case["op"] == "gla":
            s["g"] = x.channel_decay(*shape)
        else:
            s["g"] = x.decay(B, 1, H).transpose(1, 2).contiguous() * 0.1
    elif kind == "gdn_prefill":
        T, D = case["T"], case["D"]
        s["q"], s["k"], s["v"] = x.unit(1, T, H, D), x.unit(1, T, H, D), x.normal(1, T, H, D)
        s["g"], s["beta"] = x.decay(1, T, H), x.beta(1, T, H)
        s["cu"] = x.offsets(case["N"], T) if case["N"] > 1 else None
    elif kind == "retention_prefill":
        s["q"], s["k"], s["v"] = (x.normal(case["B"], H, case["T"], case["D"]) for _ in range(3))
    elif kind == "linear_attn_train":
        B, T, K, V = case["B"], case["T"], case["K"], case["V"]
        # behind a positive feature map
        s["q"], s["k"] = (x.uniform(B, H, T, K).bfloat16() for _ in range(2))
        s["v"], s["do"] = x.normal(B, H, T, V), x.normal(B, H, T, V)
        s["leaves"] = ["q", "k", "v"]
    elif kind == "gla_train":
        B, T, K, V = case["B"], case["T"], case["K"], case["V"]
        s["q"], s["k"], s["v"] = x.normal(B, H, T, K), x.normal(B, H, T, K), x.normal(B, H, T, V)
        s["g"], s["do"] = x.channel_decay(B, H, T, K), x.normal(B, H, T, V)
        s["leaves"] = ["q", "k", "v", "g"]
    elif kind in ("gdn_train", "gdn_train_packed"):
        T, D, B = case["T"], case["D"], case.get("B", 1)
        s["q"], s["k"], s["v"] = x.unit(B, T, H, D), x.unit(B, T, H, D), x.normal(B, T, H, D)
        s["g"], s["beta"], s["do"] = x.decay(B, T, H), x.beta(B, T, H), x.normal(B, T, H, D)
        s["leaves"] = ["q", "k", "v", "g", "beta"]
        if kind == "gdn_train_packed":
            s["cu"] = x.offsets(case["N"], T)
            s["h"] = x.normal(case["N"], H, D, D, dtype=torch.float32, std=0.1)
            s["dh"] = x.normal(case["N"], H, D, D, dtype=torch.float32)
            s["leaves"].append("h")
    elif kind == "gdn_layer_train":
        B, T, D = case["B"], case["T"], case["D"]
        s["qkv"], s["gate"] = x.normal(T, B, H * 3 * D), x.normal(T, B, H * D)
        s["a"], s["b"] = x.normal(B, T, H), x.normal(B, T, H)
        s["A_log"], s["dt_bias"] = torch.log(1 + 15 * x.uniform(H)), x.normal(H, dtype=torch.float32, std=0.1)
        # (with a mean, as a loss has: the sums over all tokens that dA_log and ddt_bias are would be noise without one)
        s["dy"] = x.normal(T, B, H * D) + 0.25
        s["leaves"] = ["qkv", "gate", "a", "b", "A_log", "dt_bias"]
    else:
        B, T, D, E, topk = case["B"], case["T"], case["D"], case["memories"], case["topk"]
        w, s["routes"] = torch.topk(torch.softmax(x.normal(B, T, E, dtype=torch.float32), -1), topk, dim=-1)
        s["w"] = (w / w.sum(-1, keepdim=True)).bfloat16()
        s["hidden"], s["dpacked"] = x.normal(B, T, H * D), x.normal(B * T * topk, H * D)
        # the per-memory projections of the packed rows, left out here: their results
        n = B * T * topk
        s["q"], s["k"], s["v"] = x.unit(1, n, H, D), x.unit(1, n, H, D), x.normal(1, n, H, D)
        s["g"], s["beta"], s["dy"] = x.decay(1, n, H), x.beta(1, n, H), x.normal(B, T, H, D)
        s["leaves"] = ["hidden", "q", "k", "v", "g", "beta", "w"]
    for n in s.get("leaves", ()):
        s[n].requires_grad_(True)
    return s


def _grads(s, outs, douts):
    leaves = [s[n] for n in s["leaves"]]
    return [o.detach() for o in outs] + list(torch.autograd.grad(outs, leaves, douts))


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "linear_attn_fp32":
        with torch.no_grad():
            return L.chunk_linear_attn(s["q"], s["k"], s["v"], normalize=False)[0]
    if kind == "decode":
        with torch.no_grad():
            if case["op"] == "gdn":
                return L.fused_recurrent_gated_delta_rule(s["q"], s["k"], s["v"], s["g"], s["beta"], initial_state=s["h"],
                                                          output_final_state=True, use_qk_l2norm_in_kernel=True)
            op = L.fused_recurrent_gla if case["op"] == "gla" else L.fused_recurrent_simple_gla
            return op(s["q"], s["k"], s["v"], s["g"], initial_state=s["h"], output_final_state=True)
    if kind == "gdn_prefill":
        with torch.no_grad():
            return L.chunk_gated_delta_rule(s["q"], s["k"], s["v"], s["g"], s["beta"], output_final_state=True,
                                            cu_seqlens=s["cu"])
    if kind == "retention_prefill":
        with torch.no_grad():
            return L.chunk_retention(s["q"], s["k"], s["v"], output_final_state=True)
    if kind == "linear_attn_train":
        o, _ = L.chunk_linear_attn(s["q"], s["k"], s["v"], normalize=case["normalize"])
        return _grads(s, [o], [s["do"]])
    if kind == "gla_train":
        o, _ = L.chunk_gla(s["q"], s["k"], s["v"], s["g"])
        return _grads(s, [o], [s["do"]])
    if kind == "gdn_train":
        o, _ = L.chunk_gated_delta_rule(s["q"], s["k"], s["v"], s["g"], s["beta"], head_first=False)
        return _grads(s, [o], [s["do"]])
    if kind == "gdn_train_packed":
        o, h = L.chunk_gated_delta_rule(s["q"], s["k"], s["v"], s["g"], s["beta"], initial_state=s["h"],
                                        output_final_state=True, cu_seqlens=s["cu"])
        return _grads(s, [o, h], [s["do"], s["dh"]])
    if kind == "gdn_layer_train":
        g, beta = L.gdn_gates(s["a"], s["b"], s["A_log"], s["dt_bias"])
        o = L.gdn_mixer_core(s["qkv"], g, beta, case["H"], case["D"])
        return _grads(s, [L.swish_gate_relayout(o, s["gate"])], [s["dy"]])
    plan = L.mom_plan(s["routes"], case["memories"])
    packed = L.mom_pack(s["hidden"], plan)
    o, _ = L.chunk_gated_delta_rule(s["q"], s["k"], s["v"], s["g"], s["beta"], cu_seqlens=plan.cu_seqlens)
    return _grads(s, [packed, L.mom_combine(o[0], plan, s["w"])], [s["dpacked"], s["dy"]])


def _op_flops(kind, n, K, V):
    """Matrix products of n (token, head) pairs of the chunked forward."""
    if kind.startswith(("gdn", "mom")):
        return n * (6 * CHUNK * K + 4 * CHUNK * V + 6 * K * V + CHUNK * CHUNK * 2 / 3)
    return n * (2 * CHUNK * K + 2 * CHUNK * V + 4 * K * V)


def work(case):
    """Every input read once, every output written once."""
    kind, H = case["kind"], case["H"]
    K, V = case.get("K", case.get("D")), case.get("V", case.get("D"))
    n = case.get("B", 1) * case.get("T", 1) * H                             # (token, head) pairs
    if kind == "linear_attn_fp32":
        return dict(bytes=n * (2 * K + 2 * V) * 4, flops=_op_flops(kind, n, K, V))
    if kind == "decode":
        gate = {"gdn": 6, "gla": 2 * K, "simple_gla": 4}[case["op"]]
        return dict(bytes=n * (8 * K * V + (2 * K + 2 * V) * 2 + gate), flops=n * (8 if case["op"] == "gdn" else 5) * K * V)
    if kind == "gdn_prefill":
        return dict(bytes=n * ((2 * K + 2 * V) * 2 + 6) + case["N"] * H * K * V * 4, flops=_op_flops(kind, n, K, V))
    if kind == "retention_prefill":
        return dict(bytes=n * (2 * K + 2 * V) * 2 + case["B"] * H * K * V * 4, flops=_op_flops(kind, n, K, V))
    if kind == "linear_attn_train":
        return dict(bytes=n * (4 * K + 4 * V) * 2, flops=3 * _op_flops(kind, n, K, V))
    if kind == "gla_train":
        return dict(bytes=n * (6 * K + 4 * V) * 2, flops=3 * _op_flops(kind, n, K, V))
    if kind == "gdn_layer_train":                                           # qkv, gate, dy, y and three gradients; a, b
        return dict(bytes=n * (10 * K * 2 + 8), flops=3 * _op_flops(kind, n, K, V))
    if kind == "mom_train":
        m = n * case["topk"]
        return dict(bytes=n * 4 * K * 2 + m * ((2 * K + 6 * K) * 2 + 12), flops=3 * _op_flops(kind, m, K, V))
    states = 4 * case["N"] * H * K * V * 4 if kind == "gdn_train_packed" else 0
    return dict(bytes=n * ((4 * K + 4 * V) * 2 + 12) + states, flops=3 * _op_flops(kind, n, K, V))


# About four times the largest relative error, over the outputs of the listed and forty drawn cases, of the bfloat16
# path against the same pass in float32 (decode 3.0e-3, gdn_prefill 3.1e-3, retention_prefill 2.8e-3, linear_attn_train
# 5.5e-3, gla_train 4.8e-3, gdn_train 3.1e-3, gdn_train_packed 4.9e-3, gdn_layer_train 5.9e-3, mom_train 3.6e-3), and of
# the float32 path against the token recurrence in float64 (7.0e-7).
_REL = {"linear_attn_fp32": 3e-6, "decode": 1.2e-2, "gdn_prefill": 1.2e-2, "retention_prefill": 1.1e-2,
        "linear_attn_train": 2.2e-2, "gla_train": 1.9e-2, "gdn_train": 1.2e-2, "gdn_train_packed": 2.0e-2,
        "gdn_layer_train": 2.4e-2, "mom_train": 1.4e-2}


def tolerance(case):
    return {"rel": _REL[case["kind"]]}
