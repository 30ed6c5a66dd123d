"""``chunk_gated_delta_rule`` on MI355X.

  S~_t = e^{g_t} S_{t-1};  S_t = S~_t + k_t^T beta_t (v_t - k_t S~_t);  o_t = scale q_t S_t

Keeps flash-linear-attention's call signature as the reference uses it at
``linear_moe/sequence_modeling/gated_deltanet/gated_deltanet.py:112``:
``chunk_gated_delta_rule(q, k, v, g, beta, head_first=False)`` with q, k, v ``[B,T,H,D]`` and
g, beta ``[B,T,H]``.
"""
from __future__ import annotations

import ctypes as C
from typing import Optional, Tuple

import torch

from . import _lib
from .l2norm import l2_norm
from ._host import (HEAD_DIMS, WIDE_V, seq_plan, _aligned, _check_inputs, _desc, _state_check, base_args, by_head_dim_blocks,
                    came_back, inputs_came_back, native, no_node, no_tokens, ptr, stash, stream_ptr, unstash)


def _scalar_dt(x: torch.Tensor) -> int:
    return _lib.LMOE_F32 if x.dtype == torch.float32 else _lib.LMOE_BF16


class GDNCall:
    """One call of the op: owns the argument blocks and every buffer the kernels touch.
    The autograd function and the benchmark harness (per-kernel timing through
    ``lmoe_launch_stage``) both drive the kernels through this object."""

    OP = 2  # LMOE_OP_GATED_DELTA_RULE

    def __init__(self, keep: bool = False):
        # keep=True (benchmark harness) also pins outputs and gradients so that the argument
        # blocks stay valid for lmoe_launch_stage; the autograd path must not (reference cycle)
        self.keep = keep

    def forward(self, q, k, v, g, beta, scale, initial_state, output_final_state, cu_seqlens, head_first, save=True,
                v_act=False):
        """save=False: a forward-only call (nothing requires a gradient): what only the backward reads (the
        per-chunk states, v_new, Tinv) is neither allocated nor written.
        v_act: v is the argument of the SiLU in front of the op (bfloat16 only): the kernels apply it where they
        read v, and ``backward`` returns the gradient with respect to that argument."""
        ctx = self
        lib = _lib.load()
        plan = dims = None
        if cu_seqlens is not None:
            dims = _check_inputs(q, k, v, head_first, cu_seqlens, wide_v=True)
            B, T = dims[:2]
            plan = seq_plan(B, T, cu_seqlens, q.device)
        if not self.keep and q.dtype != torch.float32:           # (4-byte elements need w and u as well)
            tables = None if plan is None else plan.tables
            r = native("forward", "chunk_gated_delta_rule forward", self.OP, q, k, v, g, beta, initial_state, tables,
                       scale, output_final_state, head_first, save, 0, 0.0, v_act)
            if r is not None:
                o, ht, *kept = r
                ctx.saved = (q, k, v, g, beta, initial_state, *kept)
                ctx.plan, ctx.dims, ctx.head_first, ctx.scale = plan, None, head_first, scale
                ctx.has_h0, ctx.v_act, self.seg_ws = initial_state is not None, bool(v_act), None
                return o, ht
        if dims is None:
            dims = _check_inputs(q, k, v, head_first, cu_seqlens, wide_v=True)
        B, T, H, K, V = dims
        q, k, v = _aligned(q), _aligned(k), _aligned(v)
        if plan is None:
            plan = seq_plan(B, T, None, q.device)
        want = (B, H, T) if head_first else (B, T, H)
        if beta is None or tuple(beta.shape) != want:
            raise ValueError(f"beta must have shape {want}")
        if g is not None and tuple(g.shape) != want:
            raise ValueError(f"g must have shape {want}, got {tuple(g.shape)}")
        if g is not None and g.dtype not in (torch.float32, torch.bfloat16):
            g = g.float()
        if beta.dtype not in (torch.float32, torch.bfloat16):
            beta = beta.float()
        h0 = _state_check(initial_state, plan.N, H, K, V, "initial_state")
        a = base_args(q, k, v, head_first, scale, plan, dims)
        a.gate = _lib.GATE_NONE if g is None else _lib.GATE_SCALAR
        if g is not None:
            a.g, a.g_dtype = _desc(g, head_first), _scalar_dt(g)
        a.beta, a.beta_dtype = _desc(beta, head_first), _scalar_dt(beta)
        a.h0 = ptr(h0)
        dev, dt = q.device, q.dtype
        # (v_act: v is a block of a wider tensor; o is a tensor of its own)
        o = torch.empty(v.shape, dtype=dt, device=dev) if v_act else torch.empty_like(v)
        ht = torch.empty(plan.N, H, K, V, dtype=torch.float32, device=dev) if output_final_state else None
        hs = torch.empty(max(plan.NT, 1), H, K, V, dtype=dt, device=dev) if save else None
        # always: the backward reads it, and the forward state pass forms w from it (8 KB per chunk and head)
        tinv = torch.empty(max(plan.NT, 1), H, 64, 64, dtype=dt, device=dev)
        # P: the bf16 forward pass forms it on the chip and stores it only for the backward
        pmat = torch.empty(max(plan.NT, 1), H, 64, 64, dtype=dt, device=dev) if (save or dt == torch.float32) else None
        gcum = torch.empty(max(plan.NT, 1), H, 5, 64, dtype=torch.float32, device=dev)
        # w, u: the bf16 state passes form them on the chip from tinv; only the fp32 forward pass reads them
        w = torch.empty(B, T, H, K, dtype=dt, device=dev) if dt == torch.float32 else None
        u = torch.empty(B, T, H, V, dtype=dt, device=dev) if dt == torch.float32 else None
        # library-side layout [chunk, head, 32-column slice, token in chunk, column] (see include/lmoe.h)
        vnew = torch.empty(max(plan.NT, 1), H, V // 32, 64, 32, dtype=dt, device=dev) if save else None
        a.o, a.ht, a.hs, a.tinv = _desc(o, head_first), ptr(ht), ptr(hs), ptr(tinv)
        a.pmat, a.gcum = ptr(pmat), gcum.data_ptr()
        a.w, a.u = _desc(w, False), _desc(u, False)
        a.vnew.ptr = ptr(vnew)
        if v_act and dt != torch.bfloat16:
            raise ValueError("v_act exists for bfloat16")
        a.v_act = int(bool(v_act))
        ctx.v_act = bool(v_act)
        seg_p = self._cut(lib, a, dev, save)
        _lib.check(lib.lmoe_chunk_gated_delta_rule_fwd(C.byref(a), stream_ptr()), "chunk_gated_delta_rule forward")
        ctx.saved = (q, k, v, g, beta, h0, hs, tinv, pmat, gcum, vnew, seg_p)
        ctx.fwd_args, ctx.fwd_keep = a, ((o, ht, w, u, seg_p, self.seg_ws) if self.keep else None)
        ctx.plan, ctx.dims, ctx.head_first, ctx.scale = plan, dims, head_first, scale
        ctx.has_h0 = initial_state is not None
        self.seg_ws = None
        return o, ht

    def came_from_native(self, q, k, v, g, beta, scale, kept):
        """What the native path keeps of a dense call on the v block of a projection (``lmoe_native.cpp``, mixer_forward)."""
        self.saved = (q, k, v, g, beta, None, *kept)
        self.plan, self.dims, self.head_first, self.scale = None, None, False, scale
        self.has_h0, self.v_act, self.seg_ws = False, True, None

    def backward_args(self, do, dht):
        """The arguments of the native backward, but for the last (``extra``)."""
        q, k, v, g, beta, h0, *kept = self.saved
        return (self.OP, q, k, v, g, beta, h0, self.plan and self.plan.tables, self.scale, do, dht, self.head_first, tuple(kept))

    def _cut(self, lib, a, dev, save=False, seg_p=None):
        """The buffers of a call whose sequences are cut along T (``lmoe_args.seg_ws``; ``seg_p``, which a call that
        saves hands to its backward), or none."""
        self.seg_ws = None
        n = lib.lmoe_split_floats(C.byref(a), self.OP, 1)
        if n <= 0:
            return None
        n_p = lib.lmoe_split_floats(C.byref(a), self.OP, 0)
        if save:
            seg_p = torch.empty(n_p, dtype=torch.float32, device=dev)
        elif seg_p is not None:
            seg_p = came_back(seg_p, (n_p,), torch.float32, dev, "seg_p")
        self.seg_ws = torch.empty(n, dtype=torch.float32, device=dev)
        a.seg_p, a.seg_ws = ptr(seg_p), self.seg_ws.data_ptr()
        return seg_p

    def backward(self, do, dht, dv_out=None, dq_out=None, dk_out=None, qk_raw=None, qk_eps=1e-6):
        """dv_out, dq_out, dk_out: where the gradients go (tensors of the shapes of v, q, k, any strides the kernels
        take: e.g. the blocks of the gradient of a fused projection); default: new tensors.  qk_raw = (q_raw, k_raw)
        (bfloat16): q and k of the forward were l2norm(silu(.)) of these rows (eps qk_eps inside the root), and dq,
        dk are returned with respect to them."""
        ctx = self
        lib = _lib.load()
        q, k, v, g, beta, h0, hs, tinv, pmat, gcum, vnew, seg_p = ctx.saved
        head_first = ctx.head_first
        dims = None
        if not self.keep:
            raw, what = (None, None) if qk_raw is None else qk_raw, "chunk_gated_delta_rule backward"
            args = (*self.backward_args(do, dht), (ctx.v_act, dq_out, dk_out, dv_out, *raw, float(qk_eps)))
            if q.dtype != torch.float32:
                r = native("backward", what, *args)
                if r is not None:
                    dq, dk, dv, dg, dbeta, dh0 = r
                    return dq, dk, dv, (dg if dg is None or dg.dtype == g.dtype else dg.to(g.dtype)), dbeta, dh0
            else:
                dims = native("intact", what, *args)
        intact = dims is not None
        if not intact:
            q, k, v, do, dims = inputs_came_back(q, k, v, do, head_first, wide_v=True)
        B, T, H, K, V = dims
        plan = ctx.plan or seq_plan(B, T, None, q.device)
        dev, dt = q.device, q.dtype
        if not intact:
            tok, nt = ((B, H, T) if head_first else (B, T, H)), max(plan.NT, 1)
            g = None if g is None else came_back(g, tok, None, dev, "g")
            beta = came_back(beta, tok, None, dev, "beta")
            if ctx.has_h0:
                h0 = came_back(h0, (plan.N, H, K, V), torch.float32, dev, "initial_state")
            hs, tinv = came_back(hs, (nt, H, K, V), dt, dev, "hs"), came_back(tinv, (nt, H, 64, 64), dt, dev, "tinv")
            pmat = came_back(pmat, (nt, H, 64, 64), dt, dev, "pmat")
            gcum = came_back(gcum, (nt, H, 5, 64), torch.float32, dev, "gcum")
            vnew = came_back(vnew, (nt, H, V // 32, 64, 32), dt, dev, "vnew")
        a = base_args(q, k, v, head_first, ctx.scale, plan, dims)
        a.gate = _lib.GATE_NONE if g is None else _lib.GATE_SCALAR
        if g is not None:
            a.g, a.g_dtype = _desc(g, head_first), _scalar_dt(g)
        a.beta, a.beta_dtype = _desc(beta, head_first), _scalar_dt(beta)
        a.h0, a.hs, a.tinv, a.pmat = ptr(h0), hs.data_ptr(), tinv.data_ptr(), pmat.data_ptr()
        a.gcum = gcum.data_ptr()
        a.vnew.ptr = vnew.data_ptr()
        a.d_o = _desc(do, head_first)
        dht = None if dht is None else dht.float().contiguous()
        a.dht = ptr(dht)
        dq = torch.empty_like(q) if dq_out is None else dq_out
        dk = torch.empty_like(k) if dk_out is None else dk_out
        dv = torch.empty_like(v) if dv_out is None else dv_out
        for n, t, like in (("dq_out", dq, q), ("dk_out", dk, k), ("dv_out", dv, v)):
            if t.shape != like.shape or t.dtype != dt or _aligned(t) is not t:
                raise ValueError(f"{n} must have the shape and dtype of its input, 16-byte aligned rows, a contiguous "
                                 "last dimension")
        a.dq, a.dk, a.dv = _desc(dq, head_first), _desc(dk, head_first), _desc(dv, head_first)
        a.v_act = int(ctx.v_act)
        if qk_raw is not None:
            q_raw, k_raw = qk_raw
            if dt != torch.bfloat16:
                raise ValueError("qk_raw exists for bfloat16")
            for t, like in ((q_raw, q), (k_raw, k)):
                if t.shape != like.shape or t.dtype != dt or _aligned(t) is not t:
                    raise ValueError("qk_raw: the shapes and dtype of q, k, 16-byte aligned rows, a contiguous last dimension")
            a.q_raw, a.k_raw, a.qk_eps = _desc(q_raw, head_first), _desc(k_raw, head_first), float(qk_eps)
        dg = torch.empty(beta.shape, dtype=torch.float32, device=dev)
        # (rounded to the type of beta by the kernel that forms it: a conversion pass cost a launch)
        dbeta = torch.empty(beta.shape, dtype=torch.bfloat16 if beta.dtype == torch.bfloat16 else torch.float32, device=dev)
        a.dbeta_bf16 = int(dbeta.dtype == torch.bfloat16)
        a.dg, a.dbeta = _desc(dg, head_first), _desc(dbeta, head_first)
        dh0 = torch.empty_like(h0) if ctx.has_h0 else None
        a.dh0 = ptr(dh0)
        dhs = torch.empty_like(hs)
        dvnew = torch.empty_like(vnew)
        a.dhs = dhs.data_ptr()
        a.dvnew.ptr = dvnew.data_ptr()
        if seg_p is not None:
            self._cut(lib, a, dev, seg_p=seg_p)
        _lib.check(lib.lmoe_chunk_gated_delta_rule_bwd(C.byref(a), stream_ptr()), "chunk_gated_delta_rule backward")
        ctx.bwd_args = a
        ctx.bwd_keep = (do, dht, dq, dk, dv, dg, dbeta, dh0, dhs, dvnew, qk_raw, self.seg_ws) if self.keep else None
        self.seg_ws = None
        dg = None if g is None else dg.to(g.dtype)
        return dq, dk, dv, dg, dbeta.to(beta.dtype), dh0


class _ChunkGatedDeltaRule(torch.autograd.Function):
    @staticmethod
    def forward(ctx, q, k, v, g, beta, scale, initial_state, output_final_state, cu_seqlens, head_first):
        call = GDNCall()
        o, ht = call.forward(q, k, v, g, beta, scale, initial_state, output_final_state, cu_seqlens, head_first,
                             save=any(ctx.needs_input_grad))
        ctx.call = call
        stash(ctx, call)
        return o, ht

    @staticmethod
    def backward(ctx, do, dht):
        unstash(ctx, ctx.call)
        try:
            dq, dk, dv, dg, dbeta, dh0 = ctx.call.backward(do, dht)
        finally:
            ctx.call.saved = None
        return dq, dk, dv, dg, dbeta, None, dh0, None, None, None


def chunk_gated_delta_rule(
    q: torch.Tensor,
    k: torch.Tensor,
    v: torch.Tensor,
    g: torch.Tensor,
    beta: torch.Tensor,
    scale: Optional[float] = None,
    initial_state: Optional[torch.Tensor] = None,
    output_final_state: bool = False,
    cu_seqlens: Optional[torch.Tensor] = None,
    head_first: bool = False,
    use_qk_l2norm_in_kernel: bool = False,
) -> Tuple[torch.Tensor, Optional[torch.Tensor]]:
    """q, k: ``[B,T,H,K]``, v: ``[B,T,H,V]``, g (log-space decay) and beta: ``[B,T,H]``
    (``[B,H,T,*]`` with ``head_first=True``).  Returns ``(o, final_state)``.  K, V of 64 or 128 and K = 128 with
    V = 256 (``expand_v = 2``) run as they are; a smaller K is zero-padded, any other V is cut into blocks of
    256 (K > 64) / 128 / 64 columns (``_host.by_head_dim_blocks``).

    ``use_qk_l2norm_in_kernel=True`` gives the results of fla's flag, not its fusion: q and k go through the ``l2_norm``
    kernel (one read and one write of each, forward and backward) in front of the op, the op's kernels do not
    normalise.  A caller that holds the fused projection of the mixer gets q^, k^ and silu(v) in one pass from
    ``layer_io.gdn_qkv_prologue`` instead."""
    if use_qk_l2norm_in_kernel:
        q = l2_norm(q)
        k = l2_norm(k)
    if q.dim() == 4 and v.dim() == 4 and (q.shape[-1] not in HEAD_DIMS or v.shape[-1] not in HEAD_DIMS) \
            and (q.shape[-1], v.shape[-1]) != WIDE_V:
        # e.g. K = 96 (padded to 128), V = 320 (a block of 256 and one of 64 columns)
        sc = q.shape[-1] ** -0.5 if scale is None else scale          # of the whole key, not of the padded one
        return by_head_dim_blocks(
            lambda q_, k_, v_, _g, h0: chunk_gated_delta_rule(q_, k_, v_, g, beta, sc, h0, output_final_state,
                                                              cu_seqlens, head_first),
            q, k, v, None, initial_state, output_final_state, False, "chunk_gated_delta_rule", wide_v=True)
    r = no_tokens(q, k, v, head_first, cu_seqlens, initial_state, output_final_state, wide_v=True)
    if r is not None:
        return r
    if no_node(q, k, v, g, beta, initial_state):
        return GDNCall().forward(q, k, v, g, beta, scale, initial_state, output_final_state, cu_seqlens, head_first, save=False)
    return _ChunkGatedDeltaRule.apply(q, k, v, g, beta, scale, initial_state, output_final_state, cu_seqlens,
                                      head_first)
