"""``chunk_gla`` on MI355X: S_t = diag(e^{g_t}) S_{t-1} + k_t^T v_t, o_t = scale q_t S_t with
per-channel log-decays g_t in R^K.

Keeps flash-linear-attention's call signature as the reference uses it at
``linear_moe/sequence_modeling/gla/gla.py:94`` (``chunk_gla(q, k, v, gk)``, ``[B,H,T,D]``) and
``linear_moe/sequence_modeling/hgrn2/hgrn2.py:76``.
"""
from __future__ import annotations

import ctypes as C
from typing import Optional, Tuple

import torch

from . import _lib
from ._host import (HEAD_DIMS, seq_plan, _aligned, _check_inputs, _desc, _state_check, base_args, by_head_dim_blocks,
                    came_back, cut_workspace, inputs_came_back, native, no_node, no_tokens, ptr, stash, stream_ptr, unstash)


class GLACall:
    """One call of the op: owns the argument blocks and every buffer the kernels touch
    (shared by the autograd function and the benchmark harness)."""

    OP = 1  # LMOE_OP_GLA

    def __init__(self, keep: bool = False):
        self.keep = keep

    def _gate(self, a, g, head_first):
        a.gate = _lib.GATE_VECTOR
        a.g = _desc(g, head_first)
        a.g_dtype = _lib.LMOE_F32 if g.dtype == torch.float32 else _lib.LMOE_BF16

    def forward(self, q, k, v, g, scale, initial_state, output_final_state, cu_seqlens, head_first, save=True):
        """save=False: a forward-only call (nothing requires a gradient): the per-chunk states are not written where
        the state pass forms the output itself (bf16); the fp32 path's output kernel reads them."""
        lib = _lib.load()
        plan = dims = None
        if cu_seqlens is not None:
            dims = _check_inputs(q, k, v, head_first, cu_seqlens)
            B, T = dims[:2]
            if g is not None and g.shape == q.shape:
                plan = seq_plan(B, T, cu_seqlens, q.device)
        if not self.keep:
            tables = None if plan is None else plan.tables
            r = native("forward", "chunk_gla forward", self.OP, q, k, v, g, None, initial_state, tables, scale,
                       output_final_state, head_first, save, 0, 0.0, False)
            if r is not None:
                o, ht, *kept = r
                self.saved = (q, k, v, g, initial_state, *kept)
                self.plan, self.dims, self.head_first, self.scale = plan, None, head_first, scale
                self.has_h0 = initial_state is not None
                return o, ht
        if dims is None:
            dims = _check_inputs(q, k, v, head_first, cu_seqlens)
        B, T, H, K, V = dims
        if g is None or tuple(g.shape) != tuple(q.shape):
            raise ValueError(f"g must have the shape of q {tuple(q.shape)}")
        # fp32 operands take an fp32 gate; bf16 operands take the gate as bf16 or fp32
        if q.dtype == torch.float32 or g.dtype not in (torch.float32, torch.bfloat16):
            g = g.float()
        q, k, v, g = _aligned(q), _aligned(k), _aligned(v), _aligned(g)
        if plan is None:
            plan = seq_plan(B, T, cu_seqlens, q.device)
        h0 = _state_check(initial_state, plan.N, H, K, V, "initial_state")
        a = base_args(q, k, v, head_first, scale, plan, dims)
        self._gate(a, g, head_first)
        a.h0 = ptr(h0)
        dev, dt = q.device, q.dtype
        o = torch.empty_like(v)
        ht = torch.empty(plan.N, H, K, V, dtype=torch.float32, device=dev) if output_final_state else None
        fused = dt == torch.bfloat16
        hs = torch.empty(max(plan.NT, 1), H, K, V, dtype=dt, device=dev) if (save or not fused) else None
        amat = torch.empty(max(plan.NT, 1), H, 64, 64, dtype=dt, device=dev)
        # gated operands of the state passes (q e^b, k e^{b_C - b}, e^{b_C}), formed once per chunk
        qe = torch.empty(max(plan.NT, 1), H, 64, K, dtype=dt, device=dev)
        ke = torch.empty_like(qe)
        gdec = torch.empty(max(plan.NT, 1), H, K, dtype=torch.float32, device=dev)
        a.o, a.ht, a.hs, a.amat = _desc(o, head_first), ptr(ht), ptr(hs), amat.data_ptr()
        a.qe, a.ke, a.gcum = qe.data_ptr(), ke.data_ptr(), gdec.data_ptr()
        seg_ws = cut_workspace(lib, a, self.OP, dev)
        _lib.check(lib.lmoe_chunk_gla_fwd(C.byref(a), stream_ptr()), "chunk_gla forward")
        self.saved = (q, k, v, g, h0, hs, amat, qe, ke, gdec)
        self.fwd_args, self.fwd_keep = a, ((o, ht, seg_ws) if self.keep else None)
        self.plan, self.dims, self.head_first, self.scale = plan, dims, head_first, scale
        self.has_h0 = initial_state is not None
        return o, ht

    def backward(self, do, dht):
        lib = _lib.load()
        q, k, v, g, h0, hs, amat, qe, ke, gdec = self.saved
        head_first = self.head_first
        if not self.keep:
            r = native("backward", "chunk_gla backward", self.OP, q, k, v, g, None, h0, self.plan and self.plan.tables,
                       self.scale, do, dht, head_first, (hs, amat, qe, ke, gdec), None)
            if r is not None:
                dq, dk, dv, dg, _, dh0 = r
                return dq, dk, dv, dg, dh0
        q, k, v, do, dims = inputs_came_back(q, k, v, do, head_first)
        B, T, H, K, V = dims
        plan = self.plan or seq_plan(B, T, None, q.device)
        dev, dt, nt = q.device, q.dtype, max(plan.NT, 1)
        g = came_back(g, q.shape, None, dev, "g")
        g = _aligned(g if dt == torch.bfloat16 else g.float())
        if self.has_h0:
            h0 = came_back(h0, (plan.N, H, K, V), torch.float32, dev, "initial_state")
        hs, amat = came_back(hs, (nt, H, K, V), dt, dev, "hs"), came_back(amat, (nt, H, 64, 64), dt, dev, "amat")
        qe, ke = came_back(qe, (nt, H, 64, K), dt, dev, "qe"), came_back(ke, (nt, H, 64, K), dt, dev, "ke")
        gdec = came_back(gdec, (nt, H, K), torch.float32, dev, "gdec")
        a = base_args(q, k, v, head_first, self.scale, plan, dims)
        self._gate(a, g, head_first)
        a.h0, a.hs, a.amat = ptr(h0), hs.data_ptr(), amat.data_ptr()
        a.qe, a.ke, a.gcum = qe.data_ptr(), ke.data_ptr(), gdec.data_ptr()
        a.d_o = _desc(do, head_first)
        dht = None if dht is None else dht.float().contiguous()
        a.dht = ptr(dht)
        dq, dk, dv = torch.empty_like(q), torch.empty_like(k), torch.empty_like(v)
        a.dq, a.dk, a.dv = _desc(dq, head_first), _desc(dk, head_first), _desc(dv, head_first)
        dg = torch.empty(g.shape, dtype=g.dtype, device=q.device)      # written in the dtype of g by the kernel
        a.dg = _desc(dg, head_first)
        dh0 = torch.empty_like(h0) if self.has_h0 else None
        a.dh0 = ptr(dh0)
        dhs = torch.empty_like(hs)
        a.dhs = dhs.data_ptr()
        seg_ws = cut_workspace(lib, a, self.OP, q.device)
        _lib.check(lib.lmoe_chunk_gla_bwd(C.byref(a), stream_ptr()), "chunk_gla backward")
        self.bwd_args = a
        self.bwd_keep = (do, dht, dq, dk, dv, dg, dh0, dhs, seg_ws) if self.keep else None
        return dq, dk, dv, dg, dh0


class _ChunkGLA(torch.autograd.Function):
    @staticmethod
    def forward(ctx, q, k, v, g, scale, initial_state, output_final_state, cu_seqlens, head_first):
        call = GLACall()
        o, ht = call.forward(q, k, v, g, scale, initial_state, output_final_state, cu_seqlens, head_first,
                             save=any(ctx.needs_input_grad))
        ctx.call, ctx.g_dtype = call, g.dtype
        stash(ctx, call)
        return o, ht

    @staticmethod
    def backward(ctx, do, dht):
        unstash(ctx, ctx.call)
        try:
            dq, dk, dv, dg, dh0 = ctx.call.backward(do, dht)
        finally:
            ctx.call.saved = None
        return dq, dk, dv, dg.to(ctx.g_dtype), None, dh0, None, None, None


def chunk_gla(
    q: torch.Tensor,
    k: torch.Tensor,
    v: torch.Tensor,
    g: torch.Tensor,
    scale: Optional[float] = None,
    initial_state: Optional[torch.Tensor] = None,
    output_final_state: bool = False,
    cu_seqlens: Optional[torch.Tensor] = None,
    head_first: bool = True,
) -> Tuple[torch.Tensor, Optional[torch.Tensor]]:
    """q, k, g: ``[B,H,T,K]``, v: ``[B,H,T,V]`` (``[B,T,H,*]`` with ``head_first=False``); g is the
    per-channel log-space decay.  Returns ``(o, final_state)``."""
    if q.dim() == 4 and v.dim() == 4 and (q.shape[-1] not in HEAD_DIMS or v.shape[-1] not in HEAD_DIMS):
        if g is None or g.shape != q.shape:
            raise ValueError("chunk_gla: g must have the shape of q")
        sc = q.shape[-1] ** -0.5 if scale is None else scale          # of the whole key, not of a block
        return by_head_dim_blocks(
            lambda q_, k_, v_, g_, h0: chunk_gla(q_, k_, v_, g_, sc, h0, output_final_state, cu_seqlens, head_first),
            q, k, v, g, initial_state, output_final_state, True, "chunk_gla")
    r = no_tokens(q, k, v, head_first, cu_seqlens, initial_state, output_final_state)
    if r is not None:
        return r
    if no_node(q, k, v, g, initial_state):
        return GLACall().forward(q, k, v, g, scale, initial_state, output_final_state, cu_seqlens, head_first, save=False)
    return _ChunkGLA.apply(q, k, v, g, scale, initial_state, output_final_state, cu_seqlens, head_first)
