"""Mixture-of-memories routing on MI355X: pack the routed tokens of all memories into one variable-length
batch, run the op once, combine the results per token.

The reference pads the tokens routed to every (memory, batch row) to a common capacity
(``transform``, ``linear_moe/sequence_modeling/mom_linear_attention.py:15-77``), calls the op once per
memory (``:369-409``) and scatters the results back (``reconstruct``, ``:79-120``).  Left padding with
zero tokens does not change a linear-attention state, so the same function is computed by one
``cu_seqlens`` call over the packed tokens: no padded rows, one launch for all memories.

    plan = mom_plan(selected_memories, num_memories, capacity)     # index tables (device)
    xp   = mom_pack(hidden, plan)                                  # [T_total, D]; rows of memory m:
                                                                   #   plan.mem_offsets[m] : plan.mem_offsets[m + 1]
    ... per-memory projections on those row ranges, then one op call with cu_seqlens = plan.cu_seqlens ...
    out  = mom_combine(op_output_rows, plan, routing_weights)      # [B, S, D']

Sequences are ordered memory-major: sequence ``m * B + b`` holds the tokens of batch row ``b`` routed to
memory ``m``, in time order, truncated to the last ``max_len`` of them exactly as the reference truncates.
"""
from __future__ import annotations

import math
from dataclasses import dataclass
from typing import Optional

import torch

from . import _lib
from ._host import came_back, native_call, stream_ptr


@dataclass
class MomPlan:
    B: int
    S: int
    topk: int
    num_memories: int
    T_total: int
    src_token: torch.Tensor     # [T_total] int32: flat token index b * S + t of every packed row
    src_choice: torch.Tensor    # [T_total] int32: flat (token, k) index of every packed row
    row_of: torch.Tensor        # [B * S, topk] int32: packed row of every (token, k), -1 if dropped
    cu_seqlens: torch.Tensor    # [num_memories * B + 1] int32 (device)
    max_len_dev: torch.Tensor   # 0-dim int64 (device): tokens kept per sequence at most
    mem_offsets_dev: torch.Tensor   # [num_memories + 1] int64 (device): row range of every memory

    # the two figures a caller may want on the host are read back only when asked for
    @property
    def max_len(self) -> int:
        return int(self.max_len_dev)

    @property
    def mem_offsets(self) -> torch.Tensor:
        return self.mem_offsets_dev.to("cpu")


def mom_plan(selected_memories: torch.Tensor, num_memories: int, capacity: Optional[float] = None,
             check: bool = False) -> MomPlan:
    """Index tables for ``selected_memories`` [B, S, topk] (as ``torch.topk`` returns them,
    mom_linear_attention.py:288).  ``capacity``: the reference's capacity factor; ``None`` keeps every token.

    Built on the device (a stable counting sort by (memory, batch row) in one to three launches; what its kernels do not take
    -- more than 1024 memories, or more than 8192 counts of a memory in 2048 choices of a batch row --
    by tensor operations), as the reference builds its tables (mom_linear_attention.py:28-66).  Without a capacity nothing is read
    back to the host: every routed token is kept, ``T_total = B * S * topk`` is known up front, and pack -> op ->
    combine can run inside a HIP graph capture with the plan in it.  With a capacity the number of surviving rows is
    the one device-to-host read of the call.  ``check`` validates the memory indices (two more reads).  Unchecked indices
    outside [0, num_memories) are a mistake of the caller: the kernels drop such a choice (``row_of`` -1; the rows behind
    ``cu_seqlens[-1]`` then belong to nobody and hold ``src_token`` -1), the tensor operations are undefined for it."""
    if selected_memories.dim() != 3:
        raise ValueError("selected_memories must be [B, S, topk]")
    B, S, topk = selected_memories.shape
    if not check:
        r = native_call("mom_plan", "mom_plan", selected_memories, num_memories, _cap(S, capacity))
        if r is not None:
            return _plan_of(r, B, S, topk, num_memories, capacity)
    dev = selected_memories.device
    sel = selected_memories.reshape(-1)                                        # flat (b, t, k)
    if check and sel.numel() and (int(sel.min()) < 0 or int(sel.max()) >= num_memories):
        raise ValueError("selected_memories out of range")
    n = sel.numel()
    if sel.is_cuda and sel.device.index == torch.cuda.current_device() and n < 2 ** 31:
        plan = _plan_native(sel, B, S, topk, num_memories, capacity)
        if plan is not None:
            return plan
    return _plan_by_sorting(sel.to(torch.int64), B, S, topk, num_memories, capacity)


def _cap(S, capacity):
    return -1 if capacity is None else max(0, min(math.ceil(S * capacity), 2 ** 31 - 1))


def _plan_of(tables, B, S, topk, num_memories, capacity):
    """The plan of the tables that the library's kernels have formed."""
    cu, longest, offsets, src_token, src_choice, row_of = tables
    T_total = B * S * topk
    if capacity is not None:
        T_total = int(cu[-1])                                                  # (the one read: how many survive)
        src_token, src_choice = src_token[:T_total], src_choice[:T_total]
    return MomPlan(B, S, topk, num_memories, T_total, src_token, src_choice, row_of, cu, longest, offsets)


def _plan_native(sel, B, S, topk, num_memories, capacity):
    """The plan from the library's kernels, or None for sizes they do not take."""
    lib = _lib.load()
    n, dev = sel.numel(), sel.device
    ints = lib.lmoe_mom_plan_ints(B, S * topk, num_memories)
    if ints == 0:
        return None
    if sel.dtype not in (torch.int32, torch.int64):
        sel = sel.to(torch.int64)
    sel = sel.contiguous()                             # (a flattened slice or expanded tensor keeps its stride)
    seqs = num_memories * B
    wide = torch.empty(num_memories + 2, dtype=torch.int64, device=dev)
    counts, cu, src_token, src_choice, row_of = (torch.empty(k, dtype=torch.int32, device=dev)
                                                 for k in (ints, seqs + 1, n, n, n))
    _lib.check(lib.lmoe_mom_plan(sel.data_ptr(), int(sel.dtype == torch.int64), B, S * topk, topk, num_memories, _cap(S, capacity),
                                 counts.data_ptr(), cu.data_ptr(), wide.data_ptr(), wide.data_ptr() + 8,
                                 src_token.data_ptr(), src_choice.data_ptr(), row_of.data_ptr(), stream_ptr()), "mom_plan")
    return _plan_of((cu, wide[0], wide[1:], src_token, src_choice, row_of.view(B * S, topk)), B, S, topk, num_memories, capacity)


def _plan_by_sorting(sel, B, S, topk, num_memories, capacity):
    dev, n = sel.device, sel.numel()
    flat = torch.arange(n, device=dev)
    b_of = flat // (S * topk)
    key = sel * B + b_of                                                       # memory-major sequences
    order = torch.argsort(key, stable=True)                                    # time order inside a sequence
    lens = torch.zeros(num_memories * B, dtype=torch.int64, device=dev).scatter_add_(0, key, torch.ones_like(key))
    longest = lens.max() if lens.numel() else torch.zeros((), dtype=torch.int64, device=dev)
    row_of = torch.full((n,), -1, dtype=torch.int32, device=dev)
    cu = torch.zeros(num_memories * B + 1, dtype=torch.int64, device=dev)
    if capacity is None:
        max_len_dev = longest
        cu[1:] = torch.cumsum(lens, 0)
        rows, T_total = order, n                                               # every (token, k), sorted
    else:
        max_len_dev = torch.clamp(longest, max=math.ceil(S * capacity))
        starts = torch.cumsum(lens, 0) - lens
        skey = key[order]
        pos = flat - starts[skey]                                              # position inside its sequence
        keep = pos >= (lens[skey] - max_len_dev)                               # the last max_len survive
        cu[1:] = torch.cumsum(torch.minimum(lens, max_len_dev), 0)
        rows = order[keep]                                                     # (the one read: how many survive)
        T_total = int(rows.numel())
    row_of[rows] = torch.arange(T_total, dtype=torch.int32, device=dev)
    return MomPlan(B, S, topk, num_memories, T_total, (rows // topk).to(torch.int32).contiguous(),
                   rows.to(torch.int32).contiguous(), row_of.view(B * S, topk).contiguous(),
                   cu.to(torch.int32).contiguous(), max_len_dev, cu[::B].contiguous())


def _dt(t):
    if t.dtype not in (torch.bfloat16, torch.float32):
        raise ValueError(f"dtype {t.dtype} unsupported (bfloat16 or float32)")
    return _lib.LMOE_F32 if t.dtype == torch.float32 else _lib.LMOE_BF16


def _rows(x: torch.Tensor, n: int, what: str) -> torch.Tensor:
    if not x.is_cuda:
        raise RuntimeError("linear_moe_amd ops are GPU only (no CPU fallback)")
    x2 = x.reshape(n, -1).contiguous()
    if x2.shape[1] % 8:
        raise ValueError(f"{what}: row length {x2.shape[1]} must be a multiple of 8")
    return x2


class _Pack(torch.autograd.Function):
    @staticmethod
    def forward(ctx, x, plan):
        ctx.plan, ctx.shape = plan, x.shape
        r = native_call("mom_gather", "mom_pack", x, plan.B * plan.S, plan.src_token)
        if r is not None:
            return r[0]
        lib = _lib.load()
        x2 = _rows(x, plan.B * plan.S, "mom_pack")
        D = x2.shape[1]
        out = torch.empty(plan.T_total, D, dtype=x.dtype, device=x.device)
        _lib.check(lib.lmoe_mom_gather(x2.data_ptr(), plan.src_token.data_ptr(), None, out.data_ptr(), plan.T_total, D,
                                       _dt(x), stream_ptr()), "mom_pack")
        return out

    @staticmethod
    def backward(ctx, dout):
        plan = ctx.plan
        r = native_call("mom_combine", "mom_pack backward", dout, plan.T_total, plan.row_of, None, plan.B * plan.S, plan.topk)
        if r is not None:
            return r[0].view(ctx.shape), None
        lib = _lib.load()
        d2 = dout.contiguous()
        D = d2.shape[1]
        dx = torch.empty(plan.B * plan.S, D, dtype=dout.dtype, device=dout.device)
        _lib.check(lib.lmoe_mom_combine(d2.data_ptr(), plan.row_of.data_ptr(), None, dx.data_ptr(), plan.B * plan.S,
                                        plan.topk, D, _dt(dout), stream_ptr()), "mom_pack backward")
        return dx.view(ctx.shape), None


class _Combine(torch.autograd.Function):
    @staticmethod
    def forward(ctx, y, w, plan):
        ctx.plan, ctx.yshape, ctx.wshape, ctx.dtype, ctx.wdtype = plan, y.shape, w.shape, y.dtype, w.dtype
        r = native_call("mom_combine", "mom_combine", y, plan.T_total, plan.row_of, w, plan.B * plan.S, plan.topk)
        if r is not None:
            ctx.saved_shapes = y.shape, w.shape
            ctx.save_for_backward(y, w)
            return r[0].view((plan.B, plan.S) + tuple(y.shape[1:]))
        lib = _lib.load()
        y2 = _rows(y, plan.T_total, "mom_combine")
        D = y2.shape[1]
        w2 = w.reshape(plan.B * plan.S, plan.topk).to(y.dtype).contiguous()
        out = torch.empty(plan.B * plan.S, D, dtype=y.dtype, device=y.device)
        _lib.check(lib.lmoe_mom_combine(y2.data_ptr(), plan.row_of.data_ptr(), w2.data_ptr(), out.data_ptr(),
                                        plan.B * plan.S, plan.topk, D, _dt(y), stream_ptr()), "mom_combine")
        ctx.saved_shapes = y2.shape, w2.shape
        ctx.save_for_backward(y2, w2)
        return out.view((plan.B, plan.S) + tuple(y.shape[1:]))

    @staticmethod
    def backward(ctx, dout):
        y2, w2 = ctx.saved_tensors
        plan = ctx.plan
        r = native_call("mom_combine_backward", "mom_combine backward", y2, plan.T_total, plan.row_of, plan.src_choice, w2, dout,
                        plan.B * plan.S, plan.topk)
        if r is not None:
            return r[0].view(ctx.yshape), r[1].view(ctx.wshape).to(ctx.wdtype), None
        lib = _lib.load()
        yshape, wshape = ctx.saved_shapes
        D = yshape[1:].numel()
        y2 = came_back(y2, yshape, ctx.dtype, dout.device, "y")
        w2 = came_back(w2, wshape, ctx.dtype, dout.device, "routing_weights")
        g = came_back(dout, (plan.B, plan.S, *ctx.yshape[1:]), ctx.dtype, dout.device, "the gradient")
        # dy[row] = w[choice(row)] * dout[token(row)];  dw[t][k] = <dout[t], y[row_of[t][k]]>
        dy, dw = torch.empty_like(y2), torch.empty_like(w2)
        _lib.check(lib.lmoe_mom_combine_bwd(y2.data_ptr(), plan.row_of.data_ptr(), plan.src_choice.data_ptr(),
                                            w2.data_ptr(), g.data_ptr(), dy.data_ptr(), dw.data_ptr(), plan.B * plan.S,
                                            plan.T_total, plan.topk, D, _dt(y2), stream_ptr()), "mom_combine backward")
        return dy.view(ctx.yshape), dw.view(ctx.wshape).to(ctx.wdtype), None


def mom_pack(x: torch.Tensor, plan: MomPlan) -> torch.Tensor:
    """x [B, S, D] -> packed rows [T_total, D] (memory-major sequences, see the module docstring)."""
    if x.shape[0] != plan.B or x.shape[1] != plan.S:
        raise ValueError("mom_pack: x must be [B, S, ...] of the plan")
    return _Pack.apply(x, plan)


def mom_combine(y: torch.Tensor, plan: MomPlan, routing_weights: torch.Tensor) -> torch.Tensor:
    """y [T_total, ...] (the op's output rows), routing_weights [B, S, topk] -> [B, S, ...]:
    ``out[b, t] = sum_k w[b, t, k] * y[row of (b, t, k)]``; tokens dropped by the capacity contribute nothing."""
    if y.shape[0] != plan.T_total:
        raise ValueError("mom_combine: y must have T_total rows")
    return _Combine.apply(y, routing_weights, plan)
