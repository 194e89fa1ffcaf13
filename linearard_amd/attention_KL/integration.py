"""Autograd boundary: ``AttnKLAlignFn`` / ``attn_kl_align`` (mirrors integration.py:6-73).

``attn_kl_align(qs, ks, qt, kt, attn_mask=None, causal=True,
sm_scale_s=None, sm_scale_t=None)`` returns the 0-d float32 SUM over rows of
KL(P_t || P_s), P_x = softmax of the (masked, causal) relation logits
sm_scale_x * q_x . k_x.  Gradients flow to qs and ks only; the teacher,
mask, causal flag and scales get None (integration.py:67).

Forward (``lard_attn_kl_forward``): stage A for both relations and stage B in
one pass over the key tiles; only the two LSE vectors are saved (O(n), as in
integration.py:40).  Backward (``lard_attn_kl_backward``): stage C as a
row-owner pass (dq) and a column-owner pass (dk), both with D = P_s - P_t cast
to the input dtype before the product like kernel_C.py:233.  For the train.py
call ``attn_kl_align(x, x, y, y)`` (q is k) the library sums dq + dk in place
and the Function returns that whole gradient of ``x`` once (None for the
second input) instead of two float32 tensors for autograd to add.

When the student needs a gradient and the operands take the throughput
kernels, the forward is ``lard_attn_kl_forward_rowgrad`` instead: the same
pass also forms the row side of the gradient (dq before dloss, a float32
[B, Hq, T, Ds] buffer kept for the backward, O(n d) like the gradient
itself), and the backward runs only the column side
(``lard_attn_kl_backward_colgrad16``), which adds that buffer to itself and
writes the gradient in the inputs' dtype (the buffer is only read: a second
backward through the same graph does the same).  For float32
inputs that need a gradient the pair is ``lard_attn_kl_forward_lse64`` /
``lard_attn_kl_backward_lse64``, which keeps both LSEs in double between the
passes.
"""

from __future__ import annotations

import ctypes
import warnings

import torch

from .. import _lib
from ._checks import check_mask, check_relations, check_scale

__all__ = ["AttnKLAlignFn", "attn_kl_align"]


def _workspace(nbytes: int, device) -> torch.Tensor:
    return torch.empty((nbytes if nbytes > 0 else 1,), device=device, dtype=torch.uint8)


PATH_NAMES = {0: "throughput", 1: "fused-forward", 2: "stage", 3: "float32"}
_WARNED = set()


def kernel_path(d, ss: float, st: float):
    """(path name, condition) of lard_attn_kl_path for the four operand descriptors."""
    L = _lib.lib()
    rc = L.lard_attn_kl_path(ctypes.byref(d[0]), ctypes.byref(d[1]), ctypes.byref(d[2]), ctypes.byref(d[3]), ss, st)
    if rc < 0:  # a path code otherwise, not a status
        _lib.check(rc, "lard_attn_kl_path")
    return PATH_NAMES[rc], L.lard_last_error().decode()


def _warn_slow_path(d, ss: float, st: float) -> str:
    """The path's name, with one RuntimeWarning per condition that moves a call
    off the throughput kernels."""
    name, why = kernel_path(d, ss, st)
    if name != "throughput" and why not in _WARNED:
        _WARNED.add(why)
        warnings.warn(f"attn_kl_align: {why}: these inputs run the {name} kernels, not the throughput "
                      f"kernels (slower)", RuntimeWarning, stacklevel=3)
    return name


def _descs(qs, ks, qt, kt):
    """The operands' descriptors (one per tensor: a self relation has two)."""
    d = [_lib.tensor4(qs), None, _lib.tensor4(qt), None]
    d[1] = d[0] if ks is qs else _lib.tensor4(ks)
    d[3] = d[2] if kt is qt else _lib.tensor4(kt)
    return d


class AttnKLAlignFn(torch.autograd.Function):
    @staticmethod
    def forward(ctx, qs, ks, qt, kt, attn_mask, causal: bool, sm_scale_s, sm_scale_t):
        """integration.py:8-45: stage A x2 + stage B."""
        B, Hq, T, Ds, Dt = check_relations(qs, ks, qt, kt)
        attn_mask = check_mask(attn_mask, qs.device, B, T)
        ss = check_scale(sm_scale_s, Ds, "sm_scale_s")
        st = check_scale(sm_scale_t, Dt, "sm_scale_t")

        L = _lib.lib()
        dev = qs.device
        rows = B * Hq * T
        lse, (lse_s, lse_t) = _lib.stat_buffer((rows, rows), dev)
        loss = torch.empty((), device=dev, dtype=torch.float32)
        d = _descs(qs, ks, qt, kt)
        p = [ctypes.byref(x) for x in d]
        path = _warn_slow_path(d, ss, st) if rows > 0 else "throughput"
        md = _lib.mask_desc(attn_mask)
        stream = _lib.stream_of(qs)
        dq_row = lse64 = None
        needs_grad = ctx.needs_input_grad[0] or ctx.needs_input_grad[1]
        row_side = path == "throughput" and rows > 0 and needs_grad
        ws_bytes = (L.lard_attn_kl_forward_rowgrad_workspace_bytes(B, Hq, ks.shape[1], kt.shape[1], T, Ds) if row_side
                    else L.lard_attn_kl_forward_workspace_bytes(B, Hq, T))
        ws = _workspace(ws_bytes, dev)
        if row_side:
            dq_row = torch.empty((B, Hq, T, Ds), device=dev, dtype=torch.float32)
            rc = L.lard_attn_kl_forward_rowgrad(*p, ctypes.byref(md), int(bool(causal)), ss, st, lse_s, lse_t,
                                                loss.data_ptr(), dq_row.data_ptr(), ws.data_ptr(), ws_bytes, stream)
            _lib.check(rc, "lard_attn_kl_forward_rowgrad")
        elif path == "float32" and needs_grad:
            lse64 = torch.empty((2, B, Hq, T), device=dev, dtype=torch.float64)
            rc = L.lard_attn_kl_forward_lse64(*p, ctypes.byref(md), int(bool(causal)), ss, st, lse_s, lse_t,
                                              loss.data_ptr(), lse64.data_ptr(), ws.data_ptr(), ws_bytes, stream)
            _lib.check(rc, "lard_attn_kl_forward_lse64")
        else:
            rc = L.lard_attn_kl_forward(*p, ctypes.byref(md), int(bool(causal)), ss, st, lse_s, lse_t,
                                        loss.data_ptr(), ws.data_ptr(), ws_bytes, stream)
            _lib.check(rc, "lard_attn_kl_forward")

        ctx.has_row_grad = dq_row is not None
        ctx.has_lse64 = lse64 is not None
        ctx.save_for_backward(qs, ks, qt, kt, lse, attn_mask, dq_row if dq_row is not None else lse64)
        ctx.causal = bool(causal)
        ctx.sm_scale_s = ss
        ctx.sm_scale_t = st
        ctx.self_relation = qs is ks
        return loss

    @staticmethod
    def backward(ctx, dloss):
        """integration.py:48-67: stage C and the chain rule with dloss."""
        qs, ks, qt, kt, lse, attn_mask, extra = ctx.saved_tensors
        if ctx.self_relation:  # saved-tensor hooks hand out a tensor for each
            ks = qs
        dloss = _lib.loss_grad(dloss)
        B, Hq, T, Ds = qs.shape
        Hkv = ks.shape[1]
        self_rel = ctx.self_relation
        dev = qs.device
        L = _lib.lib()
        ps, pk, pt, pkt = [ctypes.byref(x) for x in _descs(qs, ks, qt, kt)]
        lse_s, lse_t = _lib.stat_addresses(lse, (B * Hq * T,) * 2)
        md = _lib.mask_desc(attn_mask)
        stream = _lib.stream_of(qs)
        head = (ps, pk, lse_s, pt, pkt, lse_t)
        opts = (ctypes.byref(md), int(ctx.causal), ctx.sm_scale_s, ctx.sm_scale_t, dloss.data_ptr(), int(self_rel))
        # the row side may have come with the forward: the column side then adds
        # itself to it (self relation), or it becomes dq; both in the inputs' dtype
        dtype = qs.dtype if ctx.has_row_grad else torch.float32
        dk = torch.empty((B, Hkv, T, Ds), device=dev, dtype=dtype)
        dq = None if self_rel else torch.empty((B, Hq, T, Ds), device=dev, dtype=dtype)
        out = (None if dq is None else dq.data_ptr(), dk.data_ptr())
        if ctx.has_lse64:  # float32 inputs: the forward kept its LSEs in double
            rc = L.lard_attn_kl_backward_lse64(*head, extra.data_ptr(), *opts, *out, stream)
            _lib.check(rc, "lard_attn_kl_backward_lse64")
        else:
            ws_bytes = L.lard_attn_kl_backward_workspace_bytes(B, Hq, Hkv, T, Ds, int(self_rel))
            ws = _workspace(ws_bytes, dev)
            if ctx.has_row_grad:
                rc = L.lard_attn_kl_backward_colgrad16(*head, *opts, extra.data_ptr(), *out, ws.data_ptr(), ws_bytes,
                                                       stream)
                _lib.check(rc, "lard_attn_kl_backward_colgrad16")
            else:
                rc = L.lard_attn_kl_backward(*head, *opts, *out, ws.data_ptr(), ws_bytes, stream)
                _lib.check(rc, "lard_attn_kl_backward")
        return (dk if self_rel else dq), (None if self_rel else dk), None, None, None, None, None, None


def attn_kl_align(qs, ks, qt, kt, attn_mask=None, causal=True, sm_scale_s=None, sm_scale_t=None):
    """Drop-in for integration.py:70-73."""
    return AttnKLAlignFn.apply(qs, ks, qt, kt, attn_mask, causal, sm_scale_s, sm_scale_t)
