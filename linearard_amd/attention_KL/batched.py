"""Batched relation loss: the caller's loop over layers and Q/K/V relations.

The reference caller (train.py:369-410) computes, per aligned layer, three
self relations -- ``attn_kl_align(x_s, x_s, x_t, x_t)`` for x in Q, K, V --
divides each by ``denom`` (``B*Hq*T`` without a mask, ``mask.sum()*Hq``
with one, Hq the layer's query heads, train.py:403-406), sums them and
divides by the number of layers (train.py:410).  That is 3 L calls and
12 L kernel launches per micro-batch.

``attn_kl_align_batched(xs, xt, weights)`` computes
``sum_r weights[r] * attn_kl_align(xs[r], xs[r], xt[r], xt[r])`` with one
launch per 8 relations (``lard_attn_kl_batched_forward``):
the relations' row blocks share one grid even when their head counts differ
(Q/Q 32 heads next to K/K 8).  When the students need gradients the forward
is ``lard_attn_kl_batched_forward_rowgrad``, which also leaves the row side
of every gradient in float32 buffers, and the backward
(``lard_attn_kl_batched_backward_colgrad16``) adds the column side and writes
the gradients in the inputs' dtype (the buffers are only read, so a second
backward through the same graph does the same).  ``relation_kl_loss`` builds the weights of
the train.py formula from the layers' tensors.  Batches outside the batched
kernels (different head dims, D = 256, extreme scales) go relation by
relation through the single-relation entry points inside the same autograd
Function, so the result is the same either way.
"""

from __future__ import annotations

import ctypes

import torch

from .. import _lib
from ._checks import check_mask, check_relations, check_scale, require

__all__ = ["AttnKLBatchedFn", "attn_kl_align_batched", "relation_kl_loss"]


def _workspace(nbytes: int, device) -> torch.Tensor:
    return torch.empty((nbytes if nbytes > 0 else 1,), device=device, dtype=torch.uint8)


class AttnKLBatchedFn(torch.autograd.Function):
    """Forward: sum_r w_r KL_r.  Backward: the gradient of every student
    tensor xs[r] (teachers, weights, mask, flags and scales get None)."""

    @staticmethod
    def forward(ctx, weights, attn_mask, causal: bool, sm_scale_s, sm_scale_t, n: int, *tensors):
        xs, xt = list(tensors[:n]), list(tensors[n:])
        dev = xs[0].device
        B, _, T, _ = xs[0].shape
        for r in range(n):
            check_relations(xs[r], xs[r], xt[r], xt[r], strided_ok=True)
            require(xs[r].shape[0] == B and xs[r].shape[2] == T, "batched relations must share B and T")
        attn_mask = check_mask(attn_mask, dev, B, T)
        ss = [check_scale(sm_scale_s, x.shape[3], "sm_scale_s") for x in xs]
        st = [check_scale(sm_scale_t, x.shape[3], "sm_scale_t") for x in xt]
        weights = weights.detach().to(device=dev, dtype=torch.float32).contiguous()
        require(weights.shape == (n,), "weights must hold one value per relation")

        L = _lib.lib()
        rows = [B * x.shape[1] * T for x in xs]
        lse, at = _lib.stat_buffer(rows + rows, dev)
        lse_s, lse_t = at[:n], at[n:]
        loss = torch.empty((), device=dev, dtype=torch.float32)
        md = _lib.mask_desc(attn_mask)
        stream = _lib.stream_of(xs[0])
        batched = len(set(ss)) == 1 and len(set(st)) == 1
        row_grad = None
        if batched:
            want_grad = any(ctx.needs_input_grad[6:6 + n])
            if want_grad:
                row_grad = [torch.empty(x.shape, device=dev, dtype=torch.float32) for x in xs]
            rels = _lib.relations(xs, xt, lse_s, lse_t, row_grad and [x.data_ptr() for x in row_grad])
            ws_bytes = (L.lard_attn_kl_batched_rowgrad_workspace_bytes(rels, n) if want_grad
                        else L.lard_attn_kl_batched_workspace_bytes(rels, n))
            ws = _workspace(ws_bytes, dev)
            fn = L.lard_attn_kl_batched_forward_rowgrad if want_grad else L.lard_attn_kl_batched_forward
            rc = fn(rels, n, ctypes.byref(md), int(bool(causal)), ss[0], st[0], weights.data_ptr(), loss.data_ptr(),
                    ws.data_ptr(), ws_bytes, stream)
            if rc == _lib.LARD_ERR_UNSUPPORTED:
                batched = False
                row_grad = None
            else:
                _lib.check(rc, "lard_attn_kl_batched_forward_rowgrad" if want_grad else "lard_attn_kl_batched_forward")
        if not batched:
            # relation by relation (same kernels as attn_kl_align), summed on the device
            losses = torch.empty((n,), device=dev, dtype=torch.float32)
            for r in range(n):
                B_, H_, T_, _ = xs[r].shape
                ws_bytes = L.lard_attn_kl_forward_workspace_bytes(B_, H_, T_)
                ws = _workspace(ws_bytes, dev)
                d = [_lib.tensor4(x) for x in (xs[r], xt[r])]
                rc = L.lard_attn_kl_forward(ctypes.byref(d[0]), ctypes.byref(d[0]), ctypes.byref(d[1]),
                                            ctypes.byref(d[1]), ctypes.byref(md), int(bool(causal)), ss[r], st[r],
                                            lse_s[r], lse_t[r], losses[r:r + 1].data_ptr(),
                                            ws.data_ptr(), ws_bytes, stream)
                _lib.check(rc, "lard_attn_kl_forward")
            loss = (losses * weights).sum()

        ctx.has_row_grad = row_grad is not None
        ctx.save_for_backward(weights, attn_mask, lse, *xs, *xt, *(row_grad or []))
        ctx.n = n
        ctx.causal = bool(causal)
        ctx.ss, ctx.st = ss, st
        return loss

    @staticmethod
    def backward(ctx, dloss):
        n = ctx.n
        if not any(ctx.needs_input_grad[6:6 + n]):  # weights or teachers alone: no gradient
            return (None,) * (6 + 2 * n)
        saved = ctx.saved_tensors
        weights, attn_mask, lse = saved[:3]
        xs, xt = saved[3:3 + n], saved[3 + n:3 + 2 * n]
        at = _lib.stat_addresses(lse, [x.shape[0] * x.shape[1] * x.shape[2] for x in xs] * 2)
        lse_s, lse_t = at[:n], at[n:]
        dloss = _lib.loss_grad(dloss)
        dev = xs[0].device
        L = _lib.lib()
        md = _lib.mask_desc(attn_mask)
        stream = _lib.stream_of(xs[0])
        if ctx.has_row_grad:
            rels = _lib.relations(xs, xt, lse_s, lse_t, [x.data_ptr() for x in saved[3 + 2 * n:]])
            ws_bytes = L.lard_attn_kl_batched_workspace_bytes(rels, n)
            ws = _workspace(ws_bytes, dev)
            dxs = [torch.empty(x.shape, device=dev, dtype=x.dtype) for x in xs]
            out = (ctypes.c_void_p * n)(*(x.data_ptr() for x in dxs))
            rc = L.lard_attn_kl_batched_backward_colgrad16(rels, n, ctypes.byref(md), int(ctx.causal), ctx.ss[0],
                                                           ctx.st[0], weights.data_ptr(), dloss.data_ptr(), out,
                                                           ws.data_ptr(), ws_bytes, stream)
            _lib.check(rc, "lard_attn_kl_batched_backward_colgrad16")
            return (None, None, None, None, None, None, *dxs, *([None] * n))
        # relation by relation, as the forward
        dxs = [torch.empty(x.shape, device=dev, dtype=torch.float32) for x in xs]
        scaled = (dloss * weights).contiguous()  # dloss * w_r, one device scalar per relation
        for r in range(n):
            B_, H_, T_, D_ = xs[r].shape
            ws_bytes = L.lard_attn_kl_backward_workspace_bytes(B_, H_, H_, T_, D_, 1)
            ws = _workspace(ws_bytes, dev)
            d = [_lib.tensor4(x) for x in (xs[r], xt[r])]
            rc = L.lard_attn_kl_backward(
                ctypes.byref(d[0]), ctypes.byref(d[0]), lse_s[r], ctypes.byref(d[1]),
                ctypes.byref(d[1]), lse_t[r], ctypes.byref(md), int(ctx.causal), ctx.ss[r], ctx.st[r],
                scaled[r:r + 1].data_ptr(), 1, None, dxs[r].data_ptr(), ws.data_ptr(), ws_bytes, stream)
            _lib.check(rc, "lard_attn_kl_backward")
        return (None, None, None, None, None, None, *dxs, *([None] * n))


def attn_kl_align_batched(xs, xt, weights=None, attn_mask=None, causal=True, sm_scale_s=None, sm_scale_t=None):
    """``sum_r weights[r] * attn_kl_align(xs[r], xs[r], xt[r], xt[r], ...)``.

    ``xs``, ``xt``: sequences of [B, H_r, T, D] student / teacher tensors
    (one self relation each, as train.py:380-402 calls it), any views with a
    unit last stride (the attention hook's [B, T, H, D] projections seen as
    [B, H, T, D] need no .contiguous() copy, unlike train.py:133-142);
    ``weights``: a float32 tensor (or sequence) of one value per relation,
    default all 1.  Returns a 0-d float32 tensor; gradients flow to the
    ``xs`` tensors.
    """
    xs, xt = list(xs), list(xt)
    require(len(xs) > 0 and len(xs) == len(xt), "xs and xt must hold the same number (>= 1) of relations")
    dev = xs[0].device
    if weights is None:
        weights = torch.ones((len(xs),), device=dev, dtype=torch.float32)
    elif not isinstance(weights, torch.Tensor):
        weights = torch.tensor([float(w) for w in weights], device=dev, dtype=torch.float32)
    return AttnKLBatchedFn.apply(weights, attn_mask, causal, sm_scale_s, sm_scale_t, len(xs), *xs, *xt)


def denominators(qs, attn_mask, dev, repeat=1, fn=None):
    """float32 [len(qs) * repeat]: ``fn`` of each layer's denom (train.py:403-406:
    B * Hq * T, or mask.sum().clamp_min(1) * Hq with Hq the layer's query
    heads), each ``repeat`` times.  Layers with the same denom share one, so the
    launches do not grow with the layers."""
    valid, made, out = None, {}, []
    for q in qs:
        B, Hq, T, _ = q.shape
        key = Hq if attn_mask is not None else B * Hq * T
        if key not in made:
            if attn_mask is None:  # a fill on the device: a host tensor here would be a synchronising copy
                d = torch.full((), float(key), device=dev, dtype=torch.float32)
            else:
                if valid is None:
                    valid = attn_mask.sum().clamp_min(1).to(torch.float32)
                d = valid * Hq
            made[key] = d if fn is None else fn(d)
        out += [made[key]] * repeat
    if len(made) == 1:
        return out[0].repeat(len(out))
    return torch.stack(out)


def relation_kl_loss(qs, ks, vs, qt, kt, vt, attn_mask=None, sm_scale_s=None, sm_scale_t=None):
    """The attention-relation loss of train.py:360-410 in batched launches.

    ``qs``, ``ks``, ``vs`` (student) and ``qt``, ``kt``, ``vt`` (teacher) are
    sequences over the aligned layers of [B, H, T, D] tensors.  Per layer:
    Q/Q + K/K + V/V self relations (causal), each divided by ``denom`` =
    B * Hq * T (no mask) or mask.sum().clamp_min(1) * Hq, with Hq the layer's
    query-head count for all three (train.py:403-406); the layer sum is
    divided by max(1, L) (train.py:410).  No host synchronisation: the
    weights stay on the device.
    """
    L = len(qs)
    require(L > 0 and all(len(x) == L for x in (ks, vs, qt, kt, vt)), "one tensor per layer for each of Q, K, V")
    dev = qs[0].device
    if attn_mask is not None and attn_mask.device != dev:
        attn_mask = attn_mask.to(dev)
    xs, xt = [], []
    for layer in range(L):
        for s_, t_ in ((qs[layer], qt[layer]), (ks[layer], kt[layer]), (vs[layer], vt[layer])):
            xs.append(s_)
            xt.append(t_)
    weights = denominators(qs, attn_mask, dev, 3, lambda d: 1.0 / (d * L))
    return attn_kl_align_batched(xs, xt, weights, attn_mask=attn_mask, causal=True, sm_scale_s=sm_scale_s,
                                 sm_scale_t=sm_scale_t)
