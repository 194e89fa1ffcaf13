"""dk sums cut into parts (grouped queries on a grid below one workgroup per
CU): the autograd pair, the general backward and the stage entry point against
the float64 oracle, at ragged sizes and around every limit of the cut, and the
stage entry point without a workspace (uncut) against the cut one."""

import ctypes
import math

import numpy as np
import pytest
import torch

from linearard_amd import _lib
from oracle import attn_kl as O
from tests._inputs import make_mask, mask_to_dev, randn, to_dev
from tests._tolerance import check_grad

pytestmark = pytest.mark.gpu


def _problem(seed, dtype, B, hq, hkv, T, D, ratio):
    rng = np.random.default_rng(seed)
    shapes = [(B, hq), (B, hkv), (B, hq), (B, hkv)]
    qs, ks, qt, kt = (randn(rng, (b, h, T, D), dtype) for b, h in shapes)
    return qs, ks, qt, kt, None if ratio is None else make_mask(rng, B, T, ratio)


# key blocks of 256 rows x B x hkv, parts = group x ranges of query tiles
@pytest.mark.parametrize("dtype,B,hq,hkv,T,D,causal,ratio", [
    ("f16", 1, 4, 1, 63, 64, True, None),     # one block, one range
    ("bf16", 1, 2, 1, 257, 128, True, 0.3),   # two blocks, ranges of tiles; the second block's are short
    ("bf16", 2, 4, 2, 900, 128, False, 0.2),
    ("f16", 1, 8, 2, 1100, 64, True, None),   # five blocks, ranges shorter than the diagonal's distance
    ("bf16", 1, 6, 2, 515, 32, True, 0.4),    # group of 3
    ("bf16", 1, 4, 2, 300, 256, True, 0.2),   # the stage kernels in the autograd path
])
def test_cut_dk_matches_the_oracle(gpu_available, dtype, B, hq, hkv, T, D, causal, ratio):
    from linearard_amd.attention_KL import attn_kl_align, kl_backward, lse_stats

    qs, ks, qt, kt, mask = _problem(T + D, dtype, B, hq, hkv, T, D, ratio)
    L = _lib.lib()
    assert L.lard_kl_backward_workspace_bytes(B, hq, hkv, T, D) > 0  # the cut is taken
    a = 1 / math.sqrt(D)
    d = [to_dev(x, dtype, requires_grad=i < 2) for i, x in enumerate((qs, ks, qt, kt))]
    m = mask_to_dev(mask)
    case = f"dkparts-{dtype}-{B}-{hq}-{hkv}-{T}-{D}-c{int(causal)}-r{ratio}"
    _, rq, rk, _, _ = O.attn_kl_align(qs, ks, qt, kt, mask, causal, a, a)
    loss = attn_kl_align(d[0], d[1], d[2], d[3], attn_mask=m, causal=causal, sm_scale_s=a, sm_scale_t=a)
    two = 2.0 * loss  # dloss = 2 through the parts
    dq, dk = torch.autograd.grad(two, d[:2])
    check_grad(dq.float().cpu().numpy(), 2.0 * rq, case, "dq")
    check_grad(dk.float().cpu().numpy(), 2.0 * rk, case, "dk")
    x = [t.detach() for t in d]
    ls, lt = lse_stats(x[0], x[1], m, causal, a), lse_stats(x[2], x[3], m, causal, a)
    dq, dk = kl_backward(x[0], x[1], ls, x[2], x[3], lt, m, causal, a, a)
    check_grad(dk.cpu().numpy(), rk, case + "-stage", "dk")
    # uncut: no workspace; the sums run in another order (float32)
    dq0, dk0 = torch.empty_like(dq), torch.empty_like(dk)
    p = [ctypes.byref(_lib.tensor4(t)) for t in x]
    rc = L.lard_kl_backward(p[0], p[1], ls.data_ptr(), p[2], p[3], lt.data_ptr(), ctypes.byref(_lib.mask_desc(m)),
                            int(causal), a, a, dq0.data_ptr(), dk0.data_ptr(), _lib.stream_of(dq))
    assert rc == 0, L.lard_last_error()
    assert torch.equal(dq, dq0)
    assert float((dk - dk0).abs().max()) <= 1e-5 * float(dk0.abs().max())


# around each limit of the cut; parts: of one key block's sum
@pytest.mark.parametrize("B,hq,hkv,T,D,causal,parts,stage_parts", [
    (1, 2, 1, 2100, 16, True, 16, 16),   # 9 / 17 blocks of one group of 2: ranges of tiles, at their cap of 8
    (32, 8, 2, 250, 32, True, 4, 4),     # 64 / 128 blocks of a group of 4: one range (T < 256; 512 workgroups)
    (33, 8, 2, 250, 32, False, 4, 2),    # 66 / 132 blocks: the stage kernels take two heads a part
    (66, 8, 2, 60, 32, True, 2, 2),      # 132 blocks: two heads a part in both
    (33, 16, 2, 63, 64, True, 4, 4),     # 66 blocks of a group of 8
    (85, 9, 3, 30, 16, False, 2, 2),     # 255 blocks of a group of 3: parts of two heads and of one
    (64, 8, 4, 40, 16, True, 0, 0),      # 256 blocks: not cut
    (85, 6, 3, 129, 16, True, 2, 0),     # 255 / 510
])
def test_cut_dk_at_its_limits(gpu_available, B, hq, hkv, T, D, causal, parts, stage_parts):
    from linearard_amd.attention_KL import attn_kl_align, kl_backward, lse_stats

    qs, ks, qt, kt, mask = _problem(B + T, "f16", B, hq, hkv, T, D, 0.2)
    L = _lib.lib()
    part = B * hkv * T * D * 4
    assert L.lard_kl_backward_workspace_bytes(B, hq, hkv, T, D) == stage_parts * part
    base = L.lard_attn_kl_backward_workspace_bytes(B, hq, hq, T, D, 0)
    full = L.lard_attn_kl_backward_workspace_bytes(B, hq, hkv, T, D, 0)
    Tp = (T + 63) // 64 * 64
    layout = sum((n + 255) // 256 * 256 for n in (B * Tp, 8 * B, 4 * B * hq * Tp, 4 * B * hq * Tp, parts * part))
    assert full == max(base, layout, (stage_parts * part + 255) // 256 * 256)
    a = 1 / math.sqrt(D)
    d = [to_dev(x, "f16", requires_grad=i < 2) for i, x in enumerate((qs, ks, qt, kt))]
    m = mask_to_dev(mask)
    case = f"dklimits-{B}-{hq}-{hkv}-{T}-{D}-c{int(causal)}"
    _, rq, rk, _, _ = O.attn_kl_align(qs, ks, qt, kt, mask, causal, a, a)
    dq, dk = torch.autograd.grad(attn_kl_align(*d, attn_mask=m, causal=causal), d[:2])
    check_grad(dq.float().cpu().numpy(), rq, case, "dq")
    check_grad(dk.float().cpu().numpy(), rk, case, "dk")
    x = [t.detach() for t in d]
    ls, lt = lse_stats(x[0], x[1], m, causal, a), lse_stats(x[2], x[3], m, causal, a)
    _, dk = kl_backward(x[0], x[1], ls, x[2], x[3], lt, m, causal, a, a)
    check_grad(dk.cpu().numpy(), rk, case + "-stage", "dk")


def _general_backward(L, x, lse, mask, causal, a, dloss, self_rel):
    """lard_attn_kl_backward (both sides recomputed; no row side kept)."""
    B, hq, T, D = x[0].shape
    hkv = x[1].shape[1]
    dq = None if self_rel else torch.empty((B, hq, T, D), device="cuda")
    dk = torch.empty((B, hkv, T, D), device="cuda")
    nb = L.lard_attn_kl_backward_workspace_bytes(B, hq, hkv, T, D, int(self_rel))
    ws = torch.empty((nb,), device="cuda", dtype=torch.uint8)
    p = [ctypes.byref(_lib.tensor4(t)) for t in x]
    rc = L.lard_attn_kl_backward(p[0], p[1], lse[0].data_ptr(), p[2], p[3], lse[1].data_ptr(),
                                 ctypes.byref(_lib.mask_desc(mask)), int(causal), a, a, dloss.data_ptr(),
                                 int(self_rel), None if dq is None else dq.data_ptr(), dk.data_ptr(), ws.data_ptr(),
                                 nb, _lib.stream_of(dk))
    assert rc == 0, L.lard_last_error()
    return dq, dk


def test_backwards_accept_a_workspace_without_the_parts(gpu_available):
    """A workspace of the size for kv_heads == heads: the dk sums run uncut, equal
    to the cut ones up to the order of their float32 terms."""
    B, hq, hkv, T, D, causal = 1, 4, 2, 500, 64, True
    qs, ks, qt, kt, _ = _problem(11, "bf16", B, hq, hkv, T, D, None)
    a = 1 / math.sqrt(D)
    x = [to_dev(v, "bf16") for v in (qs, ks, qt, kt)]
    L = _lib.lib()
    p = [ctypes.byref(_lib.tensor4(t)) for t in x]
    md, st = ctypes.byref(_lib.mask_desc(None)), _lib.stream_of(x[0])
    lse = [torch.empty((B, hq, T), device="cuda") for _ in range(2)]
    out, dloss = torch.empty((), device="cuda"), torch.ones((), device="cuda")
    row = torch.empty((B, hq, T, D), device="cuda")
    ws = torch.empty((L.lard_attn_kl_forward_rowgrad_workspace_bytes(B, hq, hkv, hkv, T, D),), device="cuda",
                     dtype=torch.uint8)
    assert L.lard_attn_kl_forward_rowgrad(*p, md, int(causal), a, a, lse[0].data_ptr(), lse[1].data_ptr(),
                                          out.data_ptr(), row.data_ptr(), ws.data_ptr(), ws.numel(), st) == 0
    full = L.lard_attn_kl_backward_workspace_bytes(B, hq, hkv, T, D, 0)
    least = L.lard_attn_kl_backward_workspace_bytes(B, hq, hq, T, D, 0)
    assert least < full
    got = {}
    for size in (full, least):
        ws = torch.empty((size,), device="cuda", dtype=torch.uint8)
        head = (p[0], p[1], lse[0].data_ptr(), p[2], p[3], lse[1].data_ptr(), md, int(causal), a, a, dloss.data_ptr(), 0)
        tail = (ws.data_ptr(), size, st)
        q, k = torch.empty_like(row), torch.empty((B, hkv, T, D), device="cuda")
        q16, k16 = torch.empty_like(x[0]), torch.empty_like(x[1])
        r = row.clone()
        k2 = torch.empty_like(k)
        assert L.lard_attn_kl_backward(*head, q.data_ptr(), k.data_ptr(), *tail) == 0, L.lard_last_error()
        assert L.lard_attn_kl_backward_colgrad16(*head, row.data_ptr(), q16.data_ptr(), k16.data_ptr(),
                                                 *tail) == 0, L.lard_last_error()
        assert L.lard_attn_kl_backward_colgrad(*head, r.data_ptr(), k2.data_ptr(), *tail) == 0, L.lard_last_error()
        got[size] = q, k, k2, k16.float()
        assert L.lard_attn_kl_backward(*head, q.data_ptr(), k.data_ptr(), ws.data_ptr(), least - 1, st) == -1
    cut, uncut = got.values()
    assert torch.equal(cut[0], uncut[0])
    for c, u, bound in zip(cut[1:], uncut[1:], (1e-5, 1e-5, 2.0 ** -8)):  # float32 sums; one bfloat16 rounding
        assert float((c - u).abs().max()) <= bound * float(u.abs().max())


@pytest.mark.parametrize("dtype", ["f16", "bf16"])
@pytest.mark.parametrize("self_rel,hkv,T,D", [(True, 4, 333, 128), (True, 4, 65, 8), (False, 2, 900, 64), (False, 4, 130, 32)])
def test_gradients_in_the_input_dtype(gpu_available, dtype, self_rel, hkv, T, D):
    """colgrad16 is colgrad rounded once, bitwise, and both agree with the
    general backward (cut or not) and the oracle; a second backward of one
    graph repeats the first."""
    from linearard_amd.attention_KL import attn_kl_align

    B, hq, causal = 2, 4, True
    qs, ks, qt, kt, mask = _problem(T * 3 + D, dtype, B, hq, hkv, T, D, 0.3)
    if self_rel:
        ks, kt = qs, qt
    m = mask_to_dev(mask)
    a = 1 / math.sqrt(D)
    xq, yq = to_dev(qs, dtype, requires_grad=True), to_dev(qt, dtype)
    xk, yk = (xq, yq) if self_rel else (to_dev(ks, dtype, requires_grad=True), to_dev(kt, dtype))
    wrt = [xq] if self_rel else [xq, xk]
    loss = 1.5 * attn_kl_align(xq, xk, yq, yk, attn_mask=m, causal=causal, sm_scale_s=a, sm_scale_t=a)
    got = torch.autograd.grad(loss, wrt, retain_graph=True)
    again = torch.autograd.grad(loss, wrt)
    assert all(g.dtype == xq.dtype and torch.equal(g, h) for g, h in zip(got, again))
    L = _lib.lib()
    x = [t.detach() for t in (xq, xk, yq, yk)]
    d = [_lib.tensor4(t) for t in x]
    p = [ctypes.byref(t) for t in d]
    md, st = _lib.mask_desc(m), _lib.stream_of(x[0])
    lse = [torch.empty((B, hq, T), device="cuda") for _ in range(2)]
    out, dloss = torch.empty((), device="cuda"), torch.full((), 1.5, device="cuda")
    dq_row = torch.empty((B, hq, T, D), device="cuda")
    nb = L.lard_attn_kl_forward_rowgrad_workspace_bytes(B, hq, hkv, hkv, T, D)
    ws = torch.empty((nb,), device="cuda", dtype=torch.uint8)
    rc = L.lard_attn_kl_forward_rowgrad(*p, ctypes.byref(md), int(causal), a, a, lse[0].data_ptr(), lse[1].data_ptr(),
                                        out.data_ptr(), dq_row.data_ptr(), ws.data_ptr(), nb, st)
    assert rc == 0, L.lard_last_error()
    dk = torch.empty((B, hkv, T, D), device="cuda")
    nb = L.lard_attn_kl_backward_workspace_bytes(B, hq, hkv, T, D, int(self_rel))
    ws = torch.empty((nb,), device="cuda", dtype=torch.uint8)
    rc = L.lard_attn_kl_backward_colgrad(p[0], p[1], lse[0].data_ptr(), p[2], p[3], lse[1].data_ptr(), ctypes.byref(md),
                                         int(causal), a, a, dloss.data_ptr(), int(self_rel), dq_row.data_ptr(),
                                         dk.data_ptr(), ws.data_ptr(), nb, st)
    assert rc == 0, L.lard_last_error()
    f32 = [dk] if self_rel else [dq_row, dk]
    for g, f in zip(got, f32):
        assert torch.equal(g, f.to(g.dtype))
    gq, gk = _general_backward(L, x, lse, m, causal, a, dloss, self_rel)
    ref = O.attn_kl_align(qs, ks, qt, kt, mask, causal, a, a, dloss=1.5, self_relation=self_rel)
    case = f"grad16-{dtype}-{int(self_rel)}-{hkv}-{T}-{D}"
    for name, g, f, r in zip(("dX",) if self_rel else ("dq", "dk"), got, (gk,) if self_rel else (gq, gk), ref[1:3]):
        check_grad(g.float().cpu().numpy(), r, case, name)
        check_grad(f.cpu().numpy(), r, case + "-general", name)


def test_batched_gradients_against_the_general_batched_backward(gpu_available):
    """Autograd's batched gradients (input dtype, row side from the forward)
    and lard_attn_kl_batched_backward (both sides recomputed) agree within the
    gradient bar, relation by relation."""
    from linearard_amd.attention_KL.batched import attn_kl_align_batched

    rng = np.random.default_rng(77)
    B, T, D, heads = 2, 200, 64, [4, 1, 2]
    xs = [to_dev(randn(rng, (B, h, T, D), "bf16"), "bf16", requires_grad=True) for h in heads]
    xt = [to_dev(randn(rng, (B, h, T, D), "bf16"), "bf16") for h in heads]
    m = mask_to_dev(make_mask(rng, B, T, 0.2))
    w = torch.tensor([0.5, 2.0, 1.0], device="cuda")
    loss = attn_kl_align_batched(xs, xt, w, attn_mask=m, sm_scale_s=0.1, sm_scale_t=0.1)
    got = torch.autograd.grad(loss, xs)
    L, n = _lib.lib(), len(xs)
    s = [x.detach() for x in xs]
    lse_s = [torch.empty(x.shape[:3], device="cuda") for x in s]
    lse_t = [torch.empty(x.shape[:3], device="cuda") for x in s]
    dx = [torch.empty(x.shape, device="cuda") for x in s]
    rels = _lib.relations(s, xt, *([t.data_ptr() for t in ts] for ts in (lse_s, lse_t, dx)))
    nb = L.lard_attn_kl_batched_workspace_bytes(rels, n)
    ws = torch.empty((nb,), device="cuda", dtype=torch.uint8)
    out, one = torch.empty((), device="cuda"), torch.ones((), device="cuda")
    md = _lib.mask_desc(m)
    rc = L.lard_attn_kl_batched_forward(rels, n, ctypes.byref(md), 1, 0.1, 0.1, w.data_ptr(), out.data_ptr(),
                                        ws.data_ptr(), nb, _lib.stream_of(out))
    assert rc == 0, L.lard_last_error()
    rc = L.lard_attn_kl_batched_backward(rels, n, ctypes.byref(md), 1, 0.1, 0.1, w.data_ptr(), one.data_ptr(),
                                         ws.data_ptr(), nb, _lib.stream_of(out))
    assert rc == 0, L.lard_last_error()
    for r, (g, f) in enumerate(zip(got, dx)):
        check_grad(g.float().cpu().numpy(), f.cpu().numpy(), f"batched-general-rel{r}")
