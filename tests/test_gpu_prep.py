"""The pre-passes and the loss reduction shared by a call's relations: one
launch for every side's float16 keys (each side with its own scale), one for
every relation's row normalisers, one for the loss sum (kernel_B.py:216-218),
at the sizes where their work is cut."""

import ctypes
import math

import pytest
import torch

from linearard_amd import _lib
from linearard_amd.attention_KL import attn_kl_align
from linearard_amd.attention_KL.batched import attn_kl_align_batched

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 3, 1023, 1024, 1025, 65535, 65537, 70001])
def test_loss_is_the_sum_of_the_rows_at_slice_edges(gpu_available, n):
    """Slices of whole 1024-row units over at most 64 workgroups (n > 65536:
    two units each).  The row terms stand at the start of the workspace; their
    float64 sum is within the one rounding to float32 (2^-24 relative)."""
    L = _lib.lib()
    g = torch.Generator(device="cuda").manual_seed(n)
    T, H = (n, 1) if n < 4096 else (1, n)
    B = 1
    if H > 65536:  # B * heads is limited
        T, H = n, 1
    x = torch.randn((B, H, T, 8), device="cuda", generator=g).to(torch.float16)
    y = torch.randn((B, H, T, 8), device="cuda", generator=g).to(torch.float16)
    lse_s = torch.randn((B, H, T), device="cuda", generator=g)  # arbitrary: one-key rows then have terms too
    lse_t = torch.randn((B, H, T), device="cuda", generator=g)
    ws_bytes = L.lard_kl_forward_workspace_bytes(B, H, T)
    for _ in range(3):  # the ticket counter is cleared by every call
        ws = torch.full((ws_bytes,), 0xff, device="cuda", dtype=torch.uint8)
        loss = torch.empty((), device="cuda")
        d = [_lib.tensor4(t) for t in (x, x, y, y)]
        rc = L.lard_kl_forward(*(ctypes.byref(t) for t in d[:2]), lse_s.data_ptr(), *(ctypes.byref(t) for t in d[2:]),
                               lse_t.data_ptr(), ctypes.byref(_lib.mask_desc(None)), 1, 0.3, 0.3, loss.data_ptr(),
                               ws.data_ptr(), ws_bytes, _lib.stream_of(x))
        assert rc == 0, L.lard_last_error()
        rows = ws[:4 * n].view(torch.float32).double()
        # double sums in another order: far below the final rounding
        assert abs(loss.double() - rows.sum()) <= 2.0 ** -24 * abs(rows.sum()) + 1e-12 * rows.abs().sum()


@pytest.mark.parametrize("n", [3, 1025, 5000])
def test_loss_sum_in_a_workspace_at_8_bytes(gpu_available, n):
    """lard_kl_forward takes a workspace that a caller cut out of another at any
    multiple of 8 bytes: the same loss."""
    L = _lib.lib()
    g = torch.Generator(device="cuda").manual_seed(n)
    x, y = (torch.randn((1, 2, n, 8), device="cuda", generator=g).to(torch.float16) for _ in range(2))
    lse = torch.randn((1, 2, n), device="cuda", generator=g)
    size = L.lard_kl_forward_workspace_bytes(1, 2, n)
    ws = torch.empty((size + 16,), device="cuda", dtype=torch.uint8)
    d = [ctypes.byref(_lib.tensor4(t)) for t in (x, x, y, y)]
    loss = torch.empty((2,), device="cuda")
    for i, shift in enumerate((0, 8)):
        rc = L.lard_kl_forward(d[0], d[1], lse.data_ptr(), d[2], d[3], lse.data_ptr(), ctypes.byref(_lib.mask_desc(None)),
                               1, 0.3, 0.3, loss[i:].data_ptr(), ws.data_ptr() + shift, size, _lib.stream_of(x))
        assert rc == 0, L.lard_last_error()
    assert torch.equal(loss[0], loss[1])


@pytest.mark.parametrize("D,T", [(8, 1023), (8, 1025), (64, 127), (64, 129), (128, 63), (128, 64), (128, 65)])
@pytest.mark.parametrize("masked", [False, True])
def test_nine_relations_equal_single_calls(gpu_available, D, T, masked):
    """Nine relations (two groups) of 1-4 heads around the row blocks of the
    key conversion; relation 2's student and relation 5's teacher hold values
    beyond the float16 range, so exactly these two sides take a scale.  Losses
    and gradients equal the single-relation calls' (same kernels, same
    operands): gradients bitwise, the loss to the order of a float32 sum."""
    g = torch.Generator(device="cuda").manual_seed(D + T)
    heads = [1, 2, 4, 1, 3, 2, 1, 4, 2]
    xs, xt = [], []
    for r, H in enumerate(heads):
        t = torch.randn((2, H, T, D), device="cuda", generator=g) * 0.5
        s = t + 0.2 * torch.randn(t.shape, device="cuda", generator=g)
        if r == 2:
            s[0, 0, T // 2, 0] = 40000.0
        if r == 5:
            t[1, 0, T - 1, D - 1] = -40000.0
        xs.append(s.to(torch.bfloat16).requires_grad_(True))
        xt.append(t.to(torch.bfloat16))
    mask = None
    if masked:
        mask = torch.rand((2, T), device="cuda", generator=g) < 0.7
        mask[0, : T // 2] = False  # a left-padded sequence
    a = 1.0 / math.sqrt(D)
    loss = attn_kl_align_batched(xs, xt, attn_mask=mask, sm_scale_s=a, sm_scale_t=a)
    got = torch.autograd.grad(loss, xs)
    total = 0.0
    for s, t, dx in zip(xs, xt, got):
        one = attn_kl_align(s, s, t, t, attn_mask=mask, causal=True, sm_scale_s=a, sm_scale_t=a)
        ref, = torch.autograd.grad(one, [s])
        assert torch.equal(dx, ref)
        total += float(one.detach())
    assert abs(float(loss.detach()) - total) <= len(xs) * 2.0 ** -23 * max(1.0, abs(total))
