"""float32 inputs: the stage entry points and the autograd pair against the
float64 oracle and against float32 eager PyTorch (materialised KL).

The reference's kernels take fp16/bf16 only (kernel_A.py:195-196); the
float32 path keeps the products and D = P_s - P_t in float32.  Tolerance
(written here, from the benchmark contract): loss relative error <= 1e-5
and gradient max-abs error <= 1e-5 of the gradient's max magnitude.
"""

import math

import numpy as np
import pytest
import torch

from oracle import attn_kl as O
from tests._inputs import make_mask, mask_to_dev, randn, to_dev
from tests._tolerance import check_grad, check_loss

pytestmark = pytest.mark.gpu

F32_BAR = 1e-5  # the north star's float32 bar, for the loss and the gradients

CASES = [  # causal, ratio, B, hq, hks, hkt, T, ds, dt
    (True, None, 1, 4, 4, 4, 97, 128, 128),
    (False, 0.3, 2, 4, 2, 1, 65, 64, 64),
    (True, 0.2, 1, 8, 2, 4, 130, 32, 128),   # GQA on both sides, Ds != Dt
    (True, None, 1, 2, 2, 2, 40, 256, 8),
    (True, None, 1, 1, 1, 1, 1, 16, 16),     # one token
]


def _inputs(rng, B, hq, hks, hkt, T, ds, dt, ratio, scale=1.0):
    qs = randn(rng, (B, hq, T, ds), "f32", scale)
    ks = randn(rng, (B, hks, T, ds), "f32", scale)
    qt = randn(rng, (B, hq, T, dt), "f32", scale)
    kt = randn(rng, (B, hkt, T, dt), "f32", scale)
    mask = None if ratio is None else make_mask(rng, B, T, ratio)
    return qs, ks, qt, kt, mask


@pytest.mark.parametrize("causal,ratio,B,hq,hks,hkt,T,ds,dt", CASES)
def test_f32_stages_match_the_oracle(gpu_available, causal, ratio, B, hq, hks, hkt, T, ds, dt):
    from linearard_amd.attention_KL import kl_backward, kl_forward, lse_stats

    rng = np.random.default_rng(T * 31 + ds + dt)
    qs, ks, qt, kt, mask = _inputs(rng, B, hq, hks, hkt, T, ds, dt, ratio)
    a_s, a_t = 1 / math.sqrt(ds), 1 / math.sqrt(dt)
    d = [to_dev(x, "f32") for x in (qs, ks, qt, kt)]
    m = mask_to_dev(mask)
    lse_s = lse_stats(d[0], d[1], m, causal, a_s)
    lse_t = lse_stats(d[2], d[3], m, causal, a_t)
    rls = O.lse_stats(qs, ks, mask, causal, a_s)
    rlt = O.lse_stats(qt, kt, mask, causal, a_t)
    np.testing.assert_allclose(lse_s.cpu().numpy(), rls, rtol=1e-6, atol=1e-5)
    np.testing.assert_allclose(lse_t.cpu().numpy(), rlt, rtol=1e-6, atol=1e-5)
    loss = float(kl_forward(d[0], d[1], lse_s, d[2], d[3], lse_t, m, causal, a_s, a_t))
    ref = O.kl_forward(qs, ks, rls, qt, kt, rlt, mask, causal, a_s, a_t)
    case = f"f32-stages-c{int(causal)}-r{ratio}-T{T}-ds{ds}-dt{dt}"
    check_loss(loss, ref, case, bar=F32_BAR)
    dq, dk = kl_backward(d[0], d[1], lse_s, d[2], d[3], lse_t, m, causal, a_s, a_t)
    rq, rk = O.kl_backward(qs, ks, rls, qt, kt, rlt, mask, causal, a_s, a_t)  # D exact (no cast)
    for name, got, want in (("dq", dq, rq), ("dk", dk, rk)):
        check_grad(got.cpu().numpy(), want, case, name, bar=F32_BAR)


@pytest.mark.parametrize("ratio", [None, 0.25])
def test_f32_autograd_self_relation_matches_the_oracle(gpu_available, ratio):
    from linearard_amd.attention_KL import attn_kl_align

    rng = np.random.default_rng(17)
    B, H, T, D = 1, 4, 300, 128
    xt = randn(rng, (B, H, T, D), "f32")
    xs = (xt + 0.1 * rng.standard_normal(xt.shape)).astype(np.float32)
    mask = None if ratio is None else make_mask(rng, B, T, ratio)
    a = 1 / math.sqrt(D)
    x = to_dev(xs, "f32", requires_grad=True)
    y = to_dev(xt, "f32")
    loss = attn_kl_align(x, x, y, y, attn_mask=mask_to_dev(mask), causal=True, sm_scale_s=a, sm_scale_t=a)
    loss.backward()
    ref, rdx, _, _, _ = O.attn_kl_align(xs, xs, xt, xt, mask, True, a, a, self_relation=True)
    check_loss(loss.item(), ref, f"f32-autograd-r{ratio}", bar=F32_BAR)
    assert x.grad.dtype == torch.float32
    check_grad(x.grad.cpu().numpy(), rdx, f"f32-autograd-r{ratio}", bar=F32_BAR)


@pytest.mark.parametrize("T", [15, 16, 17, 31, 33, 63, 64, 65, 129])
@pytest.mark.parametrize("ds,dt,scale", [(8, 8, 1.0), (32, 16, 1.0), (64, 64, 3.0), (64, 128, 1.0), (128, 128, 4.0),
                                         (256, 256, 1.0)])
def test_f32_tile_edges_match_the_oracle(gpu_available, T, ds, dt, scale):
    """Around the 16 rows of a wave, the 32 of a tile and the 64 of a
    workgroup, for every kernel width (32, 64, 128, 256) and for dims below
    it (padded with zeros); inputs of scale 3 and 4 have logits over 100, whose
    exponentials underflow.  Grouped queries, a mask with holes, and a
    self relation through autograd."""
    from linearard_amd.attention_KL import attn_kl_align, kl_backward, kl_forward, lse_stats

    rng = np.random.default_rng(T * 7 + ds + dt)
    for causal, ratio in ((True, None), (False, 0.3), (True, 0.3)):
        qs, ks, qt, kt, mask = _inputs(rng, 2, 4, 2, 4, T, ds, dt, ratio, scale)
        a_s, a_t = 1 / math.sqrt(ds), 1 / math.sqrt(dt)
        d = [to_dev(x, "f32") for x in (qs, ks, qt, kt)]
        m = mask_to_dev(mask)
        lse_s, lse_t = lse_stats(d[0], d[1], m, causal, a_s), lse_stats(d[2], d[3], m, causal, a_t)
        rls, rlt = O.lse_stats(qs, ks, mask, causal, a_s), O.lse_stats(qt, kt, mask, causal, a_t)
        # a float64 value rounded once to float32
        np.testing.assert_allclose(lse_s.cpu().numpy(), rls, rtol=2.0 ** -23, atol=1e-7)
        np.testing.assert_allclose(lse_t.cpu().numpy(), rlt, rtol=2.0 ** -23, atol=1e-7)
        case = f"f32-edges-c{int(causal)}-r{ratio}-T{T}-ds{ds}-dt{dt}"
        # the stages work from float32 LSEs, whose rounding (2^-24 of logits up
        # to 200) is a relative error of P up to 1.2e-5: twice that
        bar = 2.5e-5 if scale > 1 else F32_BAR
        loss = float(kl_forward(d[0], d[1], lse_s, d[2], d[3], lse_t, m, causal, a_s, a_t))
        check_loss(loss, O.kl_forward(qs, ks, rls, qt, kt, rlt, mask, causal, a_s, a_t), case, bar=bar)
        dq, dk = kl_backward(d[0], d[1], lse_s, d[2], d[3], lse_t, m, causal, a_s, a_t)
        rq, rk = O.kl_backward(qs, ks, rls, qt, kt, rlt, mask, causal, a_s, a_t)
        for name, got, want in (("dq", dq, rq), ("dk", dk, rk)):
            check_grad(got.cpu().numpy(), want, case, name, bar=bar)
        if ds == dt and scale == 1:  # the autograd pair keeps its LSEs in double
            x = to_dev(qs, "f32", requires_grad=True)
            loss = attn_kl_align(x, x, d[2], d[2], attn_mask=m, causal=causal, sm_scale_s=a_s, sm_scale_t=a_t)
            loss.backward()
            ref, rdx, _, _, _ = O.attn_kl_align(qs, qs, qt, qt, mask, causal, a_s, a_t, self_relation=True)
            check_loss(loss.item(), ref, case + "-autograd", bar=1e-6)
            check_grad(x.grad.cpu().numpy(), rdx, case + "-autograd", bar=1e-6)


def test_f32_cfg1_against_eager_pytorch(gpu_available):
    """BASELINE cfg1: B=1, H=32, n=1024, d=128, X_t ~ N(0,1) (seed 0),
    X_s = X_t + 0.1 N(0,1), scale 1/sqrt(d), causal; against float32 eager
    PyTorch with the n x n relation maps materialised (integration.py:102-127
    as a formula: sum over rows of KL(softmax(S_t) || softmax(S_s)))."""
    from linearard_amd.attention_KL import attn_kl_align

    g = torch.Generator().manual_seed(0)
    B, H, n, d = 1, 32, 1024, 128
    xt = torch.randn((B, H, n, d), generator=g)
    xs = xt + 0.1 * torch.randn((B, H, n, d), generator=g)
    a = 1 / math.sqrt(d)
    x = xs.cuda().requires_grad_(True)
    y = xt.cuda()
    loss = attn_kl_align(x, x, y, y, causal=True, sm_scale_s=a, sm_scale_t=a)
    loss.backward()

    xr = xs.cuda().requires_grad_(True)
    causal = torch.ones((n, n), dtype=torch.bool, device="cuda").tril()
    s_s = torch.matmul(xr, xr.transpose(-1, -2).contiguous()) * a
    s_t = torch.matmul(y, y.transpose(-1, -2).contiguous()) * a
    neg = torch.tensor(float("-inf"), device="cuda")
    ls = torch.log_softmax(torch.where(causal, s_s, neg), dim=-1)
    lt = torch.log_softmax(torch.where(causal, s_t, neg), dim=-1)
    pt = lt.exp()
    ref = torch.where(causal, pt * (lt - ls), torch.zeros((), device="cuda")).sum()
    ref.backward()
    # against the float64 oracle at the float32 bar
    rl, rdx, _, _, _ = O.attn_kl_align(xs.numpy(), xs.numpy(), xt.numpy(), xt.numpy(), None, True, a, a,
                                       self_relation=True)
    check_loss(loss.item(), rl, "f32-cfg1", bar=F32_BAR)
    check_grad(x.grad.cpu().numpy(), rdx, "f32-cfg1", bar=F32_BAR)
    # against float32 eager PyTorch, whose own float32 rounding is most of the
    # difference: the bar is F32_BAR or twice eager's deviation from float64
    eager_loss = abs(ref.item() - rl) / abs(rl)
    eager_grad = float(np.abs(xr.grad.cpu().numpy() - rdx).max() / np.abs(rdx).max())
    check_loss(loss.item(), ref.item(), "f32-cfg1-vs-eager-fp32", bar=max(F32_BAR, 2 * eager_loss))
    check_grad(x.grad.cpu().numpy(), xr.grad.cpu().numpy(), "f32-cfg1-vs-eager-fp32",
               bar=max(F32_BAR, 2 * eager_grad))


def test_f32_pair_equals_the_refining_backward(gpu_available):
    """Autograd (double LSEs kept from the forward) against
    lard_attn_kl_backward (which recomputes them): the same values bitwise,
    also in a second backward of one graph."""
    import ctypes

    from linearard_amd import _lib
    from linearard_amd.attention_KL import attn_kl_align

    rng = np.random.default_rng(5)
    B, H, T, D = 2, 3, 130, 64
    mask = mask_to_dev(make_mask(rng, B, T, 0.2))
    x = to_dev(randn(rng, (B, H, T, D), "f32"), "f32", requires_grad=True)
    y = to_dev(randn(rng, (B, H, T, D), "f32"), "f32")
    loss = attn_kl_align(x, x, y, y, attn_mask=mask, causal=True, sm_scale_s=0.1, sm_scale_t=0.1)
    first, = torch.autograd.grad(loss, [x], retain_graph=True)
    second, = torch.autograd.grad(loss, [x])
    assert torch.equal(first, second)
    L = _lib.lib()
    lse = [torch.zeros((B, H, T), device="cuda") for _ in range(2)]  # finite: only their finiteness is used
    dx = torch.empty_like(y)
    nb = L.lard_attn_kl_backward_workspace_bytes(B, H, H, T, D, 1)
    ws = torch.empty((nb,), device="cuda", dtype=torch.uint8)
    d = [ctypes.byref(_lib.tensor4(t)) for t in (x.detach(), y)]
    one = torch.ones((), device="cuda")
    rc = L.lard_attn_kl_backward(d[0], d[0], lse[0].data_ptr(), d[1], d[1], lse[1].data_ptr(),
                                 ctypes.byref(_lib.mask_desc(mask)), 1, 0.1, 0.1, one.data_ptr(), 1, None,
                                 dx.data_ptr(), ws.data_ptr(), nb, _lib.stream_of(y))
    assert rc == 0, L.lard_last_error()
    assert torch.equal(first, dx)


def test_f32_needs_f32_on_both_sides(gpu_available):
    from linearard_amd.attention_KL import attn_kl_align

    x = torch.zeros((1, 2, 8, 16), device="cuda")
    y = torch.zeros((1, 2, 8, 16), device="cuda", dtype=torch.bfloat16)
    with pytest.raises(AssertionError, match="float32 on both sides"):
        attn_kl_align(x, x, y, y)


@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("pad,bad", [(0, 0), (0, 2), (0, 5), (37, 38), (37, 40), (0, 33)])
def test_a_nan_score_takes_its_rows_out(gpu_available, causal, pad, bad):
    """A NaN key makes the LSE of every row that sees it -inf, also where it is
    the first or only score of a lane (lanes hold every fourth key); such rows
    leave the loss, and the others are those of the tokens before it."""
    from linearard_amd.attention_KL import attn_kl_align, lse_stats

    rng = np.random.default_rng(bad)
    B, H, T, D = 1, 2, 70, 64
    qs, ks, qt, kt, _ = _inputs(rng, B, H, H, H, T, D, D, None)
    mask = np.ones((B, T), np.int32)
    mask[:, :pad] = 0
    a = 1 / math.sqrt(D)
    seen = bad if causal else 0  # rows before `seen` do not see the key
    ref = O.lse_stats(qs[:, :, :seen], ks[:, :, :seen], mask[:, :seen], causal, a) if seen > pad else None
    for side in (0, 1):
        x = [to_dev(v, "f32") for v in (qs, ks, qt, kt)]
        x[2 * side + 1][:, :, bad] = float("nan")
        m = mask_to_dev(mask)
        lse = lse_stats(x[2 * side], x[2 * side + 1], m, causal, a).cpu().numpy()
        assert (lse[:, :, max(seen, pad):] == -np.inf).all()
        assert (lse[:, :, :pad] == 0).all()
        if side == 0 and ref is not None:
            np.testing.assert_allclose(lse[:, :, pad:seen], ref[:, :, pad:], rtol=1e-6, atol=1e-5)
        want = (float(attn_kl_align(*(v[:, :, :seen].contiguous() for v in x), attn_mask=m[:, :seen].contiguous(),
                                    causal=causal)) if seen > pad else 0.0)
        assert float(attn_kl_align(*x, attn_mask=m, causal=causal)) == pytest.approx(want, rel=1e-6, abs=0)


@pytest.mark.parametrize("value", [float("inf"), 1e30, 1e5])
def test_a_score_far_above_its_lse_overflows_to_infinity(gpu_available, value):
    """exp(S - lse) of a caller's LSE that does not cover S: inf, as in the
    oracle's formula, not NaN, in the row KL and in D."""
    from linearard_amd.attention_KL import kl_backward, kl_forward

    B, H, T, D, key = 1, 2, 40, 32, 9
    rng = np.random.default_rng(5)
    qs, ks, qt, kt = (to_dev(np.abs(rng.standard_normal((B, H, T, D))) + 0.1, "f32") for _ in range(4))
    kt[:, :, key, 0] = value
    lse = torch.zeros((B, H, T), device="cuda")
    # the row KL exceeds float32 (and double, for inf): p_t (l_t - l_s) = inf
    assert float(kl_forward(qs, ks, lse, qt, kt, lse, None, True, 1.0, 1.0)) == math.inf
    dq, dk = kl_backward(qs, ks, lse, qt, kt, lse, None, True, 1.0, 1.0)
    # D = p_s - p_t is -inf at this key for the rows that see it, finite elsewhere
    assert bool((dq[:, :, key:] == -math.inf).all()) and bool(torch.isfinite(dq[:, :, :key]).all())
    assert bool((dk[:, :, key] == -math.inf).all()) and bool(torch.isfinite(dk[:, :, key + 1:]).all())
