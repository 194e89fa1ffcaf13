"""The stage kernels' tile ring at its edges: fewer tiles than ring buffers,
whole and partial last tiles, one and several workgroups, every dim pair with
instances of its own (equal dims and one type) and the general ones (Ds != Dt,
mixed types), and validity bits beyond one window of 32768 tokens.  Against the
float64 oracle, with the bars of tests/_tolerance.py."""

import math

import numpy as np
import pytest
import torch

from oracle import attn_kl as O
from tests._inputs import make_mask, mask_to_dev, randn, to_dev
from tests._tolerance import check_grad, check_loss

pytestmark = pytest.mark.gpu


def _check(seed, B, hq, hks, hkt, T, ds, dt, dts, dtt, causal, ratio):
    from linearard_amd.attention_KL import kl_backward, kl_forward, lse_stats

    rng = np.random.default_rng(seed)
    qs, ks = randn(rng, (B, hq, T, ds), dts), randn(rng, (B, hks, T, ds), dts)
    qt, kt = randn(rng, (B, hq, T, dt), dtt), randn(rng, (B, hkt, T, dt), dtt)
    mask = None if ratio is None else make_mask(rng, B, T, ratio)
    a_s, a_t = 1 / math.sqrt(ds), 1 / math.sqrt(dt)
    d = [to_dev(qs, dts), to_dev(ks, dts), to_dev(qt, dtt), to_dev(kt, dtt)]
    m = mask_to_dev(mask)
    lse_s, lse_t = lse_stats(d[0], d[1], m, causal, a_s), lse_stats(d[2], d[3], m, causal, a_t)
    rls, rlt = O.lse_stats(qs, ks, mask, causal, a_s), O.lse_stats(qt, kt, mask, causal, a_t)
    # float32 sums of up to T exponentials: 1e-5 absolute on values below 30
    np.testing.assert_allclose(lse_s.cpu().numpy(), rls, rtol=1e-6, atol=1e-5)
    np.testing.assert_allclose(lse_t.cpu().numpy(), rlt, rtol=1e-6, atol=1e-5)
    case = f"ring-{dts}-{dtt}-{B}-{hq}-{hks}-{hkt}-{T}-{ds}-{dt}-c{int(causal)}-r{ratio}"
    check_loss(float(kl_forward(d[0], d[1], lse_s, d[2], d[3], lse_t, m, causal, a_s, a_t)),
               O.kl_forward(qs, ks, rls, qt, kt, rlt, mask, causal, a_s, a_t), case)
    dq, dk = kl_backward(d[0], d[1], lse_s, d[2], d[3], lse_t, m, causal, a_s, a_t)
    rq, rk = O.kl_backward(qs, ks, rls, qt, kt, rlt, mask, causal, a_s, a_t, d_cast=dts)
    check_grad(dq.cpu().numpy(), rq, case, "dq")
    check_grad(dk.cpu().numpy(), rk, case, "dk")


@pytest.mark.parametrize("T", [2, 31, 32, 33, 64, 65, 96, 97, 127, 129, 161])
@pytest.mark.parametrize("ds,dt", [(8, 8), (16, 16), (32, 32), (64, 64), (128, 128), (256, 256), (64, 128), (256, 32)])
def test_tiles_and_dims(gpu_available, T, ds, dt):
    _check(T + ds, 1, 2, 2, 2, T, ds, dt, "bf16", "bf16", True, None)
    _check(T + dt, 2, 4, 2, 1, T, ds, dt, "f16", "f16", False, 0.3)


@pytest.mark.parametrize("dts,dtt", [("bf16", "f16"), ("f16", "bf16")])
@pytest.mark.parametrize("ds,dt", [(128, 128), (64, 256), (256, 256)])
def test_mixed_types(gpu_available, dts, dtt, ds, dt):
    _check(7, 1, 4, 2, 4, 130, ds, dt, dts, dtt, True, 0.2)


@pytest.mark.parametrize("D", [16, 64])
def test_validity_bits_of_a_second_window(gpu_available, D):
    """One masked head of 32768 + 200 tokens, almost all of them masked: the
    stages on the whole sequence equal the stages on the kept tokens alone
    (masked tokens take no part), bitwise in dq and dk rows up to the order of
    the sums: 1e-3 of the largest.  D = 64 refills the bits with tiles in
    flight, D = 16 with none."""
    from linearard_amd.attention_KL import kl_backward, kl_forward, lse_stats

    T, n = 32768 + 200, 300
    g = torch.Generator(device="cuda").manual_seed(3)
    keep = torch.cat([torch.randperm(32768, generator=g, device="cuda")[: n - 60],
                      32768 + torch.randperm(200, generator=g, device="cuda")[:60]]).sort().values
    mask = torch.zeros((1, T), dtype=torch.bool, device="cuda")
    mask[0, keep] = True
    x = torch.randn((1, 1, T, D), generator=g, device="cuda").to(torch.float16)
    y = torch.randn((1, 1, T, D), generator=g, device="cuda").to(torch.float16)
    xc, yc = x[:, :, keep].contiguous(), y[:, :, keep].contiguous()
    for causal in (True, False):
        out = []
        for s, t, m in ((x, y, mask), (xc, yc, None)):
            ls, lt = lse_stats(s, s, m, causal, 0.25), lse_stats(t, t, m, causal, 0.25)
            out.append((ls, lt, kl_forward(s, s, ls, t, t, lt, m, causal, 0.25, 0.25),
                        *kl_backward(s, s, ls, t, t, lt, m, causal, 0.25, 0.25)))
        a, b = out
        for i in (0, 1):
            assert float((a[i][:, :, keep] - b[i]).abs().max()) <= 1e-5
            assert float(a[i][:, :, ~mask[0]].abs().max()) == 0.0  # masked rows
        assert abs(float(a[2]) - float(b[2])) <= 1e-5 * abs(float(b[2]))
        for i in (3, 4):
            assert float((a[i][:, :, keep] - b[i]).abs().max()) <= 1e-3 * float(b[i].abs().max())
            assert float(a[i][:, :, ~mask[0]].abs().max()) == 0.0


def test_validity_bits_of_a_second_window_256_wide(gpu_available):
    """The same for the 256-wide autograd pair (its forward refills the bits of
    its own ring): loss and gradient of the kept tokens, to the bars."""
    from linearard_amd.attention_KL import attn_kl_align

    T, D, n = 32768 + 200, 256, 300
    g = torch.Generator(device="cuda").manual_seed(4)
    keep = torch.cat([torch.randperm(32768, generator=g, device="cuda")[: n - 60],
                      32768 + torch.randperm(200, generator=g, device="cuda")[:60]]).sort().values
    mask = torch.zeros((1, T), dtype=torch.bool, device="cuda")
    mask[0, keep] = True
    y = torch.randn((1, 1, T, D), generator=g, device="cuda").to(torch.float16)
    x = (y.float() + 0.3 * torch.randn(y.shape, generator=g, device="cuda")).to(torch.float16)
    for causal in (True, False):
        out = []
        for s, t, m in ((x, y, mask), (x[:, :, keep].contiguous(), y[:, :, keep].contiguous(), None)):
            s = s.clone().requires_grad_(True)
            loss = attn_kl_align(s, s, t, t, attn_mask=m, causal=causal, sm_scale_s=0.02, sm_scale_t=0.02)
            out.append((float(loss.detach()), *torch.autograd.grad(loss, [s])))
        case = f"window-256-c{int(causal)}"
        check_loss(out[0][0], out[1][0], case)
        check_grad(out[0][1][:, :, keep].float().cpu().numpy(), out[1][1].float().cpu().numpy(), case)
        assert float(out[0][1][:, :, ~mask[0]].abs().max()) == 0.0


@pytest.mark.parametrize("dtype", ["bf16", "f16"])
@pytest.mark.parametrize("ds,dt", [(8, 8), (8, 64), (64, 8)])
def test_an_infinite_key_element_does_not_reach_the_padding(gpu_available, dtype, ds, dt):
    """D = 8 runs in tiles of 16 dims: an infinite key element against queries
    of the other sign scores -inf (its weight is 0 in the LSE, and the KL with a
    student's is +inf), not NaN from the padding's zeros."""
    from linearard_amd.attention_KL import kl_forward, lse_stats

    rng = np.random.default_rng(ds + dt)
    B, H, T, key = 1, 2, 70, 40
    x = [randn(rng, (B, H, T, d), dtype) for d in (ds, ds, dt, dt)]
    m = np.ones((B, T), np.int32)
    m[:, key] = 0  # the oracle: without that key (and its row)
    rows = np.arange(T) != key
    for side, d in ((0, ds), (1, dt)):
        q, k = x[2 * side].copy(), x[2 * side + 1].copy()
        q[..., 0] = -1.0
        ref = O.lse_stats(q, k, m, False, 0.3)
        k[:, :, key, 0] = np.inf
        got = lse_stats(to_dev(q, dtype), to_dev(k, dtype), None, False, 0.3).cpu().numpy()
        np.testing.assert_allclose(got[:, :, rows], ref[:, :, rows], rtol=1e-6, atol=1e-5)
        if side == 0:
            y = [to_dev(v, dtype) for v in (q, k, x[2], x[3])]
            ls, lt = (lse_stats(y[2 * i], y[2 * i + 1], None, False, 0.3) for i in (0, 1))
            assert float(kl_forward(y[0], y[1], ls, y[2], y[3], lt, None, False, 0.3, 0.3)) == math.inf
