"""dk sums cut into parts (grouped queries on a grid below one workgroup per
CU): the autograd pair, the general backward and the stage entry point against
the float64 oracle, around the sizes where the cut changes, and the stage entry
point without a workspace (uncut) against the cut one."""

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
    for again in range(2):  # the autograd pair, then the general backward of the same graph
        dq, dk = torch.autograd.grad(two, d[:2], retain_graph=True)
        check_grad(dq.float().cpu().numpy(), 2.0 * rq, case + f"-{again}", "dq")
        check_grad(dk.float().cpu().numpy(), 2.0 * rk, case + f"-{again}", "dk")
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
