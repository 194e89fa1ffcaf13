"""The order in which causal work is dealt to the XCDs and CUs (ring.h causal_item)."""

import os
import shutil
import subprocess

import pytest
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = r"""
#include "ring.h"
#include <cstdio>
#include <vector>
int main() {
  for (int wgs = 1; wgs <= 4; ++wgs)
    for (int heads = 1; heads <= 70; ++heads)
      for (int nblk = 1; nblk <= 140; nblk += nblk < 40 ? 1 : 7) {
        const int n = heads * nblk;
        std::vector<char> seen(n, 0);
        for (int b = 0; b < n; ++b) {
          const int i = lard::causal_item(b, n, nblk, wgs);
          if (i < 0 || i >= n || seen[i]) {
            std::printf("wgs %d heads %d blocks %d: workgroup %d -> %d\n", wgs, heads, nblk, b, i);
            return 1;
          }
          seen[i] = 1;
        }
      }
  return 0;
}
"""


def test_every_item_is_dealt_once(tmp_path):
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(hipcc):
        pytest.skip("no hipcc")
    src, exe = tmp_path / "order.hip", tmp_path / "order"
    src.write_text(PROGRAM)
    subprocess.run([hipcc, "--offload-arch=gfx950", "-O1", "-std=c++17", "-Xclang", "-target-feature", "-Xclang",
                    "-packed-fp32-ops", "-I", os.path.join(ROOT, "linearard_amd", "csrc"), str(src), "-o", str(exe)],
                   check=True, capture_output=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True)
    assert out.returncode == 0, out.stdout


@pytest.mark.gpu
@pytest.mark.parametrize("B,H,T,D", [(1, 5, 1300, 128), (1, 12, 700, 64), (2, 10, 520, 256), (1, 33, 400, 128)])
def test_heads_do_not_depend_on_their_place(gpu_available, B, H, T, D):
    """Each head's gradient in a call of many equals its gradient in a call of
    its own: the same kernels and sums, only the order of the work differs
    (the loss is a sum over heads, so dloss is 1 in both)."""
    from linearard_amd.attention_KL import attn_kl_align

    g = torch.Generator(device="cuda").manual_seed(H * T)
    xs = (torch.randn(B, H, T, D, device="cuda", generator=g) * 0.7).to(torch.float16)
    xt = (xs.float() + 0.2 * torch.randn(xs.shape, device="cuda", generator=g)).to(torch.float16)

    def grad(s, t):
        s = s.contiguous().requires_grad_(True)
        t = t.contiguous()
        return torch.autograd.grad(attn_kl_align(s, s, t, t, causal=True), [s])[0]

    whole = grad(xs.clone(), xt)
    for h in range(H):
        assert torch.equal(whole[:, h:h + 1], grad(xs[:, h:h + 1].clone(), xt[:, h:h + 1])), h
