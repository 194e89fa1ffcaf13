"""Descriptors handed to the library and the loss weights, built on the host."""

import ctypes

import pytest
import torch

from linearard_amd import _lib
from linearard_amd.attention_KL.batched import denominators


@pytest.mark.parametrize("permuted", [False, True])
def test_descriptors(permuted):
    x = torch.zeros(2, 3, 5, 16, dtype=torch.bfloat16)
    y = torch.zeros(2, 3, 5, 16, dtype=torch.float16)
    if permuted:
        x, y = x.permute(0, 2, 1, 3), y[:, ::2]
    for t in (x, y):
        d = _lib.tensor4(t)
        assert (d.data, tuple(d.size), tuple(d.stride), d.dtype) == (
            t.data_ptr(), tuple(t.shape), t.stride(), _lib.DTYPE_CODES[t.dtype])
    rels = _lib.relations([x, y], [y, x], [11, 12], [21, 22])
    assert len(rels) == 2 and ctypes.sizeof(rels) == 2 * ctypes.sizeof(_lib.Relation)
    for r, (s, t) in enumerate([(x, y), (y, x)]):
        assert (rels[r].xs.data, rels[r].xt.data) == (s.data_ptr(), t.data_ptr())
        assert tuple(rels[r].xt.stride) == t.stride() and rels[r].xs.dtype == _lib.DTYPE_CODES[s.dtype]
        assert (rels[r].lse_s, rels[r].lse_t, rels[r].dxs) == (11 + r, 21 + r, None)
    assert _lib.relations([x], [y], [1], [2], [3])[0].dxs == 3
    for m in (None, torch.ones(2, 7, dtype=torch.int64), torch.ones(4, 7, dtype=torch.bool)[::2]):
        d = _lib.mask_desc(m)
        want = (None, 0, (0, 0), (0, 0)) if m is None else (m.data_ptr(), _lib.MASK_CODES[m.dtype], tuple(m.shape),
                                                            m.stride())
        assert (d.data, d.kind, tuple(d.size), tuple(d.stride)) == want
    z = torch.zeros(3, 4, 9)[:, :, :7]
    d = _lib.logits_desc(z)
    assert (d.data, tuple(d.size), tuple(d.stride), d.dtype) == (z.data_ptr(), (3, 4, 7), (36, 9, 1), 2)
    assert tuple(_lib.logits_desc(z[1]).size) == (1, 4, 7)


@pytest.mark.parametrize("sizes", [(0, 0), (1, 1), (64, 64), (65, 3, 130)])
def test_stat_buffer(sizes):
    """Disjoint arrays inside the buffer, 256-byte steps, found again from it."""
    buf, at = _lib.stat_buffer(sizes, "cpu")
    assert at == _lib.stat_addresses(buf, sizes) and at[0] == buf.data_ptr()
    ends = at[1:] + [buf.data_ptr() + 4 * buf.numel()]
    assert all((a - at[0]) % 256 == 0 and a + 4 * n <= e for a, n, e in zip(at, sizes, ends))


@pytest.mark.parametrize("heads", [[4, 4, 4], [4, 8, 4]])
@pytest.mark.parametrize("mask", [None, "ones", "zeros"])
def test_denominators(heads, mask):
    qs = [torch.zeros(2, h, 5, 8) for h in heads]
    m = None if mask is None else torch.full((2, 5), int(mask == "ones"), dtype=torch.int64)
    got = denominators(qs, m, "cpu", 3, lambda d: 1.0 / (d * 3))
    want = []
    for h in heads:
        d = torch.tensor(float(2 * h * 5)) if m is None else m.sum().clamp_min(1).to(torch.float32) * h
        want += [1.0 / (d * 3)] * 3
    assert got.dtype == torch.float32 and torch.equal(got, torch.stack(want))
