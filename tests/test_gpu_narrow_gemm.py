"""The narrow GEMM's dealing of 64-wide K slices to waves, two in flight: fewer slices than waves, uneven
shares, more than two per wave, on 4 and on 8 waves, with partial row tiles; against float64 (bound: fp16
rounding of the result and the fp32 sum's, K 2^-24 sum |x w| < 2e-4)."""

import math

import pytest
import torch

from tttj_2026_amd import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,n,k", [(33, 64, 64), (5, 128, 192), (64, 64, 320), (40, 192, 512),   # 4 waves
                                   (31, 64, 576), (64, 128, 1088), (7, 64, 2624), (65, 64, 4096)])  # 8 waves
def test_narrow_slices(m, n, k):
    g = torch.Generator().manual_seed(k)
    x, w = torch.randn(m, k, generator=g).half(), (torch.randn(n, k, generator=g) / math.sqrt(k)).half()
    b, r = torch.randn(n, generator=g).half(), torch.randn(m, n, generator=g).half()
    branch = x.double() @ w.double().t() + b.double()
    y = ops.linear(x.cuda(), w.cuda(), b.cuda(), "masked_resid", residual=r.cuda()).cpu().double()
    ref = branch + r.double()
    assert bool(((y - ref).abs() <= 2.0 ** -11 * (ref.abs() + branch.abs()) + 2e-4).all())


@pytest.mark.parametrize("m,n,k", [(40, 64, 128), (40, 192, 1024), (33, 72, 40), (5, 40, 1032), (4000, 72, 136)])
@pytest.mark.parametrize("mode", ["bias", "resid_masked"])
def test_operands_at_any_offset(device, m, n, k, mode):
    """Contiguous operands that start at any fp16 value of a buffer give what aligned ones give, bit for bit where
    both run on narrow tiles."""
    g = torch.Generator().manual_seed(1)
    at = {name: (torch.randn(*s, generator=g) * c).half().to(device)
          for name, s, c in (("x", (m, k), 1), ("w", (n, k), k ** -0.5), ("b", (n,), 1), ("r", (m, n), 1))}
    off = {}
    for i, (name, t) in enumerate(at.items()):
        buf = torch.empty(t.numel() + 8, dtype=t.dtype, device=device)
        off[name] = buf[1 + 2 * i:1 + 2 * i + t.numel()].view(t.shape).copy_(t)
        assert off[name].is_contiguous() and off[name].data_ptr() % 16 != 0
    y, want = (ops.linear(t["x"], t["w"], t["b"], mode, residual=t["r"] if mode != "bias" else None) for t in (off, at))
    if m < 100:
        assert torch.equal(y, want)
    else:  # sums of k products in another order
        assert bool(((y - want).abs().double() <= 2.0 ** -10 * want.abs().double() + 1e-4).all())
