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
