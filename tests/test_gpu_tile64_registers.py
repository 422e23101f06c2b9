"""The 64 x 64 GEMM tile staged through registers (about one tile per CU with a long K): K of one, two, three
and an odd number of 64-wide stages, partial row tiles, every epilogue; against float64 (bound: fp16 rounding of
result and branch, and the fp32 sum's)."""

import math

import pytest
import torch

from tttj_2026_amd import _lib, ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mode", ["bias", "gelu", "resid_masked", "masked_resid"])
@pytest.mark.parametrize("m,n,k", [(65, 64, 64), (130, 192, 128), (63, 128, 192), (200, 64, 832)])
def test_tile64_registers(m, n, k, mode):
    g = torch.Generator().manual_seed(k)
    x, w = torch.randn(m, k, generator=g).half(), (torch.randn(n, k, generator=g) / math.sqrt(k)).half()
    b, r = torch.randn(n, generator=g).half(), torch.randn(m, n, generator=g).half()
    valid = torch.rand(m, generator=g) > 0.3
    lib = _lib.load()
    _lib.check(lib.tt_gemm_tile_override(11), "override")
    try:
        y = ops.linear(x.cuda(), w.cuda(), b.cuda(), mode, residual=r.cuda() if "resid" in mode else None,
                       valid=valid.cuda()).cpu()
    finally:
        lib.tt_gemm_tile_override(-1)
    branch = x.double() @ w.double().t() + b.double()
    if mode == "gelu":
        branch = 0.5 * branch * (1 + torch.erf(branch / math.sqrt(2)))
    ref = branch + r.double() if "resid" in mode else branch
    err = (y.double() - ref).abs()
    assert bool((err <= 2.0 ** -11 * (ref.abs() + branch.abs()) + 2e-4)[valid].all())
    assert torch.equal(y[~valid], r[~valid] if mode == "resid_masked" else torch.zeros_like(y[~valid]))


@pytest.mark.parametrize("b,s,d,h", [(3, 100, 256, 4), (2, 72, 128, 1), (5, 16, 64, 2)])
def test_tile64_registers_qkv(b, s, d, h):
    g = torch.Generator().manual_seed(s)
    x, w = torch.randn(b, s, d, generator=g).half(), (torch.randn(3 * d, d, generator=g) / math.sqrt(d)).half()
    bias = torch.randn(3 * d, generator=g).half()
    lib = _lib.load()
    _lib.check(lib.tt_gemm_tile_override(11), "override")
    try:
        q, k, vt = ops.qkv_projection(x.cuda(), w.cuda(), bias.cuda(), h)
        torch.cuda.synchronize()
    finally:
        lib.tt_gemm_tile_override(-1)
    ref = (x.double().reshape(-1, d) @ w.double().t() + bias.double()).reshape(b, s, 3, h, d // h)
    for got, want in ((q, ref[:, :, 0].permute(0, 2, 1, 3)), (k, ref[:, :, 1].permute(0, 2, 1, 3)),
                      (vt[..., :s], ref[:, :, 2].permute(0, 2, 3, 1))):
        assert bool(((got.cpu().double() - want).abs() <= 2.0 ** -10 * want.abs() + 2e-4).all())
