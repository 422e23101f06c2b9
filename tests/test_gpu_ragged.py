"""GEMMs whose N or K is a multiple of 8 but not of 64, on every kernel the ragged rule picks: the narrow
tiles (4 and 8 waves), 64 x 64 and 128 x 128, at tile edges and K remainders, against a float64 product.

Bound: operands are fp16, products are exact in fp32 and summed in fp32, so an output differs from the
float64 value by the fp32 sum's rounding (K 2^-24 sum |x w|, below 1e-4 here) and one or two fp16 roundings
(2^-11 of the value and of the branch added to a residual)."""

import math

import pytest
import torch

from tttj_2026_amd import ops

pytestmark = pytest.mark.gpu

SHAPES = [
    (33, 72, 8),        # narrow, one K chunk; last row and column tiles partial
    (200, 40, 264),     # narrow, K % 16 == 8
    (100, 160, 1032),   # narrow on 8 waves
    (64, 64, 72),       # N whole, K ragged
    (2100, 488, 200),   # 64 x 64
    (4099, 1096, 136),  # 128 x 128
    (3000, 64, 1000),   # 64 x 64, N whole
]


def _rand(shape, seed, scale=1.0):
    g = torch.Generator().manual_seed(seed)
    return (torch.randn(*shape, generator=g) * scale).half().cuda()


def _close(got, ref, branch):
    bound = 2.0 ** -11 * (ref.abs() + branch.abs()) + 1e-4
    assert bool(((got.cpu().double() - ref).abs() <= bound).all())


@pytest.mark.parametrize("mode", ["bias", "gelu", "resid_masked", "masked_resid"])
@pytest.mark.parametrize("m,n,k", SHAPES)
def test_ragged_linear(mode, m, n, k):
    x, w, b = _rand((m, k), 1), _rand((n, k), 2, 1 / math.sqrt(k)), _rand((n,), 3, 0.5)
    r = _rand((m, n), 4)
    valid = torch.rand(m, generator=torch.Generator().manual_seed(5)) > 0.3
    x[1] = float("nan")  # a row's K remainder must not read into its neighbour's row
    x[m - 2] = float("inf")
    bad = torch.zeros(m, dtype=torch.bool)
    bad[1] = bad[m - 2] = True
    branch = x.cpu().double() @ w.cpu().double().t() + b.cpu().double()
    if mode == "gelu":
        branch = 0.5 * branch * (1 + torch.erf(branch / math.sqrt(2)))
    y = ops.linear(x, w, b, mode, residual=r if "resid" in mode else None, valid=valid.cuda()).cpu()
    ref = branch + r.cpu().double() if "resid" in mode else branch
    keep = valid & ~bad
    _close(y[keep], ref[keep], branch[keep])
    want = r.cpu()[~valid] if mode == "resid_masked" else torch.zeros_like(y[~valid])
    assert torch.equal(y[~valid], want)
    assert not torch.isfinite(y[valid & bad]).any() or not (valid & bad).any()


@pytest.mark.parametrize("b,s,d,h", [(2, 33, 40, 5), (3, 100, 96, 3), (5, 333, 160, 5), (4, 520, 264, 33),
                                     (9, 512, 480, 15)])
def test_ragged_qkv(b, s, d, h):
    x, w, bias = _rand((b, s, d), 1), _rand((3 * d, d), 2, 1 / math.sqrt(d)), _rand((3 * d,), 3, 0.5)
    q, k, vt = ops.qkv_projection(x, w, bias, h)
    ref = (x.cpu().double().reshape(-1, d) @ w.cpu().double().t() + bias.cpu().double()).reshape(b, s, 3, h, d // h)
    for got, want in ((q, ref[:, :, 0].permute(0, 2, 1, 3)), (k, ref[:, :, 1].permute(0, 2, 1, 3)),
                      (vt[..., :s], ref[:, :, 2].permute(0, 2, 3, 1))):
        _close(got, want, want)


@pytest.mark.parametrize("masked", [False, True])
@pytest.mark.parametrize("b,s,d,h", [(2, 33, 40, 10), (9, 520, 40, 10), (5, 333, 96, 8), (9, 512, 480, 40),
                                     (4, 520, 192, 16), (8, 1024, 192, 16), (16, 1024, 256, 64)])
def test_qkv_heads_off_eight(b, s, d, h, masked):
    """Head widths that are a multiple of 4 but not of 8 (4, 12), at row counts and widths of every tile;
    with a mask, whole tiles of padded rows among them."""
    x, w, bias = _rand((b, s, d), 1), _rand((3 * d, d), 2, 1 / math.sqrt(d)), _rand((3 * d,), 3, 0.5)
    valid = None
    if masked:
        valid = torch.rand(b, s, generator=torch.Generator().manual_seed(6)) > 0.3
        valid[1] = False
    q, k, vt = ops.qkv_projection(x, w, bias, h, None if valid is None else valid.cuda())
    ref = x.cpu().double().reshape(-1, d) @ w.cpu().double().t() + bias.cpu().double()
    if masked:
        ref[~valid.reshape(-1)] = 0
    ref = ref.reshape(b, s, 3, h, d // h)
    for got, want in ((q, ref[:, :, 0].permute(0, 2, 1, 3)), (k, ref[:, :, 1].permute(0, 2, 1, 3)),
                      (vt[..., :s], ref[:, :, 2].permute(0, 2, 3, 1))):
        _close(got, want, want)
