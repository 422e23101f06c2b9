"""Attention whose key tiles are shared by two groups of waves (small grids of at least 16 key tiles), against
float64: odd tile counts, a partial last tile in either group, sequences so short that the second group has no
tile, empty sequences, every mask kind.

Bound: probabilities are rounded to fp16 (2^-11 of each), the result is rounded to fp16, and Q times the
softmax factor is rounded to fp16 on load, which moves a score by up to 2^-11 sum_i |q_i k_i| hd^-1/2 <= 3.5e-3
for unit-variance inputs at head_dim 128; together below 5e-3 of what is summed."""

import pytest
import torch

from tttj_2026_amd import _lib, ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("hd", [32, 64, 128])
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("mask_kind", ["none", "prefix", "scattered"])
@pytest.mark.parametrize("s", [1024, 1030, 1100])
def test_split_attention(hd, causal, mask_kind, s):
    b, h = 4, 2
    g = torch.Generator().manual_seed(s + hd)
    q, k = (torch.randn(b, h, s, hd, generator=g).half() for _ in range(2))
    vt = torch.full((b, h, hd, (s + 63) // 64 * 64), float("nan"), dtype=torch.float16)
    vt[..., :s] = torch.randn(b, h, hd, s, generator=g).half()
    mask = None
    if mask_kind == "prefix":
        mask = torch.arange(s)[None, :] < torch.tensor([s, 40, 0, 700])[:, None]
    elif mask_kind == "scattered":
        mask = torch.rand(b, s, generator=g) > 0.4
        mask[1, 64:] = False
        mask[2] = False
        mask[3, :128] = False  # both groups' first tiles without a valid key
    args = (q.cuda(), k.cuda(), vt.cuda(), None if mask is None else mask.cuda(), causal)
    y = ops.attention(*args).cpu()
    assert torch.equal(y, ops.attention(*args).cpu())
    sc = torch.matmul(q.double(), k.double().transpose(-1, -2).contiguous()) * hd ** -0.5
    if causal:
        sc = sc.masked_fill(torch.ones(s, s, dtype=torch.bool).triu(1), float("-inf"))
    if mask is not None:
        sc = sc.masked_fill(~mask[:, None, None, :], float("-inf"))
    p = torch.softmax(sc, -1).nan_to_num(0.0)
    v = vt[..., :s].double().transpose(-1, -2).contiguous()
    ref = torch.matmul(p, v).permute(0, 2, 1, 3).reshape(b, s, h * hd)
    mag = torch.matmul(p, v.abs()).permute(0, 2, 1, 3).reshape(b, s, h * hd)
    if mask is not None:
        ref[~mask] = 0
        assert not y.view(torch.int16)[~mask].any()
    assert bool(((y.double() - ref).abs() <= 5e-3 * mag + 1e-6).all())


@pytest.mark.parametrize("hd", [8, 16, 32, 64, 128, 256])
@pytest.mark.parametrize("s", [1, 77, 1024, 1500])
def test_own_mask_summary(hd, s):
    """A masked call whose blocks summarise the mask themselves equals the call with tt_mask_info's summary bit
    for bit (16-byte and byte-wise scans, empty, prefix and scattered masks)."""
    b, h = 4, 1
    g = torch.Generator().manual_seed(s)
    q, k = (torch.randn(b, h, s, hd, generator=g).half().cuda() for _ in range(2))
    vt = torch.randn(b, h, hd, (s + 63) // 64 * 64, generator=g).half().cuda()
    mask = torch.rand(b, s, generator=g) > 0.4
    mask[1] = torch.arange(s) < (s + 1) // 2
    mask[2] = False
    mask[3] = True
    mask = mask.cuda()
    y = ops.attention(q, k, vt, mask, True)
    info = ops.mask_info(mask, b, s, q.device)
    z = torch.full_like(y, float("nan"))
    rc = _lib.load().tt_attention_fwd(q.data_ptr(), k.data_ptr(), vt.data_ptr(), mask.data_ptr(), info.data_ptr(),
                                      z.data_ptr(), b, s, h, hd, 1, torch.cuda.current_stream().cuda_stream)
    _lib.check(rc, "tt_attention_fwd")
    assert torch.equal(y, z)
