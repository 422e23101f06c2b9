"""Attention at head_dim 8 and 16 against float64, at the edges of its 16-key and 16-query tiles, 64-key
steps and 128-query blocks.  Probabilities carry fp32 precision, so beside the fp16 rounding of the result
(2^-11) an output may only differ by fp32-sized errors of the scores: their rounding, up to 2^-22 of a
score of magnitude c (c <= 60 here), is a relative error of c 2^-22 ln 2 of a probability."""

import pytest
import torch

from tttj_2026_amd import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("hd", [8, 16])
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("mask_kind", ["none", "prefix", "scattered"])
@pytest.mark.parametrize("s,scale", [(1, 1.0), (17, 1.0), (63, 3.0), (65, 1.0), (129, 3.0), (300, 1.0)])
def test_small_head_attention(hd, causal, mask_kind, s, scale):
    b, h = 3, 2
    g = torch.Generator().manual_seed(s)
    q, k = ((torch.randn(b, h, s, hd, generator=g) * scale).half() for _ in range(2))
    vt = torch.full((b, h, hd, (s + 63) // 64 * 64), float("nan"), dtype=torch.float16)
    vt[..., :s] = torch.randn(b, h, hd, s, generator=g).half()
    mask = None
    if mask_kind == "prefix":
        mask = torch.arange(s)[None, :] < torch.tensor([s, max(1, s // 2), 0])[:, None]
    elif mask_kind == "scattered":
        mask = torch.rand(b, s, generator=g) > 0.4
    y = ops.attention(q.cuda(), k.cuda(), vt.cuda(), None if mask is None else mask.cuda(), causal).cpu()
    sc = torch.matmul(q.double(), k.double().transpose(-1, -2).contiguous()) * hd ** -0.5
    if causal:
        sc = sc.masked_fill(torch.ones(s, s, dtype=torch.bool).triu(1), float("-inf"))
    if mask is not None:
        sc = sc.masked_fill(~mask[:, None, None, :], float("-inf"))
    p = torch.softmax(sc, -1).nan_to_num(0.0)
    v = vt[..., :s].double().transpose(-1, -2).contiguous()
    ref = torch.matmul(p, v).permute(0, 2, 1, 3).reshape(b, s, h * hd)
    mag = torch.matmul(p, v.abs()).permute(0, 2, 1, 3).reshape(b, s, h * hd)  # of what is summed
    if mask is not None:
        ref[~mask] = 0
        assert not y.view(torch.int16)[~mask].any()
    assert bool(((y.double() - ref).abs() <= 2.0 ** -11 * ref.abs() + 3e-5 * mag + 1e-7).all())
