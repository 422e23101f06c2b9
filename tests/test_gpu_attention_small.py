"""Attention at head_dim 8 and 16 against float64, at the edges of its 16-key and 16-query tiles, 64-key
steps and 128-query blocks.  Probabilities carry 22 bits, so beside the fp16 rounding of the result
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


@pytest.mark.parametrize("hd", [8, 16])
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("prefix", [False, True])
def test_small_head_attention_infinite_values(hd, causal, prefix):
    """An infinite V makes its feature infinite for every query that gives its key weight, the row's largest
    weight among them, and leaves all else alone: the other features, the query tiles that come before its key,
    and, at keys past the last valid one's tile, everything."""
    b, h, s, end = 2, 2, 150, 101 if prefix else 150
    g = torch.Generator().manual_seed(3)
    q, k = (torch.randn(b, h, s, hd, generator=g).half() for _ in range(2))
    vt = torch.zeros(b, h, hd, 192, dtype=torch.float16)
    vt[..., :s] = torch.randn(b, h, hd, s, generator=g).half()
    at = [(0, 0, 1.0), (1, 37, -1.0), (2, 64, 1.0), (3, 90, -1.0)]  # feature, key, sign
    k[:, :, 37] = q[:, :, 120] * 3  # the largest weight of query 120, of 37 and of others
    k[:, :, 0] = q[:, :, 37] * 3
    clean = vt.clone()
    for d, key, sign in at:
        vt[:, :, d, key] = sign * float("inf")
        clean[:, :, d, key] = 0
    if prefix:
        vt[..., (end + 15) // 16 * 16:] = float("nan")
    mask = (torch.arange(s) < end).expand(b, s).contiguous().cuda() if prefix else None
    run = lambda v: ops.attention(q.cuda(), k.cuda(), v.cuda(), mask, causal).cpu().view(b, s, h, hd)
    y, want = run(vt), run(clean)
    # both within an fp16 rounding and 3e-5 of values of magnitude 8 at most (as above) of the true ones
    near = lambda a, b: bool(((a - b).abs().double() <= 2.0 ** -10 * b.abs().double() + 5e-4).all())
    for d, key, sign in at:
        first = key if causal else 0
        assert (y[:, first:end, :, d] == sign * float("inf")).all(), (d, key)
        if causal:
            assert near(y[:, :key // 16 * 16, :, d], want[:, :key // 16 * 16, :, d])
    assert near(y[..., len(at):], want[..., len(at):])
    assert not y[:, end:].any()
