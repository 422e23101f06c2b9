"""Whole forwards of models whose widths are no multiple of 64 and which the row chain does not take: few tokens
(the LayerNorms folded into the narrow ragged GEMM tiles, with statistics slots of 32 or 8 columns) and padded
batches of many (packed variable-length rows on the ragged MFMA tiles).  The gate is the forward's own (2e-2
max, 2e-3 mean against the fp32 oracle, padded rows +0.0, two calls bit-identical)."""

import copy

import pytest
import torch

from oracle import transformer_oracle as O
from tttj_2026_amd import PLAN_LAYERWISE, _lib, make_optimized_transformer
from tttj_2026_amd.configs import build_model, make_inputs
from tttj_2026_amd.model import TransformerConfig

pytestmark = pytest.mark.gpu


def _model(cfg, device, seed):
    model = build_model(cfg, seed=seed)
    g = torch.Generator().manual_seed(seed + 1)
    with torch.no_grad():
        for name, p in model.named_parameters():
            if "norm" in name:
                p.add_(0.25 * torch.randn(p.shape, generator=g))
    return model.half().to(device).eval()


def _mask(kind, b, s, seed):
    g = torch.Generator().manual_seed(seed)
    if kind == "none":
        return None
    if kind == "prefix":
        lens = torch.randint(1, s + 1, (b,), generator=g)
        lens[0] = s
        if b > 2:
            lens[1] = 0
        return torch.arange(s)[None, :] < lens[:, None]
    m = torch.rand(b, s, generator=g) > 0.35
    m[b // 2] = False
    return m


def _inputs(cfg, kind, seed):
    x16, _ = make_inputs(cfg, False, seed)
    mask = _mask(kind, cfg.batch_size, cfg.seq_len, seed + 1)
    return (x16 if mask is None else x16.masked_fill(~mask[..., None], 0)), mask


@pytest.mark.parametrize("kind", ["none", "prefix", "scattered"])
@pytest.mark.parametrize("b,s,d,h,f,layers,scale", [
    (2, 24, 8, 1, 16, 2, 1.0),        # one statistics slot
    (1, 16, 40, 5, 80, 3, 1.0),       # five slots of 8 columns
    (2, 33, 72, 9, 144, 2, 30.0),     # nine: more than the eight lanes of a row, partial row tiles
    (3, 20, 200, 25, 400, 3, 1.0),    # 25 slots, K of eight waves in the ffn_out
    (1, 100, 224, 7, 448, 3, 30.0),   # seven slots of 32
    (1, 70, 256, 8, 40, 2, 1.0),      # d_model whole, ffn_dim ragged
])
def test_folded_layernorm_ragged(device, b, s, d, h, f, layers, scale, kind):
    cfg = TransformerConfig(b, s, d, h, f, layers, True)
    _, ctx, _ = _lib.stage_offsets(b, s, d, h, f, layers, PLAN_LAYERWISE)
    assert ctx >= 0, "shape expected to fold its LayerNorms"
    gm = _model(cfg, device, d)
    x16, mask = _inputs(cfg, kind, s)
    x16 = (x16.float() * scale).half()
    opt = make_optimized_transformer(copy.deepcopy(gm), plan=PLAN_LAYERWISE)
    with torch.inference_mode():
        md = None if mask is None else mask.to(device)
        y1, y2 = opt(x16.to(device), md).clone(), opt(x16.to(device), md)
    res = O.check_tolerance(y1, O.forward(O.params_fp32(gm), x16.float(), mask, h, True), mask)
    assert res["passed"], res
    assert torch.equal(y1, y2)


@pytest.mark.parametrize("kind", ["prefix", "scattered", "allvalid"])
@pytest.mark.parametrize("b,s,d,h,f,causal", [
    (8, 520, 72, 9, 144, False),     # head_dim 8, 64 x 64 tiles, partial column tiles of every part
    (8, 300, 288, 9, 584, True),     # S % 8 != 0, ffn_dim off the 64 grid too
    (5, 333, 480, 15, 968, False),   # odd S: V^T a value at a time
    (16, 512, 480, 15, 960, True),   # 128 x 128 tiles
])
def test_packed_rows_ragged(device, b, s, d, h, f, causal, kind):
    """The device's row count, the row map of the QKV epilogue and partial column tiles together: against the
    oracle, and bit for bit against the forward that runs every token (the same tiles' arithmetic)."""
    assert _lib.forward_packs_rows(b, s, d, h, f), "shape expected to run on packed rows"
    cfg = TransformerConfig(b, s, d, h, f, 2, causal)
    gm = _model(cfg, device, d)
    x16, mask = _inputs(cfg, "none" if kind == "allvalid" else kind, s)
    if mask is None:
        mask = torch.ones(b, s, dtype=torch.bool)
    opt = make_optimized_transformer(copy.deepcopy(gm))
    xd, md = x16.to(device), mask.to(device)
    with torch.inference_mode():
        y1, y2 = opt(xd, md).clone(), opt(xd, md).clone()
        _lib.check(_lib.load().tt_forward_packing_override(0), "packing override")
        try:
            y_pad = opt(xd, md).clone()
        finally:
            _lib.load().tt_forward_packing_override(-1)
        y_none = opt(xd, None)
    assert torch.equal(y1, y2) and torch.equal(y1, y_pad)
    if kind == "allvalid":
        assert torch.equal(y1, y_none)
    idx = torch.arange(min(b, 6))  # sequences are independent
    ref = O.forward(O.params_fp32(gm), x16[idx].float(), mask[idx], h, causal)
    res = O.check_tolerance(y1.cpu()[idx], ref, mask[idx])
    assert res["passed"], res
