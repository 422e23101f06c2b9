"""Narrow models (d_model and ffn_dim multiples of 32, d_model <= 192), whose layers run as attention plus row
chain: against the fp32 oracle at the edges of its 32- and 64-row tiles, column tiles and hidden chunks, with
every mask kind, and with more tiles than blocks.  The gate is the forward's own (2e-2 max, 2e-3 mean,
padded rows +0.0, two calls bit-identical); sequences are independent, so large batches are compared on a
sample of them."""

import pytest
import torch

from oracle import transformer_oracle as O
from tttj_2026_amd import PLAN_LAYERWISE, _lib, make_optimized_transformer
from tttj_2026_amd.configs import build_model, make_inputs
from tttj_2026_amd.model import TransformerConfig

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mask_kind", ["none", "prefix", "scattered"])
@pytest.mark.parametrize("b,s,d,h,f,layers,causal", [
    (3, 33, 32, 4, 32, 1, True),       # head_dim 8, one column tile per two waves, odd length
    (2, 40, 64, 1, 96, 2, False),      # partial hidden chunk only
    (5, 77, 96, 3, 160, 3, True),      # whole and partial chunk, rows across sequences
    (4, 128, 128, 8, 128, 4, True),    # head_dim 16, weights kept in registers
    (2, 130, 160, 5, 640, 2, False),   # two output tiles per wave, five chunks
    (1, 65, 192, 3, 1024, 2, True),    # widest
    (300, 60, 64, 2, 64, 2, True),     # 64-row tiles, more of them than blocks
    (70, 257, 32, 1, 128, 1, False),   # the same with odd sequences
    (40, 250, 128, 4, 256, 1, True),   # 64-row tiles, one per block
])
def test_row_chain(device, b, s, d, h, f, layers, causal, mask_kind):
    cfg = TransformerConfig(b, s, d, h, f, layers, causal)
    model = build_model(cfg, seed=d + s)
    g = torch.Generator().manual_seed(5)
    with torch.no_grad():
        for name, p in model.named_parameters():
            if "norm" in name:
                p.add_(0.2 * torch.randn(p.shape, generator=g))
    x16, mask = make_inputs(cfg, mask_kind == "prefix", 7, min_valid=0)
    if mask_kind == "scattered":
        mask = torch.rand(b, s, generator=g) > 0.4
        mask[b // 2] = False  # a sequence without any valid token
    gm = model.half().to(device)
    y = {}
    with torch.inference_mode():  # the automatic plan and the explicit one, both of which run the row chain
        for plan in (None, PLAN_LAYERWISE):
            opt = make_optimized_transformer(gm) if plan is None else make_optimized_transformer(gm, plan=plan)
            md = None if mask is None else mask.to(device)
            first = opt(x16.to(device), md).clone()
            y[plan] = opt(x16.to(device), md)
            assert torch.equal(first, y[plan])
    assert torch.equal(y[None], y[PLAN_LAYERWISE])
    idx = torch.arange(b) if b <= 8 else torch.tensor([0, 1, b // 2, b - 1])
    res = O.check_tolerance(y[None].cpu()[idx], O.forward(O.params_fp32(gm), x16[idx].float(),
                                                          None if mask is None else mask[idx], h, causal),
                            None if mask is None else mask[idx])
    assert res["passed"], res


def test_short_packed_weights_are_refused(device):
    """Weights without the region that the row chain reads (as the layout was before it had one)."""
    cfg = TransformerConfig(2, 40, 64, 2, 96, 2, False)
    opt = make_optimized_transformer(build_model(cfg, seed=1).half().to(device))
    x16, _ = make_inputs(cfg, False, 2)
    with torch.inference_mode():
        want = opt(x16.to(device)).clone()
        full, (_, _, final, _) = opt.packed_weights, _lib.weight_layout(64, 96, 2)
        opt.packed_weights = full[:final + 2 * 64].clone()
        with pytest.raises(ValueError, match="packed weights"):
            opt(x16.to(device))
        opt.packed_weights = full
        assert torch.equal(opt(x16.to(device)), want)
