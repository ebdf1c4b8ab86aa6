"""Inference of feed-forward sizes of no whole tile: the activation in the product's epilogue, against the two kernels."""

import pytest
import torch

from fast_llm_amd.functional.config import ActivationType, KernelConfig
from fast_llm_amd.layers.moe import DroplessMoEMLP

pytestmark = pytest.mark.gpu


# 300 tokens are products of few tiles up to 200 columns, and streamed ones from 1096 on. 3000 are streamed ones from 136 on, and tiles of
# 256 x 256 with 1096 and 4168: up to 1024 rows per expert, whose reductions start at different slices. 8000 have more rows.
WIDTHS = [(tokens, ffn) for tokens in (300, 3000) for ffn in (8, 56, 64, 72, 120, 136, 200, 1096, 1432, 2376, 4168)]
WIDTHS += [(8000, ffn) for ffn in (1096, 1432, 4168)]


@pytest.mark.parametrize(("tokens", "ffn"), WIDTHS)
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("activation", [ActivationType.silu, ActivationType.squared_relu])
def test_layer_equals_two_kernels(tokens, ffn, dtype, activation, device, monkeypatch):
    torch.manual_seed(tokens + ffn)
    layer = DroplessMoEMLP(320, ffn, 7, 2, activation=activation, init_std=0.2, dtype=dtype, device=device).eval()
    x = torch.randn(tokens, 320, device=device).to(dtype)
    with torch.no_grad():
        output = layer(x)
        monkeypatch.setattr(KernelConfig, "fuse_activation", False)
        assert torch.equal(output, layer(x))


# Reductions that the product by itself cuts into pieces (from 36 slices of 64 on): 4000 tokens have a last round of few tiles, 300 are
# few tiles in all; 700 tokens run uncut in any case, in the product of experts of few rows.
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize(("tokens", "hidden", "ffn"), [(4000, 2432, 2056), (4000, 2304, 2120), (300, 2432, 136), (700, 2432, 2056)])
def test_layer_equals_parts_where_reductions_are_cut(tokens, hidden, ffn, dtype, device, monkeypatch):
    torch.manual_seed(tokens + ffn)
    layer = DroplessMoEMLP(hidden, ffn, 8, 2, init_std=0.05, dtype=dtype, device=device).eval()
    x = torch.randn(tokens, hidden, device=device).to(dtype)
    with torch.no_grad():
        output = layer(x)
        monkeypatch.setattr(layer, "route_with_counts", lambda *args: DroplessMoEMLP.route_with_counts(layer, *args))
        assert torch.equal(output, layer(x))
