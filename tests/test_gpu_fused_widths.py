"""Inference of feed-forward sizes of no whole tile: the activation in the product's epilogue, against the two kernels."""

import pytest
import torch

from fast_llm_amd.functional.config import ActivationType, KernelConfig
from fast_llm_amd.layers.moe import DroplessMoEMLP

pytestmark = pytest.mark.gpu


# 300 tokens are products of few tiles (of 64, 128 and 256 columns as the width grows), 3000 with 1096 and more columns are not.
@pytest.mark.parametrize("tokens", [300, 3000])
@pytest.mark.parametrize("ffn", [8, 56, 64, 72, 120, 136, 200, 1096, 1432, 2376, 4168])
@pytest.mark.parametrize("activation", [ActivationType.silu, ActivationType.squared_relu])
def test_layer_equals_two_kernels(tokens, ffn, activation, device, monkeypatch):
    torch.manual_seed(tokens + ffn)
    dtype = torch.float16 if ffn % 16 else torch.bfloat16
    layer = DroplessMoEMLP(320, ffn, 7, 2, activation=activation, init_std=0.2, dtype=dtype, device=device).eval()
    x = torch.randn(tokens, 320, device=device).to(dtype)
    with torch.no_grad():
        output = layer(x)
        monkeypatch.setattr(KernelConfig, "fuse_activation", False)
        assert torch.equal(output, layer(x))
