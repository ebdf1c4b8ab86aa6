"""The inference kernels for few tokens against the oracle's dropless MLP."""

import pytest
import torch

from fast_llm_amd import _lib
from fast_llm_amd.functional import mlp
from fast_llm_amd.functional.config import ActivationType
from fast_llm_amd.layers.moe import DroplessMoEMLP
from oracle import moe_oracle
from tests.helpers import max_rel_err

pytestmark = pytest.mark.gpu

_MAX_REL = {torch.bfloat16: 1e-2, torch.float16: 2e-3}


def _expected(x, scores, top_experts, weight_1, weight_2, experts, gated, activation):
    """Per expert in fp32, rounded to the operands' type where the kernels round: before and after the activation."""
    dtype, out = x.dtype, torch.zeros(x.shape)
    for e, (w1, w2) in enumerate(zip(weight_1.chunk(experts), weight_2.chunk(experts))):
        token, slot = torch.where(top_experts == e)
        layer_1 = (x[token].float() @ w1.float().t()).to(dtype).float()
        act = moe_oracle.mlp_activation_forward(layer_1, gated, activation.value).to(dtype).float()
        out.index_add_(0, token, (act @ w2.float()) * scores[token, slot, None])
    return out


# Tokens, experts and slots on each side of where the kernels change: one workgroup row per entry or per expert, mean rows
# per expert of 10 and 24 (one, two or four groups of 16 tokens), experts with more rows than a group.
@pytest.mark.parametrize(("tokens", "experts", "slots"), [(1, 8, 2), (3, 64, 6), (16, 4, 2), (17, 4, 1), (40, 6, 3), (65, 5, 2), (99, 5, 2)])
# Sizes around the chunks (128 of K, 16 and 128 outputs), and more than one piece of layer 2's reduction.
@pytest.mark.parametrize(("hidden", "ffn"), [(64, 72), (136, 128), (264, 1032), (2056, 40)])
@pytest.mark.parametrize(("dtype", "gated", "activation"), [
    (torch.bfloat16, True, ActivationType.silu), (torch.float16, True, ActivationType.gelu),
    (torch.bfloat16, False, ActivationType.squared_relu),
])  # fmt: skip
def test_few_tokens_forward(tokens, experts, slots, hidden, ffn, dtype, gated, activation, device):
    generator = torch.Generator().manual_seed(tokens + hidden)
    x = torch.randn(tokens, hidden, generator=generator).to(dtype)
    weight_1 = torch.normal(0, 0.1, (experts * ffn * (1 + gated), hidden), generator=generator).to(dtype)
    weight_2 = torch.normal(0, 0.1, (experts * ffn, hidden), generator=generator).to(dtype)
    # Preferred experts: some get many rows, some none.
    logits = torch.randn(tokens, experts, generator=generator) + 2 * torch.randn(experts, generator=generator)
    scores, top_experts = moe_oracle.topk_routing(logits, slots)
    if tokens > 1:
        top_experts[1, 0] = -1  # an entry that selects no expert contributes nothing
    output = mlp.few_tokens_forward(
        *(t.to(device) for t in (x, scores, top_experts, weight_1, weight_2)), experts, gated, activation
    )
    expected = _expected(x, scores, top_experts, weight_1, weight_2, experts, gated, activation)
    assert output.dtype == dtype
    # The sums differ from the oracle's in their order: a value next to a rounding boundary of the activation's type may
    # fall on its other side, which the type's own bound covers.
    assert max_rel_err(output.cpu(), expected) <= _MAX_REL[dtype]


# One to four trips of 512 along the rows, whole or not, which workgroups start at different places, and longer rows, which they do not.
@pytest.mark.parametrize("hidden", [8, 512, 520, 1024, 1288, 2048, 2056])
@pytest.mark.parametrize("tokens", [1, 20, 70])
def test_every_part_of_a_row_counts_once(hidden, tokens, device):
    """Small whole numbers, whose sums are exact in any order; layer 2 picks its rows out."""
    generator = torch.Generator().manual_seed(hidden + tokens)
    experts, ffn = 3, 200
    x, weight_1 = (torch.randint(-1, 2, (rows, hidden), generator=generator).bfloat16() for rows in (tokens, experts * ffn))
    weight_2 = torch.zeros(experts, ffn, max(hidden, ffn))
    weight_2[:] = torch.eye(ffn, max(hidden, ffn))
    weight_2 = weight_2[:, :, :hidden].reshape(experts * ffn, hidden).bfloat16()
    top_experts = torch.randint(0, experts, (tokens, 1), generator=generator)
    output = mlp.few_tokens_forward(
        *(t.to(device) for t in (x, torch.ones(tokens, 1), top_experts, weight_1, weight_2)), experts, False, ActivationType.identity
    )
    layer_1 = torch.einsum("th,tfh->tf", x.float(), weight_1.float().view(experts, ffn, hidden)[top_experts[:, 0]]).bfloat16()
    assert torch.equal(output.cpu()[:, :ffn], layer_1[:, :hidden])


def test_few_tokens_forward_leaves_the_rest_to_the_sparse_layout(device):
    def call(tokens, dtype=torch.bfloat16, ffn=64):
        x, weight_1, weight_2 = (torch.zeros(rows, 64, dtype=dtype, device=device) for rows in (tokens, 8 * ffn, 4 * ffn))
        scores, top_experts = torch.ones(tokens, 2, device=device), torch.zeros(tokens, 2, dtype=torch.int64, device=device)
        return mlp.few_tokens_forward(x, scores, top_experts, weight_1, weight_2, 4, True, ActivationType.silu)

    limit = mlp.FEW_TOKENS_MAX_ROWS_PER_EXPERT * 2
    assert call(limit) is not None and call(limit + 1) is None
    assert call(4, torch.float32) is None and call(4, ffn=60) is None


def test_few_tokens_refuse_a_weight_that_does_not_fit(device):
    layer = DroplessMoEMLP(64, 128, 8, 2, device=device).eval()
    x = torch.randn(16, 64, device=device, dtype=torch.bfloat16)
    layer.layer_2 = torch.nn.Parameter(torch.cat([layer.layer_2.detach(), layer.layer_2.detach()[:4]]))
    with torch.no_grad(), pytest.raises((AssertionError, ValueError)):
        layer(x)


# The kernels take 4096 (token, slot) pairs, sizes that are multiples of 8 and aligned, contiguous inputs: what they do not take
# goes through the layer in two calls, not one launch at a time.
@pytest.mark.parametrize(("tokens", "ffn", "odd", "expected"), [
    (320, 64, None, "fm_few_tokens_forward"), (321, 64, None, "fm_moe_layer_forward"),  # 20 rows per expert
    (512, 2048, None, "fm_few_tokens_forward"), (513, 2048, None, "fm_moe_layer_forward"), (641, 64, None, "fm_moe_layer_forward"),
    (16, 60, None, "fm_moe_layer_forward"), (16, 64, "address", "fm_moe_layer_forward"), (16, 64, "strides", "fm_moe_layer_forward"),
])  # fmt: skip
def test_inference_takes_one_of_two_routes(tokens, ffn, odd, expected, device, monkeypatch):
    torch.manual_seed(0)
    layer = DroplessMoEMLP(64, ffn, 128, 8, device=device).eval()
    x = torch.randn(tokens, 64, device=device, dtype=torch.bfloat16)
    if odd == "address":
        x = torch.empty(tokens * 64 + 1, device=device, dtype=torch.bfloat16)[1:].view(tokens, 64).copy_(x)
    elif odd == "strides":
        x = x.t().contiguous().t()
    calls, call = [], _lib.call
    monkeypatch.setattr(_lib, "call", lambda name, *args, **kwargs: (calls.append(name), call(name, *args, **kwargs)))
    with torch.no_grad():
        output = layer(x)
        assert calls[-1] == expected
        scores, top_experts = layer.route(x)
        operands = (t.cpu() for t in (x, scores, top_experts, layer.layer_1, layer.layer_2))
        reference = _expected(*operands, 128, True, ActivationType.silu)
    assert max_rel_err(output.cpu(), reference) <= _MAX_REL[torch.bfloat16]


def test_layers_with_a_shared_expert_leave_the_few_token_kernels_sooner(device, monkeypatch):
    """A shared expert has a row for every token, many times the mean, and its weights are read again for each 16 to 64."""
    layer = DroplessMoEMLP(64, 64, 17, 2, shared_experts=1, device=device).eval()
    calls, call = [], _lib.call
    monkeypatch.setattr(_lib, "call", lambda name, *args, **kwargs: (calls.append(name), call(name, *args, **kwargs)))
    with torch.no_grad():
        for tokens, expected in ((56, "fm_few_tokens_forward"), (57, "fm_moe_layer_forward")):  # 10 rows per expert
            layer(torch.randn(tokens, 64, device=device, dtype=torch.bfloat16))
            assert calls[-1] == expected
