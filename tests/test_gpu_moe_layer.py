"""The layer in two library calls (`functional.moe_layer`) against its composition from the single functions, which a
kernel timer selects and the oracle tests pin."""

import pytest
import torch

from fast_llm_amd import _lib
from fast_llm_amd.functional.config import ActivationType, MLPRecomputeLevel
from fast_llm_amd.functional.routing import router_forward, router_logits
from fast_llm_amd.layers.moe import DroplessMoEMLP
from tests.helpers import max_rel_err

pytestmark = pytest.mark.gpu


def _step(layer, batches, composed):
    layer.router.grad = None
    layer.layer_1.param_grad_is_zero = layer.layer_2.param_grad_is_zero = True
    outputs, input_grads, losses = [], [], {}
    for x in batches:
        x.grad = None
        if composed:
            with _lib.KernelTimer():
                output = layer(x, grad_scale=0.5, losses=losses)
        else:
            output = layer(x, grad_scale=0.5, losses=losses)
        output.backward(torch.ones_like(output) / output.numel() ** 0.5)
        outputs.append(output.detach())
        input_grads.append(x.grad)
    return {
        "outputs": outputs,
        "losses": [value for values in losses.values() for value in values],
        "weight_grads": [layer.layer_1.grad_buffer.clone(), layer.layer_2.grad_buffer.clone()],
        "input_grads": input_grads,
        "router_grad": [layer.router.grad],
    }


@pytest.mark.parametrize("recompute_level", list(MLPRecomputeLevel))
@pytest.mark.parametrize(
    ("hidden", "ffn", "options"),
    [
        (128, 256, dict(dtype=torch.bfloat16)),
        # No instance with the activation in the product's epilogue; one shared expert; both losses trained; jitter.
        (72, 40, dict(dtype=torch.float16, shared_experts=1, z_loss_coefficient=0.1, activation=ActivationType.gelu)),
        (64, 192, dict(dtype=torch.bfloat16, gated=False, full_precision_gradients=True, dropless_dynamic_shape=True)),
        (64, 128, dict(dtype=torch.float32, dropless_dynamic_shape=True)),
    ],
)
def test_layer_in_two_calls_matches_the_composition(recompute_level, hidden, ffn, options, device):
    torch.manual_seed(0)
    layer = DroplessMoEMLP(hidden, ffn, 7, 2, recompute_level=recompute_level, init_std=0.2, device=device, **options)
    batches = [torch.randn(tokens, hidden, device=device, dtype=options["dtype"], requires_grad=True) for tokens in (300, 77)]
    one, composed = _step(layer, batches, False), _step(layer, batches, True)
    for name in ("outputs", "losses", "weight_grads"):
        assert all(torch.equal(a, b) for a, b in zip(one[name], composed[name], strict=True)), name
    # The router's linear layer sums in another order, and in fp32 its input gradient is added as it is summed.
    bound = {torch.float32: 1e-5, torch.float16: 2e-3, torch.bfloat16: 1e-2}[options["dtype"]]
    for name in ("input_grads", "router_grad"):
        assert all(max_rel_err(a, b) <= bound for a, b in zip(one[name], composed[name], strict=True)), name
    layer.eval()
    with torch.no_grad():
        x = torch.cat(batches)
        output = layer(x)
        with _lib.KernelTimer():
            assert torch.equal(output, layer(x))


# Preferred experts: input feature 0 carries log p_e in the router's weight, so its gradient is the largest of the token's by far,
# and what is rounded on the way to it shows in single elements.
@pytest.mark.parametrize("zipf", [0.6, 1.2])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize(("hidden", "experts", "options"), [
    (2048, 64, dict(shared_experts=1, recompute_level=MLPRecomputeLevel.full)), (4096, 8, dict()),
    (2048, 60, dict(jitter_eps=0.1, z_loss_coefficient=0.01)),
])  # fmt: skip
def test_layer_in_two_calls_rounds_where_the_composition_does(hidden, experts, options, dtype, zipf, device):
    torch.manual_seed(0)
    layer = DroplessMoEMLP(hidden, 512, experts + options.get("shared_experts", 0), 4, dtype=dtype, device=device, **options)
    probabilities = torch.arange(1, experts + 1, device=device) ** -zipf
    with torch.no_grad():
        layer.router[:, 0] = (probabilities / probabilities.sum()).log()
    x = torch.randn(701, hidden, device=device, dtype=dtype)
    x[:, 0] = 1
    results = []
    for composed in (False, True):
        torch.manual_seed(1)
        results.append(_step(layer, [x.requires_grad_()], composed))
    one, other = results
    for name in ("outputs", "losses", "weight_grads", "input_grads"):
        assert all(torch.equal(a, b) for a, b in zip(one[name], other[name], strict=True)), name
    # The router's weight gradient: sums of the same products in another order, rounded once. A unit in the last place of the
    # element, and 1e-5 of the largest for the order.
    a, b = one["router_grad"][0].double(), other["router_grad"][0].double()
    assert ((a - b).abs() <= torch.finfo(dtype).eps * b.abs() + 1e-5 * b.abs().max()).all()


def test_layer_in_two_calls_with_jitter_frozen_weights_and_no_input_gradient(device):
    torch.manual_seed(0)
    layer = DroplessMoEMLP(64, 128, 4, 2, jitter_eps=0.1, device=device)
    x = torch.randn(100, 64, device=device, dtype=torch.bfloat16)
    results = []
    for composed in (False, True):
        torch.manual_seed(1)
        results.append(_step(layer, [x], composed))
    assert torch.equal(results[0]["outputs"][0], results[1]["outputs"][0])
    assert results[0]["input_grads"] == [None]
    assert max_rel_err(results[0]["router_grad"][0], results[1]["router_grad"][0]) <= 1e-2
    before = layer.layer_1.grad_buffer.clone()
    layer.layer_1.requires_grad_(False)
    layer.layer_1.grad_buffer.fill_(3)
    result = _step(layer, [x.requires_grad_()], False)
    assert (layer.layer_1.grad_buffer == 3).all() and before.abs().max() > 0
    assert result["input_grads"][0].abs().max() > 0
    output = layer(x)
    output.sum().backward(retain_graph=True)
    with pytest.raises(RuntimeError, match="backward ran already"):
        output.sum().backward()


def test_layer_in_two_calls_refuses_and_accepts_what_the_composition_does(device):
    torch.manual_seed(0)
    layer = DroplessMoEMLP(64, 128, 8, 2, device=device, dtype=torch.float32)
    x = torch.randn(100, 64, device=device)
    # Autocast makes the logits half as wide as the library's call takes them.
    with torch.autocast("cuda", torch.bfloat16):
        output = layer(x)
        with _lib.KernelTimer():
            assert torch.equal(output, layer(x))
    # Nothing that autograd knows needs a gradient, but the backward runs; buffers of two types, one with strides.
    for parameter in (layer.router, layer.layer_1, layer.layer_2):
        parameter.requires_grad_(False)
    layer(x).backward(x)
    layer.layer_1.requires_grad_(True), layer.layer_2.requires_grad_(True)
    results = []
    for direct in (True, False):
        if not direct:
            layer.layer_1.grad_buffer = torch.empty_like(layer.layer_1, dtype=torch.bfloat16)
            layer.layer_2.grad_buffer = layer.layer_2.detach().t().contiguous().t()
        layer.layer_1.param_grad_is_zero = layer.layer_2.param_grad_is_zero = True
        for _ in range(2):
            layer(x).backward(x)
        results.append([layer.layer_1.grad_buffer, layer.layer_2.grad_buffer])
    assert all(max_rel_err(a, b) <= 1e-2 for a, b in zip(*results))
    layer.layer_1.grad_buffer = layer.layer_1.detach().double()
    with pytest.raises(ValueError, match="dtype"):
        layer(x).backward(x)
    # A weight that does not fit is refused.
    whole, layer.layer_1 = layer.layer_1, torch.nn.Parameter(layer.layer_1.detach()[:-8].clone())
    with pytest.raises((AssertionError, ValueError)):
        layer(x)
    layer.layer_1 = whole


@pytest.mark.parametrize("tokens", [8, 512])  # the kernels for few tokens; the layer in two calls
def test_inference_without_gradient_buffers_at_odd_addresses_and_with_a_backward(tokens, device):
    torch.manual_seed(0)
    layer = DroplessMoEMLP(64, 128, 8, 2, device=device).eval()
    x = torch.randn(tokens, 64, device=device, dtype=torch.bfloat16)
    del layer.layer_1.grad_buffer, layer.layer_2.grad_buffer
    with torch.no_grad():
        expected = layer(x)
        odd = torch.empty(tokens * 64 + 1, device=device, dtype=torch.bfloat16)[1:].view(tokens, 64).copy_(x)
        assert max_rel_err(layer(odd), expected) <= 1e-2
    output = layer(x)
    assert torch.equal(output, expected)
    with pytest.raises(RuntimeError, match="kept nothing"):
        output.sum().backward()


def test_training_step_with_an_input_at_an_odd_address(device):
    torch.manual_seed(0)
    layer = DroplessMoEMLP(64, 128, 8, 2, device=device)
    x = torch.randn(300, 64, device=device, dtype=torch.bfloat16)
    odd = torch.empty(300 * 64 + 1, device=device, dtype=torch.bfloat16)[1:].view(300, 64).copy_(x)
    results = [_step(layer, [value.requires_grad_()], False) for value in (x, odd)]
    for name in ("outputs", "input_grads", "router_grad", "weight_grads"):
        assert all(max_rel_err(a, b) <= 1e-2 for a, b in zip(results[0][name], results[1][name])), name


# Products with tile tables, written together, some of which split their last round (reductions of 38 slices and more: the input
# gradient with an ffn of 2176, both directions with 2560) and some of which do not; memory full of NaN beforehand: what padding and phantom rows hold gets nowhere.
@pytest.mark.parametrize("recompute_level", [MLPRecomputeLevel.none, MLPRecomputeLevel.full])
@pytest.mark.parametrize(("hidden", "ffn", "tokens"), [(2048, 2176, (300, 77)), (512, 2176, (1500, 40)), (2048, 192, (700, 2100)), (2432, 2560, (300, 77))])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_layer_in_two_calls_with_tile_tables(recompute_level, hidden, ffn, tokens, dtype, device):
    torch.manual_seed(0)
    layer = DroplessMoEMLP(hidden, ffn, 7, 2, recompute_level=recompute_level, init_std=0.02, device=device, dtype=dtype)
    batches = [torch.randn(count, hidden, device=device, dtype=dtype, requires_grad=True) for count in tokens]
    results = []
    for composed in (False, True):
        torch.full((1 << 28,), float("nan"), device=device)
        results.append(_step(layer, batches, composed))
    for name in ("outputs", "losses", "weight_grads"):
        assert all(torch.equal(a, b) for a, b in zip(results[0][name], results[1][name], strict=True)), name
    bound = {torch.float32: 1e-5, torch.bfloat16: 1e-2}[dtype]  # as in test_layer_in_two_calls_matches_the_composition
    for name in ("input_grads", "router_grad"):
        assert all(max_rel_err(a, b) <= bound for a, b in zip(results[0][name], results[1][name], strict=True)), name


@pytest.mark.parametrize("training", [False, True])
def test_collected_losses_keep_no_buffer_of_the_layer(training, device):
    layer = DroplessMoEMLP(64, 128, 8, 2, z_loss_coefficient=0.1, device=device).train(training)
    losses = {}
    layer(torch.randn(2000, 64, device=device, dtype=torch.bfloat16), grad_scale=1.0, losses=losses)
    assert all(value.untyped_storage().nbytes() <= 64 for values in losses.values() for value in values) and len(losses) == 2


@pytest.mark.parametrize("tokens", [8, 512])
@pytest.mark.parametrize("training", [False, True])
@pytest.mark.parametrize("subclass", [False, True])
@pytest.mark.parametrize("selected", [1, 2, 3])
def test_replaced_routing_is_honoured(tokens, training, subclass, selected, device):
    def first_experts(self, hidden_states, grad_scale=None, losses=None):
        experts = torch.arange(selected, device=hidden_states.device).expand(hidden_states.size(0), selected).contiguous()
        return torch.full(experts.shape, 0.5, device=hidden_states.device), experts, None

    torch.manual_seed(0)
    layer_class = type("FirstExperts", (DroplessMoEMLP,), {"route_with_counts": first_experts}) if subclass else DroplessMoEMLP
    layer = layer_class(64, 128, 8, 2, device=device).train(training)
    x = torch.randn(tokens, 64, device=device, dtype=torch.bfloat16)
    scores, experts, _ = first_experts(layer, x)
    with torch.no_grad():
        expected = layer(x, scores, experts)
        if not subclass:
            layer.route_with_counts = lambda *args: first_experts(layer, *args)
        assert torch.equal(layer(x), expected)


def test_undefined_output_gradient_trains_the_router_and_clears_the_buffers(device):
    class NoGradient(torch.autograd.Function):
        @staticmethod
        def forward(ctx, x):
            return x.clone()

        @staticmethod
        def backward(ctx, grad):
            return None

    torch.manual_seed(0)
    layer = DroplessMoEMLP(64, 128, 8, 2, auxiliary_loss_coefficient=1.0, z_loss_coefficient=1.0, device=device, dtype=torch.float32)
    x = torch.randn(100, 64, device=device, requires_grad=True)
    results = []
    for composed in (False, True):
        layer.router.grad = x.grad = None
        layer.layer_1.param_grad_is_zero = layer.layer_2.param_grad_is_zero = True
        layer.layer_1.grad_buffer.fill_(7), layer.layer_2.grad_buffer.fill_(7)
        if composed:
            with _lib.KernelTimer():
                output = layer(x, grad_scale=1.0)
        else:
            output = layer(x, grad_scale=1.0)
        NoGradient.apply(output).sum().backward()
        results.append((layer.router.grad, x.grad))
        assert not layer.layer_1.grad_buffer.any() and not layer.layer_2.grad_buffer.any()
    assert all(max_rel_err(a, b) <= 1e-5 and b.abs().max() > 0 for a, b in zip(*results))


@pytest.mark.parametrize("tokens", [8, 512])
@pytest.mark.parametrize("training", [False, True])
@pytest.mark.parametrize("which", ["input", "router"])
def test_tangents_are_refused_not_lost(tokens, training, which, device):
    layer = DroplessMoEMLP(64, 128, 8, 2, device=device).train(training)
    x = torch.randn(tokens, 64, device=device, dtype=torch.bfloat16)
    with torch.no_grad(), torch.autograd.forward_ad.dual_level():
        dual = torch.autograd.forward_ad.make_dual(x if which == "input" else layer.router.detach(), torch.ones_like(x if which == "input" else layer.router))
        with pytest.raises(RuntimeError, match="jvp|forward"):
            if which == "input":
                layer(dual)
            else:
                torch.func.functional_call(layer, {"router": dual}, (x,))
        layer(x)  # without a tangent nothing is lost


@pytest.mark.parametrize("tokens", [8, 512])
def test_traces_are_refused_not_wrong(tokens, device):
    """A tracer would record the space for the output and not the library calls that fill it."""
    layer = DroplessMoEMLP(64, 128, 8, 2, device=device).eval()
    x = torch.randn(tokens, 64, device=device, dtype=torch.bfloat16)
    with torch.no_grad(), pytest.raises(RuntimeError, match="requires grad"):
        torch.jit.trace(layer, x, check_trace=False)


def test_saved_tensor_hooks_see_what_the_router_saves(device):
    torch.manual_seed(0)
    layer = DroplessMoEMLP(64, 128, 8, 2, device=device, dtype=torch.float32)
    x = torch.randn(300, 64, device=device, requires_grad=True)
    results, packed = [], []

    def pack(tensor):
        packed.append(tuple(tensor.shape))
        return tensor.cpu()

    for hooks in (False, True):
        layer.router.grad = x.grad = None
        layer.layer_1.param_grad_is_zero = layer.layer_2.param_grad_is_zero = True
        if hooks:
            with torch.autograd.graph.saved_tensors_hooks(pack, lambda tensor: tensor.to(device)):
                output = layer(x, grad_scale=1.0)
        else:
            output = layer(x, grad_scale=1.0)
        output.backward(torch.ones_like(output))
        results.append((x.grad, layer.router.grad, layer.layer_1.grad_buffer.clone(), layer.layer_2.grad_buffer.clone()))
    assert {(300, 64), (8, 64), (300, 8)} <= set(packed) and len(packed) > 3  # input, router, logits, and what was selected
    assert all(torch.equal(a, b) for a, b in zip(*results))


@pytest.mark.parametrize("recompute_level", [MLPRecomputeLevel.none, MLPRecomputeLevel.full])
@pytest.mark.parametrize("gated", [False, True])
def test_layer_in_library_calls_holds_no_more_memory_than_the_composition(recompute_level, gated, device):
    """Both directions at a size where the backward lets layer 2's output go first; the composition frees every intermediate
    after its last reader. 8192 tokens in 33 792 rows of 1024: 66 MiB a row buffer."""
    torch.manual_seed(0)
    layer = DroplessMoEMLP(1024, 512, 8, 4, gated=gated, recompute_level=recompute_level, device=device)
    x = torch.randn(8192, 1024, device=device, dtype=torch.bfloat16, requires_grad=True)
    results, peaks = [], []
    for composed in (False, True, False, True):  # the first of each also pays for what the libraries keep
        torch.cuda.synchronize()
        torch.cuda.reset_peak_memory_stats()
        before = torch.cuda.memory_allocated()
        results.append(_step(layer, [x], composed))
        peaks.append(torch.cuda.max_memory_allocated() - before)
        x.grad = layer.router.grad = None
        layer.eval()
        torch.cuda.reset_peak_memory_stats()
        before = torch.cuda.memory_allocated()
        with torch.no_grad():
            if composed:
                with _lib.KernelTimer():
                    results[-1]["outputs"].append(layer(x))
            else:
                results[-1]["outputs"].append(layer(x))
        peaks.append(torch.cuda.max_memory_allocated() - before)
        layer.train()
    for name in ("outputs", "weight_grads", "input_grads"):
        assert all(torch.equal(a, b) for a, b in zip(results[2][name], results[3][name], strict=True)), name
    # What the backward's call needs beside its intermediates: the input gradient (16 MiB) and its workspace.
    assert peaks[4] <= peaks[6] + (24 << 20), [peak >> 20 for peak in peaks]
    assert peaks[5] <= peaks[7] + (1 << 20), [peak >> 20 for peak in peaks]


# The router's sums over its workgroups (16 tokens each, 256 at most) share a launch with the sparse map: fewer experts than the 8
# columns of a workgroup's threads, more than a wavefront holds, more than one batch of terms per thread.
@pytest.mark.parametrize(("tokens", "experts", "shared"), [(1, 3, 0), (17, 8, 1), (300, 64, 0), (4200, 65, 2), (5000, 300, 0), (40, 1000, 0)])
def test_losses_and_map_in_one_launch(tokens, experts, shared, device):
    torch.manual_seed(0)
    layer = DroplessMoEMLP(
        64, 64, experts + shared, 2, shared_experts=shared, z_loss_coefficient=0.1, auxiliary_loss_coefficient=0.1,
        init_std=0.2, dtype=torch.bfloat16, device=device,
    )  # fmt: skip
    x = torch.randn(tokens, 64, device=device, dtype=torch.bfloat16, requires_grad=True)
    one, composed = _step(layer, [x], False), _step(layer, [x], True)
    for name in ("outputs", "losses", "weight_grads"):
        assert all(torch.equal(a, b) for a, b in zip(one[name], composed[name], strict=True)), name
    # Against the definition: sum_e mean_t(softmax) * mean_t(selected), mean_t(logsumexp^2), in fp64.
    logits = router_logits(x.detach(), layer.router.detach())
    top_experts = router_forward(logits, None, 2, shared)[1][:, shared:]  # rounded logits may tie
    logits = logits.double()
    selected = torch.zeros_like(logits).scatter_(1, top_experts, 1)
    balance = (logits.softmax(1).mean(0) * selected.mean(0)).sum()
    z = logits.logsumexp(1).square().mean()
    # Per token fp32 exponentials and sums.
    assert abs(one["losses"][0].double() - balance) <= 1e-5 * balance
    assert abs(one["losses"][1].double() - z) <= 1e-5 * z + 1e-6
