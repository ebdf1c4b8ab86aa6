"""
The whole MoE layer, from the router's linear layer to the output, with two library calls for the forward
(`fm_moe_layer_route`, `fm_moe_layer_forward`) and one or two for the backward (`fm_moe_layer_backward`) instead of one per
kernel: the same kernels in the same order as `router` -> `get_sparse_map` -> `mlp_autograd`, without the host time of
some twenty Python launches.

Covers `MixtureOfExpertMLP._forward` (fast_llm/layers/decoder/mlp/mixture_of_experts.py:126-213) for top-k routing of the
hidden states themselves; `layers.moe.DroplessMoEMLP` composes the other cases from the parts.
"""

import dataclasses

import torch

from fast_llm_amd import _lib
from fast_llm_amd.functional.config import ActivationType, KernelConfig, MLPRecomputeLevel
from fast_llm_amd.functional.mlp import _activation_tag
from fast_llm_amd.functional.routing import router_logits
from fast_llm_amd.functional.utils import ANCHOR, Assert, is_traced, without_backward
from fast_llm_amd.tensor import accumulate_gradient, param_get_and_unset_is_zero


@dataclasses.dataclass(frozen=True)
class MoELayerOptions:
    routed_experts: int
    shared_experts: int
    experts_per_token: int
    gated: bool
    activation_type: ActivationType
    recompute_level: MLPRecomputeLevel
    dynamic_shape: bool


def moe_layer_supported(
    hidden_states: torch.Tensor,
    router: torch.Tensor,
    weight_1: torch.Tensor,
    weight_2: torch.Tensor,
    options: MoELayerOptions,
) -> bool:
    """Whether `moe_layer` takes these operands. It steps aside for what the parts offer and it does not (kernel timers,
    kernel choices other than the default ones, logits that autocast makes another type of, tracers) and for operands that do not
    fit together, which the parts refuse."""
    dtype, (experts, hidden) = hidden_states.dtype, (options.routed_experts + options.shared_experts, hidden_states.size(-1))
    ffn = weight_2.size(0) // experts
    return (
        _lib._active_timer is None
        and KernelConfig.fuse_activation is None
        and KernelConfig.grouped_gemm_workspace
        and not torch.is_autocast_enabled("cuda")
        and not is_traced()
        and hidden_states.dim() == 2
        and hidden_states.size(0) > 0
        and dtype in _lib.DTYPES
        and router.dtype == weight_1.dtype == weight_2.dtype == dtype
        and router.shape == (options.routed_experts, hidden)
        and weight_1.shape == (experts * ffn * (2 if options.gated else 1), hidden)
        and weight_2.shape == (experts * ffn, hidden)
        and router.is_contiguous()
        and weight_1.is_contiguous()
        and weight_2.is_contiguous()
    )


def _describe(
    options: MoELayerOptions,
    hidden_states: torch.Tensor,
    weight_1: torch.Tensor,
    weight_2: torch.Tensor,
    with_losses: bool,
    dynamic_rows: int = 0,
) -> _lib.MoELayer:
    tokens, hidden = hidden_states.shape
    layer = _lib.MoELayer(
        tokens,
        hidden,
        weight_2.size(0) // (options.routed_experts + options.shared_experts),
        options.routed_experts,
        options.shared_experts,
        options.experts_per_token,
        options.gated,
        _activation_tag(options.activation_type),
        _lib.DTYPES[hidden_states.dtype],
    )
    layer.with_losses, layer.dynamic_rows = with_losses, dynamic_rows
    layer.weight_1, layer.weight_2 = weight_1.data_ptr(), weight_2.data_ptr()
    _lib.check(_lib.lib().fm_moe_layer_sizes(_lib.ctypes.byref(layer)))
    return layer


def _fuses_layer_1(options: MoELayerOptions, layer: _lib.MoELayer, training: bool) -> bool:
    """Whether layer 1's product has an instance with the gated activation in its epilogue. In training for the widths only that the
    product of the parts takes: the recompute levels keep to the same kernels."""
    return options.gated and layer.dtype != 0 and layer.hidden % 64 == 0 and layer.ffn % (128 if training else 8) == 0


@dataclasses.dataclass
class _Saved:
    """What the forward keeps for the backward. An intermediate that the recompute level does not keep is None."""

    router: tuple[torch.Tensor, torch.Tensor | None, torch.Tensor]  # logits, noise, routing: autograd saves these
    sparse_input: torch.Tensor | None
    layer_1_output: torch.Tensor | None
    activation_output: torch.Tensor | None
    layer_2_output: torch.Tensor
    dynamic_rows: int


def _forward(
    options: MoELayerOptions,
    hidden_states: torch.Tensor,
    router: torch.Tensor,
    weight_1: torch.Tensor,
    weight_2: torch.Tensor,
    noise: torch.Tensor | None,
    with_losses: bool,
    training: bool,
) -> tuple[torch.Tensor, torch.Tensor | None, _Saved]:
    """(output, losses [2] or None, what the backward needs)."""
    device = _lib.require_device(hidden_states, router, weight_1, weight_2, noise)
    logits = router_logits(hidden_states, router)
    layer = _describe(options, hidden_states, weight_1, weight_2, with_losses)
    new = hidden_states.new_empty
    routing = new(layer.routing_bytes, dtype=torch.uint8)
    losses = new(2, dtype=torch.float32) if with_losses else None  # of its own: a caller may keep it long
    layer.losses = _lib.ptr(losses)
    layer.logits, layer.noise, layer.routing = logits.data_ptr(), _lib.ptr(noise), routing.data_ptr()
    if options.dynamic_shape:
        workspace = new(layer.forward_workspace_bytes, dtype=torch.uint8)
        layer.workspace = workspace.data_ptr()
        _lib.call("fm_moe_layer_route", device, _lib.ctypes.byref(layer))
        index_dtype = torch.int16 if layer.index_dtype == 0 else torch.int32
        used_rows = routing[layer.used_rows_offset : layer.used_rows_offset + index_dtype.itemsize].view(index_dtype)
        layer.dynamic_rows = used_rows.item()
        _lib.check(_lib.lib().fm_moe_layer_sizes(_lib.ctypes.byref(layer)))
    level, rows, ffn = options.recompute_level, layer.rows, layer.ffn
    keep_layer_1 = training and not level.recompute_layer_1
    workspace = new(layer.forward_workspace_bytes, dtype=torch.uint8)
    sparse_input = new((rows, layer.hidden))
    # Layer 1 is the only one to read the sparse input: where nobody keeps it, layer 2's output takes its place.
    layer_2_output = new((rows, layer.hidden)) if training and not level.recompute_sparse_input else sparse_input
    activation_output, output = new((rows, ffn)), new(hidden_states.shape)
    layer_1_output = None
    if keep_layer_1 or not _fuses_layer_1(options, layer, training):
        layer_1_output = new((rows, ffn * 2 if options.gated else ffn))
        layer.layer_1_output = layer_1_output.data_ptr()
    layer.input, layer.output, layer.workspace = hidden_states.data_ptr(), output.data_ptr(), workspace.data_ptr()
    layer.sparse_input, layer.activation_output = sparse_input.data_ptr(), activation_output.data_ptr()
    layer.layer_2_output = layer_2_output.data_ptr()
    if not options.dynamic_shape:
        _lib.call("fm_moe_layer_route", device, _lib.ctypes.byref(layer))
    try:
        _lib.call("fm_moe_layer_forward", device, _lib.ctypes.byref(layer))
    except NotImplementedError:  # a shape the fused product does not tile after all
        if layer_1_output is not None:
            raise
        layer_1_output = new((rows, ffn * 2))
        layer.layer_1_output = layer_1_output.data_ptr()
        _lib.call("fm_moe_layer_forward", device, _lib.ctypes.byref(layer))
    saved = _Saved(
        (logits, noise, routing),
        None if level.recompute_sparse_input else sparse_input,
        layer_1_output if keep_layer_1 else None,
        None if level.recompute_activation else activation_output,
        layer_2_output,
        layer.dynamic_rows,
    )
    return output, losses, saved


def _gradient_targets(weights: list[torch.Tensor]) -> list[torch.Tensor]:
    """What the library writes the gradients of `weights` to: their buffers, or where it does not take those (two types,
    strides), tensors in single precision that are added to them afterwards."""
    buffers = [weight.grad_buffer for weight in weights]
    for weight, buffer in zip(weights, buffers):
        Assert.eq(buffer.shape, weight.shape)
    one_type = len({_lib.dtype_tag(buffer.dtype) for buffer in buffers}) <= 1
    direct = one_type and all(buffer.is_contiguous() for buffer in buffers)
    return buffers if direct else [torch.empty(weight.shape, dtype=torch.float32, device=weight.device) for weight in weights]


# Layer 2's output from this size on is let go before the backward makes the rest of its buffers, at the price of a library call
# more; what is smaller is not worth the host time that small layers are bound by.
_LARGE_BUFFER = 32 << 20


class _MoELayer(torch.autograd.Function):
    # The last argument of `apply` is an empty tensor that requires a gradient: the weight gradients are side effects, the
    # node is to be visited whatever else needs one.
    @staticmethod
    def forward(ctx, hidden_states, router, weight_1, weight_2, noise, options, with_losses, loss_grads, _):
        output, losses, ctx.saved = _forward(
            options, hidden_states, router, weight_1, weight_2, noise, with_losses, training=True
        )
        # As the router's own nodes do: saved-tensor hooks see its tensors. The MLP's intermediates are the layer's.
        ctx.save_for_backward(hidden_states, router, *ctx.saved.router)
        ctx.saved.router = None
        ctx.weights, ctx.options, ctx.with_losses, ctx.loss_grads = (weight_1, weight_2), options, with_losses, loss_grads
        ctx.set_materialize_grads(False)
        if losses is not None:
            ctx.mark_non_differentiable(losses)
        return output, losses

    @staticmethod
    def backward(ctx, grad_output, _):
        hidden_states, router, logits, noise, routing = ctx.saved_tensors
        if grad_output is None:  # nothing depends on the output: the losses still train the router, the buffers become zero
            grad_output = torch.zeros_like(hidden_states)
        (weight_1, weight_2), options = ctx.weights, ctx.options
        saved, ctx.saved = ctx.saved, None  # the intermediates go when this call ends, whoever holds the graph
        if saved is None:
            raise RuntimeError("the layer's intermediates have been freed: backward ran already")
        grad_output = grad_output.contiguous()
        device = _lib.require_device(hidden_states, grad_output)
        layer = _describe(options, hidden_states, weight_1, weight_2, ctx.with_losses, saved.dynamic_rows)
        layer.auxiliary_loss_grad, layer.z_loss_grad = ctx.loss_grads
        rows, hidden, ffn = layer.rows, layer.hidden, layer.ffn
        new = hidden_states.new_empty
        grad_layer_2_output = new((rows, hidden))
        grad_scores = new(layer.tokens * (options.experts_per_token + options.shared_experts), dtype=torch.float32)
        layer.routing, layer.layer_2_output = routing.data_ptr(), saved.layer_2_output.data_ptr()
        layer.grad_output, layer.grad_layer_2_output = grad_output.data_ptr(), grad_layer_2_output.data_ptr()
        layer.grad_scores = grad_scores.data_ptr()
        if saved.layer_2_output.nbytes >= _LARGE_BUFFER:
            layer.backward_part = 1
            _lib.call("fm_moe_layer_backward", device, _lib.ctypes.byref(layer))
            saved.layer_2_output, layer.backward_part = None, 2
        workspace = new(layer.workspace_bytes, dtype=torch.uint8)
        sparse_input, layer_1_output, activation_output = saved.sparse_input, saved.layer_1_output, saved.activation_output
        if sparse_input is None:
            sparse_input, layer.recompute_input = new((rows, hidden)), True
        if layer_1_output is None:
            layer_1_output, layer.recompute_layer_1 = new((rows, ffn * 2 if options.gated else ffn)), True
        if activation_output is None:
            activation_output, layer.recompute_activation = new((rows, ffn)), True
        grad_activation_output, grad_layer_1_output = new((rows, ffn)), new(layer_1_output.shape)
        grad_logits = new(logits.shape)
        layer.logits, layer.noise, layer.input = logits.data_ptr(), _lib.ptr(noise), hidden_states.data_ptr()
        layer.workspace, layer.sparse_input = workspace.data_ptr(), sparse_input.data_ptr()
        layer.layer_1_output, layer.activation_output = layer_1_output.data_ptr(), activation_output.data_ptr()
        layer.grad_activation_output = grad_activation_output.data_ptr()
        layer.grad_layer_1_output, layer.grad_logits = grad_layer_1_output.data_ptr(), grad_logits.data_ptr()
        grad_input = None
        if ctx.needs_input_grad[0]:
            grad_input = new(hidden_states.shape)
            layer.grad_input = grad_input.data_ptr()
        trained = [weight for weight in (weight_1, weight_2) if weight.requires_grad]
        targets = _gradient_targets(trained)
        for weight, target in zip(trained, targets):
            layer.grad_dtype = _lib.DTYPES[target.dtype]
            accumulate = target is weight.grad_buffer and not param_get_and_unset_is_zero(weight)
            if weight is weight_1:
                layer.grad_weight_1, layer.accumulate_1 = target.data_ptr(), accumulate
            else:
                layer.grad_weight_2, layer.accumulate_2 = target.data_ptr(), accumulate
        # The router's linear layer: with the rest, or in torch for sizes the library does not take. Half-precision input
        # gradients of more than 128 experts are torch's too: there the library has 256 x 256 tiles for them.
        grad_router = None
        if hidden_states.data_ptr() % 16 != 0 or router.data_ptr() % 16 != 0:
            layer.router_linear = False
        if layer.router_linear:
            layer.router = router.data_ptr()
            if layer.dtype == 0:
                layer.router_input_grad = 1
            elif options.routed_experts <= 128 and layer.tokens < 2**23:
                layer.router_input_grad = 2  # rounded as torch's is
            if ctx.needs_input_grad[1]:
                grad_router = torch.empty_like(router)
                layer.grad_router = grad_router.data_ptr()
        _lib.call("fm_moe_layer_backward", device, _lib.ctypes.byref(layer))
        del saved, sparse_input, layer_1_output, activation_output, workspace
        del grad_layer_2_output, grad_activation_output, grad_layer_1_output
        for weight, target in zip(trained, targets):
            if target is not weight.grad_buffer:
                accumulate_gradient(weight, target)
        if not layer.router_linear and ctx.needs_input_grad[1]:
            grad_router = torch.mm(grad_logits.t(), hidden_states)
        if not layer.router_input_grad and grad_input is not None:
            # Rounded, then added: what autograd makes of the two gradients where the layer is composed of its parts.
            grad_input.add_(torch.mm(grad_logits, router))
        return (grad_input, grad_router) + (None,) * 7


def moe_layer(
    hidden_states: torch.Tensor,
    router: torch.Tensor,
    weight_1: torch.Tensor,
    weight_2: torch.Tensor,
    options: MoELayerOptions,
    *,
    training: bool,
    noise: torch.Tensor | None = None,
    with_losses: bool = False,
    auxiliary_loss_grad: float = 0.0,
    z_loss_grad: float = 0.0,
) -> tuple[torch.Tensor, torch.Tensor | None]:
    """
    `hidden_states` [tokens, hidden] -> (output, [load-balancing loss, z-loss] or None). Weight layouts as in
    `layers.moe.DroplessMoEMLP`; the expert weights' gradients go to their grad buffers. The two loss gradients are those
    of `functional.routing.router` and need `with_losses`. Without `training` nothing is kept for a backward.
    """
    hidden_states = hidden_states.contiguous()
    if training:
        return _MoELayer.apply(
            hidden_states, router, weight_1, weight_2, noise, options, with_losses, (auxiliary_loss_grad, z_loss_grad), ANCHOR
        )
    with torch.no_grad():
        output, losses, _ = _forward(options, hidden_states, router, weight_1, weight_2, noise, with_losses, training=False)
    return without_backward(output), losses
