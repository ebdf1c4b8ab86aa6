"""
What is measured: the dropless mixture-of-experts layer at the sizes it is used at.

Every case is one pass through `DroplessMoEMLP`, the layer that a model holds, with the router inside: an inference
forward, or a training step's forward and backward (all gradients: input, router, both expert weights). Shapes are the
benchmark's (`fast_llm_amd.workloads.WORKLOADS`) and generic ones; token counts run from one generated token to the
benchmark's 16384, mostly odd, since prompts and packed micro-batches are.
"""

import torch

from fast_llm_amd.functional.config import ActivationType, MLPRecomputeLevel
from fast_llm_amd.layers.moe import DroplessMoEMLP

_DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
# hidden, ffn, routed experts, experts per token
_MIXTRAL, _FINE_GRAINED, _WIDE = (4096, 14336, 8, 2), (2048, 1408, 64, 6), (2048, 768, 128, 8)


def _case(mode: str, tokens: int, shape: tuple[int, int, int, int], dtype: str = "bf16", **options) -> dict:
    case = {
        "mode": mode,  # "infer" or "train"
        "tokens": tokens,
        "hidden": shape[0],
        "ffn": shape[1],
        "experts": shape[2],
        "experts_per_token": shape[3],
        "dtype": dtype,
        "shared_experts": 0,
        "zipf": 0.0,  # > 0: experts are preferred by a per-expert bias log(p_e), p_e ~ (e + 1) ** -zipf
        "gated": True,
        "activation": "silu",
        "recompute": "none",
        "full_precision_gradients": False,
        "micro_batches": 1,  # accumulated in the gradient buffers
        "dynamic_shape": False,
    }
    assert set(options) <= set(case)
    return {**case, **options}


def listed() -> list[dict]:
    cases = {
        # Text generation for one user: two experts' weights are read for one token. Latency and launches count.
        "decode_1": _case("infer", 1, _MIXTRAL),
        # Batched generation: every expert is read, for a handful of tokens each.
        "decode_64": _case("infer", 64, _MIXTRAL),
        # The same with many small experts.
        "decode_wide": _case("infer", 96, _WIDE),
        # One prompt of a narrow topic, which prefers a few experts; half precision as many checkpoints are served in.
        "prefill_imbalanced": _case("infer", 1531, _MIXTRAL, "fp16", zipf=1.2),
        # Several prompts at once, many small experts.
        "prefill_fine_grained": _case("infer", 5001, _FINE_GRAINED),
        # The smallest benchmark configuration: tests and debugging runs in single precision.
        "train_tiny_fp32": _case("train", 512, (256, 512, 8, 2), "fp32"),
        # A small model trained in single precision (numerics studies, parity runs).
        "train_fp32": _case("train", 2048, (1024, 2816, 8, 2), "fp32"),
        # A short micro-batch of the widest configuration, two of them accumulated into fp32 gradients, as a training
        # engine with full-precision gradients does.
        "train_wide_short": _case("train", 1999, _WIDE, full_precision_gradients=True, micro_batches=2),
        # A feed-forward size by the 8/3 rule, rounded to what a vector load needs and to no tile; odd token count.
        "train_ragged": _case("train", 3001, (1280, 3416, 16, 2)),
        # The benchmark's headline workload.
        "train_mixtral": _case("train", 8192, _MIXTRAL),
        # Many experts of which one is shared, memory-saving training: everything recomputed, fp32 gradients.
        "train_fine_grained": _case(
            "train", 16384, _FINE_GRAINED, shared_experts=1, recompute="full", full_precision_gradients=True
        ),
        # The widest benchmark configuration.
        "train_wide": _case("train", 16384, _WIDE),
    }
    return [{"name": name, **case} for name, case in cases.items()]


def _log_uniform(rng, low: int, high: int, multiple: int = 1) -> int:
    value = low * (high / low) ** rng.random()
    return max(low, min(high, round(value / multiple) * multiple))


# No case does more than the benchmark's headline workload, in matrix products or in weights; no ragged one does more
# than the listed ragged one (layers of such sizes are small).
_MAX_FLOPS = 18 * 8192 * 2 * 4096 * 14336
_MAX_RAGGED_FLOPS = 18 * 3001 * 2 * 1280 * 3416
_MAX_WEIGHTS = 8 * 3 * 4096 * 14336


def draw(rng) -> dict:
    while True:
        kind = rng.choice(("decode", "decode", "prefill", "prefill", "train", "train", "train", "train_fp32"))
        if kind == "train_fp32":
            shape = (_log_uniform(rng, 256, 1024, 64), _log_uniform(rng, 512, 2816, 64), rng.choice((4, 8, 16)), 2)
            tokens, dtype = _log_uniform(rng, 64, 2048), "fp32"
        else:
            if rng.random() < 0.5:
                shape = rng.choice((_MIXTRAL, _FINE_GRAINED, _WIDE))
            else:
                multiple = 8 if rng.random() < 0.25 else 64
                hidden = _log_uniform(rng, 512, 4096, multiple)
                ffn = _log_uniform(rng, 512, 8192, multiple)
                # One expert per token: served, but the router's softmax over one logit has no gradient to train with.
                per_token = rng.choice((2, 4, 6, 8) if kind == "train" else (1, 2, 4, 6, 8))
                shape = (hidden, ffn, rng.choice((8, 16, 32, 60, 64, 128)), per_token)
            low, high = (1, 256) if kind == "decode" else (256, 16384)
            tokens, dtype = _log_uniform(rng, low, high), rng.choice(("bf16", "bf16", "bf16", "fp16"))
        options = {"zipf": rng.choice((0.0, 0.0, 0.6, 1.2)), "dynamic_shape": rng.random() < 0.1}
        if dtype != "fp32":
            options["shared_experts"] = rng.choice((0, 0, 0, 1))
            options["gated"] = rng.random() < 0.85
            options["activation"] = rng.choice(("silu", "silu", "gelu", "squared_relu"))
        if kind.startswith("train"):
            options["recompute"] = rng.choice(("none", "none", "activation", "activation_and_input", "full"))
            options["full_precision_gradients"] = rng.random() < 0.3
            options["micro_batches"] = rng.choice((1, 1, 2))
        case = _case("train" if kind.startswith("train") else "infer", tokens, shape, dtype, **options)
        ragged = case["hidden"] % 64 != 0 or case["ffn"] % 64 != 0
        if work(case)["flops"] <= (_MAX_RAGGED_FLOPS if ragged else _MAX_FLOPS) and _weights(case) <= _MAX_WEIGHTS:
            return case


def _weights(case: dict) -> int:
    """Elements of the expert weights."""
    experts = case["experts"] + case["shared_experts"]
    return experts * case["hidden"] * case["ffn"] * (3 if case["gated"] else 2)


def prepare(case: dict, seed: int) -> dict:
    """The layer with its weights, and the micro-batches' inputs (and output gradients)."""
    torch.manual_seed(seed)  # seeds the layer's own initialisation
    device, dtype = torch.device("cuda"), _DTYPES[case["dtype"]]
    training = case["mode"] == "train"
    layer = DroplessMoEMLP(
        case["hidden"],
        case["ffn"],
        case["experts"] + case["shared_experts"],
        case["experts_per_token"],
        gated=case["gated"],
        activation=ActivationType(case["activation"]),
        recompute_level=MLPRecomputeLevel(case["recompute"]),
        dropless_dynamic_shape=case["dynamic_shape"],
        shared_experts=case["shared_experts"],
        full_precision_gradients=case["full_precision_gradients"],
        dtype=dtype,
        device=device,
    ).train(training)
    generator = torch.Generator(device).manual_seed(seed)

    def normal() -> torch.Tensor:
        return torch.randn((case["tokens"], case["hidden"]), generator=generator, device=device).to(dtype)

    batches = []
    for _ in range(case["micro_batches"]):
        input_ = normal()
        if case["zipf"] > 0:
            input_[:, 0] = 1  # the feature that carries the router's preference
        batches.append((input_.requires_grad_(training), normal() if training else None))
    if case["zipf"] > 0:
        probabilities = torch.arange(1, case["experts"] + 1, device=device) ** -case["zipf"]
        with torch.no_grad():
            layer.router[:, 0] = (probabilities / probabilities.sum()).log()
    return {"layer": layer, "batches": batches, "training": training}


def run(state: dict):
    """One inference forward, or the forward and backward of one training step."""
    layer, batches = state["layer"], state["batches"]
    if not state["training"]:
        with torch.no_grad():
            return layer(batches[0][0])
    layer.router.grad = None
    layer.layer_1.param_grad_is_zero = layer.layer_2.param_grad_is_zero = True
    outputs, input_grads = [], []
    for input_, output_grad in batches:
        input_.grad = None
        output = layer(input_, grad_scale=1.0)
        output.backward(output_grad)
        outputs.append(output.detach())
        input_grads.append(input_.grad)
    return {
        "outputs": outputs,
        "input_grads": input_grads,
        "router_grad": layer.router.grad,
        "layer_1_grad": layer.layer_1.grad_buffer,
        "layer_2_grad": layer.layer_2.grad_buffer,
    }


def work(case: dict) -> dict:
    """Matrix products on the rows that exist (no padding), the router's included; weights of the experts that some
    token is expected to select, read once per pass, everything else that goes in and comes out once."""
    tokens, hidden, ffn = case["tokens"] * case["micro_batches"], case["hidden"], case["ffn"]
    slots = case["experts_per_token"] + case["shared_experts"]
    size = 4 if case["dtype"] == "fp32" else 2
    products = 2 * tokens * slots * hidden * ffn
    layer_1, layer_2 = products * (2 if case["gated"] else 1), products
    router = 2 * tokens * hidden * case["experts"]
    total = _weights(case)
    if case["mode"] == "infer":
        missed = (1 - case["experts_per_token"] / case["experts"]) ** tokens
        read = total * ((1 - missed) * case["experts"] + case["shared_experts"]) / (case["experts"] + case["shared_experts"])
        return {
            "flops": layer_1 + layer_2 + router,
            "bytes": size * (read + case["experts"] * hidden + 2 * tokens * hidden),
        }
    grad_size = 4 if case["full_precision_gradients"] else size
    recomputed = layer_1 if case["recompute"] == "full" else 0
    return {
        "flops": 3 * (layer_1 + layer_2 + router) + recomputed,
        "bytes": (size + grad_size) * total + size * (2 * case["experts"] * hidden + 4 * tokens * hidden),
    }


def tolerance(case: dict) -> dict:
    """About four times the distance of the layer's results from the same computation in 64 bits (largest seen over the
    listed and some drawn cases: bf16 rel 5.8e-3, max 0.22; fp16 6.6e-4, 9.8e-3; fp32 1.6e-6, 1.2e-5)."""
    return {
        "fp32": {"rel": 1e-5, "max": 5e-5},
        "bf16": {"rel": 2.3e-2, "max": 0.9},
        "fp16": {"rel": 2.6e-3, "max": 4e-2},
    }[case["dtype"]]
