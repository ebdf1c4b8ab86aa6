"""The router's logits by the kernel for few tokens, against 64 bits, and their gradients."""

import pytest
import torch
from torch._subclasses.fake_tensor import FakeTensorMode
from torch.fx.experimental.proxy_tensor import make_fx
from torch.overrides import TorchFunctionMode

from fast_llm_amd import _lib
from fast_llm_amd.functional import routing

pytestmark = pytest.mark.gpu

# Unit roundoff of the type a logit is rounded to: half a unit of the last of 24, 8 and 11 significant bits.
_ROUND = {torch.float32: 2**-24, torch.bfloat16: 2**-8, torch.float16: 2**-11}


@pytest.mark.parametrize("dtype", list(_ROUND))
@pytest.mark.parametrize(("tokens", "experts"), [(1, 1), (1, 8), (15, 16), (17, 17), (33, 60), (64, 128), (1024, 8), (1100, 3)])
@pytest.mark.parametrize("hidden", [8, 32, 40, 264, 2056, 4096])
def test_logits(dtype, tokens, experts, hidden, device):
    generator = torch.Generator(device).manual_seed(tokens + experts + hidden)
    x, weight = (torch.randn((rows, hidden), generator=generator, device=device).to(dtype) for rows in (tokens, experts))
    assert routing._few_logits(x, weight)
    logits = routing.router_logits(x, weight)
    assert logits.dtype == dtype and logits.shape == (tokens, experts)
    exact = x.double() @ weight.double().t()
    # One rounding of the result, and at most hidden + 8 of partial sums in fp32.
    bound = _ROUND[dtype] * exact.abs() + (hidden + 8) * 2**-24 * (x.double().abs() @ weight.double().abs().t())
    assert ((logits.double() - exact).abs() <= bound).all()


@pytest.mark.parametrize("dtype", list(_ROUND))
def test_gradients_are_those_of_linear(dtype, device):
    torch.manual_seed(0)
    x, weight = (torch.randn((rows, 72), device=device, dtype=dtype, requires_grad=True) for rows in (50, 24))
    grad = torch.randn((50, 24), device=device, dtype=dtype)
    results = []
    for function in (routing.router_linear, torch.nn.functional.linear):
        x.grad = weight.grad = None
        logits = function(x, weight)
        logits.backward(grad)
        results.append((x.grad, weight.grad))
    assert all(torch.equal(a, b) for a, b in zip(*results))
    with torch.no_grad():
        assert torch.equal(routing.router_linear(x, weight), routing.router_logits(x, weight))


@pytest.mark.parametrize("trained", ["input", "weight"])
def test_what_no_gradient_needs_may_change(trained, device):
    """As after torch's linear layer: the operand that no gradient is made from is neither kept nor watched."""
    x, weight = torch.randn((20, 64), device=device), torch.randn((8, 64), device=device)
    (x if trained == "input" else weight).requires_grad_()
    results = []
    for function in (routing.router_linear, torch.nn.functional.linear):
        x.grad = weight.grad = None
        x_, weight_ = (x * 1, weight) if trained == "input" else (x, weight * 1)
        kept = []
        with torch.autograd.graph.saved_tensors_hooks(lambda tensor: kept.append(tensor.data_ptr()) or tensor, lambda tensor: tensor):
            logits = function(x_, weight_)
        with torch.no_grad():
            (x_ if trained == "input" else weight_).add_(1)
        logits.sum().backward()
        results.append((x.grad if trained == "input" else weight.grad, len(kept)))
    assert torch.equal(results[0][0], results[1][0]) and results[0][1] == results[1][1] == 1


def test_what_the_kernel_does_not_take(device):
    x, weight = torch.randn((30, 68), device=device), torch.randn((8, 68), device=device)
    for operands in ((x[:, :66], weight[:, :66]), (x.t().contiguous().t(), weight), (x[:0], weight), (x[1:, 1:], weight[:, 1:])):
        assert not routing._few_logits(*operands)
        assert torch.equal(routing.router_linear(*operands), torch.nn.functional.linear(*operands))
    many = torch.randn((16 * (routing._MAX_LOGIT_BYTES // (68 * 4)) + 1, 68), device=device)
    assert not routing._few_logits(many, weight) and routing._few_logits(many[1:], weight)
    with torch.autocast("cuda", dtype=torch.bfloat16):
        assert routing.router_linear(x, weight).dtype == torch.bfloat16


@pytest.mark.parametrize(("tokens", "experts", "hidden"), [(3, 4097, 8), (3, 0, 64), (3, 8, 0)])
def test_sizes_that_the_kernel_refuses(tokens, experts, hidden, device):
    x, weight = torch.randn((tokens, hidden), device=device), torch.randn((experts, hidden), device=device)
    assert not routing._few_logits(x, weight)
    assert torch.equal(routing.router_linear(x, weight), torch.nn.functional.linear(x, weight))
    # Where tokens are few enough that only the number of experts decides.
    if experts > 0 and hidden > 0:
        assert routing._few_logits(x, weight[:4096])


def test_transforms_see_a_linear_layer(device):
    x, weight = torch.randn((20, 64), device=device), torch.randn((8, 64), device=device)
    assert routing._few_logits(x, weight)
    expected = torch.nn.functional.linear(x, weight)

    def loss(w):
        return routing.router_linear(x, w).square().sum()

    torch.testing.assert_close(torch.func.grad(loss)(weight), 2 * expected.t() @ x)
    torch.testing.assert_close(torch.func.vmap(routing.router_linear, (0, None))(x.view(4, 5, 64), weight).view(20, 8), expected)
    torch.testing.assert_close(torch.func.jvp(routing.router_linear, (x, weight), (x, weight))[1], 2 * expected)
    graph = make_fx(routing.router_linear)(x, weight)
    torch.testing.assert_close(graph(x + 1, weight), torch.nn.functional.linear(x + 1, weight))
    with FakeTensorMode():
        fake = routing.router_linear(torch.empty((20, 64), device=device), torch.empty((8, 64), device=device))
    assert fake.shape == (20, 8)
    compiled = torch.compile(routing.router_linear, backend="eager", fullgraph=True)
    torch.testing.assert_close(compiled(x, weight), expected)


class _Calls(TorchFunctionMode):
    def __init__(self):
        super().__init__()
        self.functions = []

    def __torch_function__(self, function, types, args=(), kwargs=None):
        self.functions.append(function)
        return function(*args, **(kwargs or {}))


def test_function_modes_see_a_linear_layer(device):
    x, weight = torch.randn((20, 64), device=device), torch.randn((8, 64), device=device)
    with _Calls() as mode:
        logits = routing.router_linear(x, weight)
    assert torch.nn.functional.linear in mode.functions and torch.equal(logits, torch.nn.functional.linear(x, weight))
    with torch.device(device):  # the mode of a default device looks for functions that make tensors
        assert torch.equal(routing.router_linear(x, weight), routing.router_logits(x, weight))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("experts", [8, 32, 40, 64, 72, 128])
@pytest.mark.parametrize(("tokens", "hidden"), [(1, 8), (15, 128), (17, 136), (64, 120), (257, 520), (300, 2056)])
def test_input_gradient_is_added(dtype, experts, tokens, hidden, device):
    """In place, nothing beside it touched, one rounding of the sum."""
    generator = torch.Generator(device).manual_seed(experts + tokens)
    normal = lambda *shape: torch.randn(shape, generator=generator, device=device).to(dtype)  # noqa: E731
    grad_logits, weight, around = normal(tokens, experts), normal(experts, hidden), normal(tokens + 2, hidden)
    grad_input = around.clone()[1:-1]
    whole = grad_input._base
    _lib.call(
        "fm_router_linear_backward", device, grad_logits.data_ptr(), None, weight.data_ptr(), grad_input.data_ptr(), None,
        tokens, experts, hidden, _lib.dtype_tag(dtype), None, 0,
    )  # fmt: skip
    assert torch.equal(whole[0], around[0]) and torch.equal(whole[-1], around[-1])
    exact = around[1:-1].double() + grad_logits.double() @ weight.double()
    # At most experts + 8 roundings of partial sums in fp32, and one of the result.
    partial = (experts + 8) * 2**-24 * (grad_logits.double().abs() @ weight.double().abs() + around[1:-1].double().abs())
    assert ((grad_input.double() - exact).abs() <= _ROUND[dtype] * (exact.abs() + partial) + partial).all()
