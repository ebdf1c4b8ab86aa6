"""The backward of the router's linear layer against the same products in fp64."""

import pytest
import torch

from fast_llm_amd import _lib
from tests.helpers import max_rel_err

pytestmark = pytest.mark.gpu


# One piece of the token axis and many (pieces are whole slices of 64 tokens, 128 at least), with a last slice of every kind;
# experts and columns around the tiles of 32 (fp32) and 256.
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize(
    ("tokens", "experts", "hidden"),
    [(1, 8, 64), (31, 16, 72), (33, 64, 8), (257, 72, 136), (300, 128, 56), (513, 136, 64), (5000, 8, 264), (4099, 256, 192)],
)
def test_router_linear_backward(tokens, experts, hidden, dtype, library, device):
    generator = torch.Generator().manual_seed(tokens)
    grad_logits = torch.randn(tokens, experts, generator=generator).to(dtype)
    input_ = torch.randn(tokens, hidden, generator=generator).to(dtype)
    weight = torch.randn(experts, hidden, generator=generator).to(dtype)
    previous = torch.randn(tokens, hidden, generator=generator).to(dtype)
    size = library.fm_router_linear_backward_workspace_size(tokens, experts, hidden, _lib.dtype_tag(dtype))
    workspace = torch.empty(size, dtype=torch.uint8, device=device)
    grad_input, grad_weight = previous.to(device), torch.full((experts, hidden), float("nan"), dtype=dtype, device=device)
    operands = [tensor.to(device) for tensor in (grad_logits, input_, weight)]
    _lib.check(
        library.fm_router_linear_backward(
            *(tensor.data_ptr() for tensor in (*operands, grad_input, grad_weight)), tokens, experts, hidden,
            _lib.dtype_tag(dtype), workspace.data_ptr(), size, torch.cuda.current_stream(device).cuda_stream,
        )
    )  # fmt: skip
    # One rounding to the type after sums of exact products in fp32.
    bound = {torch.float32: 1e-5, torch.bfloat16: 2**-8, torch.float16: 2**-11}[dtype]
    assert max_rel_err(grad_weight.cpu(), grad_logits.double().t() @ input_.double()) <= bound
    assert max_rel_err(grad_input.cpu(), previous.double() + grad_logits.double() @ weight.double()) <= bound


def test_router_linear_backward_refuses_what_it_cannot_vectorise(library):
    for experts, hidden in ((60, 64), (64, 60)):
        assert library.fm_router_linear_backward_workspace_size(100, experts, hidden, 1) == 0
        status = library.fm_router_linear_backward(256, 256, 256, None, 256, 100, experts, hidden, 1, 256, 1 << 20, None)
        assert status == _lib.FM_ERR_UNSUPPORTED
