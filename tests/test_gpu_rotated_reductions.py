"""Products whose experts start their reductions at different slices: small whole numbers, whose sums are exact in any order."""

import pytest
import torch

from fast_llm_amd import _lib
from fast_llm_amd.functional.config import ActivationType
from fast_llm_amd.functional.mlp import gated_layer_1_forward, gated_layer_2_input_backward, mlp_activation_backward
from fast_llm_amd.functional.sparse_linear import output_sparse_matmul
from oracle import moe_oracle
from tests.helpers import fixture_sparse_map, to_device_map

pytestmark = pytest.mark.gpu

_TOKENS = [1, 0, 128, 129, 300, 7, 256, 0, 257, 64, 5]


def _map(times=1):
    ends, used = [], 0
    for tokens in _TOKENS:
        used += -(-tokens * times // 128) * 128
        ends.append(used)
    return fixture_sparse_map({"expert_ends": ends, "tokens_per_expert": [tokens * times for tokens in _TOKENS]})


def _operands(oracle_map, columns, slices, dtype):
    """Whole numbers, NaN in the padding rows, and the product, rounded to `dtype`."""
    generator = torch.Generator().manual_seed(slices + columns)
    x = torch.randint(-1, 2, (oracle_map.num_rows, 64 * slices), generator=generator).to(dtype)
    weight = torch.randint(-1, 2, (len(_TOKENS) * columns, 64 * slices), generator=generator).to(dtype)
    # One more weight per slice that nothing but its own slice can make up for.
    weight[:, ::64] *= 3
    expected = moe_oracle.output_sparse_matmul(x.float(), weight.float().t(), oracle_map).to(dtype)
    x[~oracle_map.real_row_mask()] = float("nan")
    return x, weight, expected


# The 15 row tiles of 128 are few tiles up to 520 columns, and streamed products with 4616.
@pytest.mark.parametrize("slices", [1, 2, 3, 5, 12, 33])
@pytest.mark.parametrize("columns", [8, 264, 520, 4616])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_every_slice_counts_once(slices, columns, dtype, device):
    oracle_map = _map()
    real = oracle_map.real_row_mask()
    x, weight, expected = _operands(oracle_map, columns, slices, dtype)
    out = output_sparse_matmul(x.to(device), weight.to(device).t(), to_device_map(oracle_map, device, torch.int32))
    assert torch.equal(out.cpu()[real], expected[real])


# Five times as many rows: tiles of 256 x 256.
LARGE_TIMES, LARGE_COLUMNS = 5, 2568


@pytest.mark.parametrize("slices", [1, 2, 3, 5, 12, 33])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_every_slice_counts_once_on_large_tiles(slices, dtype, device):
    oracle_map = _map(LARGE_TIMES)
    real = oracle_map.real_row_mask()
    x, weight, expected = _operands(oracle_map, LARGE_COLUMNS, slices, dtype)
    out = output_sparse_matmul(x.to(device), weight.to(device).t(), to_device_map(oracle_map, device, torch.int32))
    assert torch.equal(out.cpu()[real], expected[real])


@pytest.mark.parametrize("slices", [1, 2, 3, 5, 12, 33])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_every_slice_counts_once_in_the_fused_products(slices, dtype, device):
    ffn, oracle_map = 256, _map()
    real, sparse_map = oracle_map.real_row_mask(), to_device_map(oracle_map, device, torch.int32)
    x, weight, expected = _operands(oracle_map, 2 * ffn, slices, dtype)
    layer_1, output = gated_layer_1_forward(x.to(device), weight.to(device), sparse_map, ActivationType.identity, True)
    assert torch.equal(layer_1.cpu()[real], expected[real])
    gate, up = expected[real].float().chunk(2, 1)
    assert torch.equal(output.cpu()[real], (gate * up).to(dtype))

    grad, weight, expected = _operands(oracle_map, ffn, slices, dtype)
    layer_1 = torch.randint(-3, 4, (oracle_map.num_rows, 2 * ffn)).to(device, dtype)
    grad_layer_1, _ = gated_layer_2_input_backward(
        grad.to(device), weight.to(device).t(), sparse_map, layer_1, ActivationType.identity, False
    )
    in_two, _ = mlp_activation_backward(expected.to(device), (layer_1, True, ActivationType.identity, sparse_map))
    assert torch.equal(grad_layer_1.cpu()[real], in_two.cpu()[real])


def test_axes_of_rows_that_overlap_start_at_their_beginning(library, device):
    """One row for all of them, of 2^21: an offset along a longer one would not fit its 32 bits. The exact sums are 0, the rounded ones
    tell in which order they were made."""
    inner, rows, columns = 2**21, 256, 8
    half = torch.randn((2, inner // 2), device=device).bfloat16()
    x, weight = torch.cat([half[0], -half[0]]), torch.cat([half[1], half[1]])
    ends = torch.tensor([128, 256], dtype=torch.int32, device=device)
    out = torch.empty((rows, columns), dtype=torch.bfloat16, device=device)
    _lib.check(
        library.fm_output_sparse_matmul(
            x.data_ptr(), weight.data_ptr(), out.data_ptr(), ends.data_ptr(), rows, columns, inner, 2, 0, 1, 1, 0, columns, 1, 0,
            _lib.dtype_tag(out.dtype), _lib.dtype_tag(out.dtype), 1, None, 0, torch.cuda.current_stream(device).cuda_stream,
        )
    )  # fmt: skip
    assert (out == out[0, 0]).all()
