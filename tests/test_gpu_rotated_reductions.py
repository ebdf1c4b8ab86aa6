"""Products whose experts start their reductions at different slices: small whole numbers, whose sums are exact in any order."""

import pytest
import torch

from fast_llm_amd.functional.sparse_linear import output_sparse_matmul
from oracle import moe_oracle
from tests.helpers import fixture_sparse_map, to_device_map

pytestmark = pytest.mark.gpu

_TOKENS = [1, 0, 128, 129, 300, 7, 256, 0, 257, 64, 5]


@pytest.mark.parametrize("slices", [1, 2, 3, 5, 12, 33])
@pytest.mark.parametrize("columns", [8, 264, 520])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_every_slice_counts_once(slices, columns, dtype, device):
    inner, experts = 64 * slices, len(_TOKENS)
    ends, used = [], 0
    for tokens in _TOKENS:
        used += -(-tokens // 128) * 128
        ends.append(used)
    oracle_map = fixture_sparse_map({"expert_ends": ends, "tokens_per_expert": _TOKENS})
    real = oracle_map.real_row_mask()
    generator = torch.Generator().manual_seed(slices + columns)
    x = torch.randint(-1, 2, (used, inner), generator=generator).to(dtype)
    weight = torch.randint(-1, 2, (experts * columns, inner), generator=generator).to(dtype)
    # One more weight per slice that nothing but its own slice can make up for.
    weight[:, ::64] *= 3
    expected = moe_oracle.output_sparse_matmul(x.float(), weight.float().t(), oracle_map).to(dtype)
    x[~real] = float("nan")
    out = output_sparse_matmul(x.to(device), weight.to(device).t(), to_device_map(oracle_map, device, torch.int32))
    assert torch.equal(out.cpu()[real], expected[real])
