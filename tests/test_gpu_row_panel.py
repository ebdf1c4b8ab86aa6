"""Weight gradients of experts of few rows: small whole numbers, whose sums are exact in any order."""

import pytest
import torch

from fast_llm_amd.functional.sparse_linear import input_row_sparse_matmul
from tests.helpers import fixture_sparse_map, to_device_map

pytestmark = pytest.mark.gpu

# Around the ends of slices (32 rows) and of what stays in LDS (160 rows).
_TOKENS = [0, 1, 31, 32, 33, 64, 97, 128, 159, 160, 161, 192, 193, 320, 325, 0]


def _map(experts):
    tokens = [_TOKENS[e % len(_TOKENS)] if e < 32 else e % 7 for e in range(experts)]
    ends, used = [], 0
    for count in tokens:
        used += -(-count // 64) * 64
        ends.append(used)
    return fixture_sparse_map({"expert_ends": ends, "tokens_per_expert": tokens})


# 256 experts of 11 x 2 tiles are the fewest that take the kernel without adding; 257 are one too many for it. 1000 columns are no
# whole lines.
GRADIENTS = [
    (256, 1288, 264, False), (256, 1408, 512, False), (17, 30728, 1000, False), (257, 1288, 264, False),
    (16, 8, 8, True), (40, 136, 264, True), (17, 392, 1000, True), (256, 128, 256, True),
]  # fmt: skip


@pytest.mark.parametrize(("experts", "rows", "columns", "accumulate"), GRADIENTS)
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_gradients_are_exact(experts, rows, columns, accumulate, dtype, device):
    oracle_map = _map(experts)
    generator = torch.Generator(device).manual_seed(experts + rows + columns)

    def whole(*shape):
        return torch.randint(-2, 3, shape, generator=generator, device=device).to(dtype)

    grad, x = whole(oracle_map.num_rows, rows), whole(oracle_map.num_rows, columns)
    previous = whole(experts * rows, columns)
    padding = ~oracle_map.real_row_mask().to(device)
    grad[padding], x[padding] = float("nan"), float("nan")
    out = previous.clone() if accumulate else torch.full_like(previous, float("nan"))
    input_row_sparse_matmul(grad.t(), x, to_device_map(oracle_map, device, torch.int32), out=out, accumulate=accumulate)
    begin = 0
    for expert in range(experts):
        end, blocks = int(oracle_map.expert_pad_begins[expert]), slice(expert * rows, (expert + 1) * rows)
        expected = grad[begin:end].float().t() @ x[begin:end].float()
        if accumulate:
            expected += previous[blocks]
        assert torch.equal(out[blocks], expected.to(dtype)), expert
        begin = int(oracle_map.expert_ends[expert])
