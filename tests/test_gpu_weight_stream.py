"""Products with the weights of experts of few rows: small whole numbers, whose sums are exact in any order."""

import pytest
import torch

from fast_llm_amd.functional.config import ActivationType, KernelConfig
from fast_llm_amd.functional.sparse_linear import input_inner_sparse_matmul, output_sparse_matmul
from fast_llm_amd.layers.moe import DroplessMoEMLP
from tests.helpers import fixture_sparse_map, to_device_map

pytestmark = pytest.mark.gpu

# Around the ends of a wavefront's rows (64; 96 in tall tiles) and of a tile (128; 192).
_FEW = [0, 1, 31, 33, 64, 65, 96, 127, 128, 129, 192, 200, 256, 257, 320, 0]
_MORE = [0, 1, 63, 65, 95, 97, 128, 129, 160, 161, 191, 192, 193, 224, 256, 257, 320, 384, 385, 577]


def _map(experts, tall):
    tokens = [_MORE[e % len(_MORE)] if tall else _FEW[e % len(_FEW)] if e < 48 else e % 7 for e in range(experts)]
    ends, used = [], 0
    for count in tokens:
        used += -(-count // 128) * 128
        ends.append(used)
    return fixture_sparse_map({"expert_ends": ends, "tokens_per_expert": tokens})


# Reductions of one slice, of no whole slice, of two and of several; columns of one tile and of a remainder.
PRODUCTS = [
    (256, 64, 1288, False), (128, 8, 1544, False), (70, 72, 2056, False), (64, 128, 2304, False), (33, 392, 4104, False),
    (128, 520, 1280, False), (40, 8, 1288, True), (64, 64, 1032, True), (20, 136, 2312, True), (40, 520, 3080, True),
]  # fmt: skip
STRIDED, STRIDED_INNER, STRIDED_COLUMNS = [(70, False), (40, True)], 136, 1288
DENSE = [(1, 64, 24840), (129, 200, 16392), (1601, 136, 2048), (3000, 64, 2568)]


@pytest.mark.parametrize(("experts", "inner", "columns", "tall"), PRODUCTS)
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_products_are_exact(experts, inner, columns, tall, dtype, device):
    oracle_map = _map(experts, tall)
    generator = torch.Generator(device).manual_seed(experts + inner + columns)

    def whole(*shape):
        return torch.randint(-2, 3, shape, generator=generator, device=device).to(dtype)

    sparse_map = to_device_map(oracle_map, device, torch.int32)
    x = whole(oracle_map.num_rows, inner)
    by_column, by_row = whole(experts * columns, inner), whole(experts * inner, columns)
    output = output_sparse_matmul(x, by_column.t(), sparse_map)
    input_ = input_inner_sparse_matmul(x, by_row, sparse_map)
    begin = 0
    for expert in range(experts):
        end = int(oracle_map.expert_ends[expert])
        rows = x[begin:end].float()
        expected = rows @ by_column[expert * columns : (expert + 1) * columns].float().t()
        assert torch.equal(output[begin:end], expected.to(dtype)), expert
        expected = rows @ by_row[expert * inner : (expert + 1) * inner].float()
        assert torch.equal(input_[begin:end], expected.to(dtype)), expert
        begin = end


@pytest.mark.parametrize(("experts", "tall"), STRIDED)
@pytest.mark.parametrize("index_dtype", [torch.int32, torch.int64])
def test_strides_and_guards(experts, tall, index_dtype, device):
    oracle_map, inner, columns = _map(experts, tall), STRIDED_INNER, STRIDED_COLUMNS
    generator = torch.Generator(device).manual_seed(experts)

    def whole(rows, width, stride):
        return torch.randint(-2, 3, (rows, stride), generator=generator, device=device).bfloat16()[:, :width]

    sparse_map = to_device_map(oracle_map, device, index_dtype)
    x = whole(oracle_map.num_rows, inner, inner + 8)
    by_column, by_row = whole(experts * columns, inner, inner + 24), whole(experts * inner, columns, columns + 16)
    kept = torch.full((2, oracle_map.num_rows + 1, columns + 8), 7.0, device=device, dtype=torch.bfloat16)
    output_sparse_matmul(x, by_column.t(), sparse_map, out=kept[0, :-1, :columns])
    input_inner_sparse_matmul(x, by_row, sparse_map, out=kept[1, :-1, :columns])
    begin = 0
    for expert in range(experts):
        end = int(oracle_map.expert_ends[expert])
        expected = x[begin:end].float() @ by_column[expert * columns : (expert + 1) * columns].float().t()
        assert torch.equal(kept[0, begin:end, :columns], expected.bfloat16()), expert
        expected = x[begin:end].float() @ by_row[expert * inner : (expert + 1) * inner].float()
        assert torch.equal(kept[1, begin:end, :columns], expected.bfloat16()), expert
        begin = end
    assert (kept[:, :, columns:] == 7).all() and (kept[:, -1] == 7).all()  # nothing outside of the results


@pytest.mark.parametrize(("rows", "inner", "columns"), DENSE)
def test_dense_products_are_exact(rows, inner, columns, device):
    generator = torch.Generator(device).manual_seed(rows)
    x = torch.randint(-2, 3, (rows, inner), generator=generator, device=device).bfloat16()
    for weight in (torch.empty(columns, inner, device=device).t(), torch.empty(inner, columns, device=device)):
        weight = torch.randint_like(weight, -2, 3).bfloat16()
        assert torch.equal(output_sparse_matmul(x, weight), (x.float() @ weight.float()).bfloat16())


# More rows in one expert than tiles x blocks of 32 rows have room for in 32 bits; columns that take tiles of 192 rows.
@pytest.mark.parametrize("columns", [128, 384])
def test_four_million_rows(columns, device):
    rows, inner = 4_000_000, 64
    generator = torch.Generator(device).manual_seed(columns)
    x = torch.randint(-2, 3, (rows, inner), generator=generator, device=device, dtype=torch.int8).bfloat16()
    weight = torch.randint(-2, 3, (columns, inner), generator=generator, device=device, dtype=torch.int8).bfloat16()
    kept = torch.full((rows + 2 * 192, columns), 7.0, device=device, dtype=torch.bfloat16)
    output_sparse_matmul(x, weight.t(), out=kept[192:-192])
    for begin in range(0, rows, 500_000):
        expected = x[begin : begin + 500_000].float() @ weight.float().t()
        assert torch.equal(kept[192 + begin : 192 + begin + 500_000], expected.bfloat16()), begin
    assert (kept[:192] == 7).all() and (kept[-192:] == 7).all()


WIDTHS = [(1000, 768), (1500, 1032), (2100, 200), (2900, 768), (3300, 1032)]


@pytest.mark.parametrize(("tokens", "ffn"), WIDTHS)
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("activation", [ActivationType.silu, ActivationType.gelu])
def test_activation_equals_two_kernels(tokens, ffn, dtype, activation, device, monkeypatch):
    torch.manual_seed(tokens + ffn)
    layer = DroplessMoEMLP(320, ffn, 128, 6, activation=activation, init_std=0.2, dtype=dtype, device=device).eval()
    x = torch.randn(tokens, 320, device=device).to(dtype)
    with torch.no_grad():
        output = layer(x)
        monkeypatch.setattr(KernelConfig, "fuse_activation", False)
        assert torch.equal(output, layer(x))
