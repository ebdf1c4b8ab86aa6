"""fp32 products on operands split into bf16 parts: every tile shape against 64 bits, and operands that the parts cannot hold."""

import itertools

import pytest
import torch

from fast_llm_amd.functional.sparse_copy import SparseMap
from fast_llm_amd.functional.sparse_linear import dense_matmul, input_inner_sparse_matmul, input_row_sparse_matmul, output_sparse_matmul

pytestmark = pytest.mark.gpu

# Columns with 200 rows (two row tiles of 128, four of 64) for tiles of 64 x 64, 128 x 64 and 128 x 128, each with a remainder, and the
# reductions from which on they are split: shorter ones are fp32 multiply-adds.
_COLUMNS = {"64x64": 12804, "128x64": 33028, "128x128": 82052}
_SPLIT_FROM = {"64x64": 256, "128x64": 192, "128x128": 128}


def _operands(columns, inner, device, rhs_along_k):
    generator = torch.Generator(device).manual_seed(columns + inner)
    lhs = torch.randn((200, inner), generator=generator, device=device)
    rhs = torch.randn((columns, inner), generator=generator, device=device)
    return lhs, rhs.t() if rhs_along_k else rhs.t().contiguous()


def _check(out, lhs, rhs, multiply_adds=False):
    """Worst case of the kernel: at most inner / 16 + 5 roundings of the large sum and as many, 2^-8 as large, of the small ones; parts
    left out are below 2^-25 of a product. Rounded up to inner / 16 + 8 units of 2^-24 of the sum of magnitudes, and the smallest
    fp32 number for results below the normal ones. fp32 multiply-adds round every two reduction indices."""
    exact = lhs.double() @ rhs.double()
    roundings = lhs.shape[1] / (2 if multiply_adds else 16) + 8
    bound = roundings * 2**-24 * (lhs.double().abs() @ rhs.double().abs()) + 2.0**-149
    assert ((out.double() - exact).abs() <= bound).all()


@pytest.mark.parametrize("tile", _COLUMNS)
@pytest.mark.parametrize("inner", [4, 16, 20, 64, 132, 192, 256, 260, 276, 324])
@pytest.mark.parametrize("rhs_along_k", [True, False])
def test_tiles(tile, inner, rhs_along_k, device):
    lhs, rhs = _operands(_COLUMNS[tile], inner, device, rhs_along_k)
    out = dense_matmul(lhs, rhs)
    _check(out, lhs, rhs, multiply_adds=inner < _SPLIT_FROM[tile])
    twice = dense_matmul(lhs, rhs, out.clone(), accumulate=True)
    assert torch.equal(twice, out + out)


@pytest.mark.parametrize("rows", [(0, 1, 200, 383), (0, 1, 1000, 2100)])
@pytest.mark.parametrize("columns", [68, 132, 1000, 2000, 4100])
def test_row_sparse(columns, rows, device):
    """Reductions of few and many rows, NaN in the padding: multiply-adds and, of many rows from 1000 columns on, the three tile shapes."""
    ends = list(itertools.accumulate(-(-count // 128) * 128 for count in rows))
    begins = [0, *ends[:-1]]
    sparse_map = SparseMap(
        None, torch.tensor(ends, dtype=torch.int32, device=device),
        torch.tensor([begin + count for begin, count in zip(begins, rows)], dtype=torch.int32, device=device), None, ends[-1], None, 4, None,
    )  # fmt: skip
    generator = torch.Generator(device).manual_seed(columns)
    x = torch.full((ends[-1], 380), float("nan"), device=device)
    y = torch.full((ends[-1], columns), float("nan"), device=device)
    for count, begin in zip(rows, begins):
        x[begin : begin + count].normal_(generator=generator)
        y[begin : begin + count].normal_(generator=generator)
    out = input_row_sparse_matmul(x.t(), y, sparse_map)
    for expert, (count, begin) in enumerate(zip(rows, begins)):
        lhs, rhs = x[begin : begin + count].t(), y[begin : begin + count]
        _check(out[expert * 380 : (expert + 1) * 380], lhs, rhs, multiply_adds=columns < 1000 or max(rows) < 1000)


# Tiles of 64 x 64, 128 x 64 and 128 x 128 by the rows that experts of the map's buffer are expected to have.
@pytest.mark.parametrize(("columns", "inner"), [(500, 772), (2500, 388), (4100, 196)])
@pytest.mark.parametrize("product", [output_sparse_matmul, input_inner_sparse_matmul])
def test_experts_of_few_rows(product, columns, inner, device):
    """0 to 40 rows, NaN in the padding."""
    rows = [7 * expert % 41 for expert in range(32)]
    ends = list(itertools.accumulate(-(-count // 128) * 128 for count in rows))
    begins = [0, *ends[:-1]]
    sparse_map = SparseMap(
        None, torch.tensor(ends, dtype=torch.int32, device=device),
        torch.tensor([begin + count for begin, count in zip(begins, rows)], dtype=torch.int32, device=device), None, ends[-1], None, 32, None,
    )  # fmt: skip
    generator = torch.Generator(device).manual_seed(columns)
    lhs = torch.full((ends[-1], inner), float("nan"), device=device)
    for count, begin in zip(rows, begins):
        lhs[begin : begin + count].normal_(generator=generator)
    weight = torch.randn((32, columns, inner), generator=generator, device=device)
    rhs = weight.flatten(0, 1).t() if product is output_sparse_matmul else weight.transpose(1, 2).reshape(-1, columns)
    out = product(lhs, rhs, sparse_map)
    for expert, (count, begin) in enumerate(zip(rows, begins)):
        _check(out[begin : begin + count], lhs[begin : begin + count], weight[expert].t())


@pytest.mark.parametrize(("rows", "cols", "inner"), [(2048, 1024, 8), (8192, 2048, 8), (16384, 8, 8), (16384, 32, 264), (24, 16384, 264)])
def test_short_reductions_and_narrow_sides_are_multiply_adds(rows, cols, inner, device):
    """Where splitting is the slower route: the same bits as in a product of one tile, which is never split."""
    lhs, rhs = torch.randn((rows, inner), device=device), torch.randn((inner, cols), device=device)
    few_rows, few_cols = lhs[:64], rhs[:, :64].contiguous()
    assert torch.equal(dense_matmul(lhs, rhs)[:64, :64], dense_matmul(few_rows, few_cols))


def test_few_gradient_tiles_are_multiply_adds(device):
    ends = torch.tensor([512, 1024, 1536, 2048], dtype=torch.int32, device=device)
    sparse_map = SparseMap(None, ends, ends, None, 2048, None, 4, None)
    x, y = torch.randn((2048, 64), device=device), torch.randn((2048, 128), device=device)
    out = input_row_sparse_matmul(x.t(), y, sparse_map)
    for expert in range(4):
        rows = slice(512 * expert, 512 * (expert + 1))
        assert torch.equal(out[64 * expert : 64 * (expert + 1)], dense_matmul(x[rows].t(), y[rows]))


@pytest.mark.parametrize("tile", _COLUMNS)
def test_values_that_bf16_parts_cannot_hold(tile, device):
    """Infinities, NaN, values that bf16 rounds to infinity and values whose parts lie below bf16: as by fp32 multiply-adds."""
    inner = 272
    lhs, rhs = _operands(_COLUMNS[tile], inner, device, True)
    infinite, nan, largest = 3, 70, 130  # rows, in different blocks
    lhs[infinite, 5] = float("inf")
    lhs[nan, 7] = float("nan")
    lhs[largest] = 0
    lhs[largest, 9] = torch.finfo(torch.float32).max
    rhs[9] = rhs[9].sign() * 0.5
    out = dense_matmul(lhs, rhs)
    assert torch.equal(out[infinite], float("inf") * rhs[5].sign())
    assert out[nan].isnan().all()
    assert torch.equal(out[largest], lhs[largest, 9] * rhs[9])
    rest = [row for row in range(200) if row not in (infinite, nan, largest)]
    _check(out[rest], lhs[rest], rhs)

    # Rows of one magnitude each, down to where the third part of a value would be below the smallest bf16.
    lhs, rhs = _operands(_COLUMNS[tile], inner, device, True)
    lhs *= 2.0 ** -torch.linspace(0, 118, 200, device=device).round()[:, None]
    _check(dense_matmul(lhs, rhs), lhs, rhs)
    lhs[:] = 0
    assert (dense_matmul(lhs, rhs) == 0).all()


# Operands with an exponent each, the smallest results below the smallest normal number. From 2^103 on (and sums from 2^80 on) the
# results are those of fp32 multiply-adds.
@pytest.mark.parametrize("tile", _COLUMNS)
@pytest.mark.parametrize(
    ("lhs_exponent", "rhs_exponent"),
    [(-112, 40), (-120, 60), (-126, 100), (100, -126), (-126, 120), (-112, 105), (60, 30), (-113, 0), (-124, 0), (0, -126), (-70, -70)],
)
def test_operands_of_all_magnitudes(tile, lhs_exponent, rhs_exponent, device):
    inner = 272
    lhs, rhs = (x.sign() * (1 + x.abs() % 1) for x in _operands(_COLUMNS[tile], inner, device, True))
    lhs, rhs = lhs * 2.0**lhs_exponent, rhs * 2.0**rhs_exponent
    multiply_adds = max(lhs_exponent, rhs_exponent) >= 102 or lhs_exponent + rhs_exponent >= 72
    _check(dense_matmul(lhs, rhs), lhs, rhs, multiply_adds)
    # Among operands of ordinary size: a row and a column of these, a row of them here and there.
    mixed_lhs, mixed_rhs = _operands(_COLUMNS[tile], inner, device, True)
    mixed_lhs[77], mixed_lhs[130, ::5], mixed_rhs[:, 33] = lhs[77], lhs[130, ::5], rhs[:, 33]
    _check(dense_matmul(mixed_lhs, mixed_rhs), mixed_lhs, mixed_rhs, multiply_adds)


def test_subnormal_operands(device):
    lhs, rhs = _operands(_COLUMNS["64x64"], 272, device, True)
    lhs *= 2.0**-140
    out = dense_matmul(lhs, rhs * 2.0**100)
    assert out.abs().max() > 0
    _check(out, lhs, rhs * 2.0**100)
