"""fp32 products on operands split into bf16 parts: every tile shape against 64 bits, and operands that the parts cannot hold."""

import pytest
import torch

from fast_llm_amd.functional.sparse_copy import SparseMap
from fast_llm_amd.functional.sparse_linear import dense_matmul, input_row_sparse_matmul

pytestmark = pytest.mark.gpu

# Columns with 200 rows (two row tiles of 128, four of 64) for tiles of 64 x 64, 128 x 64 and 128 x 128, each with a remainder.
_COLUMNS = {"64x64": 2564, "128x64": 33028, "128x128": 82052}


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
@pytest.mark.parametrize("inner", [4, 16, 20, 64, 132])
@pytest.mark.parametrize("rhs_along_k", [True, False])
def test_tiles(tile, inner, rhs_along_k, device):
    lhs, rhs = _operands(_COLUMNS[tile], inner, device, rhs_along_k)
    out = dense_matmul(lhs, rhs)
    _check(out, lhs, rhs)
    twice = dense_matmul(lhs, rhs, out.clone(), accumulate=True)
    assert torch.equal(twice, out + out)


@pytest.mark.parametrize("columns", [68, 132, 4100])
def test_row_sparse(columns, device):
    """Reductions of 0, 1, 200 and 383 rows, NaN in the padding, both tile shapes."""
    rows, ends = [0, 1, 200, 383], [0, 128, 384, 768]
    sparse_map = SparseMap(
        None, torch.tensor(ends, dtype=torch.int32, device=device),
        torch.tensor([0, 1, 128 + 200, 384 + 383], dtype=torch.int32, device=device), None, 768, None, 4, None,
    )  # fmt: skip
    generator = torch.Generator(device).manual_seed(columns)
    x = torch.full((768, 260), float("nan"), device=device)
    y = torch.full((768, columns), float("nan"), device=device)
    for end, count, begin in zip(ends, rows, [0, *ends]):
        x[begin : begin + count].normal_(generator=generator)
        y[begin : begin + count].normal_(generator=generator)
    out = input_row_sparse_matmul(x.t(), y, sparse_map)
    for expert, (count, begin) in enumerate(zip(rows, [0, *ends])):
        _check(out[expert * 260 : (expert + 1) * 260], x[begin : begin + count].t(), y[begin : begin + count])


@pytest.mark.parametrize("tile", _COLUMNS)
def test_values_that_bf16_parts_cannot_hold(tile, device):
    """Infinities, NaN, values that bf16 rounds to infinity and values whose parts lie below bf16: as by fp32 multiply-adds."""
    inner = 48
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
    inner = 48
    lhs, rhs = (x.sign() * (1 + x.abs() % 1) for x in _operands(_COLUMNS[tile], inner, device, True))
    lhs, rhs = lhs * 2.0**lhs_exponent, rhs * 2.0**rhs_exponent
    multiply_adds = max(lhs_exponent, rhs_exponent) >= 102 or lhs_exponent + rhs_exponent >= 72
    _check(dense_matmul(lhs, rhs), lhs, rhs, multiply_adds)
    # Among operands of ordinary size: a row and a column of these, a row of them here and there.
    mixed_lhs, mixed_rhs = _operands(_COLUMNS[tile], inner, device, True)
    mixed_lhs[77], mixed_lhs[130, ::5], mixed_rhs[:, 33] = lhs[77], lhs[130, ::5], rhs[:, 33]
    _check(dense_matmul(mixed_lhs, mixed_rhs), mixed_lhs, mixed_rhs, multiply_adds)


def test_subnormal_operands(device):
    lhs, rhs = _operands(_COLUMNS["64x64"], 48, device, True)
    lhs *= 2.0**-140
    out = dense_matmul(lhs, rhs * 2.0**100)
    assert out.abs().max() > 0
    _check(out, lhs, rhs * 2.0**100)
