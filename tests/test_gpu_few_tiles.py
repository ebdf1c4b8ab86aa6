"""Products of few tiles (128 rows x 64 columns), and of the kernels that take over with more columns, against fp64, at the edges of their
tiles, slices and of the rule that picks them."""

import pytest
import torch

from fast_llm_amd import _lib

pytestmark = pytest.mark.gpu

_ROUND = {torch.bfloat16: 2**-8, torch.float16: 2**-11}


# Columns: with the 7 and 8 row tiles here, few tiles up to 2056, streamed products with more; with 12296 256 x 256
# tiles in the dense product. Inner: slices of 64 that are whole, and not; one slice, two (the slots in LDS) and more.
@pytest.mark.parametrize("dtype", list(_ROUND))
@pytest.mark.parametrize("contiguous_k", [True, False], ids=["k", "columns"])
@pytest.mark.parametrize("inner", [8, 72, 128, 448])
@pytest.mark.parametrize("cols", [8, 136, 2056, 5000, 7688, 12296])
@pytest.mark.parametrize("counts", [(127, 0, 1, 129, 256), None], ids=str)
def test_against_fp64(counts, cols, inner, contiguous_k, dtype, library, device):
    _check(counts, cols, inner, contiguous_k, dtype, library, device)


# More than 256 experts, of which a third has rows: 101 and 202 tiles of 128 x 256, for tiles of 128 and 256 columns.
MANY = tuple(e * 37 % 128 + 1 if e % 3 == 0 else 0 for e in range(300))


@pytest.mark.parametrize("dtype", list(_ROUND))
@pytest.mark.parametrize("contiguous_k", [True, False], ids=["k", "columns"])
@pytest.mark.parametrize("inner", [8, 72, 128, 448])
@pytest.mark.parametrize("cols", [8, 136, 256, 264, 504])
def test_many_experts_against_fp64(cols, inner, contiguous_k, dtype, library, device):
    _check(MANY, cols, inner, contiguous_k, dtype, library, device)


def _check(counts, cols, inner, contiguous_k, dtype, library, device):
    generator = torch.Generator(device).manual_seed(cols + inner)
    experts = len(counts) if counts else 1
    pad = 128
    begins, ends, at = [], [], 0
    for count in counts or (1009,):
        begins.append(at)
        at += -(-count // pad) * pad if counts else count
        ends.append(at)
    rows = at + (pad if counts else 0)  # a static map: rows behind the last expert
    # What nobody reads is NaN: padding rows, and the rest of the last line of either operand.
    owned = torch.zeros(rows, dtype=torch.bool)
    for begin, count in zip(begins, counts or (1009,), strict=True):
        owned[begin : begin + count] = True
    owned = owned.to(device)
    lhs = torch.randn(rows, inner + 8, generator=generator, device=device).to(dtype)
    lhs[:, inner:] = lhs[~owned] = float("nan")
    rhs = torch.randn(experts, cols, inner, generator=generator, device=device).to(dtype)
    out = torch.full((rows, cols), 7.0, dtype=dtype, device=device)
    pads = torch.tensor([b + c for b, c in zip(begins, counts or (1009,), strict=True)], dtype=torch.int32, device=device)
    ends_ = torch.tensor(ends, dtype=torch.int32, device=device)
    if contiguous_k:  # output-sparse: the weights side by side
        weight = torch.full((experts * cols, inner + 8), float("nan"), dtype=dtype, device=device)
        weight[:, :inner] = rhs.reshape(-1, inner)
        _lib.check(
            library.fm_output_sparse_matmul(
                lhs.data_ptr(), weight.data_ptr(), out.data_ptr(), ends_.data_ptr() if counts else None, rows, cols, inner, experts,
                inner + 8, 1, 1, inner + 8, cols, 1, 0, _lib.dtype_tag(dtype), _lib.dtype_tag(dtype), 1, None, 0,
                torch.cuda.current_stream(device).cuda_stream,
            )
        )  # fmt: skip
    else:  # input-inner-sparse: the weights one after the other along K
        weight = torch.full((experts * inner, cols + 8), float("nan"), dtype=dtype, device=device)
        weight[:, :cols] = rhs.transpose(1, 2).reshape(-1, cols)
        _lib.check(
            library.fm_input_inner_sparse_matmul(
                lhs.data_ptr(), weight.data_ptr(), out.data_ptr(), ends_.data_ptr() if counts else None, rows, cols, inner, experts,
                inner + 8, 1, cols + 8, 1, cols, 1, 0, _lib.dtype_tag(dtype), _lib.dtype_tag(dtype), 1, None, 0,
                torch.cuda.current_stream(device).cuda_stream,
            )
        )  # fmt: skip
    for expert, (begin, count) in enumerate(zip(begins, counts or (1009,), strict=True)):
        a, b = lhs[begin : begin + count, :inner].double(), rhs[expert].double()
        exact = a @ b.t()
        # Sums of exact products in fp32, in any order, and one rounding to the type.
        bound = _ROUND[dtype] * exact.abs() + (inner + 8) * 2**-24 * (a.abs() @ b.abs().t())
        assert ((out[begin : begin + count].double() - exact).abs() <= bound).all()
    assert (out[ends[-1] :] == 7).all()  # rows of no expert
