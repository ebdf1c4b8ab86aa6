"""The GPU tests of one kernel run on that kernel: a rule that sends their products elsewhere has to bring other cases for them."""

import pytest

from tests import test_gpu_few_tiles as few_tiles
from tests import test_gpu_fused_widths as fused_widths
from tests import test_gpu_rotated_reductions as rotated
from tests import test_gpu_row_panel as row_panel
from tests import test_gpu_weight_stream as weight_stream
from tests.dispatch import INPUT_INNER_SPARSE, INPUT_ROW_SPARSE, OUTPUT_SPARSE, Dispatch


@pytest.fixture(scope="module")
def kernel(tmp_path_factory, library):
    from fast_llm_amd import _lib

    return Dispatch(tmp_path_factory.mktemp("dispatch"), _lib.LIBRARY_PATH)


def test_streamed_products(kernel):
    strided = [(experts, weight_stream.STRIDED_INNER, weight_stream.STRIDED_COLUMNS, tall) for experts, tall in weight_stream.STRIDED]
    for experts, inner, columns, tall in weight_stream.PRODUCTS + strided:
        rows = weight_stream._map(experts, tall).num_rows
        for mode in (OUTPUT_SPARSE, INPUT_INNER_SPARSE):
            assert kernel(mode, rows, columns, inner, experts) == "weight stream", (mode, experts, inner, columns)
    for rows, inner, columns in weight_stream.DENSE:
        for mode in (OUTPUT_SPARSE, INPUT_INNER_SPARSE):
            assert kernel(mode, rows, columns, inner) == "weight stream", (mode, rows, inner, columns)
    for columns in (128, 384):
        assert kernel(OUTPUT_SPARSE, 4_000_000, columns, 64) == "weight stream"
    for tokens, ffn in weight_stream.WIDTHS:
        rows = (tokens * 6 + 128 * 128) // 128 * 128
        assert kernel(OUTPUT_SPARSE, rows, 2 * ffn, 320, 128, gated=True) == "weight stream", (tokens, ffn)


def test_fused_widths(kernel):
    for tokens, ffn in fused_widths.WIDTHS:
        rows = (tokens * 2 + 7 * 128) // 128 * 128
        if tokens == 300:
            expected = "few tiles" if ffn <= 200 else "weight stream"
        elif tokens == 3000:
            expected = "few tiles" if ffn <= 120 else "large tiles" if ffn in (1096, 4168) else "weight stream"
        else:
            expected = "large tiles"
        assert kernel(OUTPUT_SPARSE, rows, 2 * ffn, 320, 7, gated=True) == expected, (tokens, ffn)


def test_rotated_reductions(kernel):
    rows, experts = rotated._map().num_rows, len(rotated._TOKENS)
    for slices in (1, 2, 3, 5, 12, 33):
        for columns, expected in ((8, "few tiles"), (264, "few tiles"), (520, "few tiles"), (4616, "weight stream")):
            assert kernel(OUTPUT_SPARSE, rows, columns, 64 * slices, experts) == expected, (slices, columns)
        many = rotated._map(rotated.LARGE_TIMES).num_rows
        assert many <= 1024 * experts  # their tiles start at different slices
        assert kernel(OUTPUT_SPARSE, many, rotated.LARGE_COLUMNS, 64 * slices, experts) == "large tiles", slices


def test_few_tiles(kernel):
    for inner in (8, 72, 128, 448):
        for columns in (8, 136, 2056, 5000, 7688, 12296):
            for mode in (OUTPUT_SPARSE, INPUT_INNER_SPARSE):
                expected = "few tiles" if columns <= 2056 else "weight stream"
                assert kernel(mode, 7 * 128, columns, inner, 5) == expected, (mode, inner, columns)
                expected = expected if columns <= 7688 else "large tiles"
                assert kernel(mode, 1009, columns, inner) == expected, (mode, inner, columns)


    for inner in (8, 72, 128, 448):
        for columns in (8, 136, 256, 264, 504):
            for mode in (OUTPUT_SPARSE, INPUT_INNER_SPARSE):
                assert kernel(mode, 101 * 128, columns, inner, len(few_tiles.MANY)) == "few tiles", (mode, inner, columns)
    # With the gated activation up to 96 tiles only.
    assert kernel(OUTPUT_SPARSE, 96 * 128, 256, 128, 300, gated=True) == "few tiles"
    assert kernel(OUTPUT_SPARSE, 97 * 128, 256, 128, 300, gated=True) == "large tiles"


def test_weight_gradients(kernel):
    for experts, size, columns, accumulate in row_panel.GRADIENTS:
        rows = row_panel._map(experts).num_rows
        expected = "row panel" if experts <= 256 else "row sparse"
        assert kernel(INPUT_ROW_SPARSE, rows, columns, size, experts, accumulate) == expected, (experts, size, columns)


# (rows, columns, inner, experts): layer 2, or layer 1's input gradient.
@pytest.mark.parametrize(("product", "expected"), [
    ((9472, 2048, 1408, 64), "weight stream"), ((16896, 704, 3712, 60), "weight stream"), ((6400, 1544, 128, 11), "large tiles"),
    ((22400, 968, 1184, 32), "weight stream"),  # a reduction of no whole slices
])  # fmt: skip
def test_weights_along_rows(kernel, product, expected):
    rows, columns, inner, experts = product
    assert kernel(INPUT_INNER_SPARSE, rows, columns, inner, experts) == expected


@pytest.mark.parametrize(("product", "expected"), [
    ((46592, 1152, 1152, 61), "large tiles"), ((99840, 768, 2048, 128), "large tiles"),  # about as many rounds of tall tiles, or more
    # Exactly 15 and 13 rounds of large ones, not one more: 427 and 405 per round, where 400 and 432 were counted.
    ((37248, 6400, 1024, 96), "large tiles"), ((32512, 6400, 1024, 64), "weight stream"),
    ((14976, 1408, 2048, 64), "weight stream"), ((15104, 1152, 2240, 17), "weight stream"),  # 1.5 and 1.1 rounds of large ones
    ((9472, 2816, 2048, 64), "weight stream"), ((18432, 1536, 2048, 128), "weight stream"),  # low ones
])  # fmt: skip
def test_weights_along_the_reduction(kernel, product, expected):
    rows, columns, inner, experts = product
    assert kernel(OUTPUT_SPARSE, rows, columns, inner, experts) == expected
