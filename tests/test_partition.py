"""How the kernels with wavefronts that only load cut rows into tiles (csrc/fm_partition.h), compiled for the host."""

import ctypes
import pathlib
import subprocess

import pytest

CSRC = pathlib.Path(__file__).resolve().parent.parent / "fast_llm_amd" / "csrc"

# 0, or the number of the first tile that is empty, out of order, too long or ends at another row than the next begins; count + 1 if
# the last does not end with the rows.
_PROGRAM = """
#include "fm_partition.h"

extern "C" int first_wrong_tile(int rows, int height) {
    const int count = (rows + height - 1) / height;
    int next = 0;
    for (int i = 0; i < count; ++i) {
        const fm::TileRows tile = fm::rows_of_tile(i, rows, count);
        if (tile.first != next || tile.last <= tile.first || tile.last - tile.first > height) return i + 1;
        next = tile.last;
    }
    return next == rows ? 0 : count + 1;
}

extern "C" int first_wrong_part(int total, int parts) {
    const int least = total / parts;
    for (int i = 0; i < parts; ++i) {
        const int length = fm::part_begin(i + 1, total, parts) - fm::part_begin(i, total, parts);
        if (length != least && length != least + 1) return i + 1;
    }
    return fm::part_begin(0, total, parts) == 0 && fm::part_begin(parts, total, parts) == total ? 0 : parts + 1;
}
"""


@pytest.fixture(scope="module")
def partition(tmp_path_factory):
    folder = tmp_path_factory.mktemp("partition")
    (folder / "partition.cpp").write_text(_PROGRAM)
    library = folder / "partition.so"
    subprocess.run(
        ["g++", "-std=c++17", "-O1", "-shared", "-fPIC", f"-I{CSRC}", str(folder / "partition.cpp"), "-o", str(library)],
        check=True,
    )
    return ctypes.CDLL(str(library))


def test_tiles_of_few_rows(partition):
    for height in (128, 192):
        for rows in range(1, 2500):
            assert partition.first_wrong_tile(rows, height) == 0, (rows, height)


# Around 3.63 million rows, where tiles x blocks passes 2^31, and the most rows that a product may have.
@pytest.mark.parametrize("rows", [3_629_760, 3_633_000, 4_000_000, 2**28 + 33, 2**30 - 1])
@pytest.mark.parametrize("height", [128, 192])
def test_tiles_of_many_rows(partition, rows, height):
    assert partition.first_wrong_tile(rows, height) == 0


# The parts of a column of tiles (128 rows each) of up to 2^30 rows, as many as there are tiles and fewer.
@pytest.mark.parametrize("total", [1, 2, 7, 46_340, 46_341, 60_000, 2**23])
def test_parts(partition, total):
    for parts in {1, min(3, total), (total + 1) // 2, max(total - 1, 1), total}:
        assert partition.first_wrong_part(total, parts) == 0, parts
