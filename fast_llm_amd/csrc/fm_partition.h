// Nearly equal parts of a length, without device code: the host compiler takes it too.
#pragma once

namespace fm {

// Where part `index` (up to `parts`, the end) of [0, total) begins; parts differ by one at most, the longer ones come first. Nothing
// here is larger than `total`: index * total would pass 32 bits from 3.6 million rows on (parts of 192 rows, counted in 32).
constexpr int part_begin(int index, int total, int parts) {
    const int longer = total % parts;
    return index * (total / parts) + (index < longer ? index : longer);
}

// The rows of tile `index` of an expert's `count` tiles that differ by 32 rows at most: [first, last).
struct TileRows {
    int first, last;
};
constexpr TileRows rows_of_tile(int index, int expert_rows, int count) {
    const int blocks = (expert_rows + 31) / 32, last = part_begin(index + 1, blocks, count) * 32;
    return {part_begin(index, blocks, count) * 32, last < expert_rows ? last : expert_rows};
}

}  // namespace fm
