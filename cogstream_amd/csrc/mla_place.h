// Which split of a sequence's keys and which 16 of its heads a workgroup of the decode attention takes (mla.hip).
//
// Launch: (x, y), x < grid_x = 8 * per_xcd, y = a cache block (sequence, group of heads). Workgroups of one x & 7 run on one XCD: the
// head tiles of a split share it, so that its L2 serves the second and later readers. Every block is launched with as many places as
// the longest one needs, so the shorter ones' last places are empty -- at the same x, block for block, unless they are moved about:
//   * split 0 goes to another XCD from block to block (behind the splits of the blocks in front), or the first XCDs have all the work;
//   * an XCD deals its workgroups out to its four shader engines in turn, empty or not: with an even number of places a block it
//     would always be the same engines that get the empty ones, so a split's place moves by one from block to block (a multiple of
//     four) or every second block; with an odd number it moves by itself.
// 32 sequences of 256 .. 8192 keys, rows of 640 columns, 16 heads, nine tiles a split (29 splits of the longest: four places): a pass
// of six layers 1160 us with the places in order, 960 so; rows of 576 columns 657 -> 612. 32 x 256 .. 8192 keys of 32 heads of 64, each
// with rows of its own (few splits, all on the first XCDs): 1870 -> 620.
#pragma once

struct MlaPlace { int split, head_tile; };

// first_part: partials of the sequences in front (their rounding up included); head_tiles: tiles of 16 heads that read one block
constexpr MlaPlace mla_place(int x, int y, int grid_x, int head_tiles, long first_part) {
    const int per_xcd = grid_x >> 3, moved = per_xcd & 1 ? 0 : per_xcd & 2 ? y >> 1 : y, k = ((x >> 3) + moved) % per_xcd;
    return {k / head_tiles * 8 + (int)((x - first_part) & 7), k % head_tiles};
}
