// Which kernel or tile a call takes where that is decided by sizes alone:
// plain functions of the sizes (no HIP), so that the rules can be checked
// without a GPU.
#pragma once
#include <stddef.h>

namespace mphip {

// Score floats of a KV head's query heads that the stand-alone single-row
// attention keeps on the chip; longer rows take theirs through global memory.
constexpr int kAttentionLdsScores = 10240;
constexpr bool attention_scores_global(int group, int length) {
    return (size_t)group * (((size_t)length + 15) & ~(size_t)15) > (size_t)kAttentionLdsScores;
}

// Whether a fast projection of `rows` x `columns` takes tiles of `row_blocks`
// x `column_blocks` blocks of 16, which read weights and activations less
// often than 16 x 16 tiles: from 7 work-groups per 4 CUs on (below, the wider
// tile leaves CUs idle: SwiGLU of 512 rows, 384 tiles of 64 x 32: 28.5 vs
// 24.0 us for 64 x 16; down at 512 rows, 288 of 64 x 16: 21.9 vs 20.0 for
// 16 x 16), and from 33 rows on: up to 32, half of a 64-row tile's matrix work
// is for padding and the weights, read once, gain from the streamed loads of
// the 16-row tiles. Whole steps of wide models (hidden 2,048 to 8,192, 7,168
// to 14,336 columns) with 64-row tiles against 16-row ones: 310 to 580 vs 260
// to 408 us at 1 to 16 rows, 312 to 593 vs 303 to 561 at 17, the same at 32,
// 350 to 700 vs 377 to 820 at 33.
constexpr int kChipCus = 256, kLargeTileRows = 33;
constexpr bool fast_large_tiles(int rows, int columns, int row_blocks, int column_blocks) {
    if (rows < kLargeTileRows || columns % (16 * column_blocks)) return false;
    const long long tiles = (long long)(((rows + 15) / 16 + row_blocks - 1) / row_blocks) * (columns / 16 / column_blocks);
    return 4 * tiles >= 7 * kChipCus;
}

}  // namespace mphip
