// Which kernel or tile a call takes where that is decided by sizes alone:
// plain functions of the sizes (no HIP), so that the rules can be checked
// without a GPU.
#pragma once
#include <stddef.h>

namespace mphip {

constexpr int kChipCus = 256;

// Score floats of a KV head's query heads that the stand-alone single-row
// attention keeps on the chip; longer rows take theirs through global memory.
constexpr int kAttentionLdsScores = 10240;
constexpr bool attention_scores_global(int group, int length) {
    return (size_t)group * (((size_t)length + 15) & ~(size_t)15) > (size_t)kAttentionLdsScores;
}

// Whether a single-row attention with 16-token pages and 64-wide heads whose
// scores stay on the chip takes the row kernel: four work-groups of a whole CU
// for each query head, against one work-group for a KV head's heads whose
// output chains take three times as long. The row kernel loses where a row is
// short, and where many heads make it take several turns of the chip. Both
// estimates are in ns, fitted over 1 to 384 heads, 1 to 8 of them per KV head,
// and 1 to 8,192 tokens (general and row kernel, us): 32 heads apart 9.3 and
// 10.6 at 64 tokens, 13 and 11.6 at 128, 36 and 19 at 503; 128 apart 9.4 and
// 20 at 64, 38 and 42 at 503, 77 and 66 at 1,000, 149 and 104 at 2,000; 256
// apart 43 and 81 at 503, 707 and 746 at 8,192; 256 on 32 KV heads 39 and 42
// at 128, 50 and 49 at 200, 102 and 71 at 503.
constexpr bool attention_row_pays(int heads, int kv_heads, int length) {
    const long long group = heads / kv_heads, turns = (4ll * heads + kChipCus - 1) / kChipCus;
    const long long general = 3500 + 2900 * group + (67 * ((group + 3) / 4) + 5 * group) * (length > 32 ? length - 32 : 0);
    const long long row = 1000 + turns * (9300 + (turns == 1 ? 14ll : 16 + 6 / group) * length);
    return row < general;
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
constexpr int kLargeTileRows = 33;
constexpr bool fast_large_tiles(int rows, int columns, int row_blocks, int column_blocks) {
    if (rows < kLargeTileRows || columns % (16 * column_blocks)) return false;
    const long long tiles = (long long)(((rows + 15) / 16 + row_blocks - 1) / row_blocks) * (columns / 16 / column_blocks);
    return 4 * tiles >= 7 * kChipCus;
}

// Whether the tiled LM head (hidden sizes other than 576) streams its weights
// past the caches: where one group of up to 64 rows reads them and they would
// not stay in the last-level cache (256 MiB) beside the rest of the model.
// Streamed against plain loads at 1 to 16 rows: 98 vs 110 us for 525 MB
// (hidden 1,024, 128,256 columns), 54.5 vs 58 for 262 MB (2,048, 32,000; in a
// model of 8 layers), but 46 vs 46 for 67 MB (4,096, 4,096; 4 layers) and 21
// vs 20 (512, 32,768; 16 layers). Two row groups share plain loads' lines:
// 331 vs 323 us at 65 rows of the first, 57 vs 53 of the last.
constexpr bool fast_head_streams(int rows, int inner, int columns) {
    return rows <= 64 && (long long)inner * columns > 32ll << 20;  // floats: 128 MiB
}

// Columns of the exact LM head per work-group (and per argmax partial): 8
// wavefronts of two columns, their weights as scalars, where a row of weights
// is whole 64-wide chunks. Elsewhere the weights go through LDS and eight
// columns share an x read: 128 instead of 203 us for 49,152 columns of hidden
// size 608 at 1 to 64 rows, 54 instead of 78 for 4,096 columns at 200 rows;
// two columns where eight leave half the chip idle (4,096 columns: 31 instead
// of 51 us up to 64 rows, 48 instead of 53 up to 128).
constexpr int kExactHeadColumns = 16;  // the fewest
constexpr int exact_head_columns(int inner, int columns, int rows) {
    const long long wide = (long long)((columns + 63) / 64) * ((rows + 63) / 64);
    return inner % 64 && 2 * wide > kChipCus ? 64 : kExactHeadColumns;
}
constexpr int exact_head_groups(int inner, int columns, int rows) {
    const int group = exact_head_columns(inner, columns, rows);
    return (columns + group - 1) / group;
}

// Whether the exact prefill attention computes a row's softmax and output one
// query head a wavefront (its own e_t and chain, V read once per head) or a KV
// head's together: apart where few tasks (rows times KV heads) leave SIMDs
// idle, and in the kernel for 16-token pages and 64-wide heads for long rows
// as well. `longest` is the step's longest row. Apart against together, us:
// 7.5 vs 12.4 for 30 rows at position 100, 127 vs 134 for 256 rows at 3,000
// and 128 vs 135 for 1,024 at 1,000, but 25.5 vs 24.2 for 256 at 256. The
// kernel for other shapes is bound by its scattered V reads, which apart it
// makes once per head: three heads of 48 dims, 256 rows, 508 vs 292 at 1,000
// and 1,283 vs 730 at 3,000; two of 32 dims 571 vs 493 and 1,478 vs 1,300;
// three of 32, 100 rows (448 tasks) 244 vs 217 at 1,000 but 30 rows (128) 178
// vs 187; four of 32 gain with 100 rows as well (246 vs 295).
constexpr bool exact_heads_apart(long long tasks, int group, int longest, bool paged16x64) {
    if (paged16x64) return tasks <= 512 || longest > 1024;
    return tasks <= (group > 3 ? 512 : 256);
}

}  // namespace mphip
