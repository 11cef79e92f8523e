// The rules of tinyinfer_amd/csrc/backend/launch_rules.h at the sizes where
// they change over.
#include "launch_rules.h"

#include <cstdio>
#include <cstdlib>
#include <initializer_list>

#define CHECK(condition)                                                                \
    do {                                                                                \
        if (!(condition)) {                                                             \
            std::fprintf(stderr, "%s:%d: %s\n", __FILE__, __LINE__, #condition);        \
            std::exit(1);                                                               \
        }                                                                               \
    } while (0)

using namespace mphip;

// Scores in global memory (of the allocation-free call: in an array that
// overlapping calls share) only where they do not fit the chip.
static void scores_in_global_memory() {
    CHECK(!attention_scores_global(1, 10240));
    CHECK(attention_scores_global(1, 10241));
    CHECK(!attention_scores_global(3, 641));
    CHECK(!attention_scores_global(3, 3408));
    CHECK(attention_scores_global(3, 3409));
    CHECK(!attention_scores_global(8, 1280));
    CHECK(attention_scores_global(8, 1281));
    CHECK(attention_scores_global(8, 2147483632));
}

// 64-row tiles where they fill the chip, and never for up to 32 rows, however
// many columns there are.
static void large_tiles() {
    for (int rows : {1, 8, 16, 17, 32})
        for (int columns = 64; columns <= 1 << 20; columns += 4032)
            for (int cb : {1, 2}) CHECK(!fast_large_tiles(rows, columns, 4, cb));
    CHECK(fast_large_tiles(33, 7168, 4, 1));   // 448 tiles
    CHECK(!fast_large_tiles(33, 7152, 4, 1));  // 447
    CHECK(!fast_large_tiles(64, 8192, 4, 2));  // 256 tiles of 32 columns
    CHECK(fast_large_tiles(64, 14336, 4, 2));  // 448
    CHECK(!fast_large_tiles(4096, 1552, 4, 2));  // 97 column blocks: no pairs
    CHECK(fast_large_tiles(4096, 1552, 4, 1));
    CHECK(!fast_large_tiles(512, 1536, 4, 2));  // the sizes measured beside the rule
    CHECK(fast_large_tiles(512, 1536, 4, 1));
    CHECK(!fast_large_tiles(512, 576, 4, 1));
    CHECK(fast_large_tiles(2147483647 - 15, 1 << 20, 4, 2));
}

// A head whose weights outgrow the caches is streamed while one group of rows
// reads it.
static void head_streams() {
    CHECK(fast_head_streams(1, 1024, 128256) && fast_head_streams(64, 1024, 128256));
    CHECK(!fast_head_streams(65, 1024, 128256));
    CHECK(fast_head_streams(16, 2048, 32000));
    CHECK(!fast_head_streams(16, 512, 32768) && !fast_head_streams(1, 4096, 4096));
    CHECK(!fast_head_streams(1, 1024, 32768) && fast_head_streams(1, 1024, 32832));
    CHECK(fast_head_streams(1, 16384, 262144));
}

static void head_columns() {
    for (int rows : {1, 64, 200})
        for (int columns : {4, 4096, 49152}) CHECK(exact_head_columns(576, columns, rows) == 16);
    CHECK(exact_head_columns(608, 49152, 1) == 64 && exact_head_columns(2020, 32000, 256) == 64);
    CHECK(exact_head_columns(608, 4096, 128) == 16 && exact_head_columns(608, 4096, 129) == 64);
    CHECK(exact_head_columns(608, 8192, 64) == 16 && exact_head_columns(608, 8196, 64) == 64);
    CHECK(exact_head_groups(576, 49152, 1) == 3072 && exact_head_groups(608, 49152, 1) == 768);
    CHECK(exact_head_groups(576, 4, 1) == 1 && exact_head_groups(576, 20, 1) == 2);
    CHECK(exact_head_groups(608, 8260, 64) == 130);
    CHECK(exact_head_columns(4, 2147483647 - 63, 2147483647 - 63) == 64);
}

// Long rows take their heads apart in the kernel for 16-token pages and
// 64-wide heads only, few rows in every kernel.
static void heads_apart() {
    for (int group = 1; group <= 8; ++group) {
        CHECK(exact_heads_apart(512, group, 64, true) && exact_heads_apart(1, group, 40000, true));
        CHECK(!exact_heads_apart(513, group, 1024, true) && exact_heads_apart(513, group, 1025, true));
        CHECK(exact_heads_apart(1, group, 40000, false) && exact_heads_apart(256, group, 64, false));
        CHECK(!exact_heads_apart(513, group, 1025, false) && !exact_heads_apart(1ll << 40, group, 32768, false));
    }
    CHECK(!exact_heads_apart(257, 3, 1000, false) && exact_heads_apart(512, 4, 1000, false));
}

// The row kernel at the measured sizes that are clear either way, and that it
// stays once a row is long enough.
static void row_kernel() {
    CHECK(attention_row_pays(9, 3, 1) && attention_row_pays(9, 3, 503) && attention_row_pays(32, 4, 1));
    CHECK(!attention_row_pays(32, 32, 64) && attention_row_pays(32, 32, 128));
    CHECK(!attention_row_pays(128, 128, 64) && !attention_row_pays(128, 128, 256) && attention_row_pays(128, 128, 1000));
    CHECK(!attention_row_pays(128, 32, 64) && attention_row_pays(128, 32, 256) && attention_row_pays(128, 16, 1));
    CHECK(!attention_row_pays(192, 192, 1000) && attention_row_pays(192, 192, 8192));
    CHECK(!attention_row_pays(256, 256, 8192) && !attention_row_pays(384, 384, 10240));
    CHECK(!attention_row_pays(256, 32, 100) && attention_row_pays(256, 32, 300));
    for (int group = 1; group <= 8; ++group)
        for (int kv_heads : {1, 3, 16}) {
            bool before = false;
            for (int length = 1; length <= 10240; ++length) {
                const bool now = attention_row_pays(group * kv_heads, kv_heads, length);
                CHECK(now || !before || length <= 32);
                before = now;
            }
            CHECK(before);
        }
    CHECK(!attention_row_pays(1 << 20, 1 << 20, 10240));
}

int main() {
    scores_in_global_memory();
    row_kernel();
    large_tiles();
    head_streams();
    head_columns();
    heads_apart();
    std::puts("ok");
    return 0;
}
