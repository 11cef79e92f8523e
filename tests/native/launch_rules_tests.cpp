// The rules of tinyinfer_amd/csrc/backend/launch_rules.h at the sizes where
// they change over.
#include "launch_rules.h"

#include <cstdio>
#include <cstdlib>

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

int main() {
    scores_in_global_memory();
    std::puts("ok");
    return 0;
}
