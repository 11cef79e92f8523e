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

}  // namespace mphip
