// Memory that outlives the call it was allocated for (no HIP here: `Memory`
// names the allocator, so that the rules can be checked without a GPU).
#pragma once
#include <stddef.h>

namespace mphip {

// Memory::allocate(out, bytes) (0: done), and once more where that fails and
// give_back() frees something. The HIP runtime keeps a failed call's error
// until it is read, and the launches of a call that succeeds after all would
// return it: Memory::clear_error() reads it after every failure.
template <typename Memory, typename GiveBack>
int allocate_with_room(void** out, size_t bytes, GiveBack&& give_back) {
    for (bool last = false;; last = true) {
        *out = nullptr;
        const int error = Memory::allocate(out, bytes);
        if (!error) return 0;
        Memory::clear_error();
        *out = nullptr;
        if (last || !give_back()) return error;
    }
}

}  // namespace mphip
