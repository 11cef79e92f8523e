// tinyinfer_amd/csrc/backend/idle_memory.h over a stand-in for the HIP
// runtime: allocations fail on request, and a failed call's error stays until
// it is read, as the runtime's does.
#include "idle_memory.h"

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

namespace {

constexpr int kOutOfMemory = 2;

struct Runtime {
    static inline int last_error = 0, failures = 0, allocations = 0, live = 0;
    static int allocate(void** out, size_t bytes) {
        ++allocations;
        if (failures > 0) {
            --failures;
            *out = reinterpret_cast<void*>(8);  // what a failed call leaves there means nothing
            return last_error = kOutOfMemory;
        }
        ++live;
        *out = std::malloc(bytes);
        return 0;
    }
    static void release(void* p) {
        --live;
        std::free(p);
    }
    static void clear_error() { last_error = 0; }
    static void reset(int fail) { last_error = 0, failures = fail, allocations = 0, live = 0; }
};

// An allocation that succeeds after memory was given back leaves no error for
// the launches that follow; one that fails leaves none either and says so.
void retry_after_giving_back() {
    void* p = nullptr;
    int given_back = 0;
    auto some = [&] { return ++given_back > 0; };
    auto none = [&] { return ++given_back < 0; };

    Runtime::reset(0);
    CHECK(allocate_with_room<Runtime>(&p, 16, some) == 0 && p && given_back == 0 && Runtime::allocations == 1);
    Runtime::release(p);

    Runtime::reset(1);
    CHECK(allocate_with_room<Runtime>(&p, 16, some) == 0 && p);
    CHECK(given_back == 1 && Runtime::allocations == 2 && Runtime::last_error == 0);
    Runtime::release(p);

    Runtime::reset(2);
    given_back = 0;
    CHECK(allocate_with_room<Runtime>(&p, 16, some) == kOutOfMemory && !p);
    CHECK(given_back == 1 && Runtime::allocations == 2 && Runtime::last_error == 0);

    Runtime::reset(1);
    given_back = 0;
    CHECK(allocate_with_room<Runtime>(&p, 16, none) == kOutOfMemory && !p);
    CHECK(given_back == 1 && Runtime::allocations == 1 && Runtime::last_error == 0 && Runtime::live == 0);
}

}  // namespace

int main() {
    retry_after_giving_back();
    std::puts("ok");
    return 0;
}
