// tinyinfer_amd/csrc/backend/idle_memory.h over a stand-in for the HIP
// runtime: allocations fail on request, and a failed call's error stays until
// it is read, as the runtime's does.
#include "idle_memory.h"

#include <cstdio>
#include <cstdlib>
#include <thread>
#include <vector>

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

// The pool as a call uses it; what allocate_with_room would have to allocate
// counts as an allocation.
using Pool = IdleMemory<Runtime>;
constexpr size_t kMiB = 1 << 20;

Pool::Buffer get(Pool& pool, size_t bytes, int gpu = 0) {
    Pool::Buffer b;
    if (pool.take(gpu, bytes, &b)) return b;
    b.bytes = bytes;
    b.gpu = gpu;
    CHECK(allocate_with_room<Runtime>(&b.data, bytes, [&] { return pool.trim(); }) == 0);
    return b;
}

int allocations_of(Pool& pool, size_t bytes, int gpu = 0) {
    const int before = Runtime::allocations;
    pool.put(get(pool, bytes, gpu));
    return Runtime::allocations - before;
}

// A caller whose calls grow past every kept buffer allocates once per size and
// nothing when a size comes again, with the pool full of smaller ones.
void growing_calls_allocate_once() {
    Runtime::reset(0);
    Pool pool;
    std::vector<Pool::Buffer> held;
    for (int i = 0; i < Pool::kBuffers + 4; ++i) held.push_back(get(pool, 100));
    for (const auto& b : held) pool.put(b);
    CHECK(Runtime::live == Pool::kBuffers);
    for (size_t mib = 1; mib <= 40; ++mib) {
        CHECK(allocations_of(pool, mib * kMiB) == 1);
        for (int again = 0; again < 3; ++again) CHECK(allocations_of(pool, mib * kMiB) == 0);
        CHECK(Runtime::live <= Pool::kBuffers);
    }
    CHECK(allocations_of(pool, 100) == 0);  // a larger idle buffer serves
    CHECK(pool.trim() && Runtime::live == 0 && !pool.trim());
}

// The smallest buffer that is large enough is taken, and only on its own GPU.
void smallest_that_fits() {
    Runtime::reset(0);
    Pool pool;
    for (size_t size : {400, 100, 300, 200}) {
        Pool::Buffer b;
        b.bytes = size;
        b.gpu = 0;
        CHECK(Runtime::allocate(&b.data, size) == 0);
        pool.put(b);
    }
    Pool::Buffer a, b, c;
    CHECK(pool.take(0, 150, &a) && a.bytes == 200);
    CHECK(pool.take(0, 150, &b) && b.bytes == 300);
    CHECK(!pool.take(0, 401, &c) && !pool.take(1, 50, &c));
    pool.put(a);
    pool.put(b);
    pool.put(Pool::Buffer{});  // a call that got no memory
    CHECK(Runtime::live == 4);
    pool.trim();
    CHECK(Runtime::live == 0);
}

// No buffer above its limit and no more than the limit together are kept, and
// the largest stay.
void bounded() {
    Runtime::reset(0);
    Pool pool;
    CHECK(allocations_of(pool, Pool::kBufferBytes + 1) == 1 && Runtime::live == 0);
    std::vector<Pool::Buffer> held;
    for (int i = 0; i < 6; ++i) held.push_back(get(pool, Pool::kBufferBytes - i * kMiB));
    for (const auto& b : held) pool.put(b);
    CHECK(Runtime::live == 4);
    Pool::Buffer b;
    CHECK(pool.take(0, 1, &b) && b.bytes == Pool::kBufferBytes - 3 * kMiB);
    pool.put(b);
    pool.trim();
    CHECK(Runtime::live == 0);
}

// What is kept gives way to another allocation that finds no memory.
void gives_way() {
    Runtime::reset(0);
    Pool pool;
    CHECK(allocations_of(pool, 50 * kMiB) == 1 && Runtime::live == 1);
    Runtime::failures = 1;
    void* p = nullptr;
    CHECK(allocate_with_room<Runtime>(&p, 16, [&] { return pool.trim(); }) == 0 && p && Runtime::live == 1);
    Runtime::release(p);
    Runtime::failures = 1;  // nothing left to give back
    CHECK(allocate_with_room<Runtime>(&p, 16, [&] { return pool.trim(); }) == kOutOfMemory && Runtime::last_error == 0);
}

struct Quiet {
    static void release(void* p) { std::free(p); }
};

// Threads never hold the same buffer at once.
void threads() {
    IdleMemory<Quiet> pool;
    std::vector<std::thread> all;
    for (int t = 0; t < 8; ++t)
        all.emplace_back([&pool, t] {
            for (int i = 0; i < 500; ++i) {
                IdleMemory<Quiet>::Buffer b;
                const size_t bytes = 64 + 64 * ((i * 7 + t) % 50);
                if (!pool.take(0, bytes, &b)) {
                    b.data = std::malloc(bytes);
                    b.bytes = bytes;
                    b.gpu = 0;
                }
                int* const mine = static_cast<int*>(b.data);
                mine[0] = t;
                mine[15] = i;
                std::this_thread::yield();
                CHECK(mine[0] == t && mine[15] == i);
                if (i % 97 == 96) pool.trim();
                pool.put(b);
            }
        });
    for (auto& t : all) t.join();
    pool.trim();
}

}  // namespace

int main() {
    retry_after_giving_back();
    growing_calls_allocate_once();
    smallest_that_fits();
    bounded();
    gives_way();
    threads();
    std::puts("ok");
    return 0;
}
