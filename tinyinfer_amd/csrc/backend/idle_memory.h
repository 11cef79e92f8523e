// Memory that outlives the call it was allocated for (no HIP here: `Memory`
// names the allocator, so that the rules can be checked without a GPU).
#pragma once
#include <stddef.h>

#include <mutex>

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

// Buffers of one kind of memory between calls. A call takes one for itself
// (any thread, any stream) and puts it back when nothing uses it any more, so
// an idle buffer is in nobody's use. take() gives the smallest idle buffer
// that is large enough; put() keeps the largest ones: at most kBuffers, of
// kBufferBytes each and kBytes together, smaller ones make room. So a caller
// whose calls grow replaces what it no longer takes, and its next call of the
// same size allocates nothing. (64 rows of the fast attention at 8,192 tokens,
// after calls at 300 to 5,000: 176 us, and 247 with the first four buffers kept
// for good, 216 with a device allocation in every call and nothing pinned.)
template <typename Memory>
class IdleMemory {
public:
    static constexpr int kBuffers = 32;
    static constexpr size_t kBufferBytes = (size_t)64 << 20, kBytes = (size_t)256 << 20;
    struct Buffer {
        void* data = nullptr;
        size_t bytes = 0;
        int gpu = -1;
    };

    bool take(int gpu, size_t bytes, Buffer* out) {
        std::lock_guard<std::mutex> lock(mutex_);
        int best = -1;
        for (int i = 0; i < count_; ++i)
            if (idle_[i].gpu == gpu && idle_[i].bytes >= bytes && (best < 0 || idle_[i].bytes < idle_[best].bytes))
                best = i;
        if (best < 0) return false;
        *out = remove(best);
        return true;
    }

    void put(const Buffer& buffer) {
        if (!buffer.data) return;
        if (buffer.bytes > kBufferBytes) {
            Memory::release(buffer.data);
            return;
        }
        Buffer out[kBuffers + 1];
        int given = 0;
        {
            std::lock_guard<std::mutex> lock(mutex_);
            idle_[count_++] = buffer;
            total_ += buffer.bytes;
            while (count_ > kBuffers || total_ > kBytes) {
                int least = 0;
                for (int i = 1; i < count_; ++i)
                    if (idle_[i].bytes < idle_[least].bytes) least = i;
                out[given++] = remove(least);
            }
        }
        for (int i = 0; i < given; ++i) Memory::release(out[i].data);
    }

    // Frees every idle buffer; whether there was one.
    bool trim() {
        Buffer out[kBuffers];
        int given = 0;
        {
            std::lock_guard<std::mutex> lock(mutex_);
            while (count_ > 0) out[given++] = remove(count_ - 1);
        }
        for (int i = 0; i < given; ++i) Memory::release(out[i].data);
        return given > 0;
    }

private:
    Buffer remove(int i) {
        const Buffer buffer = idle_[i];
        idle_[i] = idle_[--count_];
        total_ -= buffer.bytes;
        return buffer;
    }

    std::mutex mutex_;
    Buffer idle_[kBuffers + 1];
    int count_ = 0;
    size_t total_ = 0;
};

}  // namespace mphip
