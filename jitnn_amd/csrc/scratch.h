// A thread's grow-only block of device memory, as a policy over an allocator: host code without any HIP, so that it can be
// driven on a machine that has no GPU (tests/scratch_block_test.cpp).
#pragma once
#include <algorithm>
#include <cstddef>
#include <new>

namespace jitnn {

// Mem::alloc(bytes) -> address or nullptr; Mem::release(address) waits for the device, false: refused, the memory is still held.
// The destructor frees nothing (thread_local objects outlive the runtime on the process's first thread): release_all() does.
template <class Mem>
class ScratchBlock {
    struct Retired {
        void *ptr;
        size_t bytes;
        Retired *next;
    };
    void *ptr_ = nullptr;
    size_t cap_ = 0;
    size_t refused_ = (size_t)-1;  // the smallest size try_get could not have
    bool recorded_ = false;  // a stream capture has been given this block: a graph may hold its address
    Retired *retired_ = nullptr;
    size_t retired_bytes_ = 0;
    int growths_ = 0;

    static size_t round_up(size_t b) { return (b + ((size_t)1 << 20) - 1) & ~(((size_t)1 << 20) - 1); }

    // Moves to a block of `want` bytes; where there is none, the block stays as it is.  A block a graph may hold is retired, not
    // freed: it lives until release_all().
    bool grow(size_t want, bool *waited) {
        Retired *node = ptr_ ? new (std::nothrow) Retired : nullptr;
        if (ptr_ && !node) return false;
        void *p = Mem::alloc(want);
        if (!p) {
            delete node;
            return false;
        }
        if (ptr_ && !recorded_ && Mem::release(ptr_)) {
            ptr_ = nullptr;
            *waited = true;
        }
        if (ptr_) {
            *node = {ptr_, cap_, retired_};
            retired_ = node;
            retired_bytes_ += cap_;
        } else {
            delete node;
        }
        ptr_ = p;
        cap_ = want;
        recorded_ = false;
        ++growths_;
        return true;
    }
    // (a block that leaves a retired one behind is at least twice as large, so that the retired ones add up to less than it)
    bool extend(size_t bytes, bool *waited) {
        return (recorded_ && grow(round_up(std::max(bytes, 2 * cap_)), waited)) || grow(round_up(bytes), waited);
    }

public:
    // The block, of at least `bytes`, or nullptr.  recording: the caller's stream is capturing.  *waited is set where the old
    // block was freed, which waits for the device: nothing enqueued before still runs.
    // Where the device has no room beside the old block, that is given up first: what it held is of no use to this call.
    void *get(size_t bytes, bool recording, bool *waited) {
        if (bytes > cap_ && !extend(bytes, waited) && !(give_up(waited) && grow(round_up(bytes), waited))) return nullptr;
        if (recording) recorded_ = true;
        return ptr_;
    }
    // The same for a caller that can do without: nullptr leaves the block as it is, a size that was refused once is not asked
    // for again until ask_again(), and a capturing stream, whose capture an allocation would invalidate, gets no growth.
    void *try_get(size_t bytes, bool recording, bool *waited) {
        if (bytes > cap_) {
            if (recording || bytes >= refused_) return nullptr;
            if (!extend(bytes, waited)) {
                refused_ = bytes;
                return nullptr;
            }
        }
        if (recording) recorded_ = true;
        return ptr_;
    }
    void ask_again() { refused_ = (size_t)-1; }
    // Frees the block unless a graph may hold it; true: memory came back.
    bool give_up(bool *waited) {
        if (!ptr_ || recorded_ || !Mem::release(ptr_)) return false;
        ptr_ = nullptr;
        cap_ = 0;
        *waited = true;
        return true;
    }
    size_t capacity() const { return cap_; }
    size_t retired_bytes() const { return retired_bytes_; }
    int growths() const { return growths_; }  // allocations so far
    void release_all() {
        if (ptr_) (void)Mem::release(ptr_);
        while (retired_) {
            Retired *r = retired_;
            (void)Mem::release(r->ptr);
            retired_ = r->next;
            delete r;
        }
        *this = ScratchBlock{};
    }
};

// The start of a prompt pass: sizes that were refused are asked for again by whoever needs them, and where the pass knows its largest
// launches (0: it does not) both blocks move to their sizes at once, not step by step.
template <class Block>
void start_pass(Block &operands, Block &weights, size_t operand_bytes, size_t weight_bytes, bool *waited) {
    operands.ask_again();
    weights.ask_again();
    if (operand_bytes) (void)operands.try_get(operand_bytes, false, waited);
    if (weight_bytes) (void)weights.try_get(weight_bytes, false, waited);
}

}  // namespace jitnn
