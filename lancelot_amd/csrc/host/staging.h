// Page-locked staging between host values and the device, not in the reference (which copies through pageable memory).
#pragma once
#include <cstddef>

#include "cahel.h"

namespace cahel {

// The blocks of one host thread, used in turn.  A block that device work reads is guarded by an event recorded behind that
// work: it is rewritten only when the work is done, and nothing else waits for it.  Blocks grow on demand up to kMaxBytes and
// are given back when the thread ends (worker threads of a pool come and go).
class PinnedRing {
    struct Block {
        void *ptr = nullptr;
        std::size_t bytes = 0;
        he_event event = nullptr;
        bool busy = false, held = false;
    };

public:
    static constexpr int kBlocks = 4;
    static constexpr std::size_t kMaxBytes = std::size_t(16) << 20;
    PinnedRing() = default;
    PinnedRing(const PinnedRing &) = delete;
    PinnedRing &operator=(const PinnedRing &) = delete;
    ~PinnedRing() {
        for (Block &b : blocks_) {
            if (b.busy) (void)he_event_synchronize(b.event);
            if (b.event) (void)he_event_destroy(b.event);
            if (b.ptr) (void)he_host_free(b.ptr);
        }
    }
    static PinnedRing &of_thread() {
        thread_local PinnedRing ring;
        return ring;
    }
    // the next block, at least `bytes` (at most kMaxBytes) large, with no device work left on it
    void *take(std::size_t bytes) {
        if (bytes > kMaxBytes) throw std::logic_error("staging block too large");
        do current_ = (current_ + 1) % kBlocks;
        while (blocks_[current_].held);   // (at most two are)
        Block &b = blocks_[current_];
        if (b.busy) {
            check_status(he_event_synchronize(b.event), "he_event_synchronize");
            b.busy = false;
        }
        if (bytes > b.bytes) {
            void *old = b.ptr;
            b.ptr = nullptr;
            b.bytes = 0;
            if (old) check_status(he_host_free(old), "he_host_free");
            check_status(he_host_malloc(&b.ptr, bytes), "he_host_malloc");
            b.bytes = bytes;
        }
        if (!b.event) check_status(he_event_create(&b.event), "he_event_create");
        return b.ptr;
    }
    // the work enqueued on `stream` so far may read or write the block taken last
    void fence(he_stream stream) {
        Block &b = blocks_[current_];
        check_status(he_event_record(b.event, stream), "he_event_record");
        b.busy = true;
    }

    // The block taken last, which the work enqueued on `stream` so far writes, kept out of turn for what its owner does before it waits
    // for the block: other blocks may be taken, and other work enqueued, in between.
    class Held {
    public:
        Held(PinnedRing &ring, he_stream stream) : block_(&ring.blocks_[ring.current_]) {
            ring.fence(stream);
            block_->held = true;
        }
        Held(Held &&o) noexcept : block_(o.block_) { o.block_ = nullptr; }
        Held &operator=(Held &&) = delete;
        ~Held() {
            if (block_) block_->held = false;
        }
        void wait() {
            check_status(he_event_synchronize(block_->event), "he_event_synchronize");
            block_->busy = false;
        }

    private:
        Block *block_;
    };

private:
    Block blocks_[kBlocks];
    int current_ = 0;
};

}  // namespace cahel
