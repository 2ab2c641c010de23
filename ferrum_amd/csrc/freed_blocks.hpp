// Blocks of freed buffers that a device keeps for the buffers to come.  Nothing of HIP is in here: what returns a block
// to the system, and waits for the GPU by it, is the caller's.
#pragma once

#include <cstddef>
#include <iterator>
#include <list>
#include <map>
#include <mutex>

namespace fh {

class FreedBlocks {
 public:
    static constexpr size_t kPoolBytes = 256u << 20;       // most memory kept
    static constexpr size_t kPoolBlockBytes = 64u << 20;   // largest block kept
    static constexpr size_t kLeavingBytes = 64u << 20, kLeavingBlocks = 512;   // blocks that wait for the GPU together

    // Held by whoever waits for the GPU on these blocks' account, and by whoever changes whether such a wait is allowed
    // (a recording, the device's end).  Taken before `lock`, and `lock` is never held over a wait: no thread that
    // allocates or frees waits for the GPU because another one does.
    std::mutex settling;
    // `pool`, `leaving` and their sums.
    mutable std::mutex lock;

    bool take(size_t bytes, void** out) {
        std::lock_guard<std::mutex> hold(lock);
        const auto found = pool.find(bytes);
        if (found == pool.end()) return false;
        *out = found->second;
        pool_bytes -= bytes;
        pool.erase(found);
        return true;
    }

    bool fits(size_t bytes) const {
        std::lock_guard<std::mutex> hold(lock);
        return pool_bytes + bytes <= kPoolBytes;
    }

    // A block on which all that is still to be done comes before what the next buffer does; false: it stays the caller's.
    template <class May>
    bool keep(size_t bytes, void* ptr, May&& may) {
        std::lock_guard<std::mutex> hold(lock);
        return may() && pooled(bytes, ptr);
    }

    // A block that may be in use where this library does not see it; false: it stays the caller's.  `full`: it is time to settle.
    template <class May>
    bool gather(size_t bytes, void* ptr, May&& may, bool* full) {
        std::lock_guard<std::mutex> hold(lock);
        if (!may()) return false;
        try {
            leaving.push_back(Block{bytes, ptr});
        } catch (...) {   // no memory for the entry
            return false;
        }
        leaving_bytes += bytes;
        *full = leaving_bytes >= kLeavingBytes || leaving.size() >= kLeavingBlocks;
        return true;
    }

    // Gathered blocks into the pool.  `give_back` returns a block to the system and says whether it did: only then has it waited for all
    // work on the GPU, on whatever stream, that was asked for before, and nobody uses the others.  Where it is
    // refused (a stream that is being captured forbids it, also one of another device object or of the caller's) nothing
    // is known of any block: all of them, that one too, go on waiting for the next time.
    template <class May, class GiveBack>
    void settle(May&& may, GiveBack&& give_back) {
        std::lock_guard<std::mutex> alone(settling);
        std::list<Block> settled;
        {
            std::lock_guard<std::mutex> hold(lock);
            if (leaving.empty() || !may()) return;
            settled.swap(leaving);
            leaving_bytes = 0;
        }
        const bool waited = give_back(settled.back().ptr);
        if (waited) {
            settled.pop_back();
            std::lock_guard<std::mutex> hold(lock);
            for (auto block = settled.begin(); block != settled.end();)
                block = pool_bytes + block->bytes <= kPoolBytes && pooled(block->bytes, block->ptr) ? settled.erase(block) : std::next(block);
        }
        if (waited) give_back_all(settled, give_back);
        wait_on(settled);
    }

    // Everything back to the system, after `wait`; whether that was anything.
    template <class May, class Wait, class GiveBack>
    bool drain(May&& may, Wait&& wait, GiveBack&& give_back) {
        std::lock_guard<std::mutex> alone(settling);
        std::list<Block> all;
        {
            std::lock_guard<std::mutex> hold(lock);
            if ((pool.empty() && leaving.empty()) || !may()) return false;
            for (auto block = pool.begin(); block != pool.end(); block = pool.erase(block)) {
                try {
                    all.push_back(Block{block->first, block->second});
                } catch (...) {   // no memory for the entry: the rest stays
                    break;
                }
                pool_bytes -= block->first;
            }
            all.splice(all.end(), leaving);
            leaving_bytes = 0;
        }
        wait();
        const size_t before = all.size();
        give_back_all(all, give_back);
        const bool any = all.size() < before;
        wait_on(all);
        return any;
    }

    size_t held_bytes() const {
        std::lock_guard<std::mutex> hold(lock);
        return pool_bytes;
    }
    size_t waiting_bytes() const {
        std::lock_guard<std::mutex> hold(lock);
        return leaving_bytes;
    }

 private:
    struct Block {
        size_t bytes;
        void* ptr;
    };

    bool pooled(size_t bytes, void* ptr) {
        try {
            pool.emplace(bytes, ptr);
        } catch (...) {   // no memory for the entry
            return false;
        }
        pool_bytes += bytes;
        return true;
    }

    template <class GiveBack>
    static void give_back_all(std::list<Block>& blocks, GiveBack&& give_back) {
        for (auto block = blocks.begin(); block != blocks.end();)
            block = give_back(block->ptr) ? blocks.erase(block) : std::next(block);
    }

    void wait_on(std::list<Block>& blocks) {
        std::lock_guard<std::mutex> hold(lock);
        for (const Block& block : blocks) leaving_bytes += block.bytes;
        leaving.splice(leaving.end(), blocks);
    }

    std::multimap<size_t, void*> pool;
    size_t pool_bytes = 0;
    std::list<Block> leaving;
    size_t leaving_bytes = 0;
};

}  // namespace fh
