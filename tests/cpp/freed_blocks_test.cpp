// The library's own rule for freed buffers (ferrum_amd/csrc/freed_blocks.hpp) with a system that refuses: host code only.
#include <chrono>
#include <cstdio>
#include <cstdlib>
#include <future>
#include <set>

#include "../../ferrum_amd/csrc/freed_blocks.hpp"

using fh::FreedBlocks;

#define CHECK(condition)                                                            \
    do {                                                                            \
        if (!(condition)) {                                                         \
            std::printf("line %d: %s\n", __LINE__, #condition);                     \
            std::exit(1);                                                           \
        }                                                                           \
    } while (0)

static const auto always = [] { return true; };
static const auto never = [] { return false; };
static void* at(size_t i) { return reinterpret_cast<void*>(i); }

static bool gather(FreedBlocks& blocks, size_t bytes, size_t i) {
    bool full = false;
    CHECK(blocks.gather(bytes, at(i), always, &full));
    return full;
}

// A refused free has waited for nothing: no block may reach the pool, none is lost.
static void refused() {
    FreedBlocks blocks;
    for (size_t i = 1; i < 8; ++i) CHECK(!gather(blocks, 4096, i));
    int asked = 0;
    for (int round = 0; round < 3; ++round) {
        blocks.settle(always, [&](void*) { return ++asked, false; });
        CHECK(asked == round + 1);
        void* out = nullptr;
        CHECK(!blocks.take(4096, &out));
        CHECK(blocks.held_bytes() == 0 && blocks.waiting_bytes() == 7 * 4096);
    }
    std::set<void*> returned, handed;
    blocks.settle(always, [&](void* block) { return returned.insert(block).second; });
    CHECK(returned.size() == 1 && blocks.waiting_bytes() == 0 && blocks.held_bytes() == 6 * 4096);
    for (void* out; blocks.take(4096, &out);) CHECK(handed.insert(out).second && returned.count(out) == 0);
    CHECK(handed.size() == 6 && blocks.held_bytes() == 0);
}

// Others allocate and free while one thread waits; what they free meanwhile waits for the next time.
static void others_do_not_wait() {
    FreedBlocks blocks;
    CHECK(blocks.keep(8192, at(100), always));
    for (size_t i = 1; i < 4; ++i) gather(blocks, 4096, i);
    blocks.settle(always, [&](void*) {
        auto other = std::async(std::launch::async, [&] {
            void* out = nullptr;
            return blocks.take(8192, &out) && out == at(100) && !gather(blocks, 4096, 4) && blocks.keep(16384, at(101), always);
        });
        CHECK(other.wait_for(std::chrono::seconds(20)) == std::future_status::ready && other.get());
        return true;
    });
    CHECK(blocks.waiting_bytes() == 4096 && blocks.held_bytes() == 2 * 4096 + 16384);
    void* out = nullptr;
    for (int i = 0; i < 2; ++i) CHECK(blocks.take(4096, &out) && out != at(4));
    CHECK(!blocks.take(4096, &out));
}

// What the pool has no room for goes back to the system, and where that is refused it waits again.
static void a_full_pool() {
    constexpr size_t big = 48u << 20;
    for (int mode = 0; mode < 2; ++mode) {
        FreedBlocks blocks;
        for (size_t i = 1; i <= 4; ++i) CHECK(blocks.fits(big) && blocks.keep(big, at(i), always));
        bool full = false;
        for (size_t i = 11; i <= 13; ++i) full = gather(blocks, big, i);
        CHECK(full);
        int asked = 0;
        blocks.settle(always, [&](void*) { return ++asked == 1 || mode == 0; });
        CHECK(asked == 2 && blocks.held_bytes() == 5 * big && blocks.waiting_bytes() == (mode == 0 ? 0 : big));
    }
    FreedBlocks small;
    for (size_t i = 1; i < FreedBlocks::kLeavingBlocks; ++i) CHECK(!gather(small, 4096, i));
    CHECK(gather(small, 4096, FreedBlocks::kLeavingBlocks));
}

static void not_while_recording() {
    FreedBlocks blocks;
    bool full = false;
    CHECK(!blocks.keep(4096, at(1), never) && !blocks.gather(4096, at(1), never, &full));
    CHECK(blocks.keep(4096, at(1), always));
    gather(blocks, 8192, 2);
    const auto unasked = [](void*) -> bool { std::exit(1); };
    blocks.settle(never, unasked);
    CHECK(!blocks.drain(never, [] { std::exit(1); }, unasked));
    CHECK(blocks.held_bytes() == 4096 && blocks.waiting_bytes() == 8192);
}

static void drained() {
    FreedBlocks blocks;
    int waits = 0;
    const auto wait = [&] { ++waits; };
    CHECK(!blocks.drain(always, wait, [](void*) { return true; }) && waits == 0);
    CHECK(blocks.keep(4096, at(1), always));
    gather(blocks, 8192, 2);
    CHECK(!blocks.drain(always, wait, [](void*) { return false; }) && waits == 1);   // nothing is lost, nothing handed on
    void* out = nullptr;
    CHECK(!blocks.take(4096, &out) && blocks.held_bytes() == 0 && blocks.waiting_bytes() == 4096 + 8192);
    std::set<void*> returned;
    CHECK(blocks.drain(always, wait, [&](void* block) { return returned.insert(block).second; }));
    CHECK(waits == 2 && returned.size() == 2 && blocks.waiting_bytes() == 0);
}

int main() {
    refused();
    others_do_not_wait();
    a_full_pool();
    not_while_recording();
    drained();
    std::printf("ok\n");
    return 0;
}
