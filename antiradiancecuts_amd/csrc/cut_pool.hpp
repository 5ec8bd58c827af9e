// The memory of a moment cut's pool, kept between launches.  Host code without
// the device runtime, so that its rules can be run on the CPU.
#pragma once

#include <algorithm>
#include <cstddef>
#include <cstdint>
#include <memory>
#include <vector>

namespace arc {

// Device: static void* alloc(size_t) (null: refused), static void free(void*)
// and static size_t room(), the bytes that a pool may take by itself.
//
// A cut needs no pool (without one, or where it is full, tiles are cut serially),
// so a refusal is no error: the pool gets what the device has, down to nothing,
// keeps the block that it holds, and does not ask again for what was refused.
//
// A captured graph has the block's addresses in its nodes, while the pool grows
// with what the frames ask for.  So the block is shared: who owns the graph
// holds it (hold()), a new block takes its place in the frames that follow, and
// it is freed with the last graph that has it.  A capture whose owner is not
// known keeps the block for as long as the pool lives.
template <class Device>
class PoolMemory {
    struct Block {
        void* p;
        size_t bytes;
        Block(void* at, size_t size) : p(at), bytes(size) {}
        Block(const Block&) = delete;
        Block& operator=(const Block&) = delete;
        ~Block() { Device::free(p); }
    };
    std::shared_ptr<Block> block;
    std::vector<std::shared_ptr<Block>> captured;  // by graphs whose owner is not known
    size_t limit = SIZE_MAX;                       // chunks that the device did not refuse

  public:
    void* data() const { return block ? block->p : nullptr; }
    size_t bytes() const { return block ? block->bytes : 0; }
    std::shared_ptr<void> hold() const { return block; }

    void keep() {
        if (block && std::find(captured.begin(), captured.end(), block) == captured.end()) captured.push_back(block);
    }

    // At least `size` bytes, in a new block where the present one is smaller.
    // quiet() waits for the work on the present one before it may be freed.
    // False when the device refuses them: the present block stays.
    template <class Quiet>
    bool reserve(size_t size, Quiet quiet) {
        if (block && size <= block->bytes) return true;
        void* p = Device::alloc(size);
        if (!p) return false;
        if (block) quiet();
        block = std::make_shared<Block>(p, size);
        return true;
    }

    // Up to `want` chunks of `chunk` bytes beside `fixed` bytes; returns how many
    // there are.  own: the size is the pool's own choice, so it stays within the
    // device's room.  Nothing moves unless `move`.
    template <class Quiet>
    size_t fit(size_t want, size_t chunk, size_t fixed, bool own, bool move, Quiet quiet) {
        const size_t held = bytes() > fixed ? (bytes() - fixed) / chunk : 0;
        if (want <= held) return want;
        if (!move || std::min(want, limit) <= held) return held;
        size_t n = std::min(want, limit);
        if (own) {
            const size_t room = Device::room();
            n = std::min(n, room > fixed ? (room - fixed) / chunk : 0);
        }
        for (; n > held && !reserve(fixed + n * chunk, quiet); n /= 2) {
        }
        n = std::max(n, held);
        if (n < want) limit = std::min(limit, n);
        return n;
    }

    bool refused() const { return limit != SIZE_MAX; }
    void retry() { limit = SIZE_MAX; }

    void release() {
        captured.clear();
        block.reset();
    }
};

}  // namespace arc
