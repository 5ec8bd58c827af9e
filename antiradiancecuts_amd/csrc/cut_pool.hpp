// The memory of a moment cut's pool, kept between launches.  Host code without
// the device runtime, so that its rules can be run on the CPU.
#pragma once

#include <algorithm>
#include <cstddef>
#include <memory>
#include <vector>

namespace arc {

// Device: static void* alloc(size_t) (null: refused) and static void free(void*).
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

    void release() {
        captured.clear();
        block.reset();
    }
};

}  // namespace arc
