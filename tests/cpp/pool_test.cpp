// The rules of csrc/cut_pool.hpp over a device that counts its blocks.
// Prints the first rule that does not hold and ends with 1.
#include <cstdio>
#include <cstdlib>
#include <set>

#include "cut_pool.hpp"

namespace {

struct Counted {
    static std::set<void*> live;
    static size_t most;  // larger blocks are refused
    static void* alloc(size_t bytes) {
        if (bytes > most) return nullptr;
        void* p = std::malloc(bytes);
        live.insert(p);
        return p;
    }
    static void free(void* p) {
        if (!live.erase(p)) std::exit(2);  // freed twice
        std::free(p);
    }
};
std::set<void*> Counted::live;
size_t Counted::most = 1 << 20;

int failures = 0;
void check(bool ok, const char* what) {
    if (!ok && failures++ == 0) std::printf("does not hold: %s\n", what);
}
bool live(void* p) { return Counted::live.count(p) != 0; }

void growth() {
    arc::PoolMemory<Counted> m;
    int waits = 0;
    auto quiet = [&] { ++waits; };
    check(m.reserve(1000, quiet) && waits == 0, "a first block needs no wait");
    void* a = m.data();
    check(m.reserve(900, quiet) && m.data() == a, "a block that is large enough stays");
    check(m.reserve(2000, quiet) && m.data() != a && waits == 1 && !live(a), "an unused block is freed after a wait");
    m.release();
    check(Counted::live.empty(), "release frees the block");
}

void held_by_a_graph() {
    arc::PoolMemory<Counted> m;
    auto quiet = [] {};
    m.reserve(1000, quiet);
    void* a = m.data();
    std::shared_ptr<void> graph = m.hold();
    check(m.reserve(5000, quiet) && m.data() != a && live(a), "growth leaves the block that a graph holds");
    m.release();
    check(live(a) && Counted::live.size() == 1, "the pool's end leaves it too");
    graph.reset();
    check(Counted::live.empty(), "it goes with the graph");
}

void captured_by_someone() {
    arc::PoolMemory<Counted> m;
    auto quiet = [] {};
    m.reserve(1000, quiet);
    void* a = m.data();
    m.keep();
    m.keep();
    check(m.reserve(5000, quiet) && live(a), "growth leaves a block captured by an unknown owner");
    m.release();
    check(Counted::live.empty(), "it goes with the pool");
}

void refused() {
    arc::PoolMemory<Counted> m;
    auto quiet = [] {};
    m.reserve(1000, quiet);
    void* a = m.data();
    check(!m.reserve((1 << 20) + 1, quiet) && m.data() == a && live(a), "a refusal leaves the present block");
    m.release();
}

}  // namespace

int main() {
    growth();
    held_by_a_graph();
    captured_by_someone();
    refused();
    check(Counted::live.empty(), "no block is left");
    if (!failures) std::printf("pool rules hold\n");
    return failures ? 1 : 0;
}
