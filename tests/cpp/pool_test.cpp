// The rules of csrc/cut_pool.hpp over a device that counts its blocks.
// Prints the first rule that does not hold and ends with 1.
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <set>

#include "cut_pool.hpp"

namespace {

struct Counted {
    static std::set<void*> live;
    static size_t most;  // larger blocks are refused
    static size_t left;  // what a pool may take by itself
    static int asked;
    static size_t room() { return left; }
    static void* alloc(size_t bytes) {
        ++asked;
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
size_t Counted::left = SIZE_MAX;
int Counted::asked = 0;

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

// Frames that ask for chunks of 100 bytes beside 50.
void sizes() {
    arc::PoolMemory<Counted> m;
    auto quiet = [] {};
    auto frame = [&](size_t want, bool own = true, bool move = true) { return m.fit(want, 100, 50, own, move, quiet); };
    check(frame(10, true, false) == 0 && !m.data(), "nothing is allocated while the frame is captured");
    check(frame(10) == 10 && m.bytes() == 1050, "a first frame's pool");
    void* a = m.data();
    check(frame(4) == 4 && m.data() == a, "a smaller pool in the same block");
    check(frame(50, true, false) == 10 && m.data() == a, "a captured frame takes what there is");
    Counted::most = 3000;
    check(frame(50) == 25 && m.refused() && m.data() != a, "half of what was refused");
    const int asked = Counted::asked;
    a = m.data();
    for (int k = 0; k < 3; ++k) check(frame(80) == 25 && m.data() == a, "later frames keep it");
    check(Counted::asked == asked, "and do not ask again");
    Counted::most = 1 << 20;
    m.retry();
    check(frame(80) == 80 && !m.refused(), "asked again after retry");
    a = m.data();
    Counted::left = 8000;
    check(frame(1000) == 80 && m.data() == a, "no room: the block stays");
    m.retry();
    check(frame(1000, false) == 1000, "a size that the caller chose does not mind the room");
    m.release();
    m.retry();
    check(frame(1000) == 79, "a first pool within the room");
    m.release();
    m.retry();
    Counted::left = 10;
    check(frame(1000) == 0 && !m.data(), "no pool");
    Counted::left = SIZE_MAX;
    Counted::most = 0;
    m.retry();
    check(frame(1000) == 0 && frame(1000) == 0 && !m.data(), "no pool where every block is refused");
    Counted::most = 1 << 20;
    m.retry();
    m.reserve(40, quiet);
    check(frame(3) == 3, "a block smaller than the fixed part");
    m.release();
}

}  // namespace

int main() {
    growth();
    held_by_a_graph();
    captured_by_someone();
    refused();
    sizes();
    check(Counted::live.empty(), "no block is left");
    if (!failures) std::printf("pool rules hold\n");
    return failures ? 1 : 0;
}
