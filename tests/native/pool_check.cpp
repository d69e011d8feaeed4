// The blocks a device handle keeps, against a runtime of host memory.
//   pool_check <name of a check>       exit 0: it holds
#include "fake_hip.h"

#include "../../wurstrenderer_amd/csrc/wr_memory.h"

#include <cstdio>
#include <new>
#include <string>

static bool no_host_memory = false;
void *operator new(size_t n) {
    if (no_host_memory) throw std::bad_alloc();
    return std::malloc(n);
}
void operator delete(void *p) noexcept { std::free(p); }
void operator delete(void *p, size_t) noexcept { std::free(p); }

using Block = wr::BlockPool::Block;

// giving a block back happens in destructors and C entry points: it may not throw
static int give_without_host_memory() {
    wr::BlockPool pool(2, 100);
    Block b[4];
    for (Block &x : b)
        if (pool.take(50, &x) != hipSuccess) return 1;
    no_host_memory = true;
    for (Block &x : b) pool.give(x);
    pool.trim();
    no_host_memory = false;
    return fake::used == 0 ? 0 : 2;
}

// at most `keep` blocks of at most `most` bytes are kept, the largest ones; a take gets the smallest that fits
static int keeps_the_largest() {
    wr::BlockPool pool(2, 100);
    Block a, b, c, d, e;
    if (pool.take(30, &a) || pool.take(50, &b) || pool.take(40, &c) || pool.take(101, &d)) return 1;
    for (Block x : {a, b, c, d, Block{}}) pool.give(x);
    if (fake::used != 90) return 2;  // 50 and 40
    if (pool.take(35, &e) || e.p != c.p || pool.take(51, &a) || a.p == b.p) return 3;
    return 0;
}

static int close_fit() {
    wr::BlockPool pool(2, 100, true);
    Block a, b;
    if (pool.take(80, &a)) return 1;
    pool.give(a);
    if (pool.take(39, &b) || b.p == a.p) return 2;  // 80 > 2 x 39
    if (pool.take(40, &b) || b.p != a.p) return 3;
    return 0;
}

// allocations that find the device full get the idle blocks of every pool
static int full_device() {
    wr::DeviceMemory mem;
    fake::memory = 1000;
    Block a, b, c;
    if (mem.take(mem.spills, 400, &a) || mem.take(mem.geometry, 300, &b) || mem.take(mem.build_memory, 200, &c)) return 1;
    mem.spills.give(a);
    mem.geometry.give(b);
    mem.build_memory.give(c);
    void *p = nullptr;
    if (mem.idle() != 900 || mem.alloc(&p, 950) != hipSuccess || mem.idle() != 0 || fake::used != 950) return 2;
    if (mem.alloc(&p, 100) != hipErrorOutOfMemory) return 3;
    return 0;
}

int main(int argc, char **argv) {
    const std::string name = argc == 2 ? argv[1] : "";
    if (name == "give_without_host_memory") return give_without_host_memory();
    if (name == "keeps_the_largest") return keeps_the_largest();
    if (name == "close_fit") return close_fit();
    if (name == "full_device") return full_device();
    return 64;
}
