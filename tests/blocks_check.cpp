// Checks of the block cache of device memory (omc_blocks.hpp) on a simulated
// card: addresses and sizes only, nothing behind them.  Run with the name of a
// check; prints what differs and exits with 1.
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <random>

#include "omc_blocks.hpp"

constexpr size_t MiB = (size_t)1 << 20, GiB = (size_t)1 << 30;

#define EXPECT(x)                                              \
    do {                                                       \
        if (!(x)) {                                            \
            printf("line %d: not so: %s\n", __LINE__, #x);     \
            exit(1);                                           \
        }                                                      \
    } while (0)

// Two cards of `total` bytes each; an allocation is an address range of its own.
struct SimMem {
    size_t total = 100 * GiB, used[2] = {0, 0};
    int current = 0;
    std::map<char *, std::pair<size_t, int>> live;
    char *next = (char *)((size_t)1 << 44);
    int device() { return current; }
    void *get(size_t n) {
        if (used[current] + n > total) return nullptr;
        char *p = next;
        next += n;                        // touching ranges, so that a join across slabs would show
        used[current] += n;
        live[p] = {n, current};
        return p;
    }
    void put(void *p) {
        auto it = live.find((char *)p);
        EXPECT(it != live.end());
        used[it->second.second] -= it->second.first;
        live.erase(it);
    }
};
using Cache = DevBlocks<SimMem>;

// the lists of a device's cache agree with one another and with the card
static void consistent(Cache &B, int dev) {
    DevCache &C = B.caches[dev];
    size_t free_bytes = 0, listed = 0, slab_bytes = 0;
    for (auto &kv : C.slabs) {
        size_t at = 0, used = 0;
        bool was_free = false;
        EXPECT(B.mem.live.count(kv.first) && B.mem.live[kv.first].first == kv.second->size);
        while (at < kv.second->size) {
            auto it = C.blocks.find(kv.first + at);
            EXPECT(it != C.blocks.end() && it->second.slab == kv.second.get() && it->second.size > 0);
            EXPECT(!(was_free && it->second.free));            // free neighbours are joined
            was_free = it->second.free;
            (it->second.free ? free_bytes : used) += it->second.size;
            at += it->second.size;
        }
        EXPECT(at == kv.second->size && used == kv.second->used);
        slab_bytes += kv.second->size;
    }
    for (auto &f : C.free) {
        auto it = C.blocks.find(f.second);
        EXPECT(it != C.blocks.end() && it->second.free && it->second.size == f.first);
        listed += f.first;
    }
    EXPECT(listed == free_bytes && C.held == free_bytes && B.mem.used[dev] == slab_bytes);
}

// blocks are cut from larger ones, joined again, and idle slabs go back
static void cut_join_evict() {
    Cache B;
    size_t got;
    void *a = B.alloc(10 * GiB, &got), *b = B.alloc(3 * GiB + 1, &got);
    EXPECT(got == 3 * GiB + 2 * MiB);
    B.release(a);
    void *c = B.alloc(4 * GiB, &got), *d = B.alloc(5 * GiB, &got), *e = B.alloc(1 * GiB, &got);
    EXPECT(c == a && (char *)d == (char *)a + 4 * GiB && (char *)e == (char *)a + 9 * GiB);
    EXPECT(B.mem.live.size() == 2);
    consistent(B, 0);
    B.release(c);
    B.release(e);
    consistent(B, 0);
    B.trim();                                 // both slabs are in use
    EXPECT(B.mem.live.size() == 2);
    B.release(d);                             // joins both neighbours
    EXPECT(B.caches[0].free.size() == 1 && B.caches[0].held == 10 * GiB);
    B.trim();
    EXPECT(B.mem.live.size() == 1 && B.caches[0].held == 0);
    B.release(b);
    consistent(B, 0);
    B.mem.total = 400 * GiB;                  // more idle than the cache keeps: the slab idle for longest goes
    void *x = B.alloc(90 * GiB, &got), *y = B.alloc(60 * GiB, &got);
    B.release(x);
    EXPECT(B.caches[0].held == 93 * GiB + 2 * MiB);
    B.release(y);
    EXPECT(B.caches[0].held == 60 * GiB && B.mem.live.count((char *)y) && !B.mem.live.count((char *)x));
    consistent(B, 0);
}

// a request is served while any free block of the card holds it
static void full_card() {
    Cache B;
    size_t got;
    void *whole = B.alloc(90 * GiB, &got);
    B.release(whole);
    void *a = B.alloc(2 * GiB, &got);         // cut from the slab, which is in use from here on
    void *other = B.alloc(9 * GiB, &got);
    EXPECT(a == whole && other);
    B.mem.total = 90 * GiB;                   // the rest of the card is taken
    void *s = B.alloc(512 * MiB, &got);       // far less than the free 79 GiB
    EXPECT(s != nullptr);
    consistent(B, 0);
    EXPECT(B.alloc(80 * GiB, &got) == nullptr);
    B.release(s);
    B.release(other);
    B.release(a);
    consistent(B, 0);
    EXPECT(B.alloc(90 * GiB, &got) != nullptr);      // every idle byte can go back to the runtime
}

// half of what a plan counts as free or reusable can be had in one block
static void reusable() {
    Cache B;
    size_t got;
    std::vector<void *> v;
    void *whole = B.alloc(80 * GiB, &got);
    B.release(whole);
    for (int k = 0; k < 40; k++) v.push_back(B.alloc(2 * GiB, &got));
    EXPECT(B.mem.live.size() == 1);           // all cut from the one slab
    for (int k = 0; k < 40; k++)
        if (k % 4) B.release(v[k]);           // 60 GiB free, in pieces of 6
    size_t counted = B.mem.total - B.mem.used[0] + B.reusable();
    EXPECT(B.alloc(counted / 2, &got) != nullptr);

    std::mt19937 g(11);
    for (int k = 0; k < 300; k++) {
        Cache C;
        std::vector<void *> live;
        for (int j = 0; j < 60; j++) {
            if (live.size() < 12 && g() % 2) {
                size_t n = (size_t)1 << (24 + g() % 11);
                void *p = C.alloc(n + g() % n, &got);
                if (p) live.push_back(p);
            } else if (!live.empty()) {
                size_t i = g() % live.size();
                C.release(live[i]);
                live.erase(live.begin() + (long)i);
            }
        }
        const size_t grain = 2 * MiB;
        counted = C.mem.total - C.mem.used[0] + C.reusable();
        if (counted / 2 < grain) continue;
        EXPECT(C.alloc(counted / 2 / grain * grain, &got) != nullptr);
        consistent(C, 0);
    }
}

// a block goes back to the device it is of, whichever is current
static void two_devices() {
    Cache B;
    size_t got;
    void *a = B.alloc(4 * GiB, &got);
    B.mem.current = 1;
    void *b = B.alloc(6 * GiB, &got);
    B.release(a);
    EXPECT(B.caches[0].held == 4 * GiB && B.caches[1].held == 0);
    consistent(B, 0);
    consistent(B, 1);
    EXPECT(B.alloc(4 * GiB, &got) != a);
    B.mem.current = 0;
    B.release(b);
    EXPECT(B.caches[1].held == 6 * GiB && B.alloc(4 * GiB, &got) == a);
    consistent(B, 0);
    consistent(B, 1);
}

// any order of requests and releases leaves the lists in agreement
static void any_order() {
    Cache B;
    std::mt19937 g(7);
    std::vector<void *> live;
    for (int k = 0; k < 20000; k++) {
        if (live.size() < 12 && g() % 2) {
            size_t n = (size_t)1 << (g() % 34), got;
            void *p = B.alloc(n + g() % n, &got);
            if (p) live.push_back(p);
        } else if (!live.empty()) {
            size_t i = g() % live.size();
            B.release(live[i]);
            live.erase(live.begin() + (long)i);
        }
        if (k % 50 == 0) consistent(B, 0);
        if (k % 3000 == 0) B.trim();
    }
    for (void *p : live) B.release(p);
    B.trim();
    EXPECT(B.mem.live.empty() && B.caches[0].held == 0 && B.caches[0].blocks.empty());
}

int main(int argc, char **argv) {
    const struct { const char *name; void (*fn)(); } checks[] = {
        {"cut_join_evict", cut_join_evict},
        {"full_card", full_card},
        {"reusable", reusable},
        {"two_devices", two_devices},
        {"any_order", any_order},
    };
    for (auto &c : checks)
        if (argc > 1 && !strcmp(argv[1], c.name)) {
            c.fn();
            return 0;
        }
    printf("no check of that name\n");
    return 2;
}
