// Device memory of runs, kept for reuse: the blocks, their slabs and the policy,
// apart from the runtime that the memory comes from.
#pragma once
#include <algorithm>
#include <cstddef>
#include <iterator>
#include <map>
#include <memory>
#include <mutex>
#include <vector>

// Device memory of runs, kept for reuse.  A slab is one allocation of the
// runtime, cut into blocks on demand; a released block joins its free
// neighbours.  A request takes the smallest free block that holds it and gives
// back the rest, so runs of different sizes share the same memory.  (Blocks
// reused whole, by size, piled up: once plans of other sizes had filled the
// cache, every pass of the next plan mapped and unmapped its tallies anew.  In a
// process that had run other plans before, a 196-beamlet FP64 plan took 1130 ms
// a pass against 208 ms alone, 50 beamlets on 13 M voxels 1480 against 95 ms.)
// Sizes are rounded to 2 MiB.  Beyond CACHE_MAX free bytes, slabs without a
// block in use go back to the runtime, the one unused for longest first; the
// free parts of slabs in use stay.
struct Slab;
struct Block {
    Slab *slab;
    size_t size;
    bool free;
};
struct Slab {
    char *base;
    size_t size;
    size_t used = 0;                 // bytes handed out
    unsigned long long stamp = 0;    // when it was last drawn on or emptied
};
struct DevCache {
    std::mutex mu;
    std::map<char *, Block> blocks;                    // every block by address
    std::multimap<size_t, char *> free;                // the free ones by size
    std::map<char *, std::unique_ptr<Slab>> slabs;     // by address
    size_t held = 0;                                   // free bytes
    unsigned long long clock = 0;
    void drop_free(std::map<char *, Block>::iterator it) {
        for (auto f = free.lower_bound(it->second.size); f != free.end() && f->first == it->second.size; ++f)
            if (f->second == it->first) {
                free.erase(f);
                return;
            }
    }
    void add_free(std::map<char *, Block>::iterator it) { free.emplace(it->second.size, it->first); }
    // the smallest free block of at least n bytes, cut to n.  A small block is
    // not cut from a much larger one, which another run may need whole while
    // it is in use, unless the card has nothing else left (any).
    void *take(size_t n, bool any = false) {
        auto f = free.lower_bound(n);
        if (f == free.end() || (!any && f->first > std::max(64 * n, (size_t)1 << 30))) return nullptr;
        auto it = blocks.find(f->second);
        free.erase(f);
        Block &b = it->second;
        if (b.size > n) {
            auto rest = blocks.emplace(it->first + n, Block{b.slab, b.size - n, true}).first;
            add_free(rest);
            b.size = n;
        }
        b.free = false;
        b.slab->used += n;
        b.slab->stamp = ++clock;
        held -= n;
        return it->first;
    }
    // a slab that is handed out whole
    void *take_at(void *p) {
        auto it = blocks.find((char *)p);
        drop_free(it);
        it->second.free = false;
        it->second.slab->used = it->second.size;
        it->second.slab->stamp = ++clock;
        held -= it->second.size;
        return p;
    }
    void add_slab(void *p, size_t n) {
        Slab *s = new Slab{(char *)p, n};
        slabs[s->base].reset(s);
        add_free(blocks.emplace(s->base, Block{s, n, true}).first);
        held += n;
    }
    // false: not a block of this cache that is in use
    bool give(void *p) {
        auto it = blocks.find((char *)p);
        if (it == blocks.end() || it->second.free) return false;
        Slab *s = it->second.slab;
        it->second.free = true;
        s->used -= it->second.size;
        s->stamp = ++clock;
        held += it->second.size;
        auto next = std::next(it);
        if (next != blocks.end() && next->second.slab == s && next->second.free) {
            drop_free(next);
            it->second.size += next->second.size;
            blocks.erase(next);
        }
        if (it != blocks.begin()) {
            auto prev = std::prev(it);
            if (prev->second.slab == s && prev->second.free) {
                drop_free(prev);
                prev->second.size += it->second.size;
                blocks.erase(it);
                it = prev;
            }
        }
        add_free(it);
        return true;
    }
    // takes the unused slab that has been so for longest out of the cache (null: none)
    void *evict() {
        Slab *old = nullptr;
        for (auto &kv : slabs)
            if (kv.second->used == 0 && (!old || kv.second->stamp < old->stamp)) old = kv.second.get();
        if (!old) return nullptr;
        char *base = old->base;
        auto it = blocks.find(base);      // an unused slab is one free block
        drop_free(it);
        held -= it->second.size;
        blocks.erase(it);
        slabs.erase(base);
        return base;
    }
};
constexpr size_t CACHE_GRAIN = (size_t)2 << 20;
constexpr size_t CACHE_MAX = (size_t)128 << 30;
constexpr int CACHE_DEVICES = 64;

// The caches of a process, one a device.  Mem gives the memory of the current
// device: device() its number, get(n) an allocation or null, put(p) its return.
template <class Mem> struct DevBlocks {
    Mem mem;
    DevCache caches[CACHE_DEVICES];
    DevCache &here() { return caches[(unsigned)mem.device() % CACHE_DEVICES]; }

    void *alloc(size_t n, size_t *got) {
        n = (n + CACHE_GRAIN - 1) / CACHE_GRAIN * CACHE_GRAIN;
        *got = n;
        DevCache &C = here();
        {
            std::lock_guard<std::mutex> lk(C.mu);
            if (void *p = C.take(n)) return p;
        }
        void *p = mem.get(n);
        if (!p) {
            trim();
            p = mem.get(n);
        }
        std::lock_guard<std::mutex> lk(C.mu);
        if (!p) return C.take(n, true);       // a free part of a slab in use, whatever its size
        C.add_slab(p, n);
        return C.take_at(p);
    }

    // a block goes back to the cache it is of: the current device's, or
    // another's where the caller's thread has turned to another device since
    void release(void *p) {
        const unsigned at = (unsigned)mem.device() % CACHE_DEVICES;
        for (unsigned k = 0; k < CACHE_DEVICES; k++) {
            DevCache &C = caches[(at + k) % CACHE_DEVICES];
            std::vector<void *> out;
            {
                std::lock_guard<std::mutex> lk(C.mu);
                if (!C.give(p)) continue;
                while (C.held > CACHE_MAX) {
                    void *s = C.evict();
                    if (!s) break;                // what is left is in slabs that are in use
                    out.push_back(s);
                }
            }
            for (void *s : out) mem.put(s);
            return;
        }
    }

    // memory that a plan may count on beside what the runtime has free: the
    // slabs without a block in use, which can go back to it, and the largest
    // free block of the others (their smaller pieces serve no large request).
    // A request of at most half of both together is served.
    size_t reusable() {
        DevCache &C = here();
        std::lock_guard<std::mutex> lk(C.mu);
        size_t idle = 0, piece = 0;
        for (auto &kv : C.slabs)
            if (kv.second->used == 0) idle += kv.second->size;
        for (auto f = C.free.rbegin(); f != C.free.rend(); ++f)
            if (C.blocks.find(f->second)->second.slab->used != 0) {
                piece = f->first;
                break;
            }
        return idle + piece;
    }

    void trim() {
        DevCache &C = here();
        std::vector<void *> out;
        {
            std::lock_guard<std::mutex> lk(C.mu);
            while (void *s = C.evict()) out.push_back(s);
        }
        for (void *s : out) mem.put(s);
    }
};
