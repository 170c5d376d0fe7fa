// Definitions of the precision-templated launchers; included once per
// precision by omc_k32.hip and omc_k64.hip, which instantiate them.
#pragma once
#include "omc_launch.hpp"

#include <cstring>

namespace omc {

template <class R> hipError_t launch_history(const HistArgs<R> &a, int rng, bool count, int grid, int block,
                                             hipStream_t st) {
    if (a.nsplit > 1 && a.stack) {
        if (rng == RNG_REPLAY) {
            if (count) hipLaunchKernelGGL((k_history_split<R, Replay, true, true>), dim3(grid), dim3(block), 0, st, a);
            else hipLaunchKernelGGL((k_history_split<R, Replay, false, true>), dim3(grid), dim3(block), 0, st, a);
        } else {
            if (count) hipLaunchKernelGGL((k_history_split<R, Philox, true, true>), dim3(grid), dim3(block), 0, st, a);
            else hipLaunchKernelGGL((k_history_split<R, Philox, false, true>), dim3(grid), dim3(block), 0, st, a);
        }
        return hipGetLastError();
    }
    if (a.nsplit > 1) {
        if (rng == RNG_REPLAY) {
            if (count) hipLaunchKernelGGL((k_history_split<R, Replay, true, false>), dim3(grid), dim3(block), 0, st, a);
            else hipLaunchKernelGGL((k_history_split<R, Replay, false, false>), dim3(grid), dim3(block), 0, st, a);
        } else {
            if (count) hipLaunchKernelGGL((k_history_split<R, Philox, true, false>), dim3(grid), dim3(block), 0, st, a);
            else hipLaunchKernelGGL((k_history_split<R, Philox, false, false>), dim3(grid), dim3(block), 0, st, a);
        }
        return hipGetLastError();
    }
    if (rng == RNG_REPLAY) {
        if (count) hipLaunchKernelGGL((k_history<R, Replay, true>), dim3(grid), dim3(block), 0, st, a);
        else hipLaunchKernelGGL((k_history<R, Replay, false>), dim3(grid), dim3(block), 0, st, a);
    } else {
        if (count) hipLaunchKernelGGL((k_history<R, Philox, true>), dim3(grid), dim3(block), 0, st, a);
        else hipLaunchKernelGGL((k_history<R, Philox, false>), dim3(grid), dim3(block), 0, st, a);
    }
    return hipGetLastError();
}

template <class R> hipError_t launch_sampler(const SampArgs<R> &a, hipStream_t st) {
    int block = 64;
    int grid = (a.ncase + block - 1) / block;
    hipLaunchKernelGGL((k_sampler<R>), dim3(grid), dim3(block), 0, st, a);
    return hipGetLastError();
}

// One kernel of round r: its function, shape and by-value arguments.
// Part 0 samples the round's primaries, 1 transports photons, 2 charged
// particles, 3 ends the round.  Arguments depend on r only through its
// parity, which selects the input and output pools.
template <class R> struct RoundCall {
    const void *fn = nullptr;
    dim3 grid, block;
    SrcArgs<R> src;
    EvArgs<R> ev;
    EvCtl *ctl = nullptr;
    int par = 0;
    void *args[2] = {nullptr, nullptr};
    int part = 0;
    unsigned shmem = 0;                  // dynamic LDS bytes per workgroup
    // kernelParams of a graph node: pointers to the argument values above
    void **bind() {
        if (part == 0) args[0] = &src;
        else if (part == 3) { args[0] = &ctl; args[1] = &par; }
        else args[0] = &ev;
        return args;
    }
};

// The transport kernel of part 1 (photons; split: the splitting kernel) or 2
// (charged particles) with the tables of st staged in LDS.
template <class R> const void *event_kernel(int part, bool split, bool count, int st) {
#define OMC_FN(...) reinterpret_cast<const void *>(&__VA_ARGS__)
    if (part == 1 && split)
        return count ? OMC_FN(k_event_split<R, true, 0>)
                     : st ? OMC_FN(k_event_split<R, false, ST_GEOM>) : OMC_FN(k_event_split<R, false, 0>);
    if (part == 1) return count ? OMC_FN(k_event<R, true, true, 0>) : OMC_FN(k_event<R, true, false, 0>);
    if (count) return OMC_FN(k_event<R, false, true, 0>);
    // FP64 bins (24 KB a medium) are read from device memory.  Staged in a trial,
    // 1e6 histories on 60^3 water took 36.3 ms against 39.6; with four media they
    // do not fit beside a second workgroup.
    if constexpr (std::is_same<R, float>::value)
        if (st & ST_BINS)
            return st & ST_GEOM ? OMC_FN(k_event<R, false, false, ST_GEOM | ST_BINS>)
                                : OMC_FN(k_event<R, false, false, ST_BINS>);
    return st ? OMC_FN(k_event<R, false, false, ST_GEOM>) : OMC_FN(k_event<R, false, false, 0>);
#undef OMC_FN
}

template <class R> void round_call(const EvLaunch<R> &L, long r, int part, bool count, RoundCall<R> &c) {
    const int par = (int)(r & 1), nx = 1 - par;
    c.part = part;
    c.block = dim3(256);
    if (part == 0) {
        SrcArgs<R> &s = c.src;
        s = L.src;
        s.ctl = L.ctl;
        s.ebal = L.ebal;
        s.out = L.pool[par][L.src.dos.charge != 0 && !L.src.use_beamlets ? 1 : 0];
        c.fn = reinterpret_cast<const void *>(&k_source<R>);
        c.grid = dim3(L.grid_source);
    } else if (part == 1 || part == 2) {
        EvArgs<R> &a = c.ev;
        a.t = L.t;
        a.g = L.g;
        a.seed = L.seed;
        a.outp = L.pool[nx][0];
        a.oute = L.pool[nx][1];
        a.n_out = &L.ctl->cnt[nx][0];
        a.cap = L.cap;
        a.endep = L.endep;
        a.slot_stride = L.slot_stride;
        a.touched = L.touched;
        a.touch_stride = L.touch_stride;
        a.ebal = L.ebal;
        a.counters = L.counters ? L.counters + (part == 1 ? 0 : 8) : nullptr;
        a.err = &L.ctl->err;
        a.ctl = L.ctl;
        a.budget = L.budget;
        a.turns = L.turns;
        a.max_age = L.max_age;
        a.delta = L.delta;
        a.nsplit = L.nsplit > 1 ? L.nsplit : 1;
        a.ebin = L.ebin;
        // (the counting kernels read every table in device memory)
        const int st = count ? 0 : part == 2 ? L.st_charged : a.nsplit > 1 ? L.st_split : 0;
        const bool list = part == 2 && L.tlist > 0;
        a.eb_words = L.eb_words;
        a.tlist = list ? L.tlist : 0;
        a.lds = part == 2 ? L.lds_charged : L.lds_split;
        if (st == 0) a.lds.list = 0;
        a.waves = part == 2 ? L.waves_charged : L.waves_event;
        c.shmem = st ? (unsigned)a.lds.bytes : list ? (unsigned)a.tlist * c.block.x * 16u : 0u;
        a.in = L.pool[par][part - 1];
        a.n_in = &L.ctl->cnt[par][part - 1];
        a.claim = &L.ctl->claim[par][part - 1];
        c.fn = event_kernel<R>(part, a.nsplit > 1, count, st);
        c.grid = dim3(part == 2 ? L.grid_charged : L.grid_event);
    } else {
        c.ctl = L.ctl;
        c.par = par;
        c.fn = reinterpret_cast<const void *>(&k_round_end);
        c.grid = dim3(1);
        c.block = dim3(64);
    }
}

template <class R> hipError_t launch_round_part(const EvLaunch<R> &L, long r, int part, bool count, hipStream_t st) {
    RoundCall<R> c;
    round_call(L, r, part, count, c);
    return hipLaunchKernel(c.fn, c.grid, c.block, c.bind(), c.shmem, st);
}

// A graph of rounds r0 .. r0+nround-1, built node by node (no stream
// capture, so enqueues and allocations of other threads cannot disturb it):
// each kernel depends on the one before, as on a stream.
template <class R> hipError_t build_rounds_graph(const EvLaunch<R> &L, long r0, int nround, bool count,
                                                 hipGraph_t *out) {
    hipGraph_t g = nullptr;
    hipError_t e = hipGraphCreate(&g, 0);
    if (e != hipSuccess) return e;
    hipGraphNode_t prev = nullptr;
    for (long r = r0; r < r0 + nround && e == hipSuccess; r++)
        for (int part = 0; part < 4 && e == hipSuccess; part++) {
            RoundCall<R> c;
            round_call(L, r, part, count, c);
            hipKernelNodeParams p;
            memset(&p, 0, sizeof p);
            p.func = const_cast<void *>(c.fn);
            p.gridDim = c.grid;
            p.blockDim = c.block;
            p.sharedMemBytes = c.shmem;
            p.kernelParams = c.bind();
            p.extra = nullptr;
            hipGraphNode_t n = nullptr;
            e = hipGraphAddKernelNode(&n, g, prev ? &prev : nullptr, prev ? 1 : 0, &p);
            prev = n;
        }
    if (e != hipSuccess) {
        (void)hipGraphDestroy(g);
        return e;
    }
    *out = g;
    return hipSuccess;
}

template <class R> hipError_t launch_rounds(const EvLaunch<R> &L, long r0, int nround, bool count, hipStream_t st) {
    for (long r = r0; r < r0 + nround; r++)
        for (int part = 0; part < 4; part++) {
            hipError_t e = launch_round_part(L, r, part, count, st);
            if (e != hipSuccess) return e;
        }
    return hipSuccess;
}

}  // namespace omc
