// Event-queue ("batched") transport form.
//
// Particles live in structure-of-arrays pools in HBM, one pool per type
// (photons, charged particles), double-buffered by round parity.  A round is
// four launches on one stream:
//   k_source     samples this round's injected primaries into the input pool,
//   k_event<1>   transports the queued photons (persistent lanes, below;
//                k_event_split when photons are split),
//   k_event<0>   transports the queued electrons/positrons, `budget`
//                condensed-history steps (electron_run) between refills,
//   k_round_end  retires the consumed input pools and plans the next
//                injection so that the number of particles in flight stays
//                near a target.
// Queue lengths live in device memory (EvCtl), so rounds are enqueued
// without host round trips; the host reads EvCtl now and then to see whether
// the job has drained.  Surviving particles and the secondaries they produced
// are appended to the output pools with one atomic per wavefront (ballot +
// popcount for the lane offsets).  Every particle carries its own random
// stream: primaries are keyed like the plain history form, secondaries by a
// hash of the parent's stream and draw position, so a result does not
// depend on scheduling, grid size or the target.
#pragma once
#include "omc_kernels.hpp"

namespace omc {

// A queued particle: its state with the resumable state of an electron
// (demfp, sig0, phase), its tally slot (beamlet of a Dij group; batch) and its
// random stream.  A pool keeps it in POOL_VECS words of 16 bytes, word k of
// entry i at base[k * cap + i]: a wave's consecutive entries are read and
// written with 16 bytes a lane, contiguous, in 6 (FP32) or 8 (FP64) accesses
// from one base address.  (One array per field took 23 accesses of 4 or 8 bytes
// and 19 pointers a pool; three pools' pointers did not fit the scalar
// registers.)  With the exchange below: 1e7 histories on the 128^3 slab 382 ->
// 284 ms, 2e5 9 MeV electrons on a CT 66 -> 59.5 ms, nsplit 20 77 -> 69 ms, 1e6
// FP64 histories on 60^3 water 50 -> 39 ms; small jobs the same.
template <class R> struct Pool {
    uint4 *base;
    long long cap;                 // entries
};
template <class R> constexpr int POOL_VECS = sizeof(R) == 4 ? 6 : 8;

template <class R> struct Queued {
    Part<R> p;
    R demfp, sig0;
    int phase;                     // electron_run phase (bits 0-7) and the particle's requeue count (bits 8-31)
    int slot;
    uint32_t ctr;                  // draws taken from the particle's stream
    uint64_t stream;               // the stream's key
    uint4 rs;                      // the stream's generator state, where ctr > 0
};

// A particle's random stream: xoshiro128** keyed by the stream's 64-bit key,
// with the count of draws taken from it (the position that keys the
// streams of the particle's secondaries).  A particle that has drawn travels
// through the queues with its generator state; one that has not (a new
// secondary) starts from its key.
struct StreamAt {
    Xoshiro g;
    uint32_t n;
    __device__ __forceinline__ void at(uint64_t seed, uint64_t stream, uint32_t pos, const uint4 &s) {
        n = pos;
        if (pos == 0) {
            g.init(seed, stream);
        } else {
            g.s0 = s.x; g.s1 = s.y; g.s2 = s.z; g.s3 = s.w;
        }
    }
    __device__ __forceinline__ uint4 state() const { return make_uint4(g.s0, g.s1, g.s2, g.s3); }
    template <class R> __device__ __forceinline__ R next() {
        n++;
        return g.template next<R>();
    }
};

__device__ __forceinline__ uint64_t child_stream(uint64_t s, uint32_t n) {
    // splitmix64 finaliser of (parent stream, draw position)
    uint64_t z = s ^ (0x9E3779B97F4A7C15ull * ((uint64_t)n + 1ull)) ^ 0xD1B54A32D192ED03ull;
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    return z ^ (z >> 31);
}

// Device-resident control block of one job (one batch of histories).
struct EvCtl {
    unsigned long long cnt[2][2];     // [round parity][photon, charged] queued particles (charged: two bands, see wave_exchange)
    long long nhist, next_hist;       // histories of the job / injected so far
    long long inj_h0, inj_n, inj_at;  // injection of the coming round
    long long target, cap;
    long long inj_max;                // primaries injected per round at most (0: no limit)
    long long rounds, done_round;     // rounds retired; round at which the job drained (-1 while running)
    unsigned long long events[2];     // photon / charged particles taken from the queues
    unsigned long long peak;          // largest number of particles in flight
    unsigned long long claim[2][2];   // [round parity][photon, charged] queue entries claimed by lanes
    int inj_dest;                     // pool of the primaries: 0 photons, 1 charged
    int err;                          // bit 0: pool overflow; bit 1: a particle exceeded an iteration guard
    // the first particle dropped by a guard: why (Engine::aborted, 5 lane
    // trips, 6 requeues), the source line of the guard, and its state
    int drop_why, drop_site, drop_iq, drop_ix, drop_iy, drop_iz, drop_phase, drop_age;
    float drop_e;
};

// Records the first particle a guard dropped (one lane of the whole job wins).
template <class R>
__device__ __forceinline__ void note_drop(EvCtl *c, int why, int site, const Part<R> &p, int phase, int age) {
    if (atomicCAS(&c->drop_why, 0, why) == 0) {
        c->drop_site = site;
        c->drop_iq = p.iq;
        c->drop_ix = p.ix;
        c->drop_iy = p.iy;
        c->drop_iz = p.iz;
        c->drop_phase = phase;
        c->drop_age = age;
        c->drop_e = (float)p.e;
    }
}

// Dynamic LDS of an event kernel that stages the tables of st, byte offsets: the
// electron bins (ST_BINS) from 0, then the media, their cut-offs and the voxel
// planes (ST_GEOM), then the deposit lists (TallyList).  `bytes` is the whole.
struct LdsLayout { int med, ecut, planes, list, bytes; };
template <class R>
inline LdsLayout lds_layout(int st, int nmed, int nx, int ny, int nz, size_t bin_bytes, size_t list_bytes) {
    auto up = [](size_t n) { return (n + 15) / 16 * 16; };
    const size_t geom = (st & ST_GEOM) != 0;
    LdsLayout l;
    l.med = (st & ST_BINS) != 0 ? (int)up(bin_bytes) : 0;
    l.ecut = l.med + (int)(geom * up(sizeof(Med<R>) * nmed));
    l.planes = l.ecut + (int)(geom * up(sizeof(R) * MXMED));
    l.list = l.planes + (int)(geom * up(sizeof(R) * ((size_t)nx + ny + nz + 3)));
    l.bytes = l.list + (int)list_bytes;
    return l;
}

template <class R> struct EvArgs {
    const Tables<R> *t;
    const Geom<R> *g;
    uint64_t seed;
    Pool<R> in;                       // input pool of this kernel's type
    const unsigned long long *n_in;   // its length
    Pool<R> outp, oute;               // photon and charged output pools
    unsigned long long *n_out;        // [2] their lengths
    unsigned long long *claim;        // entries of the input queue claimed so far (zero at launch)
    long long cap;                    // capacity of each pool
    double *endep;                    // tally base
    long slot_stride;                 // tally stride per slot
    uint8_t *touched;                 // optional tile marks of the tallies (TallyAtomic)
    long touch_stride;                // tile marks per slot
    double *ebal;                     // optional [EB_N] energy balance (escape, lost)
    unsigned long long *counters;     // [8] event counters (optional)
    int *err;                         // EvCtl::err
    int budget;                       // electron ustep iterations between refills of a wave
    int turns;                        // electrons: refills a particle may hold its lane before it is requeued (0: no limit)
    int max_age;                      // electrons: requeues after which a particle counts as stuck (dropped, err bit 1)
    int delta;                        // photons: 1 delta tracking, 0 voxel-by-voxel flight
    int nsplit;                       // photon splitting factor (vrt.nsplit); > 1 runs k_event_split for photons
    EvCtl *ctl;                       // the job's control block (guard reports)
    const CBin<R> *ebin;              // ST_BINS kernels: the electron half of Tables::cbin
    int eb_words;                     // its size in 16-byte words
    LdsLayout lds;                    // where the staged tables and lists start
    int tlist;                        // charged kernel: deposit-list entries per lane in LDS (TallyList)
    int waves;                        // wavefronts of this launch the device holds at once (lane_share)
};

__device__ __forceinline__ uint4 pack4(float a, float b, float c, float d) {
    return make_uint4(__float_as_uint(a), __float_as_uint(b), __float_as_uint(c), __float_as_uint(d));
}
__device__ __forceinline__ uint4 pack2(double a, double b) {
    return make_uint4((uint32_t)__double2loint(a), (uint32_t)__double2hiint(a), (uint32_t)__double2loint(b),
                      (uint32_t)__double2hiint(b));
}
__device__ __forceinline__ double lo2(const uint4 &v) { return __hiloint2double((int)v.y, (int)v.x); }
__device__ __forceinline__ double hi2(const uint4 &v) { return __hiloint2double((int)v.w, (int)v.z); }

// the slot word carries the charge as well, which leaves the slot 30 bits
constexpr int MAX_SLOTS = 1 << 30;
__device__ __forceinline__ uint32_t slot_word(int slot, int iq) { return ((uint32_t)slot << 2) | (uint32_t)(iq + 1); }

__device__ __forceinline__ void load(const Pool<float> &P, long long i, Queued<float> &q) {
    const OMC_GLOBAL uint4 *b = (const OMC_GLOBAL uint4 *)P.base + i;
    uint4 v[6];
#pragma unroll
    for (int k = 0; k < 6; k++) {
        const OMC_GLOBAL uint32_t *w = (const OMC_GLOBAL uint32_t *)(b + k * P.cap);
        v[k] = make_uint4(w[0], w[1], w[2], w[3]);
    }
    q.p.e = __uint_as_float(v[0].x); q.p.x = __uint_as_float(v[0].y); q.p.y = __uint_as_float(v[0].z); q.p.z = __uint_as_float(v[0].w);
    q.p.u = __uint_as_float(v[1].x); q.p.v = __uint_as_float(v[1].y); q.p.w = __uint_as_float(v[1].z); q.p.wt = __uint_as_float(v[1].w);
    q.demfp = __uint_as_float(v[2].x); q.sig0 = __uint_as_float(v[2].y); q.p.ix = (int)v[2].z; q.p.iy = (int)v[2].w;
    q.p.iz = (int)v[3].x; q.phase = (int)v[3].y; q.slot = (int)(v[3].z >> 2); q.p.iq = (int)(v[3].z & 3u) - 1; q.ctr = v[3].w;
    q.stream = (uint64_t)v[4].x | ((uint64_t)v[4].y << 32);
    q.rs = make_uint4(v[4].z, v[4].w, v[5].x, v[5].y);
}
__device__ __forceinline__ void load(const Pool<double> &P, long long i, Queued<double> &q) {
    const OMC_GLOBAL uint4 *b = (const OMC_GLOBAL uint4 *)P.base + i;
    uint4 v[8];
#pragma unroll
    for (int k = 0; k < 8; k++) {
        const OMC_GLOBAL uint32_t *w = (const OMC_GLOBAL uint32_t *)(b + k * P.cap);
        v[k] = make_uint4(w[0], w[1], w[2], w[3]);
    }
    q.p.e = lo2(v[0]); q.p.x = hi2(v[0]); q.p.y = lo2(v[1]); q.p.z = hi2(v[1]);
    q.p.u = lo2(v[2]); q.p.v = hi2(v[2]); q.p.w = lo2(v[3]); q.p.wt = hi2(v[3]);
    q.demfp = lo2(v[4]); q.sig0 = hi2(v[4]);
    q.p.ix = (int)v[5].x; q.p.iy = (int)v[5].y; q.p.iz = (int)v[5].z; q.phase = (int)v[5].w;
    q.slot = (int)(v[6].x >> 2); q.p.iq = (int)(v[6].x & 3u) - 1; q.ctr = v[6].y;
    q.stream = (uint64_t)v[6].z | ((uint64_t)v[6].w << 32);
    q.rs = v[7];
}

__device__ __forceinline__ void put4(OMC_GLOBAL uint4 *at, const uint4 &v) {
    OMC_GLOBAL uint32_t *w = (OMC_GLOBAL uint32_t *)at;
    w[0] = v.x; w[1] = v.y; w[2] = v.z; w[3] = v.w;
}
// (a new stream, ctr 0, starts from its key: its state is not written)
__device__ __forceinline__ void store(const Pool<float> &P, long long i, const Queued<float> &q) {
    OMC_GLOBAL uint4 *b = (OMC_GLOBAL uint4 *)P.base + i;
    put4(b, pack4(q.p.e, q.p.x, q.p.y, q.p.z));
    put4(b + P.cap, pack4(q.p.u, q.p.v, q.p.w, q.p.wt));
    put4(b + 2 * P.cap, make_uint4(__float_as_uint(q.demfp), __float_as_uint(q.sig0), (uint32_t)q.p.ix, (uint32_t)q.p.iy));
    put4(b + 3 * P.cap, make_uint4((uint32_t)q.p.iz, (uint32_t)q.phase, slot_word(q.slot, q.p.iq), q.ctr));
    put4(b + 4 * P.cap, make_uint4((uint32_t)q.stream, (uint32_t)(q.stream >> 32), q.rs.x, q.rs.y));
    if (q.ctr != 0u) put4(b + 5 * P.cap, make_uint4(q.rs.z, q.rs.w, 0u, 0u));
}
__device__ __forceinline__ void store(const Pool<double> &P, long long i, const Queued<double> &q) {
    OMC_GLOBAL uint4 *b = (OMC_GLOBAL uint4 *)P.base + i;
    put4(b, pack2(q.p.e, q.p.x));
    put4(b + P.cap, pack2(q.p.y, q.p.z));
    put4(b + 2 * P.cap, pack2(q.p.u, q.p.v));
    put4(b + 3 * P.cap, pack2(q.p.w, q.p.wt));
    put4(b + 4 * P.cap, pack2(q.demfp, q.sig0));
    put4(b + 5 * P.cap, make_uint4((uint32_t)q.p.ix, (uint32_t)q.p.iy, (uint32_t)q.p.iz, (uint32_t)q.phase));
    put4(b + 6 * P.cap, make_uint4(slot_word(q.slot, q.p.iq), q.ctr, (uint32_t)q.stream, (uint32_t)(q.stream >> 32)));
    if (q.ctr != 0u) put4(b + 7 * P.cap, q.rs);
}

// Reserves an output slot for every lane with `want`, one atomic per wave.
// Reached by all lanes of the wavefront together.
__device__ __forceinline__ long long wave_reserve(unsigned long long *counter, bool want) {
    unsigned long long mask = __ballot(want);
    if (mask == 0) return -1;
    int lane = threadIdx.x & 63;
    int leader = __ffsll((unsigned long long)mask) - 1;
    unsigned long long base = 0;
    if (lane == leader) base = atomicAdd(counter, (unsigned long long)__popcll(mask));
    base = __shfl(base, leader);
    unsigned long long below = mask & ((1ull << lane) - 1ull);
    return want ? (long long)(base + __popcll(below)) : -1;
}

// Total energy (MeV) above which a charged particle joins the high band of
// the charged queue.  The queue holds two bands in one pool: particles below
// fill it from index 0 up, those above from the last index down, and the
// charged kernel takes the low band first.  A wave's lanes then hold
// particles of similar energy, whose steps branch alike: on the c3 plan
// 22.8 M histories/s against 21.6 M with one unsorted queue (thresholds 1.2
// and 1.5 alike, 2.5 slightly slower).  Where a particle sits in the queue
// does not change its track.
constexpr float CHARGED_BAND_E = 1.5f;

// Places of a wave's new queue entries, and of the entries its free lanes take
// next, from one atomic instruction: lane 0 reserves in the photon output pool,
// lane 1 in the charged one, lane 2 claims from the input queue.  (Reserved and
// claimed one after the other, each waited out an atomic of its own.)  Up to
// two particles a lane are appended: an entry goes to the photon pool or, by
// its energy, to one of the charged pool's bands; a photon of zero weight (one
// that lost the roulette of photon splitting) would deposit nothing and is not
// queued.  The charged pool's counter packs the low band's length (bits 0-31)
// and the high band's (bits 32-63); a reservation that would make the bands
// meet writes nothing and reports an overflow (the job is rerun with larger
// pools).  Reached by all lanes of the wavefront together.
enum { Q_NONE = 0, Q_PHOTON = 1, Q_LOW = 2, Q_HIGH = 3 };
template <class R> __device__ __forceinline__ int queue_of(bool want, const Part<R> &p) {
    if (!want) return Q_NONE;
    if (p.iq == 0) return p.wt != (R)0 ? Q_PHOTON : Q_NONE;
    return p.e > (R)CHARGED_BAND_E ? Q_HIGH : Q_LOW;
}
struct Places { long long a, b, next; };       // -1: none (not wanted, or an overflow)
template <class R>
__device__ __forceinline__ Places wave_exchange(const EvArgs<R> &x, int qa, int qb, bool take) {
    const unsigned long long pa = __ballot(qa == Q_PHOTON), pb = __ballot(qb == Q_PHOTON);
    const unsigned long long la = __ballot(qa == Q_LOW), lb = __ballot(qb == Q_LOW);
    const unsigned long long ha = __ballot(qa == Q_HIGH), hb = __ballot(qb == Q_HIGH);
    const unsigned long long tk = __ballot(take);
    Places r = {-1, -1, -1};
    if (!(pa | pb | la | lb | ha | hb | tk)) return r;
    const unsigned long long nph = (unsigned long long)(__popcll(pa) + __popcll(pb));
    const unsigned long long nlo = (unsigned long long)(__popcll(la) + __popcll(lb));
    const unsigned long long nhi = (unsigned long long)(__popcll(ha) + __popcll(hb));
    const unsigned long long ntk = (unsigned long long)__popcll(tk);
    const int lane = threadIdx.x & 63;
    const unsigned long long v = lane == 0 ? nph : lane == 1 ? (nlo | (nhi << 32)) : lane == 2 ? ntk : 0ull;
    unsigned long long base = 0;
    if (v) base = atomicAdd(lane == 2 ? x.claim : x.n_out + lane, v);
    const unsigned long long bph = __shfl(base, 0), bch = __shfl(base, 1), btk = __shfl(base, 2);
    const unsigned long long below = (1ull << lane) - 1ull;
    const long long lo0 = (long long)(bch & 0xffffffffull), hi0 = (long long)(bch >> 32);
    const bool fits = lo0 + (long long)nlo + hi0 + (long long)nhi <= x.cap;
    auto place = [&](int q, long long ph, long long lo, long long hi) -> long long {
        if (q == Q_NONE) return -1;
        if (q == Q_PHOTON ? ph >= x.cap : !fits) {
            atomicOr(x.err, 1);
            return -1;
        }
        return q == Q_PHOTON ? ph : q == Q_LOW ? lo : x.cap - 1 - hi;
    };
    r.a = place(qa, (long long)bph + __popcll(pa & below), lo0 + __popcll(la & below), hi0 + __popcll(ha & below));
    r.b = place(qb, (long long)bph + __popcll(pa) + __popcll(pb & below), lo0 + __popcll(la) + __popcll(lb & below),
                hi0 + __popcll(ha) + __popcll(hb & below));
    if (take) r.next = (long long)btk + __popcll(tk & below);
    return r;
}

// Copies the tables of ST to LDS; every thread of the workgroup calls it.
template <class R, int ST>
__device__ __forceinline__ Staged<R> stage(const EvArgs<R> &a, unsigned char *base) {
    Staged<R> s = {};
    if constexpr ((ST & ST_BINS) != 0) {
        uint4 *dst = reinterpret_cast<uint4 *>(base);
        const uint4 *src = reinterpret_cast<const uint4 *>(a.ebin);
        for (int i = threadIdx.x; i < a.eb_words; i += blockDim.x) dst[i] = src[i];
        s.bins = (const OMC_LDS CBin<R> *)base;
    }
    if constexpr ((ST & ST_GEOM) != 0) {
        const OMC_CONST Tables<R> &t = constant(a.t);
        const OMC_CONST Geom<R> &g = constant(a.g);
        static_assert(sizeof(Med<R>) % 4 == 0, "copied in words");
        uint32_t *dm = reinterpret_cast<uint32_t *>(base + a.lds.med);
        const uint32_t *sm = reinterpret_cast<const uint32_t *>(t.med);
        for (int i = threadIdx.x; i < t.nmed * (int)(sizeof(Med<R>) / 4); i += blockDim.x) dm[i] = gld(sm + i);
        R *ec = reinterpret_cast<R *>(base + a.lds.ecut);
        if (threadIdx.x < MXMED) ec[threadIdx.x] = g.ecut[threadIdx.x];
        R *xb = reinterpret_cast<R *>(base + a.lds.planes), *yb = xb + g.nx + 1, *zb = yb + g.ny + 1;
        for (int i = threadIdx.x; i <= g.nx; i += blockDim.x) xb[i] = gld(g.xb + i);
        for (int i = threadIdx.x; i <= g.ny; i += blockDim.x) yb[i] = gld(g.yb + i);
        for (int i = threadIdx.x; i <= g.nz; i += blockDim.x) zb[i] = gld(g.zb + i);
        s.med = (const OMC_LDS Med<R> *)dm;
        s.ecut = (const OMC_LDS R *)ec;
        s.xb = (const OMC_LDS R *)xb;
        s.yb = (const OMC_LDS R *)yb;
        s.zb = (const OMC_LDS R *)zb;
    }
    if constexpr (ST != 0) __syncthreads();
    return s;
}

// Charged kernel's tally.  Like TallyAtomic it sums a lane's consecutive
// deposits to one region in a register, but a finished sum goes to a list of
// (slot, region, energy) entries the lane holds in LDS, and the wave adds the
// lists to device memory with FP64 atomics once per pass of its loop, where
// it meets to refill.  On gfx950 a load's wait for its data also waits for
// every earlier store and atomic of the wave, so a tally atomic inside the
// step loop stalled the following steps' loads.  A full list falls back to a
// direct atomic.  The sums are the same; only their order changes.  Measured
// on the 1960-beamlet plan in FP32, two runs each on one box: 22.55 and 22.82
// against 22.51 and 22.40 M histories/s (the 10,044-beamlet plan unchanged).
// The atomics still wait where the wave meets, so the gain stays well below
// the 4.4% a copy that issued no tally atomics in the step loop ran faster.
struct TallyList {
    double *endep;       // the particle's slot (direct atomics of a full list)
    uint8_t *touched;
    int slot, cur, k, cap;
    double acc;
    int2 *key;           // this lane's entries, strided by the workgroup size
    double *val;
    int stride;
    __device__ __forceinline__ void init(double *p, uint8_t *tf, int s) {
        endep = p;
        touched = tf;
        slot = s;
        cur = -1;
        acc = 0.0;
    }
    __device__ __forceinline__ void push(int r, double v) {
        if (r < 0 || v == 0.0) return;
        if (k < cap) {
            key[k * stride] = make_int2(slot, r);
            val[k * stride] = v;
            k++;
        } else {
            atomicAdd(endep + r, v);
            if (touched) touched[r >> TALLY_TILE_LOG2] = 1;
        }
    }
    __device__ __forceinline__ void add(int region, double v) {
        if (region != cur) {
            push(cur, acc);
            cur = region;
            acc = v;
        } else {
            acc += v;
        }
    }
    __device__ __forceinline__ void flush() {
        push(cur, acc);
        cur = -1;
        acc = 0.0;
    }
    // adds the lane's list to the tallies and empties it
    __device__ __forceinline__ void drain(double *base, long slot_stride, uint8_t *tbase, long touch_stride) {
        for (int j = 0; j < k; j++) {
            const int2 kk = key[j * stride];
            atomicAdd(base + (size_t)kk.x * slot_stride + kk.y, val[j * stride]);
            if (tbase) tbase[(size_t)kk.x * touch_stride + (kk.y >> TALLY_TILE_LOG2)] = 1;
        }
        k = 0;
    }
};

template <bool COUNT>
__device__ __forceinline__ void flush_counters(unsigned long long *dst, const Counters &c) {
    if (!COUNT || !dst) return;
    unsigned long long v[7] = {c.nhowfar, c.nhownear, c.ncross, c.ndep, c.nrn, c.nphoton, c.nelectron};
#pragma unroll
    for (int k = 0; k < 7; k++) {
        unsigned long long x = v[k];
        for (int off = 32; off > 0; off >>= 1) x += __shfl_xor(x, off);
        if ((threadIdx.x & 63) == 0 && x) atomicAdd(dst + k, x);
    }
}

// The photon kernel takes the registers it needs (149 VGPRs, 3 waves per
// SIMD).  Capped at 4 waves (128 VGPRs, 12 bytes of spills) its busy time on
// the c3 plan fell by a fifth with the plan's rate unchanged, but single
// dose runs, where it has a stream to itself, ran 1% slower (c2 16.8 against
// 17.0 M histories/s).
// Occupancy hint of the charged-particle kernel (waves per SIMD).  With the
// whole engine inlined the kernel keeps its state in registers; capping it at
// 4 or 3 waves spills that state to scratch, and on gfx950 2 waves measured
// fastest (C3 subset: 6.0 M histories/s at 2, 5.9 M at 3, 4.9 M at 4).
#ifndef OMC_CHARGED_WAVES_PER_EU
#define OMC_CHARGED_WAVES_PER_EU 2
#endif

// Persistent transport of one particle type.  Every lane holds one particle
// in registers and advances it -- one photon() call, or up to a.budget
// condensed-history steps of electron_run() -- then the wave meets: lanes
// whose particle left, or turned into the other type, hand it and any
// secondary to the output queues and claim the next queued particle (one
// atomic instruction a trip, wave_exchange).  A particle of this kernel's type stays in its lane until
// it is gone, so the queues only carry new secondaries and type changes, and
// no lane idles while the queue still holds work.  The wave exits when its
// lanes are empty and the queue is exhausted.
//
// Two things keep a launch short.  A wave reads the claim counter before its
// first claim, and claims no more once a claim has come back from beyond the
// queue's end, so idle waves of an exhausted queue leave without serialising on
// that one address (8192 waves queueing on it cost ~100 us
// per launch).  And an electron that has held its lane for a.turns refills
// is handed back to the queue with its resumable state (position in its
// random stream, distance to the next discrete interaction, step phase): an
// electron in single-scattering mode along a voxel face can take thousands
// of steps, and without the hand-back it alone would hold the round -- and
// every particle queued behind the round -- open for tens of milliseconds.
// Where a particle is requeued does not change its track.  The requeue count
// travels with the particle (high bits of its phase word): a particle that
// would make no progress is dropped and reported after a.max_age requeues,
// instead of cycling through rounds until the job's round guard ends it.
template <class R, bool PHOTON, bool COUNT, int ST>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(PHOTON ? 1 : OMC_CHARGED_WAVES_PER_EU)))
k_event(EvArgs<R> a) {
    // the charged queue: low band [0, n_lo), then the high band from cap - 1 down
    const unsigned long long pk = *a.n_in;
    extern __shared__ __align__(16) unsigned char omc_lds[];
    const Staged<R> lds = stage<R, ST>(a, omc_lds);
    // FP32 charged kernel: each lane's deposit list follows the tables in LDS,
    // keys [tlist][blockDim.x] then energies [tlist][blockDim.x].  (The FP64
    // kernel, which spills registers, ran 1% slower with the lists.)
    constexpr bool LIST = !PHOTON && sizeof(R) == 4;
    using Tally = typename std::conditional<LIST, TallyList, TallyAtomic>::type;
    Tally tally;
    if constexpr (LIST) {
        unsigned char *lst = omc_lds + a.lds.list;
        tally.key = reinterpret_cast<int2 *>(lst) + threadIdx.x;
        tally.val = reinterpret_cast<double *>(lst + (size_t)a.tlist * blockDim.x * sizeof(int2)) + threadIdx.x;
        tally.stride = (int)blockDim.x;
        tally.cap = a.tlist;
        tally.k = 0;
        tally.init(a.endep, a.touched, 0);
    } else {
        tally.init(a.endep);
    }
    const long long n_lo = PHOTON ? (long long)pk : (long long)(pk & 0xffffffffull);
    const long long n = PHOTON ? (long long)pk : n_lo + (long long)(pk >> 32);
    const bool takes = (int)(threadIdx.x & 63) < lane_share(n, a.waves);
    Counters tot = {0, 0, 0, 0, 0, 0, 0};
    double eb_esc = 0.0;             // photons that left the phantom (photon kernel only)
    bool have = false;
    Part<R> p, q;
    uint64_t stream = 0;
    int slot = 0, phase = 0;
    R demfp = (R)0, sig0 = (R)0;
    StreamAt rng;
    int iters = 0, turns = 0, age = 0;
    long long idx = -1;              // the entry a free lane takes next
    bool open = false;               // the queue may hold entries nobody has claimed
    {
        const unsigned long long seen = __shfl(*(volatile const unsigned long long *)a.claim, 0);
        if ((long long)seen < n) {
            idx = wave_reserve(a.claim, takes);
            open = true;
        }
    }
    for (;;) {
        open = open && !__any(idx >= n);
        if (!have && idx >= 0 && idx < n) {
            iters = 0;
            turns = 0;
            if (!PHOTON && idx >= n_lo) idx = a.cap - 1 - (idx - n_lo);
            Queued<R> in;
            load(a.in, idx, in);
            p = in.p;
            stream = in.stream;
            slot = in.slot;
            demfp = in.demfp;
            sig0 = in.sig0;
            age = in.phase >> 8;
            phase = in.phase & 0xff;
            rng.at(a.seed, stream, in.ctr, in.rs);
            if constexpr (LIST)
                tally.init(a.endep + (size_t)slot * a.slot_stride,
                           a.touched ? a.touched + (size_t)slot * a.touch_stride : nullptr, slot);
            else
                tally.init(a.endep + (size_t)slot * a.slot_stride,
                           a.touched ? a.touched + (size_t)slot * a.touch_stride : nullptr);
            have = true;
        }
        if (!__any(have)) break;
        int d = -1;
        bool done = false;
        uint32_t qpos = 0;
        if (have) {
            Engine<R, StreamAt, Tally, ST> e{constant(a.t), constant(a.g), rng, tally, {0, 0, 0, 0, 0, 0, 0}, COUNT};
            e.nsplit = a.nsplit;          // roulette of the photons that charged particles produce
            e.lds = lds;
            if (PHOTON) {
                d = a.delta ? e.photon_delta(p, q) : e.photon(p, q);
            } else {
                typename decltype(e)::EState es;
                es.demfp = demfp;
                es.sig0 = sig0;
                es.phase = phase;
                d = e.electron_run(p, q, es, a.budget);
                demfp = es.demfp;
                sig0 = es.sig0;
                phase = es.phase;
            }
            qpos = rng.n;
            // a particle that made no progress within its guards is dropped
            // and reported (EvCtl::err bit 1), never transported forever
            if (e.aborted || ++iters > (1 << 22)) {
                atomicOr(a.err, 2);
                note_drop(a.ctl, e.aborted ? e.aborted : 5, e.abort_site, p, phase, age);
                d = -1;
            }
            // d: -1 particle gone, 0 particle continues, +1 continues with a secondary
            done = d < 0 || ((p.iq == 0) != PHOTON);
            if (!PHOTON && !done && a.turns > 0 && ++turns >= a.turns) {            // requeue, see above
                done = true;
                if (++age > a.max_age) {
                    atomicOr(a.err, 2);
                    note_drop(a.ctl, 6, 0, p, phase, age);
                    d = -1;
                }
            }
            if (done) tally.flush();
            if (PHOTON) eb_esc += e.esc;
            // dropped energy is rare (quirk Q6, guards): added where it occurs
            if (e.lost != 0.0 && a.ebal) atomicAdd(a.ebal + EB_LOST, e.lost);
            if (COUNT) {
                tot.nhowfar += e.cnt.nhowfar; tot.nhownear += e.cnt.nhownear; tot.ncross += e.cnt.ncross;
                tot.ndep += e.cnt.ndep; tot.nrn += e.cnt.nrn; tot.nphoton += e.cnt.nphoton;
                tot.nelectron += e.cnt.nelectron;
            }
        }
        // the finished sums go out first: the exchange below waits for its
        // atomic, and a wait for one covers every memory operation before it
        if constexpr (LIST) tally.drain(a.endep, a.slot_stride, a.touched, a.touch_stride);
        const int qa = queue_of(have && done && d >= 0, p), qb = queue_of(have && d == 1, q);
        if (done) have = false;
        const Places at = wave_exchange(a, qa, qb, open && takes && !have);
        if (at.a >= 0)
            store(p.iq == 0 ? a.outp : a.oute, at.a,
                  Queued<R>{p, demfp, sig0, phase | (age << 8), slot, qpos, stream, rng.state()});
        if (at.b >= 0)
            store(q.iq == 0 ? a.outp : a.oute, at.b,
                  Queued<R>{q, (R)0, (R)0, 0, slot, 0u, child_stream(stream, qpos), uint4{}});
        idx = at.next;
    }
    if (PHOTON && a.ebal) wave_add(a.ebal + EB_ESCAPE, eb_esc);
    flush_counters<COUNT>(a.counters, tot);
}

// Persistent transport of photons with splitting (src/ompmc.c:1867-2139,
// nsplit > 1).  A lane holds one photon and splits it: nsplit sub-photons of
// weight wt/nsplit fly stratified numbers of mean free paths along its ray,
// each from the interaction site of the one before; a sub-photon that leaves
// the geometry ends the split.  Charged products keep the sub-photon's
// weight and are queued.  Of the scattered photons only those of one
// randomly chosen sub-photon survive, with the full weight; there is at most
// one, and it goes back to the photon queue, with its place in its random
// stream, to be split in a later round.  (Kept in the lane, a photon that
// scatters many times held the whole launch open; requeued, it follows the
// same track.)  The reference keeps the same particles on its stack, in
// another order.
//
// The loop over sub-photons has the same trip count on every lane, so a
// wave queues the products of each sub-photon together (one atomic per
// wave).  Each product gets a random stream of its own, keyed by the
// photon's stream and its draw position after the interaction; the second
// product of a pair by the complement of the stream.
template <class R, bool COUNT, int ST>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1)))
k_event_split(EvArgs<R> a) {
    extern __shared__ __align__(16) unsigned char omc_lds[];
    const Staged<R> lds = stage<R, ST>(a, omc_lds);
    const long long n = (long long)*a.n_in;
    const int ns = a.nsplit;
    const bool takes = (int)(threadIdx.x & 63) < lane_share(n, a.waves);
    Counters tot = {0, 0, 0, 0, 0, 0, 0};
    double eb_esc = 0.0, eb_lost = 0.0;
    for (;;) {
        // every lane is free here: the wave claims a photon for each lane that takes one
        long long idx = -1;
        const unsigned long long seen = __shfl(*(volatile const unsigned long long *)a.claim, 0);
        if ((long long)seen < n) idx = wave_reserve(a.claim, takes);
        const bool have = idx >= 0 && idx < n;
        if (!__any(have)) break;
        Part<R> p;
        uint64_t stream = 0;
        int slot = 0;
        StreamAt rng;
        TallyAtomic tally;
        tally.init(a.endep);
        if (have) {
            Queued<R> in;
            load(a.in, idx, in);
            p = in.p;
            stream = in.stream;
            slot = in.slot;
            rng.at(a.seed, stream, in.ctr, in.rs);
            tally.init(a.endep + (size_t)slot * a.slot_stride,
                       a.touched ? a.touched + (size_t)slot * a.touch_stride : nullptr);
        }
        Engine<R, StreamAt, TallyAtomic, ST> e{constant(a.t), constant(a.g), rng, tally, {0, 0, 0, 0, 0, 0, 0}, COUNT};
        e.nsplit = ns;
        e.lds = lds;
        // set-up of the split (src/ompmc.c:1900-1940)
        bool live = have, surv = false;
        R eig = (R)0, gle = (R)0, eta = (R)0, d_eta = (R)0, dpmfp_old = (R)0, wtsave = (R)0;
        int i_survive = -1, imed = -1, lgle = 0;
        R cohfac = (R)0, gmfp = (R)0;
        Part<R> save = p;
        typename Engine<R, StreamAt, TallyAtomic, ST>::SplitXs xs;
        if (live) {
            if (COUNT) e.cnt.nphoton++;
            imed = e.medium(p);
            eig = p.e;
            if (eig <= e.pcut_of(imed) || p.wt == (R)0) {
                e.ausgab(p, eig);
                live = false;
            } else {
                gle = M<R>::log(eig);
                e.split_xs(gle, xs);
                R rnno = e.rnd();
                rnno /= (R)ns;
                d_eta = (R)1.0 / (R)ns;
                eta = (R)1.0 - rnno + d_eta;
                wtsave = p.wt / (R)ns;
                rnno = e.rnd();
                i_survive = (int)(rnno * (R)ns);
            }
        }
        // the sub-photons (src/ompmc.c:1942-2111)
        for (int isplit = 0; isplit < ns; isplit++) {
            if (!__any(live)) break;
            Part<R> c0, c1;
            bool w0 = false, w1 = false;
            uint32_t cpos = 0;
            if (live) {
                eta -= d_eta;
                if (eta <= (R)0.0) {
                    live = false;
                } else {
                    R dpmfp = -M<R>::log(eta) - dpmfp_old;
                    dpmfp_old += dpmfp;
                    Part<R> sp = save;
                    sp.wt = wtsave;
                    sp.iq = 0;
                    if (!e.split_fly(sp, dpmfp, xs, imed, lgle, cohfac, gmfp, ns - isplit)) {
                        live = false;
                    } else {
                        save.x = sp.x; save.y = sp.y; save.z = sp.z;
                        save.ix = sp.ix; save.iy = sp.iy; save.iz = sp.iz;
                        const bool mine = isplit == i_survive;
                        R r = e.rnd();
                        if (r <= (R)1.0 - cohfac) {
                            if (mine) {
                                sp.wt *= (R)ns;
                                e.rayleigh(sp, imed, eig, gle, lgle);
                                p = sp;
                                surv = true;
                            }
                        } else {
                            Part<R> q;
                            int k = e.interact_pcp(sp, q, imed, eig, gle, lgle);
                            if (sp.iq != 0) {
                                c0 = sp;
                                w0 = true;
                            } else if (mine) {
                                sp.wt *= (R)ns;
                                p = sp;
                                surv = true;
                            }
                            if (k == 1) {
                                if (q.iq != 0) {
                                    c1 = q;
                                    w1 = true;
                                } else if (mine) {
                                    q.wt *= (R)ns;
                                    p = q;
                                    surv = true;
                                }
                            }
                        }
                        cpos = rng.n;
                    }
                }
            }
            const Places at = wave_exchange(a, queue_of(w0, c0), queue_of(w1, c1), false);
            if (at.a >= 0)
                store(a.oute, at.a, Queued<R>{c0, (R)0, (R)0, 0, slot, 0u, child_stream(stream, cpos), uint4{}});
            if (at.b >= 0)
                store(a.oute, at.b, Queued<R>{c1, (R)0, (R)0, 0, slot, 0u, child_stream(~stream, cpos), uint4{}});
        }
        if (have && e.aborted) {
            atomicOr(a.err, 2);
            note_drop(a.ctl, e.aborted, e.abort_site, p, 0, 0);
            if (surv) e.lost += (double)p.wt * (double)p.e;
            surv = false;
        }
        tally.flush();
        eb_esc += e.esc;
        eb_lost += e.lost;
        // the survivor continues from its place in the photon's stream
        const Places at = wave_exchange(a, queue_of(have && surv, p), Q_NONE, false);
        if (at.a >= 0) store(a.outp, at.a, Queued<R>{p, (R)0, (R)0, 0, slot, rng.n, stream, rng.state()});
        if (COUNT && have) {
            tot.nhowfar += e.cnt.nhowfar; tot.nhownear += e.cnt.nhownear; tot.ncross += e.cnt.ncross;
            tot.ndep += e.cnt.ndep; tot.nrn += e.cnt.nrn; tot.nphoton += e.cnt.nphoton;
            tot.nelectron += e.cnt.nelectron;
        }
    }
    if (a.ebal) {
        wave_add(a.ebal + EB_ESCAPE, eb_esc);
        wave_add(a.ebal + EB_LOST, eb_lost);
    }
    flush_counters<COUNT>(a.counters, tot);
}

// Primaries of the coming round: histories [inj_h0, inj_h0 + inj_n) of the
// job, written to the input pool of their type from offset inj_at.
template <class R> struct SrcArgs {
    const Tables<R> *t;
    const Geom<R> *g;
    SrcDosxyz<R> dos;
    SrcBeamlets<R> bix;
    int use_beamlets;
    const long *slot_off;        // [nslot+1] first history of each tally slot in the job (nslot 0: one slot)
    const int *slot_beamlet;     // beamlet source: beamlet of each slot
    const int *slot_batch;       // beamlet source: batch of each slot (null: every slot is of `batch`)
    int nslot;
    int batch;
    long hist_base;              // dosxyz source: stream of history 0 of the job
    uint64_t seed;
    const EvCtl *ctl;
    Pool<R> out;                 // destination pool (photons or charged, by source charge)
    double *ebal;                // optional [EB_N] energy balance: the primaries' energy
};

template <class R>
__global__ void __launch_bounds__(256) k_source(SrcArgs<R> a) {
    const long n = (long)a.ctl->inj_n, h0 = (long)a.ctl->inj_h0, at = (long)a.ctl->inj_at;
    double eb_src = 0.0;
    for (long k = (long)blockIdx.x * blockDim.x + threadIdx.x; k < n; k += (long)gridDim.x * blockDim.x) {
        long h = h0 + k;
        int slot = 0, beamlet = 0;
        uint64_t stream = (uint64_t)(a.hist_base + h);
        if (a.nslot > 0) slot = find_slot(a.slot_off, a.nslot, h);
        if (a.use_beamlets) {
            beamlet = a.slot_beamlet[slot];
            stream = beamlet_stream(beamlet, a.slot_batch ? a.slot_batch[slot] : a.batch, h - a.slot_off[slot]);
        }
        StreamAt rng;
        rng.at(a.seed, stream, 0, uint4{});
        TallyNone tn;
        Engine<R, StreamAt, TallyNone> e{constant(a.t), constant(a.g), rng, tn, {0, 0, 0, 0, 0, 0, 0}, false};
        Part<R> p;
        if (a.use_beamlets) init_history(e, a.bix, beamlet, p);
        else init_history(e, a.dos, p);
        store(a.out, at + k, Queued<R>{p, (R)0, (R)0, 0, slot, rng.n, stream, rng.state()});
        eb_src += source_energy(p);
    }
    if (a.ebal) wave_add(a.ebal + EB_SOURCE, eb_src);
}

// Retires the round that read the pools of parity `par` and plans the
// injection of the next round (pools of parity 1 - par).  One thread.
__device__ __forceinline__ void round_end(EvCtl *c, int par) {
    c->events[0] += c->cnt[par][0];
    c->events[1] += (c->cnt[par][1] & 0xffffffffull) + (c->cnt[par][1] >> 32);
    c->cnt[par][0] = 0;
    c->cnt[par][1] = 0;
    c->claim[par][0] = 0;
    c->claim[par][1] = 0;
    int nx = 1 - par;
    if ((long long)c->cnt[nx][0] > c->cap) {
        c->err |= 1;
        c->cnt[nx][0] = (unsigned long long)c->cap;
    }
    {
        // an overflowing charged queue holds unwritten entries in both bands:
        // it is dropped (the job is rerun with larger pools)
        const unsigned long long pkc = c->cnt[nx][1];
        if ((long long)((pkc & 0xffffffffull) + (pkc >> 32)) > c->cap) {
            c->err |= 1;
            c->cnt[nx][1] = 0;
        }
    }
    const long long nch = (long long)((c->cnt[nx][1] & 0xffffffffull) + (c->cnt[nx][1] >> 32));
    long long inflight = (long long)c->cnt[nx][0] + nch;
    long long room = c->target - inflight;
    long long left = c->nhist - c->next_hist;
    long long space = c->cap - (c->inj_dest ? nch : (long long)c->cnt[nx][0]);
    long long n = left < room ? left : room;
    if (n > space) n = space;
    if (c->inj_max > 0 && n > c->inj_max) n = c->inj_max;
    if (n < 0) n = 0;
    c->inj_h0 = c->next_hist;
    c->inj_n = n;
    c->inj_at = c->inj_dest ? (long long)(c->cnt[nx][1] & 0xffffffffull) : (long long)c->cnt[nx][0];
    c->cnt[nx][c->inj_dest] += (unsigned long long)n;
    c->next_hist += n;
    if ((unsigned long long)(inflight + n) > c->peak) c->peak = (unsigned long long)(inflight + n);
    c->rounds++;
    if (inflight + n == 0 && c->done_round < 0) c->done_round = c->rounds;
}

static __global__ void k_round_end(EvCtl *c, int par) {
    if (blockIdx.x == 0 && threadIdx.x == 0) round_end(c, par);
}

// Starts a job: clears the queues and plans the first injection into the
// pools of parity 0.
static __global__ void k_job_start(EvCtl *c, long long nhist, long long target, long long cap, long long inj_max,
                                   int dest) {
    if (blockIdx.x != 0 || threadIdx.x != 0) return;
    c->cnt[0][0] = c->cnt[0][1] = c->cnt[1][0] = c->cnt[1][1] = 0;
    c->claim[0][0] = c->claim[0][1] = c->claim[1][0] = c->claim[1][1] = 0;
    c->nhist = nhist;
    c->next_hist = 0;
    c->target = target;
    c->cap = cap;
    c->inj_max = inj_max;
    c->rounds = -1;
    c->done_round = -1;
    c->events[0] = c->events[1] = 0;
    c->peak = 0;
    c->inj_dest = dest;
    c->err = 0;
    c->drop_why = c->drop_site = 0;
    round_end(c, 1);
}

}  // namespace omc
