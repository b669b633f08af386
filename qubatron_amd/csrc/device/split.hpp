/*
 * split.hpp - the end of a traversal launch: the rays still in flight are
 * split over the idle lanes of their wave.
 *
 * Once the work queue is dry a wave is left with its longest rays, one lane
 * each, and their steps are one serial chain while the other lanes idle. The
 * entries still pending on a ray's stack are subtrees that the ray enters
 * later, in a fixed order, and what the trace of one of them does depends on
 * nothing that happens before it: so an idle lane can trace them now. A
 * segment is such a part of a ray: it has the lane that owns the ray and an
 * interval [a, b) of keys in ray order. Every kBurst steps
 *
 *   - a segment that has pending entries and the idle lane paired with it
 *     share its work: the idle lane takes over the entries of the shallowest
 *     such level (the farthest and usually largest part) with the upper end
 *     of the key interval, copying the ray and the stack words down to that
 *     level;
 *   - a ray whose lowest unfinished key belongs to a hit has that hit as its
 *     result; one with no segment left has missed; segments beyond a hit of
 *     their ray are dropped.
 *
 * The result is the first hit in ray order, the one that the serial trace
 * reaches: same leaf, same entry point (recomputed from the same plane by
 * the same operations). Rays keep their lane's identity: the owner's outputs
 * are written by the owner.
 *
 * What bounds it: the latency of a step (about 0.9 us for a wave alone on its
 * SIMD: some 200 vector instructions and a dependent gather), times the steps
 * of the longest segment. A round costs a few dozen instructions and LDS
 * exchanges, so kBurst trades their number against the time a lane idles.
 * Measured with bursts of 4, 8 and 16 steps: k_primary + k_shadow of 320x240
 * frames of 1M points (three poses) 209, 197, 224 us, 191, 187, 188 and 104,
 * 107, 122; k_shadow of 1920x1080 frames of 10M points 357, 355, 371 us, 465,
 * 464, 482 and 112, 111, 111. Without sharing (with an earlier, longer step)
 * a shadow launch of the latter kind took 632 us against 408.
 *
 * Every step of the loop takes a segment further or ends it, no lane waits
 * for another inside a burst, and the loop ends when no ray is left.
 *
 * The iteration cap is that of the serial trace (near_cap), which takes no
 * more steps than a ray's segments together, at most 64 kBurst a round. So
 * rays are shared for half the cap's worth of rounds, if none of the wave has
 * used the other half up; a ray that still has no result then (it would take
 * a path of hundreds of thousands of nodes, or an array that is no tree)
 * starts again, unshared, and its steps are counted.
 */
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>

#ifndef QBT_HOST_BUILD
#include "qbt_internal.hpp"
#endif
#include "trace.hpp"

#pragma clang fp contract(off)

namespace qbt {

constexpr int      kBurst   = 8;           /* steps between two rounds of sharing */
constexpr uint32_t kKeyEnd  = 0x80000000u; /* keys of a whole ray: [0, kKeyEnd) */
constexpr uint32_t kNoKey   = 0xFFFFFFFFu;
constexpr int      kSegFree = 3;           /* segment state besides ST_*: the lane has none */

/* words of LDS the sharing uses per thread, after the stacks */
constexpr int kMailWords = 1;

/* LDS operations of one wave take effect in program order; this keeps the
 * compiler from moving them */
__device__ __forceinline__ void wave_order()
{
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

/* bits of m below this lane */
__device__ __forceinline__ int rank_of(uint64_t m)
{
    return (int) __builtin_amdgcn_mbcnt_hi((uint32_t) (m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t) m, 0u));
}

/* Traces the wave's rays (active lanes, each the owner of its ray) to their
 * results. mail: 64 words of LDS of this wave. finish(status) is called by
 * the owner with the result in t (ST_HIT: the leaf and its entry point) and
 * returns true if it has started another ray in r, t. Called by all 64 lanes
 * of the wave. */
template <bool CMP, bool DUAL, int SEM, bool GRID, class Finish>
__device__ __forceinline__ void drain(const SceneDev& s, Ray& r, const Stack& st, TraceState& t, bool active,
                                      uint32_t* mail, Finish&& finish)
{
    const int lane = threadIdx.x & 63;
    const int W    = DUAL ? 3 : 2; /* stack words per level and lane (stack_at) */
    bool      live = active;       /* this lane owns a ray that has no result yet */
    int       seg  = active ? (int) ST_CONT : kSegFree;
    int       own  = lane;
    uint32_t  a = 0, b = kKeyEnd;
    int       rounds = s.iter_cap / (2 * 64 * kBurst); /* left with sharing; none: rays are whole */
    if (__ballot(active && t.it > s.iter_cap / 2) != 0ull) rounds = 0;
    while (__ballot(live) != 0ull) {
        const int burst = __ballot(seg == ST_CONT && near_cap<CMP>(s, t, kBurst)) != 0ull ? 1 : kBurst;
        if (seg == ST_CONT) {
#pragma nounroll
            for (int k = 0; k < burst; k++) {
                seg = trace_step<CMP, DUAL, SEM, GRID>(s, r, st, t);
                if (seg != ST_CONT) break;
            }
            if (count_steps<CMP, DUAL>(s, t, burst)) seg = ST_ABORT;
        }
        /* the lowest hit of every ray (an aborted segment ends its ray like a
         * hit), then its lowest unfinished key */
        mail[lane] = kNoKey;
        wave_order();
        if (seg == ST_HIT || seg == ST_ABORT) atomicMin(&mail[own], a);
        wave_order();
        const uint32_t hit = mail[own];
        wave_order();
        if (seg != kSegFree && a > hit) seg = kSegFree;     /* beyond a hit of its ray */
        if (seg == ST_MISS && own != lane) seg = kSegFree;
        if (seg == ST_CONT) atomicMin(&mail[own], a);
        wave_order();
        const bool     done  = live && mail[lane] == hit; /* owner: own == lane, hit is its ray's */
        const uint64_t dmask = __ballot(done);
        if (dmask != 0ull) {
            const bool mine = seg != kSegFree && ((dmask >> own) & 1ull);
            wave_order();
            if (mine && a == hit) mail[own] = (uint32_t) lane;
            wave_order();
            const int src = done && hit != kNoKey ? (int) mail[lane] : lane;
            const int res = __shfl(seg, src, 64);
            t.entry.x     = __shfl(t.entry.x, src, 64);
            t.entry.y     = __shfl(t.entry.y, src, 64);
            t.entry.z     = __shfl(t.entry.z, src, 64);
            t.entry.w     = __shfl(t.entry.w, src, 64);
            t.ns          = __shfl(t.ns, src, 64);
            if (DUAL) t.nd = __shfl(t.nd, src, 64);
            t.ix = __shfl(t.ix, src, 64);
            t.iy = __shfl(t.iy, src, 64);
            t.iz = __shfl(t.iz, src, 64);
            if (mine) seg = kSegFree;
            if (done) {
                live = finish(hit == kNoKey ? (int) ST_MISS : res);
                if (live) seg = ST_CONT, a = 0, b = kKeyEnd;
            }
        }
        if (rounds > 0 && --rounds == 0) { /* the unfinished rays again, whole */
            seg = kSegFree;
            if (live) {
                t.entry = root_entry<SEM>(s, r, root_face(t));
                t.level = t.ix = t.iy = t.iz = t.ns = t.nd = t.it = 0;
                t.pend &= kRayBits;
                seg = ST_CONT, a = 0, b = kKeyEnd;
            }
        }
        /* share */
        if (seg == kSegFree) own = lane;
        const uint32_t below = t.pend & ((1u << t.level) - 1u);
        const bool     gives = rounds > 0 && seg == ST_CONT && below != 0u && b - a >= 2u;
        const bool     idle  = seg == kSegFree && !live;
        const uint64_t gmask = __ballot(gives), imask = __ballot(idle);
        const int      pairs = min((int) __popcll(gmask), (int) __popcll(imask));
        if (pairs > 0) {
            const int grank = rank_of(gmask), irank = rank_of(imask);
            wave_order();
            if (gives) mail[grank] = (uint32_t) lane;
            wave_order();
            const bool takes = idle && irank < pairs;
            const int  v     = takes ? (int) mail[irank] : lane;
            const int  l0    = below != 0u ? __ffs((int) below) - 1 : 0; /* the giver's shallowest pending level */
            const int  lv    = __shfl(l0, v, 64);
            const uint32_t pv = __shfl(t.pend, v, 64);
            uint32_t   cut   = (b - a) >> 3; /* the upper end goes with the entries: the giver shares more often */
            cut              = b - (cut ? cut : 1u);
            r.px = __shfl(r.px, v, 64), r.py = __shfl(r.py, v, 64), r.pz = __shfl(r.pz, v, 64);
            r.dx = __shfl(r.dx, v, 64), r.dy = __shfl(r.dy, v, 64), r.dz = __shfl(r.dz, v, 64);
            r.ix = __shfl(r.ix, v, 64), r.iy = __shfl(r.iy, v, 64), r.iz = __shfl(r.iz, v, 64);
            t.level   = __shfl(t.level, v, 64);
            t.ix = __shfl(t.ix, v, 64), t.iy = __shfl(t.iy, v, 64), t.iz = __shfl(t.iz, v, 64);
            t.it                = __shfl(t.it, v, 64);
            own                 = __shfl(own, v, 64);
            const uint32_t cutv = __shfl(cut, v, 64), bv = __shfl(b, v, 64);
            if (takes) {
                a = cutv, b = bv;
                const int off = (v - lane) * W;
#pragma nounroll
                for (int l = 0; l <= lv; l++) { /* the path down to lv, and lv's pending entries */
                    st.pw[l * st.stride] = st.pw[l * st.stride + off];
                    st.ns[l * st.stride] = st.ns[l * st.stride + off];
                    if (DUAL) st.nd[l * st.stride] = st.nd[l * st.stride + off];
                }
                const int sh = t.level - (lv + 1);
                t.ix >>= sh, t.iy >>= sh, t.iz >>= sh;
                t.level = lv + 1;
                t.pend  = (pv & kRayBits) | 1u << lv;
                seg     = trace_pop<CMP, DUAL, SEM, GRID>(s, r, st, t);
            } else if (gives && grank < pairs) {
                b = cut;
                t.pend &= ~(1u << l0);
            }
        }
    }
}

#ifndef QBT_HOST_BUILD
/* ---- work queues of the persistent launches ---------------------------- */

constexpr int kSeg    = 8;  /* work segments per launch (block b starts in segment b % kSeg: one XCD each) */
constexpr int kCtrPad = 64; /* uint32 between refill counters: each on its own 256-byte line */

__device__ __forceinline__ uint32_t seg_bound(uint32_t n, int s) { return (uint32_t) (((uint64_t) n * s) / kSeg); }

/* Blocks of the launched grid that `items` rays are given to (the others
 * end at once; the count of shadow rays is known on the device only): all of
 * them from two rays per lane on, else one lane per ray within [spread,
 * small] blocks, 2 and 4 waves per SIMD. With few rays per lane a wave's
 * steps are latency and a SIMD gains little from more than 4 waves, while
 * each wave then serves more of the rays before the queue runs dry. Measured
 * with 6 against 4 waves per SIMD: 413k camera rays (1.05 per lane) 250
 * against 235 us, 0.55M shadow rays (1.4 per lane) 440 against 418 us; 2.07M
 * camera rays (5.3 per lane) 823 against 858 us. */
struct GridRule {
    uint32_t spread, small;
    __device__ __forceinline__ uint32_t blocks(uint32_t items) const
    {
        const uint32_t full = gridDim.x, bs = blockDim.x;
        if (items >= 2u * full * bs) return full;
        const uint32_t one = (items + bs - 1u) / bs;
        return min(full, min(max(one, spread), small));
    }
};

/* Wave-uniform refill: hands consecutive work items of the wave's current
 * segment to its idle lanes. Returns the item of this lane or UINT32_MAX. */
struct Refill {
    int      seg, left;
    uint32_t n, grid; /* items; blocks that take part */
    __device__ Refill(uint32_t total, uint32_t blocks)
        : seg((int) (blockIdx.x % kSeg)), left(kSeg), n(total), grid(blocks)
    {
    }

    /* A launch with at most 64 items per wave of its grid needs no counters:
     * every wave takes an equal, contiguous share of its segment, fewer than
     * 64 items when the items are few, and the queue is dry at once (drain()
     * then gives the lanes without an item a part of the others' rays). True
     * if that is the case (uniform over the launch), and the lane's item or
     * UINT32_MAX. */
    __device__ __forceinline__ bool share(int lane, uint32_t& item)
    {
        const uint32_t wpb = blockDim.x >> 6, fewest = grid / kSeg * wpb; /* waves of the smallest segment */
        const uint32_t most = n / kSeg + 1u;                                   /* items of the largest segment */
        if (fewest == 0u || (most + fewest - 1u) / fewest > 64u) return false;
        const uint32_t lo = seg_bound(n, seg), hi = seg_bound(n, seg + 1);
        const uint32_t waves = (grid - (uint32_t) seg + kSeg - 1u) / kSeg * wpb;
        const uint32_t per   = (hi - lo + waves - 1u) / waves;
        const uint32_t i     = lo + (blockIdx.x / kSeg * wpb + (threadIdx.x >> 6)) * per + (uint32_t) lane;
        item                 = (uint32_t) lane < per && i < hi ? i : UINT32_MAX;
        left                 = 0;
        return true;
    }

    __device__ __forceinline__ uint32_t fetch(unsigned* ctr, uint64_t idle, int lane)
    {
        const uint32_t nidle  = (uint32_t) __popcll(idle);
        const int      leader = __ffsll((unsigned long long) idle) - 1;
        const uint32_t lo = seg_bound(n, seg), hi = seg_bound(n, seg + 1);
        uint32_t       base = 0;
        if (lane == leader) base = atomicAdd(&ctr[seg * kCtrPad], nidle);
        /* readlane of a uniform lane: a scalar, so seg and left stay in
         * scalar registers */
        base          = __builtin_amdgcn_readlane(base, leader);
        uint32_t item = UINT32_MAX;
        if ((idle >> lane) & 1ull) {
            uint32_t rank = (uint32_t) __popcll(idle & ((1ull << lane) - 1ull));
            uint64_t it   = (uint64_t) lo + base + rank;
            if (it < hi) item = (uint32_t) it;
        }
        if ((uint64_t) lo + base + nidle >= hi) { /* this segment is done: move on */
            seg = (seg + 1) % kSeg;
            left--;
        }
        return item;
    }
};

/* When a wave refills its idle lanes, as one word of a launch: bits 0-7 the
 * number of idle lanes at which it does, bits 8-23 the idle lane-steps since
 * the last refill (0: not looked at; step_run's WASTE). A refill costs a wave about as much as
 * three steps, whatever it fetches, and what it saves grows with the square
 * of the time since the last one: the best number of idle lanes is 12 where
 * camera rays expand 125 nodes on average, 24 at 50 and 32 and more at 17,
 * and all of these are near 180 idle lane-steps. Camera rays at 24 idle
 * lanes against 180 lane-steps or 48 lanes: 5.52 -> 5.27 ms and 3.36 -> 3.23
 * (2160p, long rays), 709 -> 696 us (1080p), 305 -> 280 us (1080p, short
 * rays). Shadow rays and ray batches: 16 lanes, no gain over that. */
__host__ __device__ __forceinline__ constexpr unsigned refill_rule(unsigned lanes, unsigned waste)
{
    return lanes | waste << 8;
}

/* Lanes with a ray step until it ends; the wave leaves the loop together at
 * its refill rule (wave-uniform; at the last ray's end once the queue is
 * dry), so that the refill test, the ballots and the merge of the ray state
 * run once per refill, not once per step. A lane whose ray ends keeps its
 * status in `fin` and its state as it is: the caller writes the results of
 * all such lanes together at the next refill point (a lane that ends would
 * otherwise run the output code with one or two lanes of its wave, in most
 * steps). */
constexpr int kRunSteps = 4096; /* most steps of a run (near_cap) */

template <bool CMP, bool DUAL, int SEM, bool GRID, bool WASTE = false>
__device__ __forceinline__ void step_run(const SceneDev& s, const Ray& r, const Stack& st, TraceState& t, bool& active,
                                         bool dry, unsigned rule, int& fin)
{
    const int keep = dry ? 1 : 65 - (int) (rule & 255u), most = dry || rule < 256u ? INT_MAX : (int) (rule >> 8);
    const int run = __ballot(near_cap<CMP>(s, t, kRunSteps)) != 0ull ? 1 : kRunSteps;
    int       steps = 0, waste = 0; /* of the wave in this call: uniform */
    for (;;) {
        const int stt = trace_step<CMP, DUAL, SEM, GRID>(s, r, st, t);
        steps++;
        if (stt != ST_CONT) {
            fin    = stt;
            active = false;
            break;
        }
        const int on = (int) __popcll(__ballot(1));
        if (WASTE) waste += 64 - on;
        if (on < keep || (WASTE && waste >= most) || steps == run) break;
    }
    if (count_steps<CMP, DUAL>(s, t, steps)) {
        fin    = ST_ABORT;
        active = false;
    }
}

/* Blocks of a persistent traversal launch over at most `items` rays: all
 * that are resident (5 or 6 waves per SIMD for the traversal kernels: VGPRs and
 * LDS stacks), at most one lane per ray, but not fewer than
 * kSpreadWavesPerSimd waves per SIMD: those then take fewer rays each
 * (Refill::share), down to one. A wave alone on its SIMD steps at its own
 * latency, so a second one is nearly free, and the lanes without a ray take
 * parts of the others' rays (drain). Measured, k_primary and k_shadow of a
 * 320x240 frame of the 1M-point scene (77k camera rays, 28k shadow rays):
 * one wave per SIMD 140 + 108 us, two 128 + 95, three 120 + 104, four 129 +
 * 124. GridRule says how many of the blocks take part. */
constexpr int kSpreadWavesPerSimd = 2;
constexpr int kSmallWavesPerSimd  = 4;

template <class K>
inline int persistent_grid(const qbt_ctx* c, K kernel, int bs, size_t lds, size_t items)
{
    int per = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, kernel, bs, lds) != hipSuccess || per <= 0) {
        (void) hipGetLastError();
        per = 1;
    }
    const int wpb  = bs / 64;
    const int one  = (int) ((items + bs - 1) / bs), few = (int) ((items + wpb - 1) / wpb);
    const int fill = std::min(few, 4 * kSpreadWavesPerSimd * c->num_cus / wpb);
    return std::min(per * c->num_cus, std::max(one, fill));
}

inline GridRule grid_rule(const qbt_ctx* c, int bs)
{
    return {(uint32_t) (4 * kSpreadWavesPerSimd * c->num_cus * 64 / bs),
            (uint32_t) (4 * kSmallWavesPerSimd * c->num_cus * 64 / bs)};
}

#endif

} // namespace qbt
