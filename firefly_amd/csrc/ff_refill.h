// ff_refill.h -- how the waves of a persistent traversal share a queue of rays:
// the segmented work counters and the rules by which a wave of the one-lane
// walk takes rays.  No HIP headers: the same code runs in the kernels and, over
// counters in host memory, in a host test.
#pragma once

#include <stdint.h>

#if defined(__HIPCC__)
#define FF_HD __host__ __device__ __forceinline__
#else
#define FF_HD inline
#endif

// Work counters of the persistent traversal kernels: the queue is split into
// FETCH_SEGS segments with one counter each, every counter on its own 128-B
// line (device-scope atomics on one address serialise at the memory side).
#define FETCH_SEGS 64
#define FETCH_STRIDE 32
#define F_EXT 0
#define F_SHD 1
#define F_TRACE 2
#define FETCH_WORDS (3 * FETCH_SEGS * FETCH_STRIDE)
#define FETCH_CHUNK 256  // largest claim of one wave from a work counter

namespace ffd {

// Segmented work fetch of the persistent traversal: queue [0, n) is split
// into FETCH_SEGS segments with a counter each; a wave draws from its current
// segment and, once that is exhausted, finds the next segment with work left
// by reading all FETCH_SEGS counters at once.  It reports `done` only when such
// a scan finds every segment exhausted.  Counters only grow, so a segment seen
// exhausted stays exhausted and a wave fails at most FETCH_SEGS times.
// Wave-uniform: every lane calls it with the same arguments.
// Counters: claim(seg, want) adds want to a segment's counter and returns its
// value before, open(fetch) returns the segments with items left (a bit each),
// uniform(v) returns v, known to be the same in every lane.
template <class Counters>
struct SegFetch {
    Counters ctr;
    uint32_t n, seg_len, seg;
    uint32_t res_first, res_left;  // items claimed by this wave and not yet handed out
    uint32_t chunk;                // items claimed per atomic
    FF_HD void init(const Counters& c, uint32_t n_, uint32_t home) {
        ctr = c;
        n = n_;
        seg_len = (n + FETCH_SEGS - 1) / FETCH_SEGS;
        seg = home % FETCH_SEGS;
        res_first = 0;
        res_left = 0;
        // a wave claims up to 1/256 of a segment (at most FETCH_CHUNK) per
        // atomic, so refills of a few lanes rarely wait on the memory-side
        // atomic, and the last claims of a segment stay small
        uint32_t c8 = seg_len >> 8;
        chunk = c8 < FETCH_CHUNK ? c8 : FETCH_CHUNK;
    }
    // Hands out up to `want` items (at least one is asked for) from the wave's
    // reservoir, refilling it from the counters when it is empty.  Same contract
    // as take().
    FF_HD uint32_t take_chunked(uint32_t want, uint32_t& got, bool& done) {
        done = false;
        if (res_left == 0) {
            uint32_t g;
            uint32_t f = take(want > chunk ? want : chunk, g, done);
            res_first = ctr.uniform(f);
            res_left = ctr.uniform(g);
        }
        got = res_left < want ? res_left : want;
        uint32_t first = res_first;
        res_first += got;
        res_left -= got;
        if (res_left > 0) done = false;
        return first;
    }
    FF_HD uint32_t seg_size(uint32_t s) const {
        uint32_t lo = s * seg_len;
        return lo < n ? (n - lo < seg_len ? n - lo : seg_len) : 0u;
    }
    // Grants up to `want` items: returns the first item and the number
    // granted; got == 0 with done == false means "try again later".
    FF_HD uint32_t take(uint32_t want, uint32_t& got, bool& done) {
        got = 0;
        done = false;
        for (int attempt = 0; attempt < 2; attempt++) {
            uint32_t len = seg_size(seg);
            if (len > 0) {
                uint32_t base = ctr.claim(seg, want);
                if (base < len) {
                    got = len - base < want ? len - base : want;
                    return seg * seg_len + base;
                }
            }
            uint64_t m = ctr.open(*this);
            if (m == 0) {
                done = true;
                return 0;
            }
            // next segment with work, searching upwards from the current one
            uint32_t sh = (seg + 1) % 64u;
            uint64_t rot = (m >> sh) | (sh ? (m << (64u - sh)) : 0ull);
            seg = (sh + (uint32_t)__builtin_ctzll(rot)) % 64u;
        }
        return 0;
    }
};

// ------------------------------------------------- refills of the wide walk --
// Lanes of a wave that hold rays, in a launch of n rays: one of fewer rays than
// lanes spreads them over this many waves (one or two to a SIMD), so that a wave
// waits for fewer of its neighbours' visits: 160x120 frame 0.99 ms with full
// waves, 0.87 ms.
constexpr uint32_t TW_SPREAD = 2048;
FF_HD uint32_t wide_lanes(uint32_t n) { return n >= TW_SPREAD * 64u ? 64u : n / TW_SPREAD + 1u; }
// Idle lanes (parked ones among them) at which a wave with `lanes` lanes refills.
constexpr uint32_t TW_REFILL = 16;
FF_HD uint32_t wide_refill_at(uint32_t lanes) { return lanes < TW_REFILL ? lanes : TW_REFILL; }
// A wave takes no more rays once PARK_MOST of its lanes, or all of them, are
// parked: its parked rays are walked as soon as no other lane has work.
constexpr uint32_t PARK_MOST = 32;
struct WideRefill {
    bool full;      // no more rays before the parked ones are walked
    uint32_t want;  // rays to ask for (none: the counters are not touched)
};
// more: the queue may hold more rays; free_lanes: lanes without a ray.
// A wave that has no ray to walk and is not full has a free lane, so it gets a
// ray or learns that there is none: every wave ends.
FF_HD WideRefill wide_refill(bool more, uint32_t parked, uint32_t free_lanes, uint32_t lanes) {
    const bool full = parked >= (lanes < PARK_MOST ? lanes : PARK_MOST);
    return {full, more && !full ? free_lanes : 0u};
}

}  // namespace ffd
