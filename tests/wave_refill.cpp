// A launch of the one-lane walk on the host: its waves take turns, one pass of
// the walk's loop each, over the kernels' own SegFetch and refill rules.  A ray
// is walked for a few passes and then ends or parks (its hit is to be found
// again in the reference's order).  Every launch has to end, with every ray
// traced once.
#include <cstdio>
#include <cstdlib>
#include <vector>

#include "ff_refill.h"

using namespace ffd;

struct HostCounters {
    std::vector<uint32_t>* c;
    uint32_t claim(uint32_t seg, uint32_t want) const {
        uint32_t v = (*c)[seg];
        (*c)[seg] += want;
        return v;
    }
    template <class F>
    uint64_t open(const F& f) const {
        uint64_t m = 0;
        for (uint32_t k = 0; k < FETCH_SEGS; k++)
            if (f.seg_size(k) > 0 && (*c)[k] < f.seg_size(k)) m |= 1ull << k;
        return m;
    }
    uint32_t uniform(uint32_t v) const { return v; }
};

struct Wave {
    SegFetch<HostCounters> F;
    uint32_t ray[64], left[64];
    bool busy[64] = {}, parked[64] = {}, more = true, ended = false;
};

// passes in which a launch must end: a wave takes at most every ray, walks each
// for up to 3 passes, and looks for more up to FETCH_SEGS times
static bool launch(uint32_t n, uint32_t waves, uint32_t park_every) {
    std::vector<uint32_t> ctr(FETCH_SEGS, 0u), traced(n, 0u);
    std::vector<Wave> w(waves);
    for (uint32_t i = 0; i < waves; i++) w[i].F.init(HostCounters{&ctr}, n, i);
    const uint32_t lanes = wide_lanes(n), refill = wide_refill_at(lanes);
    uint32_t running = waves;
    for (uint64_t pass = 0; running; pass++) {
        if (pass > 8ull * n + 4ull * FETCH_SEGS) return false;
        for (Wave& v : w) {
            if (v.ended) continue;
            uint32_t parked = 0, idle = 0, walking = 0;
            for (uint32_t l = 0; l < 64; l++) {
                parked += v.parked[l];
                idle += l < lanes && !v.busy[l];
                walking += v.busy[l] && !v.parked[l];
            }
            if (idle + parked >= refill) {
                const WideRefill take = wide_refill(v.more, parked, idle, lanes);
                if (take.want) {
                    uint32_t got;
                    bool done;
                    const uint32_t first = v.F.take_chunked(take.want, got, done);
                    if (done) v.more = false;
                    for (uint32_t l = 0, k = 0; l < lanes && k < got; l++)
                        if (!v.busy[l]) {
                            v.busy[l] = true;
                            v.ray[l] = first + k++;
                            v.left[l] = 1u + v.ray[l] % 3u;
                            walking++;
                        }
                }
                if (walking == 0) {
                    if (v.more && !take.full) continue;
                    for (uint32_t l = 0; l < 64; l++)
                        if (v.parked[l]) {
                            traced[v.ray[l]]++;
                            v.parked[l] = v.busy[l] = false;
                        }
                    if (!v.more) {
                        v.ended = true;
                        running--;
                    }
                    continue;
                }
            }
            for (uint32_t l = 0; l < 64; l++)
                if (v.busy[l] && !v.parked[l] && --v.left[l] == 0) {
                    v.parked[l] = park_every && v.ray[l] % park_every == 0;
                    if (!v.parked[l]) {
                        traced[v.ray[l]]++;
                        v.busy[l] = false;
                    }
                }
        }
    }
    for (uint32_t t : traced)
        if (t != 1) return false;
    return true;
}

int main() {
    std::vector<uint32_t> sizes;
    for (uint32_t n = 1; n <= 70000; n += n < 300 ? 1 : 1 + n / 12) sizes.push_back(n);
    for (uint32_t k = 1; k <= 64; k++)  // where a wave's number of lanes changes
        for (uint32_t n : {TW_SPREAD * k - 1, TW_SPREAD * k, TW_SPREAD * k + 1})
            if (k < 8 || k % 8 < 2) sizes.push_back(n);
    sizes.push_back(200000);
    for (uint32_t n : sizes)
        for (uint32_t park : {0u, 1u, 2u, 7u}) {
            const uint32_t own = n / wide_lanes(n) + 1;         // a launch for n rays
            for (uint32_t waves : {own < 6144u ? own : 6144u, 6144u})  // a late bounce of a large call
                if (!launch(n, waves, park)) {
                    std::printf("%u rays, every %u parked, %u waves: does not end\n", n, park, waves);
                    return 1;
                }
        }
    std::printf("%zu sizes\n", sizes.size());
    return 0;
}
