// ff_kernels.hip -- gfx950 kernels of the wavefront path tracer and their
// host launchers.  Stage structure follows the reference's wavefront
// (CRT/kernel.cu:283-676): generate, extend, shadow, logic, material queues,
// plus the FP64 environment CDF build and the film resolve.
//
// Every stage kernel serves a table of render requests: a path slot knows its
// request (scene, environment, camera, depth, film) through P.preq, so one
// wavefront renders a single frame or many uneven requests at once.  The
// batch index lives in device memory (P.bstate) so the per-sample sequence of
// launches is identical from batch to batch and can be replayed as a graph.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <map>
#include <mutex>
#include <utility>

#include "ff_device.h"
#include "ff_internal.h"

using namespace ffd;

namespace {

__device__ __forceinline__ uint32_t gtid() { return blockIdx.x * blockDim.x + threadIdx.x; }
__device__ __forceinline__ uint32_t gstride() { return gridDim.x * blockDim.x; }

__device__ __forceinline__ Bvh bvh_of(const ff_dev_scene& S) {
    Bvh b;
    b.nodes = S.nodes;
    b.nodes4 = S.nodes4;
    b.leaf_count = S.leaf_count;
    b.root = S.root;
    return b;
}

// With UNI every request of the call shades the same scene and environment:
// they are read from request 0, so their pointers stay in scalar registers.
template <bool UNI>
__device__ __forceinline__ const ff_dev_scene& scene_of(const ff_paths& P, const ff_dev_request& R) {
    return UNI ? P.reqs[0].S : R.S;
}
template <bool UNI>
__device__ __forceinline__ const ff_dev_env& env_of(const ff_paths& P, const ff_dev_request& R) {
    return UNI ? P.reqs[0].E : R.E;
}

__device__ __forceinline__ EnvView env_view(const ff_dev_env& e) {
    EnvView v;
    v.rgbp = e.rgbp; v.marg_y = e.marg_y; v.conds = e.conds; v.w = e.w; v.h = e.h;
    v.guide_m = e.guide_m; v.guide_c = e.guide_c;
    return v;
}

// this workgroup's replica of the ray statistics
__device__ __forceinline__ unsigned long long* stats_rep(const ff_paths& P) {
    return P.stats + (size_t)(blockIdx.x % S_REPLICAS) * S_STRIDE;
}

// request of a path: a one-request call does not store it
__device__ __forceinline__ uint32_t req_of(const ff_paths& P, uint32_t id) {
    return P.n_req == 1 ? 0u : P.preq[id];
}

// the queue counters of iteration parity q: entries traced in it
__device__ __forceinline__ int ext_counter(int q) { return q == 0 ? C_EXT0 : C_EXT1; }
__device__ __forceinline__ int shadow_counter(int q) { return q == 0 ? C_SHD0 : C_SHD1; }
__device__ __forceinline__ int mat_counter(int q) { return q == 0 ? C_MAT0 : C_MAT1; }  // the first of four

// request owning a slot: last r with slot_base <= id
__device__ __forceinline__ uint32_t find_req(const ff_dev_request* __restrict__ reqs, uint32_t n, uint32_t id) {
    uint32_t lo = 0, hi = n;
    while (hi - lo > 1) {
        uint32_t mid = (lo + hi) >> 1;
        if (reqs[mid].slot_base <= id) lo = mid;
        else hi = mid;
    }
    return lo;
}

// ============================================================ batch state
// Starts a batch: batch index += 1, queue and work counters
// cleared, and the extension queue laid out for the batch's new samples:
// request r's active slots (its first min(K, spp - b*K) layers, a contiguous
// slot range) occupy queue entries [qbase[r], qbase[r] + count), so
// generate places every path without an atomic.
__global__ void k_batch_begin(ff_paths P) {
    uint32_t i = threadIdx.x;
    if (i < C_COUNT) P.counters[i] = 0;
    for (uint32_t k = i; k < 3 * FETCH_SEGS; k += blockDim.x) P.fetch[(size_t)k * FETCH_STRIDE] = 0;
    __syncthreads();
    if (i == 0) {
        uint32_t b = P.bstate[B_BATCH] + 1u;
        P.bstate[B_BATCH] = b;
        uint32_t q = 0;
        for (uint32_t r = 0; r < P.n_req; r++) {
            const ff_dev_request& R = P.reqs[r];
            int64_t rem = (int64_t)R.spp - (int64_t)b * R.K;
            uint32_t layers = rem <= 0 ? 0u : (rem < (int64_t)R.K ? (uint32_t)rem : R.K);
            P.qbase[r] = q;
            q += layers * R.W * R.H;
        }
        P.qbase[P.n_req] = q;
        P.counters[C_EXT0] = q;
    }
}
// Starts a pass over the batches: the next k_batch_begin makes the batch index
// 0.  A call of one request carries it (and its gradient targets) here, so that
// the host waits for nothing before it launches the call.
__global__ __launch_bounds__(FF_BLOCK) void k_begin(ff_paths P, ff_begin B) {
    if (threadIdx.x == 0) P.bstate[B_BATCH] = 0xffffffffu;
    if (B.clear_stats)
        for (uint32_t i = threadIdx.x; i < S_WORDS; i += FF_BLOCK) P.stats[i] = 0ull;
    if (B.n_req) {
        uint32_t* dst = (uint32_t*)P.reqs;
        for (uint32_t i = threadIdx.x; i < sizeof(ff_dev_request) / 4; i += FF_BLOCK) dst[i] = ((const uint32_t*)&B.req)[i];
        if (threadIdx.x < (uint32_t)B.n_gt) B.gt_dst[threadIdx.x] = B.gt[threadIdx.x];
    }
}

// ================================================================ generate
// wf_generate + dCamera::gen_ray (CRT/kernel.cu:457-485): every active slot
// of the batch starts its next sample; its extension-queue entry is
// qbase[request] + (slot - slot_base), so the queue is in slot order.
__global__ __launch_bounds__(FF_BLOCK) void k_generate(ff_paths P) {
    const uint32_t b = P.bstate[B_BATCH];
    for (uint32_t id = gtid(); id < P.n_slots; id += gstride()) {
        uint32_t r = find_req(P.reqs, P.n_req, id);
        const ff_dev_request& R = P.reqs[r];
        uint32_t WH = R.W * R.H, local = id - R.slot_base;
        uint32_t layer = local / WH, pix = local % WH;
        int64_t rem = (int64_t)R.spp - (int64_t)b * R.K;
        bool act = rem > 0 && (int64_t)layer < rem && layer < R.K;
        if (!act) continue;
        uint32_t sample = R.sample_offset + b * R.K + layer;
        uint32_t base = rng_base(R.seed, pix, sample);
        f3 o, d;
        gen_ray(R.C, (int)R.W, (int)R.H, (int)(pix % R.W), (int)(pix / R.W), base, o, d);
        P.ray[2 * id] = f4(o, __uint_as_float(base));
        P.ray[2 * id + 1] = f4(d, 0.f);  // state word 0: outside every surface
        if (P.n_req > 1) P.preq[id] = r;
        if (R.mode & RQ_ADJOINT) {
            // replay: L_rem starts as the stored radiance of this path
            P.beta[id] = make_float4(1.f, 1.f, 1.f, __uint_as_float(ST_PREV_DELTA));
            uint32_t sl = b * R.K + layer;
            P.Lp[id] = R.path_L[(size_t)sl * WH + pix];
            float4 g = R.d_img[pix];
            P.dlt[id] = make_float4(g.x * R.inv_spp, g.y * R.inv_spp, g.z * R.inv_spp, 0.f);
        }
        // a forward camera path starts at beta = 1, L = 0, state ST_PREV_DELTA:
        // wf_logic's first pass takes those as constants, so they are not stored
        P.q_ext[0][P.qbase[r] + local] = id;
    }
}

// =============================================================== traversal
// Ray sources of the persistent traversal kernels: load_ray() binds queue
// entry k to a path (or ray) and its ray, load_again() reads that ray once
// more, hit() / occluded() write the result.  kUniform: every ray of the launch
// uses one scene (its pointers then stay in scalar registers).
template <bool UNI>
struct ExtSrc {  // wf_extend (CRT/kernel.cu:487-523): closest hit of every queued path
    static constexpr bool kUniform = UNI;
    static constexpr bool kChain = false;
    const ff_paths& P;
    const uint32_t* queue;
    __device__ __forceinline__ const ff_dev_scene& scene(uint32_t id) const {
        return UNI ? P.reqs[0].S : P.reqs[req_of(P, id)].S;
    }
    __device__ __forceinline__ void load_ray(uint32_t k, uint32_t& id, uint32_t& aux, f3& o, f3& d, bool& two) const {
        id = queue[k];
        load_again(id, aux, o, d, two);
    }
    __device__ __forceinline__ void load_again(uint32_t id, uint32_t, f3& o, f3& d, bool& two) const {
        o = xyz(P.ray[2 * id]);
        float4 r1 = P.ray[2 * id + 1];
        d = xyz(r1);
        two = (__float_as_uint(r1.w) & ST_INSIDE) != 0;
    }
    __device__ __forceinline__ void hit(uint32_t id, const Hit& h) const {
        P.hit[id] = make_float4(h.t, h.u, h.v, __int_as_float(h.id));
    }
    __device__ __forceinline__ void occluded(uint32_t, uint32_t, bool) const {}
    __device__ __forceinline__ bool advance(uint32_t&, bool, uint32_t&) const { return false; }
    __device__ __forceinline__ void load_next(uint32_t, uint32_t, f3&, f3&) const {}
    __device__ __forceinline__ void count(uint32_t, uint32_t) const {}
};
// Flag of a vertex's light ray (its .w): the BRDF-sample visibility ray runs
// along the continuation, as a one-lobe material's does, and is read from it
// instead of being stored (32 of the 152 B that shading a diffuse event writes:
// 1080p frame 57.9 -> 56.6 ms).  Were the flag in the continuation's own record,
// its load would come before the ray's (shadow rays 15.2 -> 17.4 ms).
constexpr uint32_t AUX_ALONG = 16u;
// where a BRDF-sample visibility ray starts
__device__ __forceinline__ f3 sample_origin(f3 P, f3 w) { return vadd(P, vscl(w, 0.001f)); }
// A shadow-queue entry is one shading event, path << 2 | needS | needD << 1:
// its light ray first, then -- only when the light ray is unoccluded, since
// its visibility gates the whole NEE sum -- the BRDF-sample visibility rays
// (spec, then diffuse) in the same lane.  aux = ray (0 light, 1 spec,
// 2 diffuse) | rays still to trace << 2.  The reference traces the BRDF-sample
// rays inside BRDF_L either way (CRT/dMaterial.cu:404-448); where the light
// ray is occluded their results are never used, so no pixel changes.
template <bool UNI>
struct ShadowSrc {  // wf_shadow (CRT/kernel.cu:525-543): any hit of every queued shadow ray
    static constexpr bool kUniform = UNI;
    static constexpr bool kChain = true;
    const ff_paths& P;
    __device__ __forceinline__ const ff_dev_scene& scene(uint32_t id) const {
        return UNI ? P.reqs[0].S : P.reqs[req_of(P, id)].S;
    }
    __device__ __forceinline__ void load_ray(uint32_t k, uint32_t& id, uint32_t& aux, f3& o, f3& d, bool& two) const {
        uint32_t e = P.q_shadow[k];
        id = e >> 2;
        const float4 r0 = P.sray[6 * id];
        aux = (e & 3u) << 2 | __float_as_uint(r0.w);
        o = xyz(r0);
        d = xyz(P.sray[6 * id + 1]);
        two = false;
    }
    __device__ __forceinline__ void load_again(uint32_t id, uint32_t aux, f3& o, f3& d, bool&) const {
        load_next(id, aux, o, d);
    }
    __device__ __forceinline__ void hit(uint32_t, const Hit&) const {}
    __device__ __forceinline__ void occluded(uint32_t id, uint32_t aux, bool occ) const {
        P.vis[3 * id + (aux & 3u)] = occ ? 0 : 1;
    }
    // after a ray with result occ: whether the path has another ray (aux then names it)
    __device__ __forceinline__ bool advance(uint32_t& aux, bool occ, uint32_t& gated) const {
        uint32_t cur = aux & 3u, rest = aux >> 2 & 3u;
        if (cur == 0u && occ) gated += (uint32_t)__popc(rest);
        if ((cur == 0u && occ) || rest == 0u) return false;
        uint32_t nxt = (rest & 1u) ? 1u : 2u;
        aux = nxt | ((rest & ~nxt) << 2) | (aux & AUX_ALONG);
        return true;
    }
    __device__ __forceinline__ void load_next(uint32_t id, uint32_t aux, f3& o, f3& d) const {
        const bool along = (aux & AUX_ALONG) != 0u && (aux & 3u) != 0u;
        const float4* r = along ? P.ray + 2 * id : P.sray + 6 * id + 2 * (aux & 3u);
        const f3 p = xyz(ldg4(r));
        d = xyz(ldg4(r + 1));
        const f3 q = sample_origin(p, d);
        o = V3(along ? q.x : p.x, along ? q.y : p.y, along ? q.z : p.z);
    }
    __device__ __forceinline__ void count(uint32_t rays, uint32_t gated) const {
        wave_sum_add(stats_rep(P) + S_SHADOW, rays);
        wave_sum_add(stats_rep(P) + S_SHD_GATED, gated);
    }
};
struct RaySrc {  // a plain ray array (ff_trace_closest / ff_trace_any)
    static constexpr bool kUniform = true;
    static constexpr bool kChain = false;
    ff_dev_scene S;
    const float4* rays;
    float4* hits;
    uint8_t* occ;
    int two_sided;
    __device__ __forceinline__ const ff_dev_scene& scene(uint32_t) const { return S; }
    __device__ __forceinline__ void load_ray(uint32_t k, uint32_t& id, uint32_t& aux, f3& o, f3& d, bool& two) const {
        id = k;
        load_again(id, aux, o, d, two);
    }
    __device__ __forceinline__ void load_again(uint32_t id, uint32_t, f3& o, f3& d, bool& two) const {
        o = xyz(rays[2 * id]);
        d = xyz(rays[2 * id + 1]);
        two = two_sided != 0;
    }
    __device__ __forceinline__ void hit(uint32_t id, const Hit& h) const {
        hits[id] = make_float4(h.t, h.u, h.v, __int_as_float(h.id));
    }
    __device__ __forceinline__ void occluded(uint32_t id, uint32_t, bool o) const { occ[id] = o ? 1 : 0; }
    __device__ __forceinline__ bool advance(uint32_t&, bool, uint32_t&) const { return false; }
    __device__ __forceinline__ void load_next(uint32_t, uint32_t, f3&, f3&) const {}
    __device__ __forceinline__ void count(uint32_t, uint32_t) const {}
};

// Persistent traversal of the reference's tree in the reference's order, for
// traces that count the boxes and triangles it tests (and for the rare scene
// whose wide stacks exceed the fixed trace scratch).  The grid holds only the lanes the chip keeps
// resident; a lane whose ray is finished takes the next queue entry from the
// segmented work counters (per wave: one ballot and one atomic for all idle
// lanes), so a wave no longer lasts as long as its slowest ray and no second
// round of waves is needed.  A wave refills once REFILL of its lanes are idle
// (or all are), trading idle lanes against refill stalls.  Every wave leaves
// the loop once all segments are exhausted and its own rays are finished.
// WW selects the loop shape: 0 = one step (interior record or leaf) per
// lane per iteration; 1 = "while-while": lanes at interior records step
// until every busy lane has reached a leaf, then all leaves are tested
// together (fewer divergent switches between the two code paths);
// 2 = speculative while-while (Aila and Laine, "Understanding the Efficiency
// of Ray Traversal on GPUs", HPG 2009): a lane that reaches a leaf while it
// holds none postpones it and keeps walking interior records until every
// lane holds a leaf or has no interior record left, then the postponed (and
// current) leaves are tested together.  Each lane still tests its leaves in
// its visit order, so hits are those of the other shapes; pruning then sees
// the closest hit of the leaves already tested, so the boxes tested depend
// on the lanes that share the wave.  3 = leaf batching: a lane standing on a
// leaf queues it (two at most) and keeps walking; the queued leaves are
// tested together once 8 lanes hold one, or when no lane can walk on -- the
// leaf code then runs for many lanes at once instead of for the few that
// reach a leaf in any one step.  Leaves are still tested in each lane's visit
// order.  5, 6, 7 = one queued leaf per lane (fewer registers), tested
// together once 8, 4 or 16 lanes hold one.
// WIDE walks the 4-wide records (half the dependent interior steps, same
// leaf order) instead of the two-child records.
template <int BS, int LDS, int REFILL, bool ANY, int WW, bool WIDE>
__device__ __forceinline__ void trav_persistent(const RaySrc& src, uint32_t n, uint32_t* fetch, int32_t* ovf,
                                                unsigned long long* cnt, int* smem) {
    SegFetch<DevCounters> F;
    F.init(DevCounters{fetch}, n, blockIdx.x * (BS / 64) + (threadIdx.x >> 6));
    Stack st;
    st.lds = (lds_int*)&smem[threadIdx.x];
    st.lds_stride = BS;
    st.lds_entries = LDS;
    st.ovf = (glb_int*)(ovf + gtid());
    st.ovf_stride = FF_TRAV_THREADS;
    uint32_t cn = 0, ct = 0, id = 0, aux = 0;
    bool busy = false, more = true, two = false;
    bool walk = false;  // WW >= 2: the lane has records or leaves left to visit
    int pend = 0;       // WW >= 2: postponed leaf (0 = none; leaf refs are negative)
    int pend2 = 0;      // WW >= 3: a second postponed leaf, tested after pend
    const Bvh B = bvh_of(src.S);
    const float* const tris = src.S.tris;
    TravRay R;
    Hit h = no_hit();  // closest hit: h.t here, u, v and slot in the lane's LDS words (hs)
    float lim = prune_lim(h.t);  // pruning limit of the closest hit so far (kept beside it)
    HitSlots hs;  // closest-hit kernels allocate LDS * BS + 3 * BS words of smem
    hs.u = ANY ? nullptr : (lds_float*)&smem[LDS * BS + threadIdx.x];
    hs.v = ANY ? nullptr : (lds_float*)&smem[LDS * BS + BS + threadIdx.x];
    hs.id = ANY ? nullptr : (lds_int*)&smem[LDS * BS + 2 * BS + threadIdx.x];
    // closest-hit sources: the lane's leaf test, the hit reset and the result
    auto leaf_c = [&](const TravRay& L) {
        leaf_closest_slots(B, tris, L, h.t, hs, two, ct);
        lim = prune_lim(h.t);
    };
    auto reset_hit = [&]() {
        h = no_hit();
        lim = prune_lim(h.t);
        if (!ANY) {
            *hs.u = h.u;
            *hs.v = h.v;
            *hs.id = h.id;
        }
    };
    auto hit_out = [&]() {
        Hit r;
        r.t = h.t;
        r.u = *hs.u;
        r.v = *hs.v;
        r.id = *hs.id;
        src.hit(id, r);
    };
    auto end_any = [&](bool occ) { src.occluded(id, aux, occ); };
    for (;;) {
        uint64_t idle = __ballot(!busy);
        uint32_t n_idle = (uint32_t)__popcll(idle);
        if (more && n_idle >= (uint32_t)REFILL) {
            uint32_t rank = __builtin_amdgcn_mbcnt_hi((uint32_t)(idle >> 32),
                                                      __builtin_amdgcn_mbcnt_lo((uint32_t)idle, 0u));
            uint32_t got;
            bool done;
            uint32_t first = F.take_chunked(n_idle, got, done);
            if (done) more = false;
            if (!busy && rank < got) {
                f3 o, d;
                src.load_ray(first + rank, id, aux, o, d, two);
                if (!ANY) reset_hit();
                busy = trav_begin(B, o, d, R, st, cn);
                walk = busy;
                pend = 0;
                pend2 = 0;
                if (!busy) {
                    if (ANY) end_any(false);
                    else hit_out();
                }
            }
        }
        if (__ballot(busy) == 0) {
            if (!more) break;
            continue;
        }
        if (WW == 2) {
            for (;;) {
                if (busy && walk && R.ref < 0 && pend == 0) {  // postpone the first leaf
                    pend = R.ref;
                    if (st.sp == 0) walk = false;
                    else R.ref = st.pop();
                }
                bool at_int = busy && walk && R.ref >= 0;
                bool seeking = busy && walk && pend == 0;
                if (__ballot(at_int) == 0 || __ballot(seeking) == 0) break;
                if (at_int && !visit_node<WIDE, !ANY>(B, R, lim, st, cn)) {
                    if (st.sp == 0) walk = false;
                    else R.ref = st.pop();
                }
            }
            if (busy) {
                bool occ = false;
                if (pend != 0) {  // the postponed leaf, then the current one
                    TravRay L = R;
                    L.ref = pend;
                    if (ANY) occ = leaf_any(B, tris, L, ct);
                    else leaf_c(L);
                    pend = 0;
                }
                if (!occ && walk && R.ref < 0) {
                    if (ANY) occ = leaf_any(B, tris, R, ct);
                    else leaf_c(R);
                    if (st.sp == 0) walk = false;
                    else R.ref = st.pop();
                }
                if (occ || !walk) {
                    if (ANY) end_any(occ);
                    else hit_out();
                    busy = false;
                }
            }
        } else if (WW >= 3) {
            // leaf batching: a lane standing on a leaf queues it (two at most)
            // and walks on; the queued leaves are tested together once
            // LEAF_T lanes hold one, or when no lane can walk on.  Each lane
            // tests its leaves in its visit order.
            constexpr uint32_t LEAF_T = WW == 7 ? 16u : (WW == 6 ? 4u : 8u);
            constexpr bool TWO = WW == 3;  // shapes 5-7 queue one leaf per lane
            if (busy && walk && R.ref < 0 && (TWO ? pend2 == 0 : pend == 0)) {
                if (pend == 0) pend = R.ref;
                else pend2 = R.ref;
                if (st.sp == 0) walk = false;
                else R.ref = st.pop();
            }
            if (busy && walk && R.ref >= 0 && !visit_node<WIDE, !ANY>(B, R, lim, st, cn)) {
                if (st.sp == 0) walk = false;
                else R.ref = st.pop();
            }
            bool has = busy && pend != 0;
            uint32_t n_pend = (uint32_t)__popcll(__ballot(has));
            bool occ = false;
            if (n_pend >= LEAF_T || (n_pend > 0 && __ballot(busy && walk && R.ref >= 0) == 0)) {
                if (has) {
                    TravRay L = R;
                    L.ref = pend;
                    if (ANY) occ = leaf_any(B, tris, L, ct);
                    else leaf_c(L);
                    pend = TWO ? pend2 : 0;
                    pend2 = 0;
                }
            }
            if (busy && (occ || (!walk && pend == 0))) {
                if (ANY) end_any(occ);
                else hit_out();
                busy = false;
            }
        } else if (WW == 1) {
            for (;;) {  // interior records until every busy lane is at a leaf
                bool at_int = busy && R.ref >= 0;
                if (__ballot(at_int) == 0) break;
                if (at_int && !visit_node<WIDE, !ANY>(B, R, lim, st, cn)) {
                    if (st.sp == 0) {
                        if (ANY) end_any(false);
                        else hit_out();
                        busy = false;
                    } else {
                        R.ref = st.pop();
                    }
                }
            }
            if (busy) {  // at a leaf
                if (ANY) {
                    bool occ = leaf_any(B, tris, R, ct);
                    if (occ || st.sp == 0) {
                        end_any(occ);
                        busy = false;
                    } else {
                        R.ref = st.pop();
                    }
                } else {
                    leaf_c(R);
                    if (st.sp == 0) {
                        hit_out();
                        busy = false;
                    } else {
                        R.ref = st.pop();
                    }
                }
            }
        } else if (busy) {
            if (ANY) {
                int r = any_step<WIDE>(B, tris, R, st, cn, ct);
                if (r != 0) {
                    end_any(r == 1);
                    busy = false;
                }
            } else {
                // one step, with the hit's u, v and slot in LDS
                bool cont = true;
                if (R.ref >= 0 && visit_node<WIDE, true>(B, R, lim, st, cn)) {
                } else {
                    if (R.ref < 0) leaf_c(R);
                    if (st.sp == 0) cont = false;
                    else R.ref = st.pop();
                }
                if (!cont) {
                    hit_out();
                    busy = false;
                }
            }
        }
    }
    if (cnt) {
        wave_sum_add(&cnt[0], cn);
        wave_sum_add(&cnt[1], ct);
    }
}

// Launch shape of the wide walk.  Measured on the 1920x1080, 64-sample frame
// (extension / shadow stage): 6 waves per SIMD 24.1 / 15.1 ms, 5 waves 24.3 /
// 15.1, 8 waves (64 VGPRs, spills) 27.6 / 19.1; refilling at 8 idle lanes 26.1,
// at 16 24.2, at 48 29.1; testing held triangles once 2, 4, 8 or 16 lanes hold
// one is alike there (24.1-24.4), and 2 is best where a launch lasts as long as
// its slowest ray (160x120 frame: 0.86 ms, 0.87 at 4, 1.03 at 16).
constexpr int TW_BLOCK = 256, TW_LEAF = 2, TW_OCC = 6;  // (TW_REFILL: ff_refill.h)
// Launches of at most QUAD_MAX rays give every ray four lanes: at 19200 rays a
// launch takes 50 us instead of 70, at 131072 (16 rays on each of 8192 waves)
// the two are even, at 262144 rays four lanes cost 1.2x (8 spheres, 256x256).
constexpr uint32_t QUAD_MAX = 131072;
// Waves that such a launch spreads its rays over (TW_SPREAD, of the one-lane
// walk: ff_refill.h): 160x120 frame over 1024 waves 0.725 ms, over 2048 0.737,
// over 4096 0.78.
constexpr uint32_t QUAD_SPREAD = 1024;

// Persistent traversal of the compressed wide records (see ff_device.h), with
// the same work distribution: a lane owns a ray, a wave refills its idle lanes
// once REFILL of them are idle.  A lane that reaches a triangle holds it and
// walks on; the held triangles are tested together once LEAF lanes hold one,
// or when no lane can walk on.
template <int BS, bool ANY, class Src>
__device__ __forceinline__ void trav_wide(const Src& src, uint32_t n, uint32_t block, uint32_t* fetch,
                                          int32_t* ovf, unsigned long long* cnt, lds_u32* again_lds, int* smem) {
    constexpr uint32_t IDLE = 0xffffffffu;
    constexpr int LDS = FF_LDS_STACK;
    SegFetch<DevCounters> F;
    F.init(DevCounters{fetch}, n, block * (BS / 64) + (threadIdx.x >> 6));
    Stack st;
    st.lds = (lds_int*)&smem[threadIdx.x];
    st.lds_stride = BS;
    st.lds_entries = LDS;
    st.ovf = (glb_int*)(ovf + gtid());
    st.ovf_stride = FF_TRAV_THREADS;
    st.sp = 1;
    st.lds[0] = 0;  // popping the bottom ends the walk
    uint32_t cn = 0, ct = 0, c_rays = 0, c_gated = 0;  // of the wave
    bool more = true, two = false;
    uint32_t id = IDLE, aux = 0;
    bool nxt = false;
    uint32_t cur = 0;   // reference to visit next (0: none left)
    uint32_t pend = 0;  // held triangle (0: none; record 0 is no triangle)
    const float4* rec = nullptr;
    if (Src::kUniform) rec = src.scene(0).wide;
    WideRay R;
    R.fl = 0u;
    float t_hit = K_HUGE;
    HitSlots hs;
    hs.u = ANY ? nullptr : (lds_float*)&smem[LDS * BS + threadIdx.x];
    hs.v = ANY ? nullptr : (lds_float*)&smem[LDS * BS + BS + threadIdx.x];
    hs.id = ANY ? nullptr : (lds_int*)&smem[LDS * BS + 2 * BS + threadIdx.x];
    hs.redo = ANY ? nullptr : (lds_float*)&smem[LDS * BS + 3 * BS + threadIdx.x];
    auto start = [&](f3 o, f3 d) {
        wide_begin(o, d, R);
        if (!ANY) {
            t_hit = K_HUGE;
            *hs.u = 0.f;
            *hs.v = 0.f;
            *hs.id = -1;
            *hs.redo = INFINITY;
        }
        st.sp = 1;
        cur = WREF_ROOT;
        pend = 0;
    };
    // Rays whose outcome the reference's visit order decides (two triangles at
    // one distance, a NaN plane distance, an early hit) park their lane; once many lanes are
    // parked, or no other work is left, those rays walk the binary records with
    // every other lane idle (the walk's registers then add nothing to the loop).
    bool parked = false;
    const uint32_t lanes = wide_lanes(n), refill = wide_refill_at(lanes);
    const bool mine = __lane_id() < lanes;
    for (;;) {
        for (;;) {
            if (Src::kChain) {
                uint64_t chained = __ballot(nxt);
                if (chained != 0) {
                    c_rays += (uint32_t)__popcll(chained);
                    if (nxt) {
                        f3 o, d;
                        src.load_next(id, aux, o, d);
                        start(o, d);
                        nxt = false;
                    }
                }
            }
            uint64_t idle = __ballot(mine && (id == IDLE || parked));
            if ((uint32_t)__popcll(idle) >= refill) {
                idle = __ballot(mine && id == IDLE);
                const WideRefill take =
                    wide_refill(more, (uint32_t)__popcll(__ballot(parked)), (uint32_t)__popcll(idle), lanes);
                if (take.want != 0u) {
                    uint32_t rank = __builtin_amdgcn_mbcnt_hi((uint32_t)(idle >> 32),
                                                              __builtin_amdgcn_mbcnt_lo((uint32_t)idle, 0u));
                    uint32_t got;
                    bool done;
                    uint32_t first = F.take_chunked(take.want, got, done);
                    if (done) more = false;
                    c_rays += got;
                    if (mine && id == IDLE && rank < got) {
                        f3 o, d;
                        src.load_ray(first + rank, id, aux, o, d, two);
                        if (!Src::kUniform) rec = src.scene(id).wide;
                        start(o, d);
                    }
                }
                if (__ballot(id != IDLE && !parked) == 0) {
                    if (!more || take.full) break;
                    continue;
                }
            }
            // a triangle: held, and the walk goes on
            if (cur != 0u && pend == 0u && wide_is_leaf(cur)) {
                pend = cur;
                cur = (uint32_t)st.pop();
            }
            bool inner = (cur & 3u) < (cur >> 29);
            cn += (uint32_t)__popcll(__ballot(inner));
            if (inner) {
                float tn[4], tf[4];
                const uint32_t w = visit_wide<!ANY>(rec, cur, R, t_hit + t_hit * PRUNE_REL + PRUNE_ABS, tn, tf);
                // Entries are stored whether they count or not, and the top is
                // moved on by those that do: the next store overwrites the
                // others.  Near the end of the LDS stack they are pushed singly.
                const bool room = __ballot(st.sp > LDS - 4) == 0;
                lds_int* top = st.lds + st.sp * BS;
                auto put = [&](uint32_t r, bool in) {
                    if (room) {
                        *top = (int)r;
                        top += in ? BS : 0;
                    } else if (in) {
                        st.push((int)r);
                    }
                };
                if (ANY) {  // an occluder anywhere ends the ray: no order, triangles first
#pragma unroll
                    for (int k = 0; k < 4; k++) put(w | (uint32_t)k, !(tn[k] > tf[k]));
                    if (room) st.sp = (int)(top - st.lds) / BS;
                    cur = (uint32_t)st.pop();
                } else {
                    int key[4];
                    wide_order(tn, tf, key);
#pragma unroll
                    for (int k = 3; k > 0; k--) put(w | ((uint32_t)key[k] & 3u), key[k] != WKEY_MISS);
                    if (room) st.sp = (int)(top - st.lds) / BS;
                    cur = w | ((uint32_t)key[0] & 3u);
                    if (key[0] == WKEY_MISS) cur = (uint32_t)st.pop();
                }
                inner = (cur & 3u) < (cur >> 29);
            }
            uint64_t has = __ballot(pend != 0u);
            int occ = 0;
            if (has != 0 && ((uint32_t)__popcll(has) >= (uint32_t)TW_LEAF || __ballot(inner) == 0)) {
                ct += (uint32_t)__popcll(has);
                if (pend != 0u) {
                    if (ANY) occ = wide_leaf_any(rec, pend, R);
                    else wide_leaf_closest(rec, pend, R, t_hit, hs, two);
                    pend = 0;
                }
            }
            const bool fin = occ || (id != IDLE && !parked && (cur | pend) == 0u);
            uint32_t gated = 0;
            if (fin) {
                cur = 0;
                pend = 0;
                if (ANY) {
                    parked = occ == 2;
                    if (!parked) {
                        src.occluded(id, aux, occ != 0);
                        nxt = Src::kChain && src.advance(aux, occ != 0, gated);
                        if (!nxt) id = IDLE;
                    }
                } else {
                    Hit h;
                    h.id = *hs.id;
                    h.t = t_hit;
                    h.u = *hs.u;
                    h.v = *hs.v;
                    parked = *hs.redo <= t_hit;
                    if (!parked) {
                        src.hit(id, h);
                        id = IDLE;
                    }
                }
            }
            if (Src::kChain) c_gated += (uint32_t)(__popcll(__ballot(gated & 1u)) + 2 * __popcll(__ballot(gated & 2u)));
        }
        if (__ballot(parked) == 0) break;
        while (__ballot(parked) != 0) {
            uint32_t gated = 0;
            bool again = false;
            if (parked) {
                const ff_dev_scene& S = src.scene(id);
                f3 o, d;
                src.load_again(id, aux, o, d, two);
                const Hit h = reference_walk<ANY>(bvh_of(S), S.tris, o, d, two, st, again_lds);
                if (ANY) {
                    const bool occ = h.id >= 0;
                    src.occluded(id, aux, occ);
                    again = Src::kChain && src.advance(aux, occ, gated);
                } else {
                    src.hit(id, h);
                }
                st.lds[0] = 0;
                if (!again) id = IDLE;
                parked = again;
            }
            c_rays += (uint32_t)__popcll(__ballot(again));
            c_gated += (uint32_t)(__popcll(__ballot(gated & 1u)) + 2 * __popcll(__ballot(gated & 2u)));
        }
        if (!more) break;
        // nothing of an idle lane's walk lives across this
        R = WideRay{};
        t_hit = K_HUGE;
        cur = 0;
        pend = 0;
        aux = 0;
        two = false;
        nxt = false;
        st.sp = 1;
    }
    if (cnt && __lane_id() == 0) add_tested(cnt, cn, ct, again_lds);
    src.count(__lane_id() == 0 ? c_rays : 0u, __lane_id() == 0 ? c_gated : 0u);
}

// Rays that a wave of the four-lane walk holds at once: where rays are few,
// fewer to a wave, so that a wave waits for fewer others.
__host__ __device__ __forceinline__ uint32_t quad_rays(uint32_t n) {
    return n >= QUAD_SPREAD * 16u ? 16u : n / QUAD_SPREAD + 1u;
}
// Waves that hold all n rays at once take theirs by their own number: the work
// counters are not touched, so a query needs no launch that clears them first
// (two queries of 77 rays: 51 -> 38 us; a 160x120 4-bounce
// render 0.384 -> 0.342 ms, a 320x180 one 0.451 -> 0.385 ms, where every one of
// up to 6144 waves asked a counter first and then looked for more).
__host__ __device__ __forceinline__ bool quad_fixed(uint32_t n, uint32_t waves) {
    return (uint64_t)waves * quad_rays(n) >= n;
}
// The same walk with four lanes to a ray, for launches of few rays: there a
// launch lasts as long as its slowest ray's chain of dependent visits, and a
// visit is a third of the instructions when every lane tests one child.
// Triangles that a visit reaches are tested at once, a lane each, before the
// walk goes on.  A ray's stack lies in the LDS columns of its wave (no
// overflow area: the launcher takes this walk only where LDS * 4 entries hold
// the deepest stack).
template <int BS, bool ANY, class Src>
__device__ __forceinline__ void trav_quad(const Src& src, uint32_t n, uint32_t block, uint32_t blocks, uint32_t* fetch,
                                          unsigned long long* cnt, lds_u32* again_lds, int* smem) {
    constexpr uint32_t IDLE = 0xffffffffu;
    const uint32_t wave = block * (BS / 64) + (threadIdx.x >> 6);
    SegFetch<DevCounters> F;
    F.init(DevCounters{fetch}, n, wave);
    const uint32_t lane = __lane_id(), k = lane & 3u, lead = lane & ~3u;
    const uint64_t below = ((1ull << lead) - 1ull) & 0x1111111111111111ull;
    QuadStack<BS> st;
    st.col = (lds_int*)&smem[(threadIdx.x & ~63u) + (lane >> 2)];
    st.sp = 0;
    auto quad_mask = [&](bool b) { return (uint32_t)(__ballot(b) >> lead) & 15u; };
    uint32_t cn = 0, ct = 0, c_rays = 0, c_gated = 0;  // of the wave
    bool more = true, two = false, nxt = false;
    uint32_t id = IDLE, aux = 0;
    uint32_t cur = 0;
    const float4* rec = nullptr;
    if (Src::kUniform) rec = src.scene(0).wide;
    WideRay R;
    R.fl = 0u;
    float t_hit = K_HUGE;           // of the quad
    Hit best = no_hit();            // of the lane
    float redo_t = INFINITY;        // smallest t whose outcome the reference's order decides (ANY: 0, if it does)
    const uint32_t cap = quad_rays(n);
    const bool fixed = quad_fixed(n, blocks * (BS / 64));
    const bool mine = (lane >> 2) < cap;
    auto start = [&](f3 o, f3 d) {
        wide_begin(o, d, R);
        t_hit = K_HUGE;
        best = no_hit();
        redo_t = INFINITY;
        *st.at(0) = 0;  // popping the bottom ends the walk
        st.sp = 1;
        cur = WREF_ROOT;
    };
    for (;;) {
        if (Src::kChain) {
            uint64_t chained = __ballot(nxt);
            if (chained != 0) {
                c_rays += (uint32_t)__popcll(chained) / 4u;
                if (nxt) {
                    f3 o, d;
                    src.load_next(id, aux, o, d);
                    start(o, d);
                    nxt = false;
                }
            }
        }
        const uint64_t idle = __ballot(mine && id == IDLE && k == 0u);
        if (idle != 0) {
            if (more) {
                uint32_t got, first;
                bool done = true;
                if (fixed) {
                    first = wave * cap;
                    got = first < n ? (n - first < cap ? n - first : cap) : 0u;
                } else {
                    first = F.take_chunked((uint32_t)__popcll(idle), got, done);
                }
                if (done) more = false;
                c_rays += got;
                const uint32_t rank = (uint32_t)__popcll(idle & below);
                if (mine && id == IDLE && rank < got) {
                    f3 o, d;
                    src.load_ray(first + rank, id, aux, o, d, two);
                    if (!Src::kUniform) rec = src.scene(id).wide;
                    start(o, d);
                }
            }
            if (__ballot(id != IDLE) == 0) {
                if (!more) break;
                continue;
            }
        }
        cn += (uint32_t)__popcll(__ballot(cur != 0u)) / 4u;
        bool occ = false, tri = false;
        if (cur != 0u) {
            float tn, tf;
            const uint32_t w = visit_quad<!ANY>(rec, cur, R, t_hit + t_hit * PRUNE_REL + PRUNE_ABS, k, tn, tf);
            bool in = !(tn > tf);
            tri = in && k >= (w >> 29);
            if (__ballot(tri) != 0) {
                int r = 0;
                float t = K_HUGE;
                if (tri) {
                    if (ANY) {
                        r = wide_leaf_any(rec, w | k, R);
                    } else {
                        WideTri T = load_wide_tri(rec, w | k);
                        float u = 0.f, v = 0.f;
                        bool ok = two ? mt_two(T.T, R.o, R.d, t, u, v) : mt_cull(T.T, R.o, R.d, t, u, v), nanx;
                        float entry;
                        if (ok && !(t < 0.f) && t <= t_hit && wide_leaf_box(T, R, nanx, entry)) {
                            const bool early = early_hit(t, entry);
                            if (early || nanx || t == t_hit) redo_t = fminf(redo_t, t);
                            if (!early && t < t_hit) {
                                best.t = t;
                                best.u = u;
                                best.v = v;
                                best.id = T.slot;
                            }
                        }
                    }
                }
                if (ANY) {
                    occ = quad_mask(r == 1) != 0u;
                    if (!occ && quad_mask(r == 2) != 0u) redo_t = 0.f;
                } else {
                    t_hit = fminf(best.t, quad_xor<1>(best.t));
                    t_hit = fminf(t_hit, quad_xor<2>(t_hit));
                    in = in && !(tn > t_hit + t_hit * PRUNE_REL + PRUNE_ABS);
                }
                in = in && !tri;
            }
            const uint32_t m = quad_mask(in);
            if (m != 0u) {
                if (ANY) {
                    const uint32_t f = (uint32_t)__ffs((int)m) - 1u;
                    cur = w | f;
                    if (in && k != f) *st.at(st.sp + __popc(m & ((1u << k) - 1u)) - 1) = (int)(w | k);
                } else {
                    const int key = in ? ((__float_as_int(tn) & ~3) | (int)k) : WKEY_MISS;
                    const int k1 = quad_xor<1>(key), k2 = quad_xor<2>(key), k3 = quad_xor<3>(key);
                    const int rank = (k1 < key ? 1 : 0) + (k2 < key ? 1 : 0) + (k3 < key ? 1 : 0);
                    cur = w | ((uint32_t)imin(imin(key, k1), imin(k2, k3)) & 3u);
                    if (in && rank > 0) *st.at(st.sp + __popc(m) - 1 - rank) = (int)(w | k);
                }
                st.sp += __popc(m) - 1;
                // The quad's lanes pop what any of them pushed.  A wave's LDS
                // operations are carried out in order; the fence (no instruction)
                // keeps the compiler from moving a pop above the pushes.
                __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront", "local");
                __builtin_amdgcn_wave_barrier();
            } else {
                cur = (uint32_t)st.pop();
            }
        }
        ct += (uint32_t)__popcll(__ballot(tri));
        const bool fin = id != IDLE && (occ || cur == 0u);
        if (__ballot(fin) == 0) continue;
        const bool redo = quad_mask(ANY ? redo_t == 0.f && !occ : redo_t <= t_hit) != 0u ||
                          (!ANY && __popc(quad_mask(best.id >= 0 && best.t == t_hit)) > 1);
        uint32_t gated = 0;
        if (fin) {
            cur = 0;
            bool win = ANY ? k == 0u : (best.id >= 0 ? best.t == t_hit : (k == 0u && !(t_hit < K_HUGE)));
            if (redo) {  // in the reference's order, by the quad's first lane
                win = k == 0u;
                if (win) {
                    const ff_dev_scene& S = src.scene(id);
                    best = reference_walk<ANY>(bvh_of(S), S.tris, R.o, R.d, two, st, again_lds);
                    if (ANY) occ = best.id >= 0;
                }
            }
            if (ANY) {
                occ = quad_mask(occ) != 0u;
                if (win) src.occluded(id, aux, occ);
                nxt = Src::kChain && src.advance(aux, occ, gated);
                if (!nxt) id = IDLE;
            } else {
                if (win) src.hit(id, best);
                id = IDLE;
            }
        }
        if (Src::kChain)
            c_gated += (uint32_t)(__popcll(__ballot(gated & 1u)) + 2 * __popcll(__ballot(gated & 2u))) / 4u;
    }
    if (cnt && lane == 0) add_tested(cnt, cn, ct, again_lds);
    src.count(lane == 0 ? c_rays : 0u, lane == 0 ? c_gated : 0u);
}

// block: the workgroup's number among the `blocks` that draw from the same queue
// (its waves start on the queue's segments in turn)
template <bool ANY, class Src>
__device__ __forceinline__ void traverse(const Src& src, uint32_t n, uint32_t block, uint32_t blocks, bool quad,
                                         uint32_t* fetch, int32_t* ovf, unsigned long long* cnt, lds_u32* again_lds,
                                         int* smem) {
    if (quad && n <= QUAD_MAX) trav_quad<TW_BLOCK, ANY>(src, n, block, blocks, fetch, cnt, again_lds, smem);
    else trav_wide<TW_BLOCK, ANY>(src, n, block, fetch, ovf, cnt, again_lds, smem);
}
// LDS words of a traversal workgroup: the stacks, for closest hits the hit words too
constexpr int TW_LDS_ANY = FF_LDS_STACK * TW_BLOCK, TW_LDS_CLOSEST = (FF_LDS_STACK + 4) * TW_BLOCK;

// the words in which a workgroup counts what rays traced again test
__device__ __forceinline__ void clear_again(uint32_t* again, uint32_t n) {
    if (threadIdx.x < n) again[threadIdx.x] = 0u;
    __syncthreads();
}
// SMALL: a call with at most QUAD_MAX paths in flight
template <bool UNI, bool SMALL>
__device__ __forceinline__ void extend_rays(const ff_paths& P, int q, uint32_t block, uint32_t blocks, int* smem,
                                            lds_u32* again) {
    // the counters that the coming stages of the iteration add to (nothing
    // reads them during the traversal; those it reads are cleared by the logic)
    if (block == 0 && threadIdx.x < 6)
        P.counters[threadIdx.x < 4 ? mat_counter(q) + threadIdx.x
                                   : (threadIdx.x == 4 ? ext_counter(1 - q) : shadow_counter(1 - q))] = 0u;
    const ExtSrc<UNI> src{P, P.q_ext[q]};
    const uint32_t n = P.counters[ext_counter(q)];
    uint32_t* const fetch = P.fetch + F_EXT * FETCH_SEGS * FETCH_STRIDE;
    unsigned long long* const cnt = stats_rep(P) + S_EXT_NODES;
    if (SMALL) trav_quad<TW_BLOCK, false>(src, n, block, blocks, fetch, cnt, again, smem);
    else traverse<false>(src, n, block, blocks, P.quad != 0, fetch, P.ovf, cnt, again, smem);
}
template <bool UNI, bool SMALL>
__device__ __forceinline__ void shadow_rays(const ff_paths& P, int q, uint32_t block, uint32_t blocks, int* smem,
                                            lds_u32* again) {
    const ShadowSrc<UNI> src{P};
    const uint32_t n = P.counters[shadow_counter(q)];
    uint32_t* const fetch = P.fetch + F_SHD * FETCH_SEGS * FETCH_STRIDE;
    unsigned long long* const cnt = stats_rep(P) + S_SHD_NODES;
    if (SMALL) trav_quad<TW_BLOCK, true>(src, n, block, blocks, fetch, cnt, again, smem);
    else traverse<true>(src, n, block, blocks, P.quad != 0, fetch, P.ovf_shd, cnt, again, smem);
}
template <bool UNI>
__global__ __launch_bounds__(TW_BLOCK, TW_OCC) void k_extend(ff_paths P, int q) {
    __shared__ int smem[TW_LDS_CLOSEST];
    __shared__ uint32_t again[2];
    clear_again(again, 2);
    extend_rays<UNI, false>(P, q, blockIdx.x, gridDim.x, smem, (lds_u32*)again);
}
template <bool UNI>
__global__ __launch_bounds__(TW_BLOCK, TW_OCC) void k_shadow(ff_paths P, int q) {
    __shared__ int smem[TW_LDS_ANY];
    __shared__ uint32_t again[2];
    clear_again(again, 2);
    shadow_rays<UNI, false>(P, q, blockIdx.x, gridDim.x, smem, (lds_u32*)again);
}
// An iteration's extension rays and its vertices' shadow rays (both come from
// the previous shading pass) in one launch: workgroups alternate between the
// two queues by eights (one to each XCD), and each goes on to the other queue,
// so that either queue's waves fill the other's tail.
//
// OCC, waves a SIMD: a call of few paths lasts as long as its slowest rays, and
// 5 waves (96 VGPRs) spill nothing; a call of many is bound by the latency of
// its visits, and 7 waves (72 VGPRs) hide more of it, spills and all.  5, 6 and
// 7 waves at 256 k paths (spheres, 16 samples): 3.10, 3.25, 3.45 ms; at 33 M
// (327 k triangles): 16.0, 15.4, 15.0; at 133 M: 62.3, 59.2, 58.0.  Between
// these sizes the three are within 3 % of one another, and not always in that
// order (460 k, 327 k triangles: 1.57, 1.61, 1.56; 4.7 M: 4.02, 3.99, 4.06): the
// limits lie there.
constexpr uint32_t EXTEND_FEW = 2u << 20, EXTEND_MANY = 16u << 20;
template <bool UNI, int OCC>
__global__ __launch_bounds__(TW_BLOCK, OCC) void k_extend_shadow(ff_paths P, int q) {
    __shared__ int smem[TW_LDS_CLOSEST];
    __shared__ uint32_t again[4];
    clear_again(again, 4);
    const uint32_t blocks = gridDim.x / 2u;
    for (uint32_t ph = 0; ph < 2; ph++) {
        // (a queue's guests are numbered after its own workgroups, whose waves
        // may hold all its rays by their number)
        const uint32_t block = (blockIdx.x >> 4) * 8u + (blockIdx.x & 7u) + ph * blocks;
        if ((((blockIdx.x >> 3) + ph) & 1u) == 0u) extend_rays<UNI, false>(P, q, block, blocks, smem, (lds_u32*)again);
        else shadow_rays<UNI, false>(P, q, block, blocks, smem, (lds_u32*)again + 2);
    }
}
// The same for a call with at most QUAD_MAX paths in flight: each queue has
// workgroups enough, so they keep to one, and hold the four-lane walk only.
template <bool UNI>
__global__ __launch_bounds__(TW_BLOCK, TW_OCC) void k_extend_shadow_small(ff_paths P, int q) {
    __shared__ int smem[TW_LDS_ANY];
    __shared__ uint32_t again[2];
    clear_again(again, 2);
    const uint32_t block = (blockIdx.x >> 4) * 8u + (blockIdx.x & 7u);
    if (blockIdx.x & 8u) shadow_rays<UNI, true>(P, q, block, gridDim.x / 2u, smem, (lds_u32*)again);
    else extend_rays<UNI, true>(P, q, block, gridDim.x / 2u, smem, (lds_u32*)again);
}

// clears the work counters of the standalone traces (a kernel: graph-safe)
__global__ void k_reset_fetch(uint32_t* fetch) {
    if (threadIdx.x < FETCH_SEGS) fetch[(size_t)(F_TRACE * FETCH_SEGS + threadIdx.x) * FETCH_STRIDE] = 0;
}
// the counters that the iteration's traversals have consumed, cleared by the
// first workgroup of the logic that follows them
__device__ __forceinline__ void clear_traversed(const ff_paths& P) {
    if (blockIdx.x != 0) return;
    static_assert(F_EXT == 0 && F_SHD == 1 && 2 * FETCH_SEGS <= FF_BLOCK, "one thread per work counter");
    if (threadIdx.x < 2 * FETCH_SEGS) P.fetch[(size_t)threadIdx.x * FETCH_STRIDE] = 0;
}

// =================================================================== logic
// wf_logic (CRT/kernel.cu:297-455): NEE accumulation gated by the light
// ray's visibility, throughput update, Russian roulette for len > 3,
// environment radiance for escaped rays after the camera (or a delta event),
// termination into the film, routing of live paths to material queues.
// Each thread takes two paths of a 512-entry tile (entries t and t + 256, so
// every load of a wave stays coalesced), and the loads are issued level by
// level for both before any result is used: queue -> path record -> what the
// record asks for (material word, direction, visibilities with the NEE terms
// they gate, throughput factor, RNG base) -> the rare third level (escaped
// delta rays' environment lookup, inside-absorption triangle).  The NEE terms
// are read with their visibility bytes rather than after them.  The
// arithmetic of every path is the one-path wf_logic's, operation for
// operation.  In the first batch of a samples-in-flight request every slot is
// written exactly once (each slot holds one path per batch and every path
// terminates within its batch), so the layer is stored without being read.
// A path that survives its first vertex still holds the start record
// (beta = 1, L = 0): iteration 1 does not store it, and iteration 2 (and the
// first shading pass) use the constants instead of reading it.
struct LogicCounts {  // of a thread
    uint32_t prim = 0, ext = 0, paths = 0;
};
template <bool UNI, int NP>
__device__ __forceinline__ void logic_paths(const ff_paths& P, int iter, bool first_batch, const bool* live,
                                            const uint32_t* id, int* route, LogicCounts& c) {
    const bool primary = iter == 1;
    // level 1: the path record
    float4 bw[NP], lp4[NP], hh[NP], fe[NP];
    uint32_t rq[NP];
#pragma unroll
    for (int j = 0; j < NP; j++) {
        // a camera path's record is the constant start state (not stored)
        bw[j] = make_float4(1.f, 1.f, 1.f, __uint_as_float(ST_PREV_DELTA));
        lp4[j] = make_float4(0.f, 0.f, 0.f, 0.f);
        if (iter > 2) {
            bw[j] = P.beta[id[j]];
            lp4[j] = P.Lp[id[j]];
        }
        hh[j] = P.hit[id[j]];
        rq[j] = req_of(P, id[j]);
        // after a shading pass the state word travels in fext.w:
        // (f * cos / pdf of the continuation, state | ST_DEAD where f or pdf is zero)
        fe[j] = make_float4(0.f, 0.f, 0.f, 0.f);
        if (!primary) fe[j] = P.fext[id[j]];
    }
    // level 2: what the record asks for
    uint32_t stw[NP], len[NP], mw[NP], rb[NP];
    int slot[NP];
    bool found[NP], need_d[NP];
    f3 d[NP], nL[NP], nS[NP], nD[NP];
    uint8_t v0[NP], v1[NP], v2[NP];
#pragma unroll
    for (int j = 0; j < NP; j++) {
        const ff_dev_request& R = P.reqs[rq[j]];
        const ff_dev_scene& S = scene_of<UNI>(P, R);
        stw[j] = __float_as_uint(primary ? bw[j].w : fe[j].w);
        len[j] = (stw[j] & ST_LEN_MASK) + 1;
        slot[j] = __float_as_int(hh[j].w);
        found[j] = live[j] && slot[j] >= 0;
        need_d[j] = live[j] && ((found[j] && (stw[j] & ST_INSIDE)) || (!found[j] && (stw[j] & ST_PREV_DELTA)));
        mw[j] = 0u;
        if (found[j]) mw[j] = ldg(S.mat + slot[j]);
        d[j] = V3(0.f, 0.f, 0.f);
        if (need_d[j]) d[j] = xyz(P.ray[2 * id[j] + 1]);
        bool ext = live[j] && len[j] > 1;
        v0[j] = v1[j] = v2[j] = 0;
        nL[j] = nS[j] = nD[j] = V3(0.f, 0.f, 0.f);
        if (ext && (stw[j] & ST_NEED_L)) {
            v0[j] = P.vis[3 * id[j] + 0];
            nL[j] = xyz(P.nee[3 * id[j]]);
        }
        if (ext && (stw[j] & ST_NEED_S)) {
            v1[j] = P.vis[3 * id[j] + 1];
            nS[j] = xyz(P.nee[3 * id[j] + 1]);
        }
        if (ext && (stw[j] & ST_NEED_D)) {
            v2[j] = P.vis[3 * id[j] + 2];
            nD[j] = xyz(P.nee[3 * id[j] + 2]);
        }
        rb[j] = 0u;
        if (ext && found[j] && len[j] > 3) rb[j] = __float_as_uint(ldg(&P.ray[2 * id[j]].w));
    }
    // the NEE sum of the previous vertex, gated by its visibilities
    f3 lb[NP];
    bool visL[NP];
#pragma unroll
    for (int j = 0; j < NP; j++) {
        uint32_t sw = stw[j];
        visL[j] = live[j] && len[j] > 1 && (sw & ST_NEED_L) && v0[j];
        lb[j] = nL[j];
        if ((sw & ST_NEED_S) && v1[j]) lb[j] = vadd(lb[j], nS[j]);
        if ((sw & ST_NEED_D) && v2[j]) lb[j] = vadd(lb[j], nD[j]);
    }
    // level 3 and the per-path arithmetic, in wf_logic's order: an escaped
    // ray's environment term, then the NEE sum, then (a hit) throughput
    // and roulette
#pragma unroll
    for (int j = 0; j < NP; j++) {
        route[j] = -1;
        if (!live[j]) continue;
        const ff_dev_request& R = P.reqs[rq[j]];
        const ff_dev_scene& S = scene_of<UNI>(P, R);
        uint32_t sw = stw[j], ln = len[j];
        f3 beta = xyz(bw[j]);
        f3 Lp = xyz(lp4[j]);
        bool tm = (ln > R.depth) || !found[j];
        int mtype = -1;
        if (found[j]) {
            mtype = (int)(mw[j] >> MAT_TYPE_SHIFT);
            if ((sw & ST_INSIDE) && mtype != MAT_DIELECTRIC) {
                Tri T = load_tri(S.tris, slot[j]);
                if (!(vdot(d[j], vcross(T.e1, T.e2)) < 0.f)) tm = true;  // absorbed
            }
            if (visL[j]) Lp = vadd(Lp, vmul(lb[j], beta));
            if (ln > 1) {
                if (sw & ST_DEAD) {
                    tm = true;
                } else {
                    beta = vmul(beta, xyz(fe[j]));
                    if (ln > 3) {
                        float qrr = fmaxf(0.05f, 1.f - beta.y);
                        if (rng(rb[j], ln, DIM_RR) < qrr) tm = true;
                    }
                }
            }
        } else {
            if (sw & ST_PREV_DELTA) Lp = vadd(Lp, vmul(beta, env_L(env_view(env_of<UNI>(P, R)), d[j])));
            if (visL[j]) Lp = vadd(Lp, vmul(lb[j], beta));
        }
        if (tm) {
            uint32_t local = id[j] - R.slot_base, WH = R.W * R.H;
            if (R.K > 1 && first_batch) {
                stg4(R.layers + local, make_float4(0.f + Lp.x, 0.f + Lp.y, 0.f + Lp.z, 0.f + 1.f));
            } else {
                float4* acc = R.K > 1 ? &R.layers[local] : &R.film[local % WH];
                float4 L = ldg4(acc);
                stg4(acc, make_float4(L.x + Lp.x, L.y + Lp.y, L.z + Lp.z, L.w + 1.f));
            }
            if (R.mode & RQ_STORE_PATHS) {
                uint32_t sl = P.bstate[B_BATCH] * R.K + local / WH;
                stg4(R.path_L + (size_t)sl * WH + local % WH, f4(Lp, 0.f));
            }
        } else {
            uint32_t nst = (sw & (ST_INSIDE | ST_PREV_DELTA)) | ln;
            if (!primary) {
                P.beta[id[j]] = f4(beta, __uint_as_float(nst));
                P.Lp[id[j]] = f4(Lp, 0.f);
            }
            route[j] = mtype;
        }
        c.prim += ln == 1 ? 1u : 0u;
        c.ext += ln == 1 ? 0u : 1u;
        c.paths += tm ? 1u : 0u;
    }
}
__device__ __forceinline__ void add_counts(const ff_paths& P, const LogicCounts& c) {
    unsigned long long* sr = stats_rep(P);
    wave_sum_add(sr + S_PRIMARY, c.prim);
    wave_sum_add(sr + S_EXTENSION, c.ext);
    wave_sum_add(sr + S_PATHS, c.paths);
}
template <bool UNI>
__global__ __launch_bounds__(FF_BLOCK, 5) void k_logic(ff_paths P, int q, int iter) {
    constexpr int NP = 2;
    __shared__ QStage<FF_BLOCK, 4, QSTAGE_CAP> st;
    const int qidx[4] = {mat_counter(q), mat_counter(q) + 1, mat_counter(q) + 2, mat_counter(q) + 3};
    uint32_t* const qs[4] = {P.q_mat[0], P.q_mat[1], P.q_mat[2], P.q_mat[3]};
    st.init();
    clear_traversed(P);
    const uint32_t n = P.counters[ext_counter(q)];
    const uint32_t* queue = P.q_ext[q];
    const bool first_batch = P.bstate[B_BATCH] == 0;
    constexpr uint32_t TILE = NP * FF_BLOCK;
    const uint32_t n_round = (n + TILE - 1) / TILE * TILE;  // uniform trip count per workgroup
    LogicCounts c;
    for (uint32_t t0 = blockIdx.x * TILE; t0 < n_round; t0 += gridDim.x * TILE) {
        bool live[NP];
        uint32_t id[NP];
        int route[NP];
#pragma unroll
        for (int j = 0; j < NP; j++) {
            uint32_t i = t0 + (uint32_t)j * FF_BLOCK + threadIdx.x;
            live[j] = i < n;
            id[j] = live[j] ? queue[i] : 0u;
        }
        logic_paths<UNI, NP>(P, iter, first_batch, live, id, route, c);
#pragma unroll
        for (int j = 0; j < NP; j++) st.add(route[j], id[j]);
        st.flush_if_full(P.counters, qidx, qs, NP);  // room for the next tile's NP adds
    }
    st.flush(P.counters, qidx, qs);
    add_counts(P, c);
}

// ======================================================= material queues
// Every shaded event continues to the next extension stage, so the extension
// queue of parity 1 - q is the material queues of q one after another: material
// queue TYPE starts after the entries of the types below it.
template <int TYPE>
__device__ __forceinline__ uint32_t ext_base(const ff_paths& P, int q) {
    uint32_t b = 0u;
#pragma unroll
    for (int t = 0; t < TYPE; t++) b += P.counters[mat_counter(q) + t];
    return b;
}
// The first workgroup adds a material queue's n entries to the extension
// counter (one atomic per launch).
__device__ __forceinline__ void add_extensions(const ff_paths& P, int next_q, uint32_t n) {
    if (blockIdx.x == 0 && threadIdx.x == 0 && n) atomicAdd(&P.counters[ext_counter(next_q)], n);
}

// Everything the shading of one vertex produces.  With GRAD the partial
// derivatives of its terms are produced too (path-replay adjoint).
struct ShadeOut {
    f3 A, Bs, Cd;       // light-sample term and BRDF-sampled spec / diffuse terms (before visibility)
    f3 wi, wi_s, wi_d;  // their directions
    f3 lo, so, dd_o;    // shadow ray origins
    bool needL, needS, needD;
    f3 fext;
    float pdf_ext, cos_ext;
    f3 next_o, next_d;
    uint32_t nst;       // state of the continuation
    uint32_t base;      // the path's rng base (rides with the continuation ray)
    // GRAD only
    bool a_on, rough_live;
    int at, rt;
    float tu, tv;
    f3 dA_alb, dB_alb, dC_alb, dA_r, dB_r;  // d term_c / d albedo_c, d term_c / d roughness
    f3 kA, kB, kC;                         // d term_c / d Le_c
    f3 dext_alb, dext_r;
};

// Shading of one material class (wf_mat_mix / wf_mat_diffuse / wf_mat_cook,
// CRT/kernel.cu:545-651, lobes of CRT/dMaterial.cu).  The environment light
// sample of wf_logic (CRT/kernel.cu:435-439) is drawn here; the visibility
// rays of BRDF_L's BRDF-sampled MIS terms (CRT/dMaterial.cu:404-448) are
// deferred to the shadow stage with their contributions kept per path.
// Where a vertex's state word comes from (length, inside, previous delta):
#define SW_RECORD 0   // the path record's beta.w (adjoint replay)
#define SW_START 1    // the first vertex of a forward path: the start record's
#define SW_RAY 2      // a later forward vertex: the ray's .w holds the previous
                      // shading word, which wf_logic turns into this vertex's
                      // word by adding one to the length and keeping the flags
struct Vertex {
    float4 hit, r0, r1;  // hit record; ray that found it
};
__device__ __forceinline__ Vertex load_vertex(const ff_paths& P, uint32_t id) {
    return {P.hit[id], P.ray[2 * id], P.ray[2 * id + 1]};
}
template <int TYPE, bool GRAD, bool UNI>
__device__ __forceinline__ void shade_core(const ff_paths& P, uint32_t id, const Vertex& vx, ShadeOut& so,
                                           int sw_src = SW_RECORD) {
    const ff_dev_request& R = P.reqs[req_of(P, id)];
    const ff_dev_scene& S = scene_of<UNI>(P, R);
    EnvView E = env_view(env_of<UNI>(P, R));
    const float4 hh = vx.hit, r0 = vx.r0, r1 = vx.r1;
    int slot = __float_as_int(hh.w);
    f3 o = xyz(r0), d = xyz(r1);
    uint32_t stw;
    if (sw_src == SW_START) {
        stw = ST_PREV_DELTA | 1u;
    } else if (sw_src == SW_RAY) {
        uint32_t w = __float_as_uint(r1.w);
        stw = (w & (ST_INSIDE | ST_PREV_DELTA)) | ((w & ST_LEN_MASK) + 1u);
    } else {
        stw = __float_as_uint(P.beta[id].w);
    }
    uint32_t len = stw & ST_LEN_MASK;
    bool inside = (stw & ST_INSIDE) != 0;
    uint32_t base = __float_as_uint(r0.w);
    so.base = base;
    f3 Pp = vadd(o, vscl(d, hh.x));
    // the slot's 64-B shading record: normals n0 n1 n2, uvs t0 t1 t2, material word
    const float4* A = S.attr + (size_t)slot * 4;
    float4 a0 = ldg4(A), a1 = ldg4(A + 1), a2 = ldg4(A + 2), a3 = ldg4(A + 3);
    float w0 = (1.f - hh.y) - hh.z;
    f3 nrm = vnorm(vadd(vadd(vscl(V3(a0.w, a1.x, a1.y), hh.y), vscl(V3(a1.z, a1.w, a2.x), hh.z)),
                        vscl(V3(a0.x, a0.y, a0.z), w0)));
    float tu = (a2.w * hh.y + a3.y * hh.z) + a2.y * w0;
    float tv = (a3.x * hh.y + a3.z * hh.z) + a2.z * w0;
    // the 64-B material record (64-B aligned) as four 16-B loads
    const float4* M = (const float4*)(S.mats + (size_t)(__float_as_uint(a3.w) & MAT_INDEX_MASK) * FF_MAT_FLOATS_DEV);
    float4 m0 = ldg4(M), m1 = ldg4(M + 1), m2 = ldg4(M + 2), m3 = ldg4(M + 3);
    f3 alb = V3(m0.y, m0.z, m0.w);
    float rough = m1.x, metal = m1.y;
    f3 fres = V3(m1.z, m1.w, m2.x);
    int at = (int)m2.z, rt = (int)m2.w, mt = (int)m3.x;
    bool rough_live = false;
    if (at >= 0) {
        ff_tex_desc td = S.tex[at];
        float t3[3];
        bilinear(td.data, td.w, td.h, 3, tu, tv, t3);
        alb = ld3(t3);
    }
    if (rt >= 0) {
        ff_tex_desc td = S.tex[rt];
        float t1[1];
        bilinear(td.data, td.w, td.h, 1, tu, tv, t1);
        rough = fmaxf(t1[0], 0.01f);
        rough_live = t1[0] > 0.01f;
    }
    if (mt >= 0) {
        ff_tex_desc td = S.tex[mt];
        float t1[1];
        bilinear(td.data, td.w, td.h, 1, tu, tv, t1);
        metal = t1[0];
    }
    // the light shadow ray leaves along the interpolated normal (CRT/kernel.cu:437);
    // everything else uses the normal-mapped one (get_normal, CRT/dMaterial.cu:61-87)
    f3 n_geo = nrm;
    int nt = (int)m3.y;
    if (nt >= 0) {
        const float* T = S.tan + (size_t)slot * 18;
        f3 tg = vnorm(vadd(vadd(vscl(ld3(T + 6), hh.y), vscl(ld3(T + 12), hh.z)), vscl(ld3(T), w0)));
        f3 bt = vnorm(vadd(vadd(vscl(ld3(T + 9), hh.y), vscl(ld3(T + 15), hh.z)), vscl(ld3(T + 3), w0)));
        ff_tex_desc td = S.tex[nt];
        float t3[3];
        bilinear(td.data, td.w, td.h, 3, tu, tv, t3);
        float mx = t3[0] * 2.f - 1.f, my = t3[1] * 2.f - 1.f, mz = t3[2] * 2.f - 1.f;
        nrm = vnorm(vadd(vadd(vscl(tg, mx), vscl(bt, my)), vscl(nrm, mz)));
    }
    f3 wo = vneg(d);
    f3 zero = V3(0, 0, 0);
    so.A = zero; so.Bs = zero; so.Cd = zero;
    so.wi = zero; so.wi_s = zero; so.wi_d = zero;
    so.lo = Pp; so.so = Pp; so.dd_o = Pp;
    so.needL = so.needS = so.needD = false;
    if (GRAD) {
        so.a_on = false;
        so.rough_live = rough_live;
        so.at = at; so.rt = rt; so.tu = tu; so.tv = tv;
        so.dA_alb = zero; so.dB_alb = zero; so.dC_alb = zero; so.dA_r = zero; so.dB_r = zero;
        so.kA = zero; so.kB = zero; so.kC = zero; so.dext_alb = zero; so.dext_r = zero;
    }
    uint32_t nst = (stw & (ST_INSIDE | ST_PREV_DELTA | ST_LEN_MASK));
    if (TYPE == MAT_DIELECTRIC) {
        Tri T = load_tri(S.tris, slot);
        f3 gn = vnorm(vcross(T.e1, T.e2));
        float cs = vdot(d, gn);
        bool entering = cs < 0.f;
        f3 nn = entering ? gn : vneg(gn);
        float cos_i = fabsf(cs);
        if (cos_i > 1.f) cos_i = 1.f;
        float ior = m2.y;
        float eta_i = entering ? 1.f : ior, eta_t = entering ? ior : 1.f;
        float F = fresnel_dielectric(cos_i, eta_i, eta_t);
        if (rng(base, len, DIM_DIEL) < F) {
            so.next_d = vnorm(vadd(d, vscl(nn, 2.f * cos_i)));
            so.next_o = vadd(Pp, vscl(nn, 1e-4f));
        } else {
            float eta = eta_i / eta_t;
            float k = 1.f - eta * eta * (1.f - cos_i * cos_i);
            float cos_t = sqrtf(fmaxf(k, 0.f));
            so.next_d = vnorm(vadd(vscl(d, eta), vscl(nn, eta * cos_i - cos_t)));
            so.next_o = vsub(Pp, vscl(nn, 1e-4f));
            inside = !inside;
        }
        so.fext = V3(1.f, 1.f, 1.f);
        so.pdf_ext = 1.f;
        so.cos_ext = 1.f;
        so.nst = (nst & ST_LEN_MASK) | ST_PREV_DELTA | (inside ? ST_INSIDE : 0u);
        return;
    }
    constexpr bool do_spec = (TYPE == MAT_MIX || TYPE == MAT_CONDUCTOR);
    constexpr bool do_diff = (TYPE == MAT_MIX || TYPE == MAT_DIFFUSE);
    f3 wi = env_sample(E, Pp, rng(base, len, DIM_EX), rng(base, len, DIM_EY));
    so.wi = wi;
    double diff_pdf = (double)(1.f / (2.f * F_PI));
    // light-sample term of BRDF_L (CRT/dMaterial.cu:376-402)
    float ndwi = vdot(nrm, wi);
    if (ndwi > 0.f) {
        float eu, ev;
        sph_map(wi, eu, ev);
        f3 Li = env_L(E, eu, ev);
        double sp = do_spec ? (double)spec_pdf(nrm, wi, wo, rough) : 0.0;
        double lp = (double)env_pdf(E, wi, eu, ev);
        // lp is infinite where sin(acos(wi.z)) == 0; the term's limit there is 0
        if (lp > 0.f && lp < (double)INFINITY && !vzero(Li)) {
            double dwt = power_heur(lp, diff_pdf), swt = power_heur(lp, sp);
            if (do_spec) {
                f3 f = vscl(spec_f(nrm, wi, wo, rough, metal, alb, fres), ndwi);
                if (!vzero(f)) {
                    so.A = vadd(so.A, vdiv(vmul(vscl(f, (float)swt), Li), (float)lp));
                    if (GRAD) {
                        LobeGrad g = spec_grad(nrm, wi, wo, rough, metal, alb, fres);
                        float s = ndwi * (float)swt / (float)lp;
                        so.a_on = true;
                        so.kA = vadd(so.kA, vscl(f, (float)swt / (float)lp));
                        so.dA_alb = vadd(so.dA_alb, vmul(vscl(g.da, s), Li));
                        so.dA_r = vadd(so.dA_r, vmul(vscl(g.dr, s), Li));
                    }
                }
            }
            if (do_diff) {
                f3 f = vscl(diff_f(wi, wo, metal, alb, fres), ndwi);
                if (!vzero(f)) {
                    so.A = vadd(so.A, vdiv(vmul(vscl(f, (float)dwt), Li), (float)lp));
                    if (GRAD) {
                        f3 da = diff_grad(wi, wo, metal, alb, fres);
                        float s = ndwi * (float)dwt / (float)lp;
                        so.a_on = true;
                        so.kA = vadd(so.kA, vscl(f, (float)dwt / (float)lp));
                        so.dA_alb = vadd(so.dA_alb, vmul(vscl(da, s), Li));
                    }
                }
            }
        }
    }
    // BRDF-sampled MIS terms (CRT/dMaterial.cu:404-448)
    f3 wi_s = zero, wi_d = zero;
    if (do_spec) wi_s = spec_sample(nrm, wo, rough, rng(base, len, DIM_S0), rng(base, len, DIM_S1));
    if (do_diff) wi_d = diff_sample(nrm, rng(base, len, DIM_D0), rng(base, len, DIM_D1));
    so.wi_s = wi_s;
    so.wi_d = wi_d;
    if (do_spec) {
        float nd = vdot(nrm, wi_s);
        if (nd > 0.f) {
            float eu, ev;
            sph_map(wi_s, eu, ev);
            double sp = (double)spec_pdf(nrm, wi_s, wo, rough);
            double lp = (double)env_pdf(E, wi_s, eu, ev);
            double wt = power_heur(sp, lp);
            f3 f = vscl(spec_f(nrm, wi_s, wo, rough, metal, alb, fres), nd);
            f3 L2 = env_L(E, eu, ev);
            if (!vzero(f) && sp > 0.f && !vzero(L2)) {
                so.Bs = vdiv(vscl(vmul(f, L2), (float)wt), (float)sp);
                so.needS = true;
                so.so = sample_origin(Pp, wi_s);
                if (GRAD) {
                    LobeGrad g = spec_grad(nrm, wi_s, wo, rough, metal, alb, fres);
                    float s = nd * (float)wt / (float)sp;
                    so.kB = vscl(f, (float)wt / (float)sp);
                    so.dB_alb = vmul(vscl(g.da, s), L2);
                    so.dB_r = vmul(vscl(g.dr, s), L2);
                }
            }
        }
    }
    if (do_diff) {
        float nd = vdot(nrm, wi_d);
        if (nd > 0.f) {
            float eu, ev;
            sph_map(wi_d, eu, ev);
            double lp = (double)env_pdf(E, wi_d, eu, ev);
            double wt = power_heur(diff_pdf, lp);
            f3 f = vscl(diff_f(wi_d, wo, metal, alb, fres), nd);
            f3 L3 = env_L(E, eu, ev);
            if (!vzero(f) && diff_pdf > 0.f && !vzero(L3)) {
                so.Cd = vdiv(vscl(vmul(f, L3), (float)wt), (float)diff_pdf);
                so.needD = true;
                // the mixed material offsets this ray along wi_spec (CRT/dMaterial.cu:431)
                so.dd_o = sample_origin(Pp, TYPE == MAT_MIX ? wi_s : wi_d);
                if (GRAD) {
                    f3 da = diff_grad(wi_d, wo, metal, alb, fres);
                    float s = nd * (float)wt / (float)diff_pdf;
                    so.kC = vscl(f, (float)wt / (float)diff_pdf);
                    so.dC_alb = vmul(vscl(da, s), L3);
                }
            }
        }
    }
    so.needL = !vzero(so.A) || so.needS || so.needD;
    so.lo = vadd(Pp, vscl(n_geo, 0.001f));
    f3 dir;
    if (TYPE == MAT_MIX) {
        dir = (rng(base, len, DIM_LOBE) < 0.5f) ? wi_d : wi_s;
        so.fext = vadd(spec_f(nrm, dir, wo, rough, metal, alb, fres), diff_f(dir, wo, metal, alb, fres));
        float spf = spec_pdf(nrm, dir, wo, rough);
        float dpf = (float)diff_pdf;
        so.pdf_ext = (float)(0.5 * (double)(spf + dpf));
    } else if (TYPE == MAT_DIFFUSE) {
        dir = wi_d;
        so.fext = diff_f(dir, wo, metal, alb, fres);
        so.pdf_ext = (float)diff_pdf;
    } else {
        dir = wi_s;
        so.fext = spec_f(nrm, dir, wo, rough, metal, alb, fres);
        so.pdf_ext = spec_pdf(nrm, dir, wo, rough);
    }
    if (GRAD) {
        if (do_spec) {
            LobeGrad g = spec_grad(nrm, dir, wo, rough, metal, alb, fres);
            so.dext_alb = g.da;
            so.dext_r = g.dr;
        }
        if (do_diff) so.dext_alb = vadd(so.dext_alb, diff_grad(dir, wo, metal, alb, fres));
    }
    so.cos_ext = fmaxf(0.0f, vdot(nrm, dir));
    so.next_o = Pp;
    so.next_d = dir;
    so.nst = (nst & (ST_LEN_MASK | ST_INSIDE)) | (so.needL ? ST_NEED_L : 0u) | (so.needS ? ST_NEED_S : 0u) |
             (so.needD ? ST_NEED_D : 0u);
}

// shades one path; true: its shadow rays are to be traced, queue entry `shadow`
template <int TYPE, bool UNI>
__device__ __forceinline__ bool shade_path(const ff_paths& P, uint32_t id, bool first, uint32_t& shadow) {
    ShadeOut so;
    shade_core<TYPE, false, UNI>(P, id, load_vertex(P, id), so, first ? SW_START : SW_RAY);
    const bool needL = so.needL, needS = so.needS, needD = so.needD;
    if (needL) {
        P.sray[6 * id + 0] = f4(so.lo, __uint_as_float(TYPE == MAT_MIX ? 0u : AUX_ALONG));
        P.sray[6 * id + 1] = f4(so.wi, 0.f);
    }
    if (TYPE == MAT_MIX && needS) {
        P.sray[6 * id + 2] = f4(so.so, 0.f);
        P.sray[6 * id + 3] = f4(so.wi_s, 0.f);
    }
    if (TYPE == MAT_MIX && needD) {
        P.sray[6 * id + 4] = f4(so.dd_o, 0.f);
        P.sray[6 * id + 5] = f4(so.wi_d, 0.f);
    }
    // wf_logic reads a term only where the state word asks for it
    // (needS and needD imply needL)
    if (needL) P.nee[3 * id] = f4(so.A, 0.f);
    if (needS) P.nee[3 * id + 1] = f4(so.Bs, 0.f);
    if (needD) P.nee[3 * id + 2] = f4(so.Cd, 0.f);
    // the throughput factor wf_logic applies, f * cos / pdf, formed here
    // with the same operations (logic then reads 16 B instead of 32)
    // and the continuation's state word rides in its w (the path
    // record's beta is left to wf_logic)
    bool dead = vzero(so.fext) || so.pdf_ext == 0.f;
    uint32_t sw = dead ? so.nst | ST_DEAD : so.nst;
    P.fext[id] = dead ? make_float4(0.f, 0.f, 0.f, __uint_as_float(sw))
                      : f4(vdiv(vscl(so.fext, so.cos_ext), so.pdf_ext), __uint_as_float(sw));
    P.ray[2 * id] = f4(so.next_o, __uint_as_float(so.base));
    P.ray[2 * id + 1] = f4(so.next_d, __uint_as_float(sw));
    shadow = (id << 2) | (needS ? 1u : 0u) | (needD ? 2u : 0u);
    return needL;
}

template <int TYPE, bool UNI>
__global__ __launch_bounds__(FF_BLOCK) void k_shade(ff_paths P, int next_q, int first) {
    __shared__ QStage<FF_BLOCK, 1, QSTAGE_CAP> st;
    const uint32_t n = P.counters[mat_counter(1 - next_q) + TYPE];
    const uint32_t* queue = P.q_mat[TYPE];
    const uint32_t n_round = (n + FF_BLOCK - 1) / FF_BLOCK * FF_BLOCK;
    const int qidx[1] = {shadow_counter(next_q)};
    uint32_t* const qs[1] = {P.q_shadow};
    const uint32_t ebase = ext_base<TYPE>(P, 1 - next_q);
    add_extensions(P, next_q, n);
    st.init();
    for (uint32_t i = gtid(); i < n_round; i += gstride()) {
        const bool live = i < n;
        uint32_t shadow = 0;
        bool need = false;
        if (live) {
            const uint32_t id = queue[i];
            need = shade_path<TYPE, UNI>(P, id, first, shadow);
            // every event continues (wf_logic decides its fate): the material
            // queues follow one another in the next extension queue
            P.q_ext[next_q][ebase + i] = id;
        }
        // one shadow-queue entry per event with a light ray (needS / needD
        // imply needL); the shadow stage traces and counts its rays
        st.add(need ? 0 : -1, shadow);
        st.flush_if_full(P.counters, qidx, qs);
    }
    st.flush(P.counters, qidx, qs);
}

// A wave's entries into an LDS list.  Every lane of the wave calls it.
__device__ __forceinline__ void lds_append(uint32_t* list, uint32_t* count, bool on, uint32_t v) {
    const uint64_t m = __ballot(on);
    if (m == 0) return;
    uint32_t first = 0;
    if (__lane_id() == 0) first = atomicAdd(count, (uint32_t)__popcll(m));
    first = (uint32_t)__builtin_amdgcn_readfirstlane((int)first);
    if (on) list[first + __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u))] = v;
}
// The ids of a tile's continuing paths (route >= 0) in the tile's order after
// the n_ext entries that the stage holds; live_in: how many each wave has.
template <int NP, int BS>
__device__ __forceinline__ void place_in_order(uint32_t* ext, uint32_t& n_ext, const uint32_t (*live_in)[BS / 64],
                                               uint32_t wave, const int* route, const uint32_t* id) {
#pragma unroll
    for (int j = 0; j < NP; j++) {
        const uint64_t m = __ballot(route[j] >= 0);
        uint32_t at = n_ext + __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
#pragma unroll
        for (uint32_t v = 0; v < BS / 64; v++) {
            const uint32_t l = live_in[j][v];
            at += v < wave ? l : 0u;
            n_ext += l;
        }
        if (route[j] >= 0) ext[at] = id[j];
    }
}
// Appends the staged extension and shadow entries to the queues of the next
// iteration, one atomic a queue.  After a barrier; before another.
template <int BS>
__device__ __forceinline__ void flush_entries(const ff_paths& P, int q, const uint32_t* ext, uint32_t& n_ext,
                                              const uint32_t* shd, uint32_t& n_shd, uint32_t* base) {
    const uint32_t ns = n_shd;
    if (threadIdx.x == 0) base[0] = n_ext ? atomicAdd(&P.counters[ext_counter(1 - q)], n_ext) : 0u;
    if (threadIdx.x == 64) base[1] = ns ? atomicAdd(&P.counters[shadow_counter(1 - q)], ns) : 0u;
    __syncthreads();
    for (uint32_t k = threadIdx.x; k < n_ext; k += BS) P.q_ext[1 - q][base[0] + k] = ext[k];
    for (uint32_t k = threadIdx.x; k < ns; k += BS) P.q_shadow[base[1] + k] = shd[k];
    if (threadIdx.x == 0) n_shd = 0u;
    n_ext = 0;
}
// wf_logic and the material kernels of an iteration in one launch.  Apart, a
// path's id went through a material queue in memory, its hit was fetched
// twice, every launch (one per material type) had its own start and tail, and
// the next extension queue held the types one after another.  Here a workgroup
// routes a tile of TILE paths into LDS lists by type and its waves shade them
// in full chunks of 64 of one type; what is left over (under 64 a type) waits
// for the next tile, and the last tile shades everything.  The extension queue
// keeps the tile's order, so that the records of neighbouring entries lie
// together in the next iteration, which is worth more than directions that
// agree: entries sorted by the octant of their ray's direction inside a
// workgroup's run cost a 1080p frame 6 % (59.7 -> 63.3 ms).  Entries are staged
// in LDS (CAP) and appended with one atomic a queue and run.
//
// Bound by the paths' records in memory at large sizes (a diffuse event moves
// about 0.4 KB, at 3.5 TB/s), by the chain of dependent loads at small ones.
// Against separate launches: 1080p 64 samples 61.3 -> 59.4 ms, 1021x577 8
// samples 5.05 -> 4.10 ms, eight uneven views 13.7 -> 12.2 ms, 160x120
// 0.404 -> 0.377 ms, 320x180 with three material types 0.60 -> 0.50 ms.
template <bool UNI, int BS, int TILE, int NP, int CAP>
__global__ __launch_bounds__(BS, 4) void k_logic_shade(ff_paths P, int q, int iter, int last) {
    static_assert(NP * BS == TILE && TILE % 64 == 0 && CAP >= TILE + 4 * 63, "a tile's entries fit the stage");
    __shared__ uint32_t list[4][TILE + 64], ext[CAP], shd[CAP];
    __shared__ uint32_t fill[4], n_shd, base[2], live_in[NP][BS / 64];
    constexpr uint32_t ADD = TILE + 4 * 63;  // most paths that one round shades
    if (threadIdx.x < 4) fill[threadIdx.x] = 0u;
    if (threadIdx.x == 0) n_shd = 0u;
    uint32_t n_ext = 0;
    clear_traversed(P);
    const uint32_t n = P.counters[ext_counter(q)];
    const uint32_t* queue = P.q_ext[q];
    const bool first_batch = P.bstate[B_BATCH] == 0;
    const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), lane = __lane_id();
    LogicCounts cnt;
    __syncthreads();
    for (uint32_t t0 = blockIdx.x * TILE; t0 < n; t0 += gridDim.x * TILE) {
        const bool fin = n - t0 <= gridDim.x * TILE;  // the workgroup's last tile
        bool live[NP];
        uint32_t id[NP];
        int route[NP];
#pragma unroll
        for (int j = 0; j < NP; j++) {
            const uint32_t i = t0 + (uint32_t)j * BS + threadIdx.x;
            live[j] = i < n;
            id[j] = live[j] ? queue[i] : 0u;
        }
        logic_paths<UNI, NP>(P, iter, first_batch, live, id, route, cnt);
        if (last) continue;  // nothing survives the last vertex
#pragma unroll
        for (int j = 0; j < NP; j++)
#pragma unroll
            for (int t = 0; t < 4; t++) lds_append(list[t], &fill[t], route[j] == t, id[j]);
#pragma unroll
        for (int j = 0; j < NP; j++) {
            const uint64_t m = __ballot(route[j] >= 0);
            if (lane == 0) live_in[j][wave] = (uint32_t)__popcll(m);
        }
        __syncthreads();
        place_in_order<NP, BS>(ext, n_ext, live_in, wave, route, id);
        uint32_t chunks[4], total = 0;
#pragma unroll
        for (int t = 0; t < 4; t++) {
            const uint32_t have = (uint32_t)__builtin_amdgcn_readfirstlane((int)fill[t]);
            chunks[t] = fin ? (have + 63u) / 64u : have / 64u;
            total += chunks[t];
        }
        for (uint32_t w = wave; w < total; w += BS / 64) {
            uint32_t k = w, t = 0;
#pragma unroll
            for (uint32_t u = 0; u < 3; u++)
                if (t == u && k >= chunks[u]) {
                    k -= chunks[u];
                    t = u + 1;
                }
            const uint32_t have = (uint32_t)__builtin_amdgcn_readfirstlane((int)fill[t]);
            // (a full chunk is taken from the list's end: the rest stays in front)
            const uint32_t i = (fin ? 0u : have & 63u) + k * 64u + lane;
            const bool on = i < have;
            const uint32_t pid = on ? list[t][i] : 0u;
            uint32_t shadow = 0;
            bool need = false;
            if (on) {
                switch (t) {
                    case MAT_MIX: need = shade_path<MAT_MIX, UNI>(P, pid, iter == 1, shadow); break;
                    case MAT_DIFFUSE: need = shade_path<MAT_DIFFUSE, UNI>(P, pid, iter == 1, shadow); break;
                    case MAT_CONDUCTOR: need = shade_path<MAT_CONDUCTOR, UNI>(P, pid, iter == 1, shadow); break;
                    default: need = shade_path<MAT_DIELECTRIC, UNI>(P, pid, iter == 1, shadow); break;
                }
            }
            lds_append(shd, &n_shd, need, shadow);
        }
        __syncthreads();
        if (threadIdx.x < 4) fill[threadIdx.x] = fin ? 0u : fill[threadIdx.x] & 63u;
        if (fin || n_ext + TILE > CAP || n_shd + ADD > CAP) flush_entries<BS>(P, q, ext, n_ext, shd, n_shd, base);
        __syncthreads();
    }
    add_counts(P, cnt);
}

// ================================================== path-replay adjoint
// The adjoint replays every stored forward path with the same random
// numbers (same camera ray, same hits, same samples) and, at each event,
// moves d loss / d radiance onto the parameters the event's radiance depends
// on: Le through environment texels, f through albedo / roughness texels.
// L_rem (in Lp) starts as the path's stored radiance and loses each term as
// it is replayed, so at a vertex it is the radiance that flows through the
// vertex's continuation; its derivative w.r.t. f is L_rem * (df/dtheta) / f
// (path replay backpropagation).  Sampling is detached: directions, pdfs,
// MIS weights and Russian roulette are those of the forward.

// d loss / d parameter into gradient target element i: the terms v and u (0:
// none).  The deterministic sums take each term by itself, as 64-bit fixed
// point; the float sum takes both at once.
__device__ __forceinline__ void grad_add(const ff_paths& P, float* buf, uint64_t off, uint32_t i, float v, float u) {
    if (P.gmode == GM_FLOAT) {
        const float s = v + u;
        if (s != 0.f) unsafeAtomicAdd(buf + i, s);
        return;
    }
    if (v == 0.f && u == 0.f) return;
    const uint64_t a = off + i;
    if (P.gmode == GM_BOUND) {
        const uint32_t bv = __float_as_uint(fabsf(v)), bu = __float_as_uint(fabsf(u));
        atomicMax(&P.g_max[a], bv > bu ? bv : bu);
        atomicAdd(&P.g_cnt[a], (v != 0.f ? 1u : 0u) + (u != 0.f ? 1u : 0u));
    } else {
        const int e = fixed_exponent(P.g_max[a], P.g_cnt[a]);
        const long long q = __double2ll_rn(ldexp((double)v, e)) + __double2ll_rn(ldexp((double)u, e));
        atomicAdd(&P.g_fx[a], (unsigned long long)q);
    }
}
// Scatter of bilinear footprints onto gradient texels, the wave together.
// Atomics run at the memory side at about 15 G requests/s, however many
// elements a request carries.  With a lane issuing its footprint's 4 x C
// elements one by one, each is a request of its own; here the footprints go
// through LDS and consecutive lanes take consecutive elements, so the texels
// of a row (2 C floats side by side) leave in one request.
struct Scatter {  // of one wave
    uint32_t idx[4][64];
    float w[4][64];
    float val[3][64], more[3][64];
    float* buf[64];
    uint64_t off[64];
};
// on: the lane has a footprint tp of target T with value val[0..C) (per
// channel, before the tap weights).  TWO: with the values of two terms, whose
// atomics are shared: in float they are added first, in the deterministic sums
// they stay apart.  Every lane of the wave calls it.
template <int C, bool TWO = false>
__device__ __forceinline__ void scatter(const ff_paths& P, Scatter& S, bool on, const ff_dev_gtarget& T,
                                        const Taps& tp, f3 val, f3 more = V3(0.f, 0.f, 0.f)) {
    const uint64_t m = __ballot(on);
    if (m == 0) return;
    const bool apart = TWO && P.gmode != GM_FLOAT;
    if (on) {
        const uint32_t f = __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
        if (TWO && !apart) val = vadd(val, more);
        if (apart) {
            S.more[0][f] = more.x;
            S.more[1][f] = more.y;
            S.more[2][f] = more.z;
        }
#pragma unroll
        for (int k = 0; k < 4; k++) {
            S.idx[k][f] = tp.i[k];
            S.w[k][f] = tp.w[k];
        }
        S.val[0][f] = val.x;
        S.val[1][f] = val.y;
        S.val[2][f] = val.z;
        S.buf[f] = T.buf;
        S.off[f] = T.off;
    }
    __threadfence_block();
    __builtin_amdgcn_wave_barrier();
    const uint32_t total = (uint32_t)__popcll(m) * (4u * C);
    for (uint32_t e = __lane_id(); e < total; e += 64u) {
        const uint32_t f = e / (4u * C), r = e % (4u * C), k = r / C, c = r % C;
        const float w = S.w[k][f];
        grad_add(P, S.buf[f], S.off[f], C * S.idx[k][f] + c, w * S.val[c][f], apart ? w * S.more[c][f] : 0.f);
    }
    __threadfence_block();
    __builtin_amdgcn_wave_barrier();
}
// d loss / d Le(dir) = val (per channel) onto the environment texels
__device__ __forceinline__ void scatter_env(const ff_paths& P, Scatter& S, bool on, const ff_dev_request& R, f3 dir,
                                            f3 val) {
    ff_dev_gtarget T{nullptr, 0};
    Taps tp{};
    if (on) T = R.gt[GT_ENV];
    on = on && T.buf;
    if (on) {
        float u, v;
        sph_map(dir, u, v);
        tp = taps_of(R.E.w, R.E.h, u, v);
    }
    scatter<3>(P, S, on, T, tp, val);
}
// d loss / d (texture t value at (u, v)) = val + more (C channels) onto its texels
template <int C>
__device__ __forceinline__ void scatter_tex(const ff_paths& P, Scatter& S, bool on, const ff_dev_request& R, int t,
                                            float u, float v, f3 val, f3 more) {
    ff_dev_gtarget T{nullptr, 0};
    Taps tp{};
    if (on) T = R.gt[1 + t];
    on = on && T.buf;
    if (on) {
        const ff_tex_desc& td = R.S.tex[t];
        tp = taps_of(td.w, td.h, u, v);
    }
    scatter<C, true>(P, S, on, T, tp, val, more);
}

// wf_logic of the replay: same termination, Russian roulette and routing as
// k_logic; an escaping delta/camera ray's Le term is replayed.  The vertex's
// NEE terms and throughput update were replayed by k_shade_adj.
// Every lane of the wave calls it; returns the path's material type (-1: ended).
template <bool UNI>
__device__ __forceinline__ int replay_logic(const ff_paths& P, Scatter& sc, bool live, uint32_t id, LogicCounts& c) {
    int route = -1;
    bool term = false, primary = false;
    bool esc = false;  // an escaped camera or delta ray: its Le term
    f3 d = V3(0.f, 0.f, 0.f), gval = d;
    const ff_dev_request& R = P.reqs[req_of(P, id)];
    if (live) {
        const ff_dev_scene& S = scene_of<UNI>(P, R);
        float4 bw = P.beta[id];
        uint32_t stw = __float_as_uint(bw.w);
        uint32_t len = (stw & ST_LEN_MASK) + 1;
        primary = len == 1;
        f3 beta = xyz(bw);
        f3 Lrem = xyz(P.Lp[id]);
        float4 hh = P.hit[id];
        int slot = __float_as_int(hh.w);
        bool found = slot >= 0;
        term = (len > R.depth) || !found || (stw & ST_DEAD);
        int mtype = -1;
        // the direction is read only by the two cases that use it
        if ((found && (stw & ST_INSIDE)) || (!found && (stw & ST_PREV_DELTA))) d = xyz(P.ray[2 * id + 1]);
        if (found) {
            mtype = (int)(S.mat[slot] >> MAT_TYPE_SHIFT);
            if ((stw & ST_INSIDE) && mtype != MAT_DIELECTRIC) {
                Tri T = load_tri(S.tris, slot);
                if (!(vdot(d, vcross(T.e1, T.e2)) < 0.f)) term = true;  // absorbed
            }
        }
        if (!found && (stw & ST_PREV_DELTA)) {
            Lrem = vsub(Lrem, vmul(beta, env_L(env_view(env_of<UNI>(P, R)), d)));
            esc = true;
            gval = vmul(xyz(P.dlt[id]), beta);
        }
        if (!(stw & ST_DEAD) && len > 3) {
            float qrr = fmaxf(0.05f, 1.f - beta.y);
            if (rng(__float_as_uint(ldg(&P.ray[2 * id].w)), len, DIM_RR) < qrr) term = true;
        }
        if (!term) {
            uint32_t nst = (stw & (ST_INSIDE | ST_PREV_DELTA)) | len;
            P.beta[id] = f4(beta, __uint_as_float(nst));
            P.Lp[id] = f4(Lrem, 0.f);
            route = mtype;
        }
    }
    scatter_env(P, sc, esc, R, d, gval);
    c.prim += (live && primary) ? 1u : 0u;
    c.ext += (live && !primary) ? 1u : 0u;
    c.paths += (live && term) ? 1u : 0u;
    return route;
}
template <bool UNI>
__global__ __launch_bounds__(FF_BLOCK) void k_logic_adj(ff_paths P, int q) {
    __shared__ QStage<FF_BLOCK, 4, QSTAGE_CAP> st;
    __shared__ Scatter sc[FF_BLOCK / 64];
    const int qidx[4] = {mat_counter(q), mat_counter(q) + 1, mat_counter(q) + 2, mat_counter(q) + 3};
    uint32_t* const qs[4] = {P.q_mat[0], P.q_mat[1], P.q_mat[2], P.q_mat[3]};
    st.init();
    clear_traversed(P);
    const uint32_t n = P.counters[ext_counter(q)];
    const uint32_t* queue = P.q_ext[q];
    const uint32_t n_round = (n + FF_BLOCK - 1) / FF_BLOCK * FF_BLOCK;  // uniform trip count per workgroup
    LogicCounts c;
    for (uint32_t i = gtid(); i < n_round; i += gstride()) {
        const bool live = i < n;
        const uint32_t id = live ? queue[i] : 0u;
        const int route = replay_logic<UNI>(P, sc[threadIdx.x >> 6], live, id, c);
        st.add(route, id);
        st.flush_if_full(P.counters, qidx, qs);
    }
    st.flush(P.counters, qidx, qs);
    add_counts(P, c);
}

// Replay of a vertex's rays: the shadow rays and the continuation that k_shade
// queues.  The vertex itself (its hit and the ray that found it) is kept in the
// path's NEE terms, which the replay does not store, for k_shade_adj, which
// follows the rays' traversal.  (A dielectric vertex has no more to replay.)
// true: its shadow rays are to be traced, queue entry `shadow`.
template <int TYPE, bool UNI>
__device__ __forceinline__ bool replay_rays(const ff_paths& P, uint32_t id, uint32_t& shadow) {
    bool needL = false, needS = false, needD = false;
    ShadeOut so;
    const Vertex vx = load_vertex(P, id);
    shade_core<TYPE, false, UNI>(P, id, vx, so);
    uint32_t nst = so.nst;
    if (TYPE != MAT_DIELECTRIC) {
        needL = so.needL; needS = so.needS; needD = so.needD;
        if (needL) {
            P.sray[6 * id + 0] = f4(so.lo, __uint_as_float(TYPE == MAT_MIX ? 0u : AUX_ALONG));
            P.sray[6 * id + 1] = f4(so.wi, 0.f);
        }
        if (TYPE == MAT_MIX && needS) {
            P.sray[6 * id + 2] = f4(so.so, 0.f);
            P.sray[6 * id + 3] = f4(so.wi_s, 0.f);
        }
        if (TYPE == MAT_MIX && needD) {
            P.sray[6 * id + 4] = f4(so.dd_o, 0.f);
            P.sray[6 * id + 5] = f4(so.wi_d, 0.f);
        }
        nst &= ST_LEN_MASK | ST_INSIDE;
        P.nee[3 * id] = vx.hit;
        P.nee[3 * id + 1] = vx.r0;
        P.nee[3 * id + 2] = f4(xyz(vx.r1), __int_as_float(TYPE));
    } else {
        P.beta[id].w = __uint_as_float(nst);
        P.nee[3 * id + 2].w = __int_as_float(TYPE);
    }
    P.ray[2 * id] = f4(so.next_o, __uint_as_float(so.base));
    P.ray[2 * id + 1] = f4(so.next_d, __uint_as_float(nst));
    shadow = (id << 2) | (needS ? 1u : 0u) | (needD ? 2u : 0u);
    return needL;
}
template <int TYPE, bool UNI>
__global__ __launch_bounds__(FF_BLOCK) void k_shade_nee(ff_paths P, int next_q) {
    __shared__ QStage<FF_BLOCK, 1, QSTAGE_CAP> st;
    const uint32_t n = P.counters[mat_counter(1 - next_q) + TYPE];
    const uint32_t* queue = P.q_mat[TYPE];
    const uint32_t n_round = (n + FF_BLOCK - 1) / FF_BLOCK * FF_BLOCK;
    const int qidx[1] = {shadow_counter(next_q)};
    uint32_t* const qs[1] = {P.q_shadow};
    const uint32_t ebase = ext_base<TYPE>(P, 1 - next_q);
    add_extensions(P, next_q, n);
    st.init();
    for (uint32_t i = gtid(); i < n_round; i += gstride()) {
        uint32_t shadow = 0;
        bool need = false;
        if (i < n) {
            const uint32_t id = queue[i];
            need = replay_rays<TYPE, UNI>(P, id, shadow);
            P.q_ext[next_q][ebase + i] = id;
        }
        if (TYPE == MAT_DIELECTRIC) continue;
        st.add(need ? 0 : -1, shadow);
        st.flush_if_full(P.counters, qidx, qs);
    }
    st.flush(P.counters, qidx, qs);
}

// Replay of a vertex once its shadow rays are traced: its visibility-gated
// NEE terms leave L_rem (with their gradients), then the continuation's
// gradient L_rem * (df/dtheta) / f and the throughput update of wf_logic.  Every
// lane of the wave calls it.
template <int TYPE, bool UNI>
__device__ __forceinline__ void replay_gradients(const ff_paths& P, Scatter& S, bool live, uint32_t id) {
    // what the vertex scatters: NEE terms onto the environment (light, spec,
    // diffuse direction), NEE and continuation onto its albedo and roughness
    const ff_dev_request& R = P.reqs[req_of(P, id)];
    ShadeOut so;
    bool visL = false, visS = false, visD = false, alb_on = false, rough_on = false;
    f3 w = V3(0.f, 0.f, 0.f), g_alb = w, g_rough = w;  // NEE
    f3 h_alb = w, h_rough = w;                         // continuation
    if (live) {
        shade_core<TYPE, true, UNI>(P, id, {P.nee[3 * id], P.nee[3 * id + 1], P.nee[3 * id + 2]}, so);
        f3 beta = xyz(P.beta[id]);
        uint32_t nst = so.nst;
        f3 Lrem = xyz(P.Lp[id]);
        f3 dl = xyz(P.dlt[id]);
        visL = so.needL && P.vis[3 * id + 0];
        visS = visL && so.needS && P.vis[3 * id + 1];
        visD = visL && so.needD && P.vis[3 * id + 2];
        alb_on = so.at >= 0;
        rough_on = so.rt >= 0 && so.rough_live;
        if (visL) {
            f3 lb = so.A;
            if (visS) lb = vadd(lb, so.Bs);
            if (visD) lb = vadd(lb, so.Cd);
            Lrem = vsub(Lrem, vmul(lb, beta));
            w = vmul(dl, beta);
            f3 ga = so.dA_alb;
            if (visS) ga = vadd(ga, so.dB_alb);
            if (visD) ga = vadd(ga, so.dC_alb);
            g_alb = vmul(w, ga);
            f3 gr = so.dA_r;
            if (visS) gr = vadd(gr, so.dB_r);
            g_rough.x = vdot(w, gr);
        }
        bool dead = vzero(so.fext) || so.pdf_ext == 0.f;
        if (!dead) {
            f3 qv = V3(so.fext.x != 0.f ? dl.x * Lrem.x / so.fext.x : 0.f,
                       so.fext.y != 0.f ? dl.y * Lrem.y / so.fext.y : 0.f,
                       so.fext.z != 0.f ? dl.z * Lrem.z / so.fext.z : 0.f);
            h_alb = vmul(qv, so.dext_alb);
            h_rough.x = vdot(qv, so.dext_r);
            beta = vmul(beta, vdiv(vscl(so.fext, so.cos_ext), so.pdf_ext));
        }
        nst = (nst & (ST_LEN_MASK | ST_INSIDE)) | (dead ? ST_DEAD : 0u);
        P.Lp[id] = f4(Lrem, 0.f);
        P.beta[id] = f4(beta, __uint_as_float(nst));
    }
    scatter_tex<3>(P, S, alb_on, R, so.at, so.tu, so.tv, g_alb, h_alb);
    if (TYPE != MAT_DIFFUSE) scatter_tex<1>(P, S, rough_on, R, so.rt, so.tu, so.tv, g_rough, h_rough);
    scatter_env(P, S, visL && so.a_on, R, so.wi, vmul(w, so.kA));
    if (TYPE != MAT_DIFFUSE) scatter_env(P, S, visS, R, so.wi_s, vmul(w, so.kB));
    if (TYPE != MAT_CONDUCTOR) scatter_env(P, S, visD, R, so.wi_d, vmul(w, so.kC));
}
// (the paths are those of extension queue q's part for TYPE)
template <int TYPE, bool UNI>
__global__ __launch_bounds__(FF_BLOCK) void k_shade_adj(ff_paths P, int q) {
    __shared__ Scatter sc[FF_BLOCK / 64];
    const uint32_t n = P.counters[mat_counter(1 - q) + TYPE];
    const uint32_t* queue = P.q_ext[q] + ext_base<TYPE>(P, 1 - q);
    const uint32_t n_round = (n + FF_BLOCK - 1) / FF_BLOCK * FF_BLOCK;
    for (uint32_t i = gtid(); i < n_round; i += gstride())
        replay_gradients<TYPE, UNI>(P, sc[threadIdx.x >> 6], i < n, i < n ? queue[i] : 0u);
}

// The replay's stages of an iteration in one launch, as k_logic_shade has the
// forward's: a workgroup finishes its tile's previous vertices by type, routes
// the paths, and shades the next vertices by type.  The previous vertex's type
// is kept with it.  Bound by the memory side's atomics (the gradients of a tile
// overlap the routing and shading of others now) and by the path records; three
// waves a SIMD (167 VGPRs).  Against a launch for every stage and type: eight
// 192x192 views with gradients 7.95 -> 7.19 ms, 512x512 16 samples 8.09 -> 7.95,
// a deterministic 201x151 render 3.27 -> 3.20 ms.
template <bool UNI, int BS, int TILE, int NP, int CAP>
__global__ __launch_bounds__(BS, 3) void k_replay(ff_paths P, int q, int iter, int last) {
    static_assert(NP * BS == TILE && TILE % 64 == 0 && CAP >= TILE + 4 * 63, "a tile's entries fit the stage");
    __shared__ uint32_t done[3][TILE], list[4][TILE + 64], ext[CAP], shd[CAP];
    __shared__ uint32_t ended[3], fill[4], n_shd, base[2], live_in[NP][BS / 64];
    __shared__ Scatter sc[BS / 64];
    constexpr uint32_t ADD = TILE + 4 * 63;  // most paths that one round shades
    if (threadIdx.x < 4) fill[threadIdx.x] = 0u;
    if (threadIdx.x < 3) ended[threadIdx.x] = 0u;
    if (threadIdx.x == 0) n_shd = 0u;
    uint32_t n_ext = 0;
    clear_traversed(P);
    const uint32_t n = P.counters[ext_counter(q)];
    const uint32_t* queue = P.q_ext[q];
    const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), lane = __lane_id();
    Scatter& S = sc[wave];
    LogicCounts cnt;
    __syncthreads();
    for (uint32_t t0 = blockIdx.x * TILE; t0 < n; t0 += gridDim.x * TILE) {
        const bool fin = n - t0 <= gridDim.x * TILE;  // the workgroup's last tile
        bool live[NP];
        uint32_t id[NP];
        int route[NP];
#pragma unroll
        for (int j = 0; j < NP; j++) {
            const uint32_t i = t0 + (uint32_t)j * BS + threadIdx.x;
            live[j] = i < n;
            id[j] = live[j] ? queue[i] : 0u;
        }
        if (iter > 1) {
#pragma unroll
            for (int j = 0; j < NP; j++) {
                const int type = live[j] ? __float_as_int(P.nee[3 * id[j] + 2].w) : -1;
#pragma unroll
                for (int t = 0; t < 3; t++) lds_append(done[t], &ended[t], type == t, id[j]);
            }
            __syncthreads();
            uint32_t chunks[3], total = 0;
#pragma unroll
            for (int t = 0; t < 3; t++) {
                chunks[t] = ((uint32_t)__builtin_amdgcn_readfirstlane((int)ended[t]) + 63u) / 64u;
                total += chunks[t];
            }
            for (uint32_t w = wave; w < total; w += BS / 64) {
                uint32_t k = w, t = 0;
#pragma unroll
                for (uint32_t u = 0; u < 2; u++)
                    if (t == u && k >= chunks[u]) {
                        k -= chunks[u];
                        t = u + 1;
                    }
                const uint32_t i = k * 64u + lane;
                const bool on = i < (uint32_t)__builtin_amdgcn_readfirstlane((int)ended[t]);
                const uint32_t pid = on ? done[t][i] : 0u;
                switch (t) {
                    case MAT_MIX: replay_gradients<MAT_MIX, UNI>(P, S, on, pid); break;
                    case MAT_DIFFUSE: replay_gradients<MAT_DIFFUSE, UNI>(P, S, on, pid); break;
                    default: replay_gradients<MAT_CONDUCTOR, UNI>(P, S, on, pid); break;
                }
            }
            __syncthreads();  // (the records that other waves have finished are read next)
            if (threadIdx.x < 3) ended[threadIdx.x] = 0u;
        }
#pragma unroll
        for (int j = 0; j < NP; j++) route[j] = replay_logic<UNI>(P, S, live[j], id[j], cnt);
        if (last) {
            __syncthreads();
            continue;
        }
#pragma unroll
        for (int j = 0; j < NP; j++)
#pragma unroll
            for (int t = 0; t < 4; t++) lds_append(list[t], &fill[t], route[j] == t, id[j]);
#pragma unroll
        for (int j = 0; j < NP; j++) {
            const uint64_t m = __ballot(route[j] >= 0);
            if (lane == 0) live_in[j][wave] = (uint32_t)__popcll(m);
        }
        __syncthreads();
        place_in_order<NP, BS>(ext, n_ext, live_in, wave, route, id);
        uint32_t chunks[4], total = 0;
#pragma unroll
        for (int t = 0; t < 4; t++) {
            const uint32_t have = (uint32_t)__builtin_amdgcn_readfirstlane((int)fill[t]);
            chunks[t] = fin ? (have + 63u) / 64u : have / 64u;
            total += chunks[t];
        }
        for (uint32_t w = wave; w < total; w += BS / 64) {
            uint32_t k = w, t = 0;
#pragma unroll
            for (uint32_t u = 0; u < 3; u++)
                if (t == u && k >= chunks[u]) {
                    k -= chunks[u];
                    t = u + 1;
                }
            const uint32_t have = (uint32_t)__builtin_amdgcn_readfirstlane((int)fill[t]);
            const uint32_t i = (fin ? 0u : have & 63u) + k * 64u + lane;
            const bool on = i < have;
            const uint32_t pid = on ? list[t][i] : 0u;
            uint32_t shadow = 0;
            bool need = false;
            if (on) {
                switch (t) {
                    case MAT_MIX: need = replay_rays<MAT_MIX, UNI>(P, pid, shadow); break;
                    case MAT_DIFFUSE: need = replay_rays<MAT_DIFFUSE, UNI>(P, pid, shadow); break;
                    case MAT_CONDUCTOR: need = replay_rays<MAT_CONDUCTOR, UNI>(P, pid, shadow); break;
                    default: need = replay_rays<MAT_DIELECTRIC, UNI>(P, pid, shadow); break;
                }
            }
            lds_append(shd, &n_shd, need, shadow);
        }
        __syncthreads();
        if (threadIdx.x < 4) fill[threadIdx.x] = fin ? 0u : fill[threadIdx.x] & 63u;
        if (fin || n_ext + TILE > CAP || n_shd + ADD > CAP) flush_entries<BS>(P, q, ext, n_ext, shd, n_shd, base);
        __syncthreads();
    }
    add_counts(P, cnt);
}

// Adjoint-mode converter: fixed-point sums -> caller's float gradients.
__global__ void k_fixed_to_float(const unsigned long long* fx, const uint32_t* mx, const uint32_t* cnt,
                                 uint64_t n, float* out) {
    for (uint64_t i = gtid(); i < n; i += gstride()) {
        long long v = (long long)fx[i];
        if (v == 0) continue;
        int e = fixed_exponent(mx[i], cnt[i]);
        out[i] += (float)ldexp((double)v, -e);
    }
}

// ============================================================ film layers
__global__ void k_fill4(float4* p, uint32_t n) {
    for (uint32_t i = gtid(); i < n; i += gstride()) p[i] = make_float4(0.f, 0.f, 0.f, 0.f);
}
__global__ void k_fill_u32(uint32_t* p, uint64_t n) {
    for (uint64_t i = gtid(); i < n; i += gstride()) p[i] = 0u;
}
// film[pixel] += sum over layers k (in k order) of layers[k*WH + pixel]
__global__ void k_resolve_layers(const float4* layers, uint32_t K, uint32_t WH, float4* film) {
    for (uint32_t p = gtid(); p < WH; p += gstride()) {
        float4 s = layers[p];
        for (uint32_t k = 1; k < K; k++) {
            float4 l = layers[(size_t)k * WH + p];
            s.x = s.x + l.x; s.y = s.y + l.y; s.z = s.z + l.z; s.w = s.w + l.w;
        }
        float4 f = film[p];
        film[p] = make_float4(f.x + s.x, f.y + s.y, f.z + s.z, f.w + s.w);
    }
}

// ======================================================== standalone stages
struct TraceArgs {  // one ff_trace_closest / ff_trace_any call
    ff_dev_scene S;
    const float4* rays;
    uint32_t n;
    float4* hits;
    uint8_t* occ;
    int two_sided;
    uint32_t* fetch;
    int32_t* ovf;
    unsigned long long* counts;
};
template <int BS, int LDS, int RF, int WW, bool WIDE>
__global__ __launch_bounds__(BS, (WW == 0 && !WIDE && LDS <= 16 && BS >= 128) ? 7 : 1) void k_trace_closest(
    TraceArgs a) {
    __shared__ int smem[LDS * BS + 3 * BS];  // stack, then the hit words
    RaySrc src{a.S, a.rays, a.hits, nullptr, a.two_sided};
    trav_persistent<BS, LDS, RF, false, WW, WIDE>(src, a.n, a.fetch, a.ovf, a.counts, smem);
}
template <int BS, int LDS, int RF, int WW, bool WIDE>
__global__ __launch_bounds__(BS) void k_trace_any(TraceArgs a) {
    __shared__ int smem[LDS * BS];
    RaySrc src{a.S, a.rays, nullptr, a.occ, 0};
    trav_persistent<BS, LDS, RF, true, WW, WIDE>(src, a.n, a.fetch, a.ovf, a.counts, smem);
}
__global__ __launch_bounds__(TW_BLOCK, TW_OCC) void k_trace_closest_wide(TraceArgs a) {
    __shared__ int smem[TW_LDS_CLOSEST];
    RaySrc src{a.S, a.rays, a.hits, nullptr, a.two_sided};
    traverse<false>(src, a.n, blockIdx.x, gridDim.x, quad_fits(a.S.wide_levels, a.S.max_depth), a.fetch, a.ovf, nullptr, nullptr, smem);
}
__global__ __launch_bounds__(TW_BLOCK, TW_OCC) void k_trace_any_wide(TraceArgs a) {
    __shared__ int smem[TW_LDS_ANY];
    RaySrc src{a.S, a.rays, nullptr, a.occ, 0};
    traverse<true>(src, a.n, blockIdx.x, gridDim.x, quad_fits(a.S.wide_levels, a.S.max_depth), a.fetch, a.ovf, nullptr, nullptr, smem);
}
__global__ void k_gen_rays(ff_dev_camera cam, int32_t W, int32_t H, uint32_t seed, uint32_t sample,
                           float4* rays) {
    uint32_t WH = (uint32_t)W * (uint32_t)H;
    for (uint32_t pix = gtid(); pix < WH; pix += gstride()) {
        f3 o, d;
        gen_ray(cam, W, H, (int)(pix % (uint32_t)W), (int)(pix / (uint32_t)W), rng_base(seed, pix, sample), o, d);
        rays[2 * pix] = f4(o, 0.f);
        rays[2 * pix + 1] = f4(d, 0.f);
    }
}

// ========================================================= environment CDF
// FP64 CDF build replacing the serial <<<1,1>>> passes of
// g_compute_pdf_denom / g_compute_marginal_dist / g_compute_conditional_dist /
// g_write_pdf_texture (CRT/kernel.cu:65-149).  Same per-texel terms; sums are
// fixed-order tree reductions and blocked scans (deterministic, FP64).  Three
// launches: rows, conditionals (with denom, guides, pdf and render-time
// texels), marginal; 48 us for 2048 x 1024 texels, where about 100 MB have to
// move (22 us); with every part a launch of its own (seven) it took 105 us.
__device__ __forceinline__ double block_sum(double v, double* red) {
    red[threadIdx.x] = v;
    __syncthreads();
    for (int s = FF_BLOCK / 2; s > 0; s >>= 1) {
        if ((int)threadIdx.x < s) red[threadIdx.x] = red[threadIdx.x] + red[threadIdx.x + s];
        __syncthreads();
    }
    double r = red[0];
    __syncthreads();
    return r;
}

// One workgroup per row: the row's luminances, and
// row_sum[j] = sum_i lum(i,j) * sin_theta_j
__global__ __launch_bounds__(FF_BLOCK) void k_env_rows(const float* rgb, int32_t w, int32_t h, float* lum,
                                                       double* row_sum) {
    __shared__ double red[FF_BLOCK];
    int j = blockIdx.x;
    float v = (float)j / (float)h;
    double st = (double)f_sin(F_PI * v);
    double acc = 0.0;
    for (int i = threadIdx.x; i < w; i += FF_BLOCK) {
        float s[3];
        bilinear(rgb, w, h, 3, (float)i / (float)w, v, s);
        const float l = lum_of(s);
        lum[(size_t)j * w + i] = l;
        acc += (double)l * st;
    }
    double s = block_sum(acc, red);
    if (threadIdx.x == 0) row_sum[j] = s;
}

// Guide table of an environment's inverse-CDF search, formed with the list
// itself.  Entry g is the upper bound of g / ENV_GUIDE (first element greater,
// compared in double as the sampler compares), so the upper bound of any val
// in [g, g+1) / ENV_GUIDE lies in [entry g, entry g+1].  In a list that never
// decreases, element x + 1 is the upper bound from the first entry that is not
// below element x on: every element marks that entry, and the running maximum
// of the marks is the table.  (A search of the list for each of 4097 entries of
// 1024 rows of 2048 took 39 us; letting each element's thread write all its
// entries takes as long as the brightest texel has entries: 93 us for a whole
// build's rows.)  A list with a NaN or a decreasing step gets flagged entries
// (searched whole).  Every entry also carries list[0] != 0 and list[1] != 0
// (ENV_GUIDE_NZ0 / ENV_GUIDE_NZ1).
constexpr uint32_t GUIDE_PER = ENV_GUIDE / FF_BLOCK + 1;  // entries of a thread (odd: no bank conflicts)
static_assert(GUIDE_PER % 2 == 1 && GUIDE_PER * FF_BLOCK > ENV_GUIDE, "one run of entries for each thread");
struct CdfScan {  // of one workgroup
    double red[FF_BLOCK];
    uint32_t mark[GUIDE_PER * FF_BLOCK], wave[FF_BLOCK / 64];
    uint32_t nz;
};
// list[i] = the sum of term(0..i): thread t owns elements [t*c, (t+1)*c), the
// threads' sums are added up in order by one thread, eight loads at a time.
template <class Term>
__device__ __forceinline__ void cdf_scan(CdfScan& S, int size, Term term, double* list, uint32_t* guide) {
    const int c = (size + FF_BLOCK - 1) / FF_BLOCK;
    const int lo = threadIdx.x * c, hi = lo + c < size ? lo + c : size;
    double local = 0.0;
    int x = lo;
    for (; x + 4 <= hi; x += 4) {  // (four at a time: one wide load)
        double q[4];
#pragma unroll
        for (int k = 0; k < 4; k++) q[k] = term(x + k);
#pragma unroll
        for (int k = 0; k < 4; k++) local += q[k];
    }
    for (; x < hi; x++) local += term(x);
    S.red[threadIdx.x] = local;
    for (uint32_t g = threadIdx.x; g < GUIDE_PER * FF_BLOCK; g += FF_BLOCK) S.mark[g] = 0u;
    if (threadIdx.x == 0) S.nz = 0u;
    __syncthreads();
    if (threadIdx.x == 0) {
        double run = 0.0;
        for (int t = 0; t < FF_BLOCK; t += 8) {
            double q[8];
#pragma unroll
            for (int k = 0; k < 8; k++) q[k] = S.red[t + k];
#pragma unroll
            for (int k = 0; k < 8; k++) {
                S.red[t + k] = run;
                run += q[k];
            }
        }
    }
    __syncthreads();
    double run = S.red[threadIdx.x], head = 0.0;
    int bad = 0;
    uint32_t nz = 0u;
    auto element = [&](int i, double q) {  // adds q; the list's element i
        const double prev = run;
        run += q;
        if (i == lo) head = run;
        if (run != run || (i > lo && run < prev)) bad = 1;
        if (i < 2 && run != 0.0) nz |= i == 0 ? ENV_GUIDE_NZ0 : ENV_GUIDE_NZ1;
        const double e = ceil(run * (double)ENV_GUIDE);  // (the first entry not below the element; exact)
        if (e <= (double)ENV_GUIDE) atomicMax(&S.mark[e > 0.0 ? (int)e : 0], (uint32_t)i + 1u);
        return run;
    };
    x = lo;
    for (; x + 4 <= hi; x += 4) {
        double q[4];
#pragma unroll
        for (int k = 0; k < 4; k++) q[k] = term(x + k);
#pragma unroll
        for (int k = 0; k < 4; k++) q[k] = element(x + k, q[k]);
#pragma unroll
        for (int k = 0; k < 4; k++) list[x + k] = q[k];
    }
    for (; x < hi; x++) list[x] = element(x, term(x));
    if (nz) atomicOr(&S.nz, nz);
    __syncthreads();
    S.red[threadIdx.x] = run;  // the thread's last element
    __syncthreads();
    if (lo > 0 && lo < hi && head < S.red[threadIdx.x - 1]) bad = 1;
    // running maximum: of the thread's entries, of the wave's threads, of the waves
    uint32_t* const m = S.mark + threadIdx.x * GUIDE_PER;
    uint32_t top = 0u;
    for (uint32_t k = 0; k < GUIDE_PER; k++) {
        top = m[k] > top ? m[k] : top;
        m[k] = top;
    }
    const uint32_t lane = __lane_id(), w = threadIdx.x >> 6;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const uint32_t o = __shfl_up(top, off);
        if (lane >= (uint32_t)off && o > top) top = o;
    }
    if (lane == 63u) S.wave[w] = top;
    bad = __syncthreads_or(bad);
    uint32_t before = __shfl_up(top, 1);
    if (lane == 0u) before = 0u;
    for (uint32_t k = 0; k < w; k++) before = S.wave[k] > before ? S.wave[k] : before;
    for (uint32_t k = 0; k < GUIDE_PER; k++) m[k] = m[k] > before ? m[k] : before;
    __syncthreads();
    for (uint32_t g = threadIdx.x; g <= ENV_GUIDE; g += FF_BLOCK)
        guide[g] = (bad ? ENV_GUIDE_FULL : S.mark[g]) | S.nz;
}

// One workgroup per row: denom = the sum of the row sums, marginal_p[y] =
// sum_x lum * (sin_theta_y / denom) (g_compute_marginal_dist's term), then the
// row's conditional CDF (blocked scan of lum * sin_theta_y / (denom *
// marginal_p[y])) with its guide table, its pdf texels and its render-time
// texels (r, g, b, pdf).  Every workgroup forms denom itself (h values from the
// L2), which spares a launch of one workgroup.
__global__ __launch_bounds__(FF_BLOCK) void k_env_conditional(const float* rgb, const float* lum, int32_t w, int32_t h,
                                                              const double* row_sum, double* denom_out,
                                                              double* marg_p, double* conds, float* pdf,
                                                              uint32_t* guide_c, float4* rgbp) {
    __shared__ CdfScan S;
    int y = blockIdx.x;
    double acc = 0.0;
    for (int j = threadIdx.x; j < h; j += FF_BLOCK) acc += row_sum[j];
    const double denom = block_sum(acc, S.red);
    if (y == 0 && threadIdx.x == 0) *denom_out = denom;
    float v = (float)y / (float)h;
    double st = (double)f_sin(F_PI * v);
    const float* row = lum + (size_t)y * w;
    double stn = st / denom;
    double mp = 0.0;
    float scale = (float)(w * h) / (2.f * F_PI * F_PI);
    for (int x = threadIdx.x; x < w; x += FF_BLOCK) {
        const float l = row[x];
        mp += (double)l * stn;
        float p = (float)(((double)l * st) / denom);
        p *= scale;
        const size_t k = (size_t)y * w + x;
        pdf[k] = p;
        rgbp[k] = make_float4(rgb[3 * k], rgb[3 * k + 1], rgb[3 * k + 2], p);
    }
    mp = block_sum(mp, S.red);
    if (threadIdx.x == 0) marg_p[y] = mp;
    const double val = st / (denom * mp);
    cdf_scan(S, w, [&](int x) { return (double)row[x] * val; }, conds + (size_t)y * w,
             guide_c + (size_t)y * (ENV_GUIDE + 1));
}

// single workgroup: marginal_y = inclusive scan of marginal_p, and its guide table
__global__ __launch_bounds__(FF_BLOCK) void k_env_marginal(const double* marg_p, int32_t h, double* marg_y,
                                                           uint32_t* guide_m) {
    __shared__ CdfScan S;
    cdf_scan(S, h, [&](int j) { return marg_p[j]; }, marg_y, guide_m);
}

// ============================================================ film resolve
// Resolve of wf_logic (CRT/kernel.cu:447-454): average, exposure, Reinhard,
// (int)(255*c) per channel.
__global__ void k_film_resolve(const float4* film, uint32_t n, float exposure, float* avg, uint8_t* rgba) {
    for (uint32_t p = gtid(); p < n; p += gstride()) {
        float4 f = film[p];
        float cnt = f.w;
        float r = 0.f, g = 0.f, b = 0.f;
        if (cnt >= 1.f) { r = f.x / cnt; g = f.y / cnt; b = f.z / cnt; }
        if (avg) { avg[3 * p] = r; avg[3 * p + 1] = g; avg[3 * p + 2] = b; }
        if (rgba) {
            float cr = r * exposure, cg = g * exposure, cb = b * exposure;
            cr = cr / (cr + 1.f); cg = cg / (cg + 1.f); cb = cb / (cb + 1.f);
            rgba[4 * p] = (uint8_t)(int)(255 * cr);
            rgba[4 * p + 1] = (uint8_t)(int)(255 * cg);
            rgba[4 * p + 2] = (uint8_t)(int)(255 * cb);
            rgba[4 * p + 3] = 255;
        }
    }
}

inline uint32_t grid_for(uint64_t n, uint32_t cap) {
    uint64_t g = (n + FF_BLOCK - 1) / FF_BLOCK;
    if (g < 1) g = 1;
    return (uint32_t)(g < cap ? g : cap);
}

// Workgroups of a traversal kernel that the current device keeps resident:
// CUs x blocks per CU at the kernel's occupancy, capped so every lane has its
// overflow stack column.  Cached per (kernel, device).
template <class K>
uint32_t resident_grid(K kernel, int bs) {
    static std::mutex mu;
    static std::map<std::pair<const void*, int>, uint32_t> cache;
    int dev = 0;
    (void)hipGetDevice(&dev);
    std::lock_guard<std::mutex> lock(mu);
    auto key = std::make_pair((const void*)kernel, dev);
    auto it = cache.find(key);
    if (it != cache.end()) return it->second;
    int nb = 0, cus = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, kernel, bs, 0) != hipSuccess || nb < 1) nb = 1;
    if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus < 1) cus = 1;
    uint64_t g = (uint64_t)nb * (uint64_t)cus, cap = FF_TRAV_THREADS / bs;
    if (g > cap) g = cap;
    cache[key] = (uint32_t)g;
    return (uint32_t)g;
}

// Workgroups of a wide traversal launch of at most n_max rays a queue: the
// resident ones, or as many as such a launch spreads its rays over.
template <class K>
uint32_t traverse_grid(K kernel, uint32_t n_max) {
    const uint32_t res = resident_grid(kernel, TW_BLOCK);
    auto waves = [&](uint32_t spread, uint32_t rays) {
        uint32_t per = n_max / spread + 1 < rays ? n_max / spread + 1 : rays;
        return n_max / per + 1;
    };
    uint32_t w = waves(TW_SPREAD, 64);
    if (n_max <= QUAD_MAX && waves(QUAD_SPREAD, 16) > w) w = waves(QUAD_SPREAD, 16);
    const uint32_t g = (w + TW_BLOCK / 64 - 1) / (TW_BLOCK / 64);
    return g < res ? g : res;
}

// counted traversal variants (block size, LDS stack entries, refill threshold, loop
// shape 0-4, BVH record width)
#define FF_TRAV_VARIANT_LIST(X)  \
    X(0, 256, 16, 32, 0, false)  \
    X(1, 256, 16, 16, 0, false)  \
    X(2, 256, 16, 64, 0, false)  \
    X(3, 128, 16, 32, 0, false)  \
    X(4, 256, 8, 32, 0, false)   \
    X(5, 256, 24, 32, 0, false)  \
    X(6, 64, 32, 32, 0, false)   \
    X(7, 128, 24, 32, 0, false)  \
    X(8, 256, 16, 32, 1, false)  \
    X(9, 64, 32, 32, 1, false)   \
    X(10, 256, 16, 16, 1, false) \
    X(11, 128, 24, 32, 1, false) \
    X(12, 256, 16, 64, 0, true)  \
    X(13, 256, 16, 32, 0, true)  \
    X(14, 64, 32, 32, 0, true)   \
    X(15, 256, 16, 32, 1, true)  \
    X(16, 256, 16, 64, 2, false) \
    X(17, 256, 16, 32, 2, false) \
    X(18, 256, 16, 8, 0, false)  \
    X(19, 256, 24, 16, 0, false) \
    X(20, 256, 16, 16, 3, false) \
    X(21, 256, 16, 32, 3, false) \
    X(22, 256, 16, 16, 5, false) \
    X(23, 256, 16, 32, 5, false) \
    X(24, 256, 16, 16, 6, false) \
    X(25, 256, 16, 16, 7, false) \
    X(26, 128, 16, 16, 5, false)

// which: 3 ff_trace_closest, 4 ff_trace_any
template <int BS, int LDS, int RF, int WW, bool WIDE>
hipError_t trav_launch(int which, const TraceArgs& T, hipStream_t s) {
    if (which == 3) {
        uint32_t g = resident_grid(k_trace_closest<BS, LDS, RF, WW, WIDE>, BS);
        hipLaunchKernelGGL((k_trace_closest<BS, LDS, RF, WW, WIDE>), dim3(g), dim3(BS), 0, s, T);
    } else {
        uint32_t g = resident_grid(k_trace_any<BS, LDS, RF, WW, WIDE>, BS);
        hipLaunchKernelGGL((k_trace_any<BS, LDS, RF, WW, WIDE>), dim3(g), dim3(BS), 0, s, T);
    }
    return hipGetLastError();
}

hipError_t trav_dispatch(int which, int variant, const TraceArgs& T, hipStream_t s) {
    switch (variant) {
#define FF_TRAV_CASE(v, bs, lds, rf, ww, wide) \
    case v: return trav_launch<bs, lds, rf, ww, wide>(which, T, s);
        FF_TRAV_VARIANT_LIST(FF_TRAV_CASE)
#undef FF_TRAV_CASE
        default: return hipErrorInvalidValue;
    }
}

}  // namespace

// ================================================== fixed trace scratch
// Device memory of ff_trace_closest_noalloc, the entry point for callers
// that cannot allocate (graph capture, serving loops): the traversal work
// counters (FETCH_WORDS words) followed by the stack overflow area
// (FF_STATIC_OVF_ENTRIES entries for each of the FF_TRAV_THREADS lanes a
// persistent traversal grid holds).  Every device the library runs on holds
// its own copy until the process ends; calls on one device share it, so such
// calls must not overlap there.  Host code uses the address from
// hipGetSymbolAddress, never the array's name.
static __device__ __align__(256) int32_t scratch[FETCH_WORDS + (size_t)FF_STATIC_OVF_ENTRIES * FF_TRAV_THREADS];

// ===================================================================== host
namespace ffk {

#define FF_TRAV_ONE(v, bs, lds, rf, ww, wide) +1
const int kTravVariants = 0 FF_TRAV_VARIANT_LIST(FF_TRAV_ONE);
#undef FF_TRAV_ONE
#define FF_TRAV_BS(v, bs, lds, rf, ww, wide) bs,
#define FF_TRAV_LDS(v, bs, lds, rf, ww, wide) lds,
#define FF_TRAV_RF(v, bs, lds, rf, ww, wide) rf,
#define FF_TRAV_WW(v, bs, lds, rf, ww, wide) ww,
#define FF_TRAV_WIDTH(v, bs, lds, rf, ww, wide) (wide ? 4 : 2),
const int kTravBlock[] = {FF_TRAV_VARIANT_LIST(FF_TRAV_BS)};
const int kTravLds[] = {FF_TRAV_VARIANT_LIST(FF_TRAV_LDS)};
const int kTravRefill[] = {FF_TRAV_VARIANT_LIST(FF_TRAV_RF)};
const int kTravWhileWhile[] = {FF_TRAV_VARIANT_LIST(FF_TRAV_WW)};
const int kTravWidth[] = {FF_TRAV_VARIANT_LIST(FF_TRAV_WIDTH)};
#undef FF_TRAV_BS
#undef FF_TRAV_LDS
#undef FF_TRAV_RF
#undef FF_TRAV_WW
#undef FF_TRAV_WIDTH

// every request of the call shades the same scene and environment
static bool uni_shading(const ff_paths& P) { return P.uni_scene && P.uni_env; }

hipError_t launch_begin(const ff_paths& P, const ff_begin& B, hipStream_t s) {
    hipLaunchKernelGGL(k_begin, dim3(1), dim3(FF_BLOCK), 0, s, P, B);
    return hipGetLastError();
}
hipError_t launch_batch_begin(const ff_paths& P, hipStream_t s) {
    hipLaunchKernelGGL(k_batch_begin, dim3(1), dim3(256), 0, s, P);
    return hipGetLastError();
}
hipError_t launch_generate(const ff_paths& P, hipStream_t s) {
    hipLaunchKernelGGL(k_generate, dim3(grid_for(P.n_slots, FF_GRID_CAP)), dim3(FF_BLOCK), 0, s, P);
    return hipGetLastError();
}
hipError_t launch_extend(const ff_paths& P, int q, hipStream_t s) {
    if (P.uni_scene)
        hipLaunchKernelGGL(k_extend<true>, dim3(traverse_grid(k_extend<true>, P.n_slots)), dim3(TW_BLOCK), 0, s, P, q);
    else
        hipLaunchKernelGGL(k_extend<false>, dim3(traverse_grid(k_extend<false>, P.n_slots)), dim3(TW_BLOCK), 0, s, P, q);
    return hipGetLastError();
}
hipError_t launch_shadow(const ff_paths& P, int q, hipStream_t s) {
    if (P.uni_scene)
        hipLaunchKernelGGL(k_shadow<true>, dim3(traverse_grid(k_shadow<true>, P.n_slots)), dim3(TW_BLOCK), 0, s, P, q);
    else
        hipLaunchKernelGGL(k_shadow<false>, dim3(traverse_grid(k_shadow<false>, P.n_slots)), dim3(TW_BLOCK), 0, s, P, q);
    return hipGetLastError();
}
template <bool UNI>
hipError_t extend_shadow_launch(const ff_paths& P, int q, hipStream_t s) {
    if (P.n_slots <= QUAD_MAX && P.quad) {
        const uint32_t g = (traverse_grid(k_extend_shadow_small<UNI>, P.n_slots) + 7u) / 8u * 16u;
        hipLaunchKernelGGL(k_extend_shadow_small<UNI>, dim3(g), dim3(TW_BLOCK), 0, s, P, q);
    } else {
        auto launch = [&](auto kernel) {
            const uint32_t g = std::min((traverse_grid(kernel, P.n_slots) + 7u) / 8u * 16u,
                                        std::max(resident_grid(kernel, TW_BLOCK) / 16u, 1u) * 16u);
            hipLaunchKernelGGL(kernel, dim3(g), dim3(TW_BLOCK), 0, s, P, q);
        };
        if (P.n_slots <= EXTEND_FEW) launch(k_extend_shadow<UNI, 5>);
        else if (P.n_slots < EXTEND_MANY) launch(k_extend_shadow<UNI, 6>);
        else launch(k_extend_shadow<UNI, 7>);
    }
    return hipGetLastError();
}
hipError_t launch_extend_shadow(const ff_paths& P, int q, hipStream_t s) {
    return P.uni_scene ? extend_shadow_launch<true>(P, q, s) : extend_shadow_launch<false>(P, q, s);
}
// One tile of 256 paths to a workgroup up to LOGIC_SHADE_SMALL paths in flight:
// the large form's resident workgroups take 524 k paths at once, and below that
// some CUs have none (256 k paths: 0.93 against 1.03 ms a render of glossy
// spheres, 1.41 against 1.55 ms of a textured scene; 512 k: 1.23
// against 1.19, 1.59 against 1.61).  Above it every workgroup's append waits its
// turn at two counters, and the large form appends runs of up to 4000 entries
// (4.7 M paths: 6.1 against 4.1 ms).
constexpr uint32_t LOGIC_SHADE_SMALL = 384 * 1024;
template <bool UNI>
constexpr auto k_logic_shade_small = k_logic_shade<UNI, 256, 256, 1, 256 + 4 * 63>;
template <bool UNI>
constexpr auto k_logic_shade_large = k_logic_shade<UNI, 512, 1024, 2, 4000>;
template <bool UNI>
hipError_t logic_shade_launch(const ff_paths& P, int q, int iter, int last, hipStream_t s) {
    if (P.n_slots <= LOGIC_SHADE_SMALL) {
        hipLaunchKernelGGL(k_logic_shade_small<UNI>, dim3((P.n_slots + 255u) / 256u), dim3(256), 0, s, P, q, iter, last);
    } else {
        const uint32_t g = std::min((P.n_slots + 1023u) / 1024u, resident_grid(k_logic_shade_large<UNI>, 512));
        hipLaunchKernelGGL(k_logic_shade_large<UNI>, dim3(g), dim3(512), 0, s, P, q, iter, last);
    }
    return hipGetLastError();
}
hipError_t launch_logic_shade(const ff_paths& P, int q, int iter, int last, hipStream_t s) {
    return uni_shading(P) ? logic_shade_launch<true>(P, q, iter, last, s) : logic_shade_launch<false>(P, q, iter, last, s);
}
// (the same limit: the large form's 768 resident workgroups take 384 k paths at once)
template <bool UNI>
constexpr auto k_replay_small = k_replay<UNI, 256, 256, 1, 256 + 4 * 63>;
template <bool UNI>
constexpr auto k_replay_large = k_replay<UNI, 256, 512, 2, 1792>;
template <bool UNI>
hipError_t replay_launch(const ff_paths& P, int q, int iter, int last, hipStream_t s) {
    if (P.n_slots <= LOGIC_SHADE_SMALL) {
        hipLaunchKernelGGL(k_replay_small<UNI>, dim3((P.n_slots + 255u) / 256u), dim3(256), 0, s, P, q, iter, last);
    } else {
        const uint32_t g = std::min((P.n_slots + 511u) / 512u, resident_grid(k_replay_large<UNI>, 256));
        hipLaunchKernelGGL(k_replay_large<UNI>, dim3(g), dim3(256), 0, s, P, q, iter, last);
    }
    return hipGetLastError();
}
hipError_t launch_replay(const ff_paths& P, int q, int iter, int last, hipStream_t s) {
    return uni_shading(P) ? replay_launch<true>(P, q, iter, last, s) : replay_launch<false>(P, q, iter, last, s);
}
void prepare_launches() {
    (void)resident_grid(k_extend<true>, TW_BLOCK);
    (void)resident_grid(k_extend<false>, TW_BLOCK);
    (void)resident_grid(k_shadow<true>, TW_BLOCK);
    (void)resident_grid(k_shadow<false>, TW_BLOCK);
    (void)resident_grid(k_extend_shadow<true, 5>, TW_BLOCK);
    (void)resident_grid(k_extend_shadow<false, 5>, TW_BLOCK);
    (void)resident_grid(k_extend_shadow<true, 6>, TW_BLOCK);
    (void)resident_grid(k_extend_shadow<false, 6>, TW_BLOCK);
    (void)resident_grid(k_extend_shadow<true, 7>, TW_BLOCK);
    (void)resident_grid(k_extend_shadow<false, 7>, TW_BLOCK);
    (void)resident_grid(k_extend_shadow_small<true>, TW_BLOCK);
    (void)resident_grid(k_extend_shadow_small<false>, TW_BLOCK);
    (void)resident_grid(k_logic_shade_large<true>, 512);
    (void)resident_grid(k_logic_shade_large<false>, 512);
    (void)resident_grid(k_replay_large<true>, 256);
    (void)resident_grid(k_replay_large<false>, 256);
}
template <bool UNI>
hipError_t logic_launch(const ff_paths& P, int q, int iter, uint32_t n_max, hipStream_t s) {
    hipLaunchKernelGGL(k_logic<UNI>, dim3(grid_for(n_max, FF_GRID_CAP)), dim3(FF_BLOCK), 0, s, P, q, iter);
    return hipGetLastError();
}
hipError_t launch_logic(const ff_paths& P, int q, int iter, uint32_t n_max, hipStream_t s) {
    return uni_shading(P) ? logic_launch<true>(P, q, iter, n_max, s) : logic_launch<false>(P, q, iter, n_max, s);
}
template <bool UNI>
hipError_t shade_launch(int type, const ff_paths& P, int next_q, int first, uint32_t n_max, hipStream_t s) {
    dim3 g(grid_for(n_max, FF_GRID_CAP)), b(FF_BLOCK);
    switch (type) {
        case MAT_MIX: hipLaunchKernelGGL((k_shade<MAT_MIX, UNI>), g, b, 0, s, P, next_q, first); break;
        case MAT_DIFFUSE: hipLaunchKernelGGL((k_shade<MAT_DIFFUSE, UNI>), g, b, 0, s, P, next_q, first); break;
        case MAT_CONDUCTOR: hipLaunchKernelGGL((k_shade<MAT_CONDUCTOR, UNI>), g, b, 0, s, P, next_q, first); break;
        default: hipLaunchKernelGGL((k_shade<MAT_DIELECTRIC, UNI>), g, b, 0, s, P, next_q, first); break;
    }
    return hipGetLastError();
}
hipError_t launch_shade(int type, const ff_paths& P, int next_q, int first, uint32_t n_max, hipStream_t s) {
    return uni_shading(P) ? shade_launch<true>(type, P, next_q, first, n_max, s)
                          : shade_launch<false>(type, P, next_q, first, n_max, s);
}
template <bool UNI>
hipError_t logic_adj_launch(const ff_paths& P, int q, uint32_t n_max, hipStream_t s) {
    hipLaunchKernelGGL(k_logic_adj<UNI>, dim3(grid_for(n_max, FF_GRID_CAP)), dim3(FF_BLOCK), 0, s, P, q);
    return hipGetLastError();
}
hipError_t launch_logic_adj(const ff_paths& P, int q, uint32_t n_max, hipStream_t s) {
    return uni_shading(P) ? logic_adj_launch<true>(P, q, n_max, s) : logic_adj_launch<false>(P, q, n_max, s);
}
template <bool UNI>
hipError_t shade_nee_launch(int type, const ff_paths& P, int next_q, uint32_t n_max, hipStream_t s) {
    dim3 g(grid_for(n_max, FF_GRID_CAP)), b(FF_BLOCK);
    switch (type) {
        case MAT_MIX: hipLaunchKernelGGL((k_shade_nee<MAT_MIX, UNI>), g, b, 0, s, P, next_q); break;
        case MAT_DIFFUSE: hipLaunchKernelGGL((k_shade_nee<MAT_DIFFUSE, UNI>), g, b, 0, s, P, next_q); break;
        case MAT_CONDUCTOR: hipLaunchKernelGGL((k_shade_nee<MAT_CONDUCTOR, UNI>), g, b, 0, s, P, next_q); break;
        default: hipLaunchKernelGGL((k_shade_nee<MAT_DIELECTRIC, UNI>), g, b, 0, s, P, next_q); break;
    }
    return hipGetLastError();
}
hipError_t launch_shade_nee(int type, const ff_paths& P, int next_q, uint32_t n_max, hipStream_t s) {
    return uni_shading(P) ? shade_nee_launch<true>(type, P, next_q, n_max, s)
                          : shade_nee_launch<false>(type, P, next_q, n_max, s);
}
template <bool UNI>
hipError_t shade_adj_launch(int type, const ff_paths& P, int q, uint32_t n_max, hipStream_t s) {
    dim3 g(grid_for(n_max, FF_GRID_CAP)), b(FF_BLOCK);
    switch (type) {
        case MAT_MIX: hipLaunchKernelGGL((k_shade_adj<MAT_MIX, UNI>), g, b, 0, s, P, q); break;
        case MAT_DIFFUSE: hipLaunchKernelGGL((k_shade_adj<MAT_DIFFUSE, UNI>), g, b, 0, s, P, q); break;
        case MAT_CONDUCTOR: hipLaunchKernelGGL((k_shade_adj<MAT_CONDUCTOR, UNI>), g, b, 0, s, P, q); break;
        default: break;  // a dielectric vertex ends with its rays
    }
    return hipGetLastError();
}
hipError_t launch_shade_adj(int type, const ff_paths& P, int q, uint32_t n_max, hipStream_t s) {
    return uni_shading(P) ? shade_adj_launch<true>(type, P, q, n_max, s)
                          : shade_adj_launch<false>(type, P, q, n_max, s);
}
hipError_t launch_fixed_to_float(const unsigned long long* fx, const uint32_t* mx, const uint32_t* cnt, uint64_t n,
                                 float* out, hipStream_t s) {
    hipLaunchKernelGGL(k_fixed_to_float, dim3(grid_for(n, FF_GRID_CAP)), dim3(FF_BLOCK), 0, s, fx, mx, cnt, n, out);
    return hipGetLastError();
}
hipError_t launch_fill4(float4* p, uint32_t n, hipStream_t s) {
    hipLaunchKernelGGL(k_fill4, dim3(grid_for(n, FF_GRID_CAP)), dim3(FF_BLOCK), 0, s, p, n);
    return hipGetLastError();
}
hipError_t launch_fill_u32(uint32_t* p, uint64_t n, hipStream_t s) {
    hipLaunchKernelGGL(k_fill_u32, dim3(grid_for(n, FF_GRID_CAP)), dim3(FF_BLOCK), 0, s, p, n);
    return hipGetLastError();
}
hipError_t launch_resolve_layers(const float4* layers, uint32_t K, uint32_t WH, float4* film, hipStream_t s) {
    hipLaunchKernelGGL(k_resolve_layers, dim3(grid_for(WH, FF_GRID_CAP)), dim3(FF_BLOCK), 0, s, layers, K, WH,
                       film);
    return hipGetLastError();
}
// a query's launch: its workgroups, after one that clears the work counters if
// it uses them
template <class K>
static hipError_t trace_wide(K kernel, const TraceArgs& T, uint32_t* fetch, hipStream_t s) {
    const uint32_t g = traverse_grid(kernel, T.n);
    if (!(T.n <= QUAD_MAX && quad_fits(T.S.wide_levels, T.S.max_depth) && quad_fixed(T.n, g * (TW_BLOCK / 64))))
        hipLaunchKernelGGL(k_reset_fetch, dim3(1), dim3(64), 0, s, fetch);
    hipLaunchKernelGGL(kernel, dim3(g), dim3(TW_BLOCK), 0, s, T);
    return hipGetLastError();
}
hipError_t launch_trace_closest(const ff_dev_scene& S, const float4* rays, uint32_t n, float4* hits,
                                int two_sided, uint32_t* fetch, int32_t* ovf, unsigned long long* counts,
                                int variant, hipStream_t s) {
    TraceArgs T{S, rays, n, hits, nullptr, two_sided, fetch + F_TRACE * FETCH_SEGS * FETCH_STRIDE, ovf, counts};
    if (!counts && S.wide) return trace_wide(k_trace_closest_wide, T, fetch, s);
    hipLaunchKernelGGL(k_reset_fetch, dim3(1), dim3(64), 0, s, fetch);
    return trav_dispatch(3, variant, T, s);
}
// Device address of `scratch` on `device` (looked up once per device, with
// that device current, by ff_context_create).
hipError_t static_scratch(int device, int32_t** out) {
    static std::mutex mu;
    static std::map<int, int32_t*> addr;
    std::lock_guard<std::mutex> lock(mu);
    *out = nullptr;
    auto it = addr.find(device);
    if (it != addr.end()) {
        *out = it->second;
        return hipSuccess;
    }
    int cur = -1;
    hipError_t e = hipGetDevice(&cur);
    if (e != hipSuccess) return e;
    if (cur != device && (e = hipSetDevice(device)) != hipSuccess) return e;
    void* p = nullptr;
    e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (cur != device) (void)hipSetDevice(cur);
    if (e != hipSuccess) return e;
    if (p == nullptr) return hipErrorInvalidSymbol;
    addr[device] = (int32_t*)p;
    *out = (int32_t*)p;
    return hipSuccess;
}
hipError_t launch_trace_any(const ff_dev_scene& S, const float4* rays, uint32_t n, uint8_t* occ, uint32_t* fetch,
                            int32_t* ovf, unsigned long long* counts, int variant, hipStream_t s) {
    TraceArgs T{S, rays, n, nullptr, occ, 0, fetch + F_TRACE * FETCH_SEGS * FETCH_STRIDE, ovf, counts};
    if (!counts && S.wide) return trace_wide(k_trace_any_wide, T, fetch, s);
    hipLaunchKernelGGL(k_reset_fetch, dim3(1), dim3(64), 0, s, fetch);
    return trav_dispatch(4, variant, T, s);
}
hipError_t launch_gen_rays(const ff_dev_camera& cam, int W, int H, uint32_t seed, uint32_t sample, float4* rays,
                           hipStream_t s) {
    hipLaunchKernelGGL(k_gen_rays, dim3(grid_for((uint64_t)W * H, FF_GRID_CAP)), dim3(FF_BLOCK), 0, s, cam, W, H,
                       seed, sample, rays);
    return hipGetLastError();
}
hipError_t launch_env_build(const float* rgb, int w, int h, float* lum, double* row_sum, double* denom,
                            double* marg_p, double* marg_y, double* conds, float* pdf, uint32_t* guide_m,
                            uint32_t* guide_c, float4* rgbp, hipStream_t s) {
    hipLaunchKernelGGL(k_env_rows, dim3(h), dim3(FF_BLOCK), 0, s, rgb, w, h, lum, row_sum);
    hipLaunchKernelGGL(k_env_conditional, dim3(h), dim3(FF_BLOCK), 0, s, rgb, lum, w, h, row_sum, denom, marg_p, conds,
                       pdf, guide_c, rgbp);
    hipLaunchKernelGGL(k_env_marginal, dim3(1), dim3(FF_BLOCK), 0, s, marg_p, h, marg_y, guide_m);
    return hipGetLastError();
}
hipError_t launch_film_resolve(const float4* film, uint32_t n, float exposure, float* avg, uint8_t* rgba,
                               hipStream_t s) {
    hipLaunchKernelGGL(k_film_resolve, dim3(grid_for(n, FF_GRID_CAP)), dim3(FF_BLOCK), 0, s, film, n, exposure,
                       avg, rgba);
    return hipGetLastError();
}

}  // namespace ffk
