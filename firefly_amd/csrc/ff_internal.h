// ff_internal.h -- host-side declarations shared by the C ABI implementation,
// the host BVH builder and the kernel launchers.  Not part of the public ABI.
#pragma once

#include <functional>
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <vector>

#include "ff_layout.h"

namespace ffk {
extern const int kTravVariants;
extern const int kTravLds[];
extern const int kTravBlock[];
extern const int kTravRefill[];
extern const int kTravWhileWhile[];
extern const int kTravWidth[];  // BVH record width of the variant (2 or 4)
// computes the grid sizes of the wavefront's resident kernels (call before a graph capture)
void prepare_launches();
hipError_t launch_begin(const ff_paths& P, const ff_begin& B, hipStream_t s);
hipError_t launch_batch_begin(const ff_paths& P, hipStream_t s);
hipError_t launch_generate(const ff_paths& P, hipStream_t s);
hipError_t launch_extend(const ff_paths& P, int q, hipStream_t s);
hipError_t launch_shadow(const ff_paths& P, int q, hipStream_t s);
hipError_t launch_replay(const ff_paths& P, int q, int iter, int last, hipStream_t s);
hipError_t launch_logic_shade(const ff_paths& P, int q, int iter, int last, hipStream_t s);
hipError_t launch_extend_shadow(const ff_paths& P, int q, hipStream_t s);
hipError_t launch_logic(const ff_paths& P, int q, int iter, uint32_t n_max, hipStream_t s);
hipError_t launch_shade(int type, const ff_paths& P, int next_q, int first, uint32_t n_max, hipStream_t s);
hipError_t launch_logic_adj(const ff_paths& P, int q, uint32_t n_max, hipStream_t s);
hipError_t launch_shade_nee(int type, const ff_paths& P, int next_q, uint32_t n_max, hipStream_t s);
hipError_t launch_shade_adj(int type, const ff_paths& P, int q, uint32_t n_max, hipStream_t s);
hipError_t launch_fixed_to_float(const unsigned long long* fx, const uint32_t* mx, const uint32_t* cnt, uint64_t n,
                                 float* out, hipStream_t s);
hipError_t launch_fill4(float4* p, uint32_t n, hipStream_t s);
hipError_t launch_fill_u32(uint32_t* p, uint64_t n, hipStream_t s);
hipError_t launch_resolve_layers(const float4* layers, uint32_t K, uint32_t WH, float4* film, hipStream_t s);
hipError_t launch_trace_closest(const ff_dev_scene& S, const float4* rays, uint32_t n,
                                float4* hits, int two_sided, uint32_t* fetch, int32_t* ovf,
                                unsigned long long* counts, int variant, hipStream_t s);
hipError_t launch_trace_any(const ff_dev_scene& S, const float4* rays, uint32_t n, uint8_t* occ,
                            uint32_t* fetch, int32_t* ovf, unsigned long long* counts, int variant,
                            hipStream_t s);
// device address of the fixed trace scratch on `device` (FETCH_WORDS work
// counter words, then FF_STATIC_OVF_ENTRIES * FF_TRAV_THREADS overflow entries)
hipError_t static_scratch(int device, int32_t** out);
hipError_t launch_gen_rays(const ff_dev_camera& cam, int W, int H, uint32_t seed,
                           uint32_t sample, float4* rays, hipStream_t s);
hipError_t launch_env_build(const float* rgb, int w, int h, float* lum, double* row_sum,
                            double* denom, double* marg_p, double* marg_y, double* conds,
                            float* pdf, uint32_t* guide_m, uint32_t* guide_c, float4* rgbp,
                            hipStream_t s);
hipError_t launch_film_resolve(const float4* film, uint32_t n, float exposure, float* avg,
                               uint8_t* rgba, hipStream_t s);
}  // namespace ffk

namespace ffh {
// 32-byte node as stored in HBM (CRT/BVH.h:63-72 field order).
struct BvhNode {
    float bmin[3];
    float bmax[3];
    int32_t offset;
    uint16_t n_prims;
    uint8_t axis;
    uint8_t pad;
};
static_assert(sizeof(BvhNode) == 32, "BVH node must stay 32 bytes");

// SAH BVH over triangles (positions [n][3][3]); returns nodes in flattened
// depth-first order and the slot -> triangle permutation.
void build_bvh_sah(const float* positions, int32_t n, int32_t max_prims,
                   std::vector<BvhNode>& nodes, std::vector<int32_t>& ordered);
int32_t bvh_max_depth(const std::vector<BvhNode>& nodes);
}  // namespace ffh

namespace ffk {
// Pieces of one device allocation: take() them all with base null for the
// size, allocate, and take() them again.
struct Carver {
    char* base = nullptr;
    size_t off = 0;
    template <class T>
    T* take(size_t n) {
        T* p = (T*)(base + off);
        off += (n * sizeof(T) + 255) / 256 * 256;
        return p;
    }
};

// A binary tree on the device, in the SAH builder's node format; `mem` is the
// one allocation that holds it.
struct DevBvh {
    void* mem = nullptr;
    ffh::BvhNode* nodes = nullptr;
    int32_t* ordered = nullptr;
    float* pos = nullptr;  // [n][3][3], the caller's order
    int32_t n_nodes = 0, max_depth = 0, max_leaf = 1;
};
// Linear BVH on the GPU (Morton order, Karras hierarchy); positions on the
// host (gpu_ms, if given: device time of the build kernels; meanwhile: host
// work to do while the GPU builds).
hipError_t build_lbvh(const float* positions, int32_t n, int32_t max_prims, DevBvh& out, float* gpu_ms = nullptr,
                      const std::function<void()>& meanwhile = nullptr);
// PLOC tree on the GPU (locally-ordered clustering of the Morton-sorted
// triangles, SAH leaf collapse), same arguments.
hipError_t build_ploc(const float* positions, int32_t n, int32_t max_prims, DevBvh& out, float* gpu_ms = nullptr,
                      const std::function<void()>& meanwhile = nullptr);
// A host tree and its positions on the device.
hipError_t upload_bvh(const std::vector<ffh::BvhNode>& nodes, const std::vector<int32_t>& ordered, int32_t max_depth,
                      const float* positions, DevBvh& out);

// Host arrays of a scene that packing reads (uv, tan may be null).
struct SceneArrays {
    const float *nrm, *uv, *tan, *mats;
    const int32_t* mid;
    int32_t n, n_mats;
};
// A scene's traversal and shading arrays, in one allocation (`mem`).
struct ScenePack {
    void* mem = nullptr;
    float4 *nodes = nullptr, *nodes4 = nullptr, *wide = nullptr, *attr = nullptr;
    int32_t* leaf_count = nullptr;
    float *root = nullptr, *tris = nullptr, *tan = nullptr, *mats = nullptr;
    uint32_t* mat = nullptr;
    int32_t wide_levels = 0;
};
// Packing's scratch, which holds the uploaded arrays (`mem`: one allocation;
// pack_scene frees it).
struct PackScratch {
    void *mem = nullptr, *q0 = nullptr, *q1 = nullptr;
    uint32_t* rank = nullptr;
    float *nrm = nullptr, *uv = nullptr, *tan = nullptr;
    int32_t* mid = nullptr;
    char* scan_tmp = nullptr;
};
hipError_t upload_arrays(const SceneArrays& a, PackScratch& tmp);
hipError_t pack_scene(const DevBvh& bvh, const SceneArrays& a, PackScratch& tmp, ScenePack& out);
}  // namespace ffk
