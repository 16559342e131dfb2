// ff_device.h -- device math, RNG, BSDF lobes, environment light and BVH
// traversal for the gfx950 wavefront path tracer.
//
// Every routine restates a reference routine (JakeKurtz/Firefly,
// CUDA-RayTracer/ = CRT/) cited beside it.  The whole library is compiled
// with -ffp-contract=off so each float/double operation is rounded on its own
// as the reference's arithmetic is written; the traversal results are
// therefore bit-identical to a host evaluation of the same expressions.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "ff_layout.h"
#include "ff_refill.h"

namespace ffd {

// ------------------------------------------------------------ constants --
// Float constants as the reference declares them (CRT/dMath.cuh:78-128).
constexpr float F_PI = 3.14159265358979323846f;
constexpr float F_2PI = 6.28318530717958647692f;
constexpr float F_PI_2 = 1.57079632679489661923f;
constexpr float F_PI_4 = 0.785398163397448309615f;
constexpr float F_1_PI = 0.318309886183790671538f;
constexpr float F_1_2PI = 0.159154943091895335769f;
constexpr float K_EPS = 1e-6f;
constexpr float K_HUGE = 1e32f;

// RNG dimensions: bounce 0 is the camera, bounce L the L-th path vertex.
enum : uint32_t {
    DIM_JX = 0, DIM_JY = 1, DIM_LX = 2, DIM_LY = 3,
    DIM_RR = 0, DIM_EX = 1, DIM_EY = 2, DIM_S0 = 3, DIM_S1 = 4,
    DIM_D0 = 5, DIM_D1 = 6, DIM_LOBE = 7, DIM_DIEL = 8
};

// Conservative distance pruning added to the reference traversal (which
// tests every box the ray's line crosses).  Order of visits is unchanged, so
// the first closest candidate is the same triangle the reference returns.
constexpr float PRUNE_REL = 0x1p-12f;
constexpr float PRUNE_ABS = 1e-6f;
constexpr float PRUNE_BEHIND = 1e-4f;
// TravRay::negm flag: 1/d.x or o.x is not finite, so a slab's x distance can be NaN
constexpr uint32_t XNAN_RAY = 8u;

// Transcendentals are evaluated in double and rounded to float: the CUDA
// math library of the reference is closed.  The double routines below are
// this project's own, and the host oracle evaluates the same operations in
// the same order, so host and device agree bit for bit; they are within a
// few ulp of the C library in double, so after rounding to float they nearly
// always equal the correctly rounded value.  They need far fewer registers
// and instructions than general library routines (one division per atan2).
// Every sin/cos argument of a render is an angle of at most 2 pi or a NaN.
//
// sin and cos: Cody-Waite reduction modulo pi/2 with a three-part split of
// pi/2 (33 + 33 + 53 bits, so k * part is exact for |k| < 2^20), then the
// Taylor series of sin to r^17 and of cos to r^18 on |r| <= pi/4 (first
// omitted terms below 1e-19; coefficients 1/n! rounded to double).  For
// |x| < 2^19 (the host's routine gives larger arguments to the C library).
// One straight line without branches, so that the sine and the cosine of one
// angle, asked for separately, share the work: with a branch for zero and an
// out-of-line call for large arguments the compiler evaluated each anew, and
// the call's frame (48 B of scratch, 16 more registers) was paid by every
// shading kernel.  Together with one sph_map a direction this took the
// double-precision instructions of a diffuse event from 1381 to 850 and the
// shading of a 256x256 16-sample glossy render from 0.55 to 0.47 ms.
__device__ __forceinline__ void sincos_d(double x, double& s, double& c) {
    double kf = rint(x * 0x1.45f306dc9c883p-1);  // x * 2/pi
    int q = (int)kf & 3;
    double r = ((x - kf * 0x1.921fb544p+0) - kf * 0x1.0b4611a6p-34) - kf * 0x1.3198a2e037073p-69;
    double z = r * r;
    double ps = 0x1.952c77030ad4ap-49;
    ps = -0x1.ae7f3e733b81fp-41 + z * ps;
    ps = 0x1.6124613a86d09p-33 + z * ps;
    ps = -0x1.ae64567f544e4p-26 + z * ps;
    ps = 0x1.71de3a556c734p-19 + z * ps;
    ps = -0x1.a01a01a01a01ap-13 + z * ps;
    ps = 0x1.1111111111111p-7 + z * ps;
    ps = -0x1.5555555555555p-3 + z * ps;
    double pc = -0x1.6827863b97d97p-53;
    pc = 0x1.ae7f3e733b81fp-45 + z * pc;
    pc = -0x1.93974a8c07c9dp-37 + z * pc;
    pc = 0x1.1eed8eff8d898p-29 + z * pc;
    pc = -0x1.27e4fb7789f5cp-22 + z * pc;
    pc = 0x1.a01a01a01a01ap-16 + z * pc;
    pc = -0x1.6c16c16c16c17p-10 + z * pc;
    pc = 0x1.5555555555555p-5 + z * pc;
    pc = -0.5 + z * pc;
    double sr = r + (r * z) * ps, cr = 1.0 + z * pc;
    s = q == 0 ? sr : (q == 1 ? cr : (q == 2 ? -sr : -cr));
    if (x == 0.0) s = x;  // keeps the sign of a zero
    c = q == 0 ? cr : (q == 1 ? -sr : (q == 2 ? -cr : sr));
}
// atan on [0, 1]: above tan(pi/12) the addition formula
// atan t = pi/6 + atan((t*sqrt3 - 1)/(t + sqrt3)); then the Taylor series to
// u^27 on |u| <= tan(pi/12) (first omitted term below 1e-18; coefficients
// (-1)^n/(2n+1) rounded to double).
__device__ __forceinline__ double atan_unit(double t) {
    bool shift = t > 0x1.126145e9ecd56p-2;
    double u = shift ? (t * 0x1.bb67ae8584caap+0 - 1.0) / (t + 0x1.bb67ae8584caap+0) : t;
    double z = u * u;
    double p = -0x1.2f684bda12f68p-5;
    p = 0x1.47ae147ae147bp-5 + z * p;
    p = -0x1.642c8590b2164p-5 + z * p;
    p = 0x1.8618618618618p-5 + z * p;
    p = -0x1.af286bca1af28p-5 + z * p;
    p = 0x1.e1e1e1e1e1e1ep-5 + z * p;
    p = -0x1.1111111111111p-4 + z * p;
    p = 0x1.3b13b13b13b14p-4 + z * p;
    p = -0x1.745d1745d1746p-4 + z * p;
    p = 0x1.c71c71c71c71cp-4 + z * p;
    p = -0x1.2492492492492p-3 + z * p;
    p = 0x1.999999999999ap-3 + z * p;
    p = -0x1.5555555555555p-2 + z * p;
    double r = u + (u * z) * p;
    return shift ? 0x1.0c152382d7366p-1 + r : r;
}
// atan: odd symmetry; |x| > 1 by atan x = pi/2 - atan(1/x)
__device__ __forceinline__ double atan_d(double x) {
    if (x != x) return x;
    double a = fabs(x);
    bool inv = a > 1.0;
    double r = atan_unit(inv ? 1.0 / a : a);
    if (inv) r = 0x1.921fb54442d18p+0 - r;
    return copysign(r, x);
}
// atan2 with the C library's conventions for zeros, signs and infinities:
// theta = atan(min/max) of the magnitudes (one division), reflected to
// pi/2 - theta above the diagonal and to pi - theta for x < 0, signed by y
__device__ __forceinline__ double atan2_d(double y, double x) {
    if (y != y || x != x) return x + y;
    double a = fabs(y), b = fabs(x);
    if (isinf(a) || isinf(b)) {
        double t = isinf(a) ? (isinf(b) ? (x > 0.0 ? 0x1.921fb54442d18p-1 : 0x1.2d97c7f3321d2p+1)
                                        : 0x1.921fb54442d18p+0)
                            : (x > 0.0 ? 0.0 : 0x1.921fb54442d18p+1);
        return copysign(t, y);
    }
    if (b == 0.0) {
        if (a == 0.0) return signbit(x) ? copysign(0x1.921fb54442d18p+1, y) : y;
        return copysign(0x1.921fb54442d18p+0, y);
    }
    bool inv = a > b;
    double r = atan_unit(inv ? b / a : a / b);
    if (inv) r = 0x1.921fb54442d18p+0 - r;
    if (signbit(x)) r = 0x1.921fb54442d18p+1 - r;
    return copysign(r, y);
}
// asin and acos through atan2 of (x, sqrt((1 - x)(1 + x)))
__device__ __forceinline__ double asin_d(double x) {
    if (!(fabs(x) <= 1.0)) return (x - x) / (x - x);
    return atan2_d(x, sqrt((1.0 - x) * (1.0 + x)));
}
__device__ __forceinline__ double acos_d(double x) {
    if (!(fabs(x) <= 1.0)) return (x - x) / (x - x);
    return atan2_d(sqrt((1.0 - x) * (1.0 + x)), x);
}
__device__ __forceinline__ double sin_d(double x) { double s, c; sincos_d(x, s, c); return s; }
__device__ __forceinline__ double cos_d(double x) { double s, c; sincos_d(x, s, c); return c; }
__device__ __forceinline__ float f_sin(float x) { return (float)sin_d((double)x); }
__device__ __forceinline__ float f_cos(float x) { return (float)cos_d((double)x); }
__device__ __forceinline__ float f_atan(float x) { return (float)atan_d((double)x); }
__device__ __forceinline__ float f_atan2(float y, float x) { return (float)atan2_d((double)y, (double)x); }
__device__ __forceinline__ float f_asin(float x) { return (float)asin_d((double)x); }
__device__ __forceinline__ float f_acos(float x) { return (float)acos_d((double)x); }

// --------------------------------------------------------------- vectors --
struct f3 { float x, y, z; };
__device__ __forceinline__ f3 V3(float a, float b, float c) { f3 r; r.x = a; r.y = b; r.z = c; return r; }
__device__ __forceinline__ f3 vadd(f3 a, f3 b) { return V3(a.x + b.x, a.y + b.y, a.z + b.z); }
__device__ __forceinline__ f3 vsub(f3 a, f3 b) { return V3(a.x - b.x, a.y - b.y, a.z - b.z); }
__device__ __forceinline__ f3 vmul(f3 a, f3 b) { return V3(a.x * b.x, a.y * b.y, a.z * b.z); }
__device__ __forceinline__ f3 vscl(f3 a, float s) { return V3(a.x * s, a.y * s, a.z * s); }
__device__ __forceinline__ f3 vdiv(f3 a, float s) { return V3(a.x / s, a.y / s, a.z / s); }
__device__ __forceinline__ f3 vneg(f3 a) { return V3(-a.x, -a.y, -a.z); }
__device__ __forceinline__ float vdot(f3 a, f3 b) { return a.x * b.x + a.y * b.y + a.z * b.z; }
__device__ __forceinline__ f3 vcross(f3 a, f3 b) {
    return V3(a.y * b.z - a.z * b.y, a.z * b.x - a.x * b.z, a.x * b.y - a.y * b.x);
}
// normalize with 1/sqrtf (the reference's host rsqrtf, CRT/dMath.cuh:70-73,1300-1304)
__device__ __forceinline__ f3 vnorm(f3 v) { float inv = 1.0f / sqrtf(vdot(v, v)); return vscl(v, inv); }
__device__ __forceinline__ bool vzero(f3 a) { return a.x == 0.f && a.y == 0.f && a.z == 0.f; }
__device__ __forceinline__ f3 vreflect(f3 i, f3 n) { return vsub(i, vscl(vscl(n, 2.0f), vdot(n, i))); }
__device__ __forceinline__ f3 vlerp(f3 a, f3 b, float t) { return vadd(a, vscl(vsub(b, a), t)); }
__device__ __forceinline__ f3 xyz(float4 v) { return V3(v.x, v.y, v.z); }
__device__ __forceinline__ float4 f4(f3 a, float w) { return make_float4(a.x, a.y, a.z, w); }
// Loads through the global address space (global_load instead of flat_load:
// the scene pointers come from memory, so the compiler cannot infer it).
template <class T>
__device__ __forceinline__ T ldg(const T* p) {
    return *(const __attribute__((address_space(1))) T*)p;
}
typedef float v4f __attribute__((ext_vector_type(4)));
typedef int v4i __attribute__((ext_vector_type(4)));
__device__ __forceinline__ float4 ldg4(const float4* p) {
    v4f v = *(const __attribute__((address_space(1))) v4f*)p;
    return make_float4(v.x, v.y, v.z, v.w);
}
__device__ __forceinline__ int4 ldg4i(const int4* p) {
    v4i v = *(const __attribute__((address_space(1))) v4i*)p;
    return make_int4(v.x, v.y, v.z, v.w);
}
// a float4 store through the global address space
__device__ __forceinline__ void stg4(float4* p, float4 v) {
    v4f w = {v.x, v.y, v.z, v.w};
    *(__attribute__((address_space(1))) v4f*)p = w;
}
__device__ __forceinline__ f3 ld3(const float* p) { return V3(ldg(p), ldg(p + 1), ldg(p + 2)); }

// ------------------------------------------------------------------- RNG --
// Counter RNG keyed by (seed, pixel, sample, bounce, dim); replaces the
// clock()-seeded wang_hash of CRT/dRandom.cu:20-27.  Mixer: "lowbias32"
// (C. Wellons, hash-prospector, public domain).
__device__ __forceinline__ uint32_t mix32(uint32_t x) {
    x ^= x >> 16; x *= 0x7feb352dU; x ^= x >> 15; x *= 0x846ca68bU; x ^= x >> 16;
    return x;
}
__device__ __forceinline__ uint32_t rng_base(uint32_t seed, uint32_t pixel, uint32_t sample) {
    uint32_t h = mix32(seed ^ 0x5bd1e995U);
    h = mix32(h ^ pixel);
    h = mix32(h + sample * 0x9E3779B9U);
    return h;
}
__device__ __forceinline__ float rng(uint32_t base, uint32_t bounce, uint32_t dim) {
    uint32_t h = mix32(mix32(base ^ ((bounce << 8) | dim)));
    return (float)(h >> 8) * (1.0f / 16777216.0f);
}

// ------------------------------------------------------------- textures --
// Texel columns and rows of a wrap-addressed bilinear tap: with the
// coordinate's fraction in [0, 1], floor(x) lies in [-1, w - 1], so the
// wrap is one conditional add (an index out of range, from a NaN
// coordinate, is taken as 0).
__device__ __forceinline__ void wrap_texels(float fx, float fy, int w, int h, int& i0, int& j0, int& i1,
                                            int& j1) {
    i0 = (int)fx;
    j0 = (int)fy;
    if (i0 < 0) i0 += w;
    if (j0 < 0) j0 += h;
    if ((unsigned)i0 >= (unsigned)w) i0 = 0;
    if ((unsigned)j0 >= (unsigned)h) j0 = 0;
    i1 = i0 + 1 == w ? 0 : i0 + 1;
    j1 = j0 + 1 == h ? 0 : j0 + 1;
}
// Software bilinear filter, wrap addressing on normalized coordinates
// (replaces tex2DLod on linear/wrap texture objects, CRT/dTexture.cu:251-255).
__device__ __forceinline__ void bilinear(const float* __restrict__ tex, int w, int h, int c,
                                         float u, float v, float* out) {
    float uu = u - floorf(u), vv = v - floorf(v);
    float x = uu * (float)w - 0.5f, y = vv * (float)h - 0.5f;
    float fx = floorf(x), fy = floorf(y);
    float a = x - fx, b = y - fy;
    int i0, j0, i1, j1;
    wrap_texels(fx, fy, w, h, i0, j0, i1, j1);
    float w00 = (1.f - a) * (1.f - b), w10 = a * (1.f - b), w01 = (1.f - a) * b, w11 = a * b;
    for (int k = 0; k < c; k++) {
        float t00 = ldg(tex + ((size_t)j0 * w + i0) * c + k), t10 = ldg(tex + ((size_t)j0 * w + i1) * c + k);
        float t01 = ldg(tex + ((size_t)j1 * w + i0) * c + k), t11 = ldg(tex + ((size_t)j1 * w + i1) * c + k);
        out[k] = ((w00 * t00 + w10 * t10) + w01 * t01) + w11 * t11;
    }
}
// luminance (CRT/dMath.cuh:1503-1507): double expression returned as float
__device__ __forceinline__ float lum_of(const float* s) {
    return (float)(0.299 * (double)s[0] + 0.587 * (double)s[1] + 0.114 * (double)s[2]);
}

// ------------------------------------------------------------ env light --
// sample_spherical_direction / sample_spherical_map (CRT/dMath.cuh:1483-1501)
__device__ __forceinline__ f3 sph_dir(float u, float v) {
    float theta = F_2PI * u, phi = F_PI * v;
    float x = f_cos(theta) * f_sin(phi), y = f_cos(phi), z = f_sin(theta) * f_sin(phi);
    return V3(-x, -y, -z);
}
// The asin argument is clamped to [-1, 1]: a normalised float direction can
// have |y| = 1 + 1 ulp, where the reference's asin gives NaN radiance.
__device__ __forceinline__ void sph_map(f3 d, float& u, float& v) {
    u = f_atan2(d.z, d.x) * F_1_2PI + 0.5f;
    v = f_asin(fminf(fmaxf(d.y, -1.f), 1.f)) * F_1_PI + 0.5f;
}
// upper_bound with the trailing list[left <= val] adjustment (CRT/Helpers.cu:16-31)
__device__ __forceinline__ int upper_bound_ref(const double* __restrict__ list, int size, float val) {
    int left = 0, right = size;
    while (left < right) {
        int middle = (right - left) / 2 + left;
        if ((double)val >= ldg(list + middle)) left = middle + 1;
        else right = middle;
    }
    if (left < size && ldg(list + (((float)left <= val) ? 1 : 0)) != 0.0) left++;
    return left;
}

struct EnvView {
    const float4* rgbp;    // [h][w] (r, g, b, pdf)
    const double* marg_y;  // [h]
    const double* conds;   // [h][w]
    const uint32_t* guide_m, *guide_c;
    int w, h;
};
// upper_bound_ref over a non-decreasing list, starting from its guide table:
// the guide brackets the first element greater than val (the bracket of
// val's bucket), so the loop below finds the same index as a search of the
// whole list.  The trailing adjustment tests list[(float)left <= val], which
// for val in [0, 1) is list[1] when left == 0 and list[0] otherwise; the
// guide entries carry both tests.  Lists that are not monotone (guide entries
// flagged) are searched whole, and values outside [0, 1) are searched whole
// with the adjustment read from the list, exactly as upper_bound_ref does.
__device__ __forceinline__ int upper_bound_guided(const double* __restrict__ list, int size,
                                                  const uint32_t* __restrict__ guide, float val) {
    int left = 0, right = size;
    if (!(val >= 0.f && val < 1.f)) return upper_bound_ref(list, size, val);
    uint32_t g = (uint32_t)(val * (float)ENV_GUIDE);  // exact: ENV_GUIDE is a power of two
    if (g > ENV_GUIDE - 1) g = ENV_GUIDE - 1;
    typedef uint32_t v2u __attribute__((ext_vector_type(2), aligned(4)));
    // both ends of the bracket in one load (a lane's scattered loads are what a
    // shading kernel's address path spends its time on, whatever their width)
    const v2u ab = *(const __attribute__((address_space(1))) v2u*)(guide + g);
    const uint32_t a = ab.x, b = ab.y;
    if (((a | b) & ENV_GUIDE_FULL) == 0) {
        left = (int)(a & ENV_GUIDE_INDEX);
        right = (int)(b & ENV_GUIDE_INDEX);
    }
    while (left < right) {
        int middle = (right - left) / 2 + left;
        if ((double)val >= ldg(list + middle)) left = middle + 1;
        else right = middle;
    }
    if (left < size && (a & (left == 0 ? ENV_GUIDE_NZ1 : ENV_GUIDE_NZ0)) != 0u) left++;
    return left;
}
// dEnvironmentLight::L (CRT/dEnvironmentLight.cu:66-76): bilinear() over the
// (r, g, b) of the interleaved texels, one 16-B load per texel
// (u, v): sph_map of the direction, which its pdf shares
__device__ __forceinline__ f3 env_L(const EnvView& e, float u, float v) {
    float uu = u - floorf(u), vv = v - floorf(v);
    float x = uu * (float)e.w - 0.5f, y = vv * (float)e.h - 0.5f;
    float fx = floorf(x), fy = floorf(y);
    float a = x - fx, b = y - fy;
    int i0, j0, i1, j1;
    wrap_texels(fx, fy, e.w, e.h, i0, j0, i1, j1);
    float w00 = (1.f - a) * (1.f - b), w10 = a * (1.f - b), w01 = (1.f - a) * b, w11 = a * b;
    float4 t00 = ldg4(e.rgbp + (size_t)j0 * e.w + i0), t10 = ldg4(e.rgbp + (size_t)j0 * e.w + i1);
    float4 t01 = ldg4(e.rgbp + (size_t)j1 * e.w + i0), t11 = ldg4(e.rgbp + (size_t)j1 * e.w + i1);
    return V3(((w00 * t00.x + w10 * t10.x) + w01 * t01.x) + w11 * t11.x,
              ((w00 * t00.y + w10 * t10.y) + w01 * t01.y) + w11 * t11.y,
              ((w00 * t00.z + w10 * t10.z) + w01 * t01.z) + w11 * t11.z);
}
__device__ __forceinline__ f3 env_L(const EnvView& e, f3 wi) {
    float u, v;
    sph_map(wi, u, v);
    return env_L(e, u, v);
}
// dEnvironmentLight::get_pdf(isect, wi) (CRT/dEnvironmentLight.cu:83-103)
__device__ __forceinline__ float env_pdf(const EnvView& e, f3 wi, float u, float v) {
    int px = (int)(u * (float)(e.w - 1)), py = (int)(v * (float)(e.h - 1));
    px = px < 0 ? 0 : (px > e.w - 1 ? e.w - 1 : px);
    py = py < 0 ? 0 : (py > e.h - 1 ? e.h - 1 : py);
    float z = wi.z < -1.f ? -1.f : (wi.z > 1.f ? 1.f : wi.z);
    return ldg4(e.rgbp + (size_t)py * e.w + px).w / f_sin(f_acos(z));
}
// dEnvironmentLight::get_direction (CRT/dEnvironmentLight.cu:41-58);
// indices clamped at 0 where the reference would index out of range.
__device__ __forceinline__ f3 env_sample(const EnvView& e, f3 P, float ex, float ey) {
    int y = (int)((float)upper_bound_guided(e.marg_y, e.h, e.guide_m, ey) - 1.f);
    if (y < 0) y = 0;
    int x = (int)((float)upper_bound_guided(e.conds + (size_t)y * e.w, e.w, e.guide_c + (size_t)y * (ENV_GUIDE + 1),
                                            ex) - 1.f);
    if (x < 0) x = 0;
    f3 dir = sph_dir((float)x / (float)e.w, (float)y / (float)e.h);
    f3 spt = vadd(V3(0.f, 0.f, 0.f), vscl(dir, 10000.f));
    return vnorm(vsub(spt, P));
}

// -------------------------------------------------------------- camera --
// dCamera::gen_ray (CRT/dCamera.cu:10-36) with Matrix4x4*float4
// (CRT/dMatrix.cuh:61-69) and ConcentricSampleDisk (CRT/dRandom.cu:104-126).
__device__ __forceinline__ void gen_ray(const ff_dev_camera& cam, int width, int height, int px,
                                        int py, uint32_t base, f3& o, f3& d) {
    float nx = (float)(2.0f * (((double)px + 0.5) / (double)width) - 1.0f);
    float ny = (float)(1.0f - 2.0f * (((double)py + 0.5) / (double)height));
    const float* m = cam.inv_vp;
    float a[4] = {nx, ny, -1.f, 1.f}, b[4] = {nx, ny, 1.f, 1.f}, pa[4], pb[4];
#pragma unroll
    for (int r = 0; r < 4; r++) {
        pa[r] = m[0 * 4 + r] * a[0] + m[1 * 4 + r] * a[1] + m[2 * 4 + r] * a[2] + m[3 * 4 + r] * a[3];
        pb[r] = m[0 * 4 + r] * b[0] + m[1 * 4 + r] * b[1] + m[2 * 4 + r] * b[2] + m[3 * 4 + r] * b[3];
    }
    f3 pn = V3(pa[0] / pa[3], pa[1] / pa[3], pa[2] / pa[3]);
    f3 pf = V3(pb[0] / pb[3], pb[1] / pb[3], pb[2] / pb[3]);
    float sx = rng(base, 0, DIM_JX) * 0.005f, sy = rng(base, 0, DIM_JY) * 0.005f;
    o = vadd(pn, V3(sx, sy, 0.f));
    d = vnorm(vsub(pf, pn));
    if (cam.lens_radius > 0.f) {
        f3 pfoc = vadd(o, vscl(d, cam.focal));
        float u0 = rng(base, 0, DIM_LX), u1 = rng(base, 0, DIM_LY);
        float ox = 2.f * u0 - 1.f, oy = 2.f * u1 - 1.f, lx = 0.f, ly = 0.f;
        if (!(ox == 0 && oy == 0)) {
            float theta, r;
            if (fabsf(ox) > fabsf(oy)) { r = ox; theta = F_PI_4 * (oy / ox); }
            else { r = oy; theta = F_PI_2 - F_PI_4 * (ox / oy); }
            lx = r * f_cos(theta);
            ly = r * f_sin(theta);
        }
        o = vadd(o, V3(lx * cam.lens_radius, ly * cam.lens_radius, 0.f));
        d = vnorm(vsub(pfoc, o));
    }
}

// ---------------------------------------------------------------- BSDFs --
__device__ __forceinline__ float pow5(float x) { float x2 = x * x; return (x2 * x2) * x; }
// fresnel (CRT/dMaterial.cu:90-92)
__device__ __forceinline__ f3 fresnel_s(f3 f0, f3 h, f3 wo) {
    float p = pow5(1.f - fmaxf(0.f, vdot(h, wo)));
    return vadd(f0, vscl(V3(1.f - f0.x, 1.f - f0.y, 1.f - f0.z), p));
}
// power_heuristic with nf = ng = 1 (CRT/dMaterial.cu:114-119)
__device__ __forceinline__ double power_heur(double f, double g) { return (f * f) / (f * f + g * g); }
// ggxtr_ndf (CRT/dMaterial.cu:120-125)
__device__ __forceinline__ double ggx_ndf(f3 n, f3 h, float r) {
    double a2 = (double)(r * r * r * r);
    float nh = fmaxf(0.0f, vdot(n, h));
    double nh2 = (double)(nh * nh);
    double q = nh2 * (a2 - 1.0) + 1.0;
    return a2 / ((double)F_PI * (q * q));
}
// geo_atten (CRT/dMaterial.cu:126-137)
__device__ __forceinline__ double geo_att(f3 wi, f3 wo, f3 n, float r) {
    float rp = r + 1.f;
    double k = (double)((rp * rp) / 8.f);
    double nl = (double)fmaxf(vdot(n, wi), 0.0f), nv = (double)fmaxf(vdot(n, wo), 0.0f);
    double g1 = nl / (nl * (1.0 - k) + k), g2 = nv / (nv * (1.0 - k) + k);
    return g1 * g2;
}
// spec_get_pdf (CRT/dMaterial.cu:255-265)
__device__ __forceinline__ float spec_pdf(f3 n, f3 wi, f3 wo, float r) {
    f3 wh = vnorm(vadd(wo, wi));
    double whn = (double)fmaxf(vdot(wh, n), 0.f), wowh = (double)fmaxf(vdot(wo, wh), 0.f);
    double D = ggx_ndf(n, wh, r);
    float den = fmaxf((float)(4.0 * wowh), 0.001f);
    return (float)((D * whn) / (double)den);
}
// spec_f (CRT/dMaterial.cu:266-288)
__device__ __forceinline__ f3 spec_f(f3 n, f3 wi, f3 wo, float r, float m, f3 alb, f3 fres) {
    f3 f0 = vlerp(fres, alb, m);
    f3 wh = vnorm(vadd(wo, wi));
    double ndwi = (double)fmaxf(vdot(n, wi), 0.f), ndwo = (double)fmaxf(vdot(n, wo), 0.f);
    double D = ggx_ndf(n, wh, r), G = geo_att(wi, wo, n, r);
    f3 F = fresnel_s(f0, wh, wi);
    float den = fmaxf((float)(4.0 * ndwo * ndwi), 0.001f);
    return vdiv(vscl(F, (float)(D * G)), den);
}
// diff_f (CRT/dMaterial.cu:164-178)
__device__ __forceinline__ f3 diff_f(f3 wi, f3 wo, float m, f3 alb, f3 fres) {
    f3 f0 = vlerp(fres, alb, m);
    f3 wh = vnorm(vadd(wo, wi));
    f3 F = fresnel_s(f0, wh, wi);
    f3 kd = V3(1.f - F.x, 1.f - F.y, 1.f - F.z);
    kd = vscl(kd, (float)(1.0 - (double)m));
    return vscl(vmul(kd, alb), F_1_PI);
}
// get_orthogonal_vec (CRT/dMath.cuh:1450-1463)
__device__ __forceinline__ f3 ortho_axis(f3 in) {
    if (fabsf(in.x) < 0.57735026919f) return V3(1, 0, 0);
    if (fabsf(in.y) < 0.57735026919f) return V3(0, 1, 0);
    return V3(0, 0, 1);
}
// diff_sample (CRT/dMaterial.cu:139-159)
__device__ __forceinline__ f3 diff_sample(f3 N, float e0, float e1) {
    float sin_t = sqrtf(1.f - e0 * e0);
    float phi = 2.f * F_PI * e1;
    float x = sin_t * f_cos(phi), z = sin_t * f_sin(phi);
    f3 T = vnorm(vcross(N, ortho_axis(N)));
    f3 B = vnorm(vcross(N, T));
    return vnorm(vadd(vadd(vscl(T, x), vscl(N, e0)), vscl(B, z)));
}
// spec_sample (CRT/dMaterial.cu:229-254)
__device__ __forceinline__ f3 spec_sample(f3 N, f3 wo, float r, float e0, float e1) {
    double theta = (double)f_atan(r * r * sqrtf(e0 / (1.f - e0)));
    double phi = (double)((2 * F_PI) * e1);
    double st, ct, sp, cp;
    sincos_d(theta, st, ct);
    sincos_d(phi, sp, cp);
    f3 h = V3((float)(st * cp), (float)ct, (float)(st * sp));
    f3 T = vnorm(vcross(N, ortho_axis(N)));
    f3 B = vnorm(vcross(N, T));
    f3 smp = vadd(vadd(vscl(T, h.x), vscl(N, h.y)), vscl(B, h.z));
    return vneg(vreflect(wo, vnorm(smp)));
}
// Exact Fresnel reflectance of a smooth dielectric (textbook Fresnel
// equations).  No reference counterpart (the reference has no dielectric).
__device__ __forceinline__ float fresnel_dielectric(float cos_i, float eta_i, float eta_t) {
    float sin_i = sqrtf(fmaxf(0.f, 1.f - cos_i * cos_i));
    float sin_t = eta_i / eta_t * sin_i;
    if (sin_t >= 1.f) return 1.f;
    float cos_t = sqrtf(fmaxf(0.f, 1.f - sin_t * sin_t));
    float rpar = (eta_t * cos_i - eta_i * cos_t) / (eta_t * cos_i + eta_i * cos_t);
    float rper = (eta_i * cos_i - eta_t * cos_t) / (eta_i * cos_i + eta_t * cos_t);
    return 0.5f * (rpar * rpar + rper * rper);
}

// ------------------------------------------------------------- adjoint --
// Partial derivatives of the BSDF values for the path-replay adjoint.  The
// sampling (directions, pdfs, MIS weights) is detached, so only the values
// of spec_f / diff_f depend on albedo and roughness.  No reference
// counterpart (the reference is not differentiable).
struct LobeGrad {
    f3 da;  // d f_c / d albedo_c
    f3 dr;  // d f_c / d roughness
};
// spec_f = F * D * G / den with F = f0 + (1 - f0) p, f0 = fres + (albedo - fres) m,
// D = a2 / (pi q^2), a2 = r^4, q = nh^2 (a2 - 1) + 1, G = g(n.wi) g(n.wo),
// g(x) = x / (x (1 - k) + k), k = (r + 1)^2 / 8.
__device__ __forceinline__ LobeGrad spec_grad(f3 n, f3 wi, f3 wo, float r, float m, f3 alb, f3 fres) {
    // D and G in FP64 as ggx_ndf / geo_att evaluate them (q loses all float
    // precision near the lobe peak at low roughness)
    f3 f0 = vlerp(fres, alb, m);
    f3 wh = vnorm(vadd(wo, wi));
    double ndwi = (double)fmaxf(vdot(n, wi), 0.f), ndwo = (double)fmaxf(vdot(n, wo), 0.f);
    float nh = fmaxf(0.f, vdot(n, wh));
    double rd = (double)r;
    double a2 = (double)(r * r * r * r), nh2 = (double)(nh * nh);
    double q = nh2 * (a2 - 1.0) + 1.0;
    double D = a2 / ((double)F_PI * (q * q));
    double dD = 4.0 * rd * rd * rd * (q - 2.0 * a2 * nh2) / ((double)F_PI * q * q * q);
    float rp = r + 1.f;
    double k = (double)((rp * rp) / 8.f), dk = 0.25 * (rd + 1.0);
    double d1 = ndwi * (1.0 - k) + k, d2 = ndwo * (1.0 - k) + k;
    double g1 = ndwi / d1, g2 = ndwo / d2;
    double dg1 = -ndwi * (1.0 - ndwi) / (d1 * d1), dg2 = -ndwo * (1.0 - ndwo) / (d2 * d2);
    double G = g1 * g2, dG = (dg1 * g2 + g1 * dg2) * dk;
    float p = pow5(1.f - fmaxf(0.f, vdot(wh, wi)));
    float den = fmaxf((float)(4.0 * ndwo * ndwi), 0.001f);
    f3 F = vadd(f0, vscl(V3(1.f - f0.x, 1.f - f0.y, 1.f - f0.z), p));
    LobeGrad g;
    float sa = (float)((double)(m * (1.f - p)) * D * G / (double)den);
    g.da = V3(sa, sa, sa);
    g.dr = vscl(F, (float)((dD * G + D * dG) / (double)den));
    return g;
}
// diff_f = (1 - F) (1 - m) albedo / pi
__device__ __forceinline__ f3 diff_grad(f3 wi, f3 wo, float m, f3 alb, f3 fres) {
    f3 f0 = vlerp(fres, alb, m);
    f3 wh = vnorm(vadd(wo, wi));
    float p = pow5(1.f - fmaxf(0.f, vdot(wh, wi)));
    f3 F = vadd(f0, vscl(V3(1.f - f0.x, 1.f - f0.y, 1.f - f0.z), p));
    float c = (1.f - m) * F_1_PI, s = m * (1.f - p);
    return V3(c * ((1.f - F.x) - alb.x * s), c * ((1.f - F.y) - alb.y * s), c * ((1.f - F.z) - alb.z * s));
}

// The four texels and weights bilinear() reads at (u, v) (same arithmetic).
struct Taps {
    uint32_t i[4];
    float w[4];
};
__device__ __forceinline__ Taps taps_of(int w, int h, float u, float v) {
    float uu = u - floorf(u), vv = v - floorf(v);
    float x = uu * (float)w - 0.5f, y = vv * (float)h - 0.5f;
    float fx = floorf(x), fy = floorf(y);
    float a = x - fx, b = y - fy;
    int i0, j0, i1, j1;
    wrap_texels(fx, fy, w, h, i0, j0, i1, j1);
    Taps t;
    t.i[0] = (uint32_t)(j0 * w + i0); t.i[1] = (uint32_t)(j0 * w + i1);
    t.i[2] = (uint32_t)(j1 * w + i0); t.i[3] = (uint32_t)(j1 * w + i1);
    t.w[0] = (1.f - a) * (1.f - b); t.w[1] = a * (1.f - b); t.w[2] = (1.f - a) * b; t.w[3] = a * b;
    return t;
}

// Scale exponent of one fixed-point gradient element: every partial sum of
// its terms is bounded by count * max|term| < 2^k, so terms are kept in
// units of 2^-(61 - k) and the int64 sum cannot overflow.
__device__ __forceinline__ int fixed_exponent(uint32_t max_bits, uint32_t count) {
    double b = (double)__uint_as_float(max_bits) * (double)count;
    if (!(b > 0.0)) return 0;
    int k;
    (void)frexp(b, &k);
    return 61 - k;
}

// ------------------------------------------------------------ traversal --

// Bounds3f::hit(ray, invDir, dirIsNeg) (CRT/Bounds3f.h:128-160) on one box:
// the line test without [0, tmax] clipping; returns the final tmin/tmax.
// The reference's comparisons are evaluated branch-free (all six plane
// distances first): same values, same outcome, and no load or branch is
// left waiting on the x/y test.
__device__ __forceinline__ bool slab(float lx, float ly, float lz, float hx, float hy, float hz, f3 o,
                                     f3 inv, bool nx, bool ny, bool nz, float& tn, float& tf) {
    float tmin = ((nx ? hx : lx) - o.x) * inv.x;
    float tmax = ((nx ? lx : hx) - o.x) * inv.x;
    float tymin = ((ny ? hy : ly) - o.y) * inv.y;
    float tymax = ((ny ? ly : hy) - o.y) * inv.y;
    float tzmin = ((nz ? hz : lz) - o.z) * inv.z;
    float tzmax = ((nz ? lz : hz) - o.z) * inv.z;
    bool ok_xy = !((tmin > tymax) || (tymin > tmax));
    float t1 = (tymin > tmin) ? tymin : tmin;
    float t2 = (tymax < tmax) ? tymax : tmax;
    bool ok_z = !((t1 > tzmax) || (tzmin > t2));
    tn = (tzmin > t1) ? tzmin : t1;
    tf = (tzmax < t2) ? tzmax : t2;
    return ok_xy & ok_z;
}

// The same test in fewer instructions, for boxes with lo <= hi (every box of
// a scene with finite vertices) and rays whose x distances cannot be NaN
// (finite 1/d.x and o.x): entry = max, exit = min of the three slab
// distances, hit = !(entry > exit).  A NaN y or z distance (0 * inf: origin
// on a slab plane, zero direction component) drops out of the reference's
// comparisons and out of fmaxf/fminf alike, so the outcome, entry and exit
// equal slab()'s.  (A NaN x distance would also hide the y distance from
// the reference's z comparison; such rays take slab().)
__device__ __forceinline__ bool slab_box(float lx, float ly, float lz, float hx, float hy, float hz, f3 o,
                                         f3 inv, bool nx, bool ny, bool nz, float& tn, float& tf) {
    float x0 = ((nx ? hx : lx) - o.x) * inv.x;
    float x1 = ((nx ? lx : hx) - o.x) * inv.x;
    float y0 = ((ny ? hy : ly) - o.y) * inv.y;
    float y1 = ((ny ? ly : hy) - o.y) * inv.y;
    float z0 = ((nz ? hz : lz) - o.z) * inv.z;
    float z1 = ((nz ? lz : hz) - o.z) * inv.z;
    tn = fmaxf(fmaxf(x0, y0), z0);
    tf = fminf(fminf(x1, y1), z1);
    return !(tn > tf);
}

// Triangle record in BVH-slot order: v0, e1 = v1 - v0, e2 = v2 - v0 (the
// edges the reference forms per test, CRT/dTriangle.cu:35-36).
struct Tri { f3 v0, e1, e2; };
__device__ __forceinline__ Tri load_tri(const float* __restrict__ t, int slot) {
    const float* p = t + (size_t)slot * 9;
    Tri r;
    r.v0 = V3(ldg(p + 0), ldg(p + 1), ldg(p + 2));
    r.e1 = V3(ldg(p + 3), ldg(p + 4), ldg(p + 5));
    r.e2 = V3(ldg(p + 6), ldg(p + 7), ldg(p + 8));
    return r;
}
// dTriangle::intersect, TEST_CULL branch (CRT/dTriangle.cu:34-62)
__device__ __forceinline__ bool mt_cull(const Tri& T, f3 o, f3 d, float& t, float& u, float& v) {
    f3 pvec = vcross(d, T.e2);
    float detf = vdot(T.e1, pvec);
    if (detf < K_EPS) return false;
    f3 tvec = vsub(o, T.v0);
    float uf = vdot(tvec, pvec);
    if (uf < 0.f || uf > detf) return false;
    f3 qvec = vcross(tvec, T.e1);
    float vf = vdot(d, qvec);
    if (vf < 0.f || (uf + vf) > detf) return false;
    float tf = vdot(T.e2, qvec);
    double inv_det = 1.0 / (double)detf;
    t = (float)((double)tf * inv_det);
    u = (float)((double)uf * inv_det);
    v = (float)((double)vf * inv_det);
    return true;
}
// dTriangle::intersect, non-culling branch (CRT/dTriangle.cu:63-80)
__device__ __forceinline__ bool mt_two(const Tri& T, f3 o, f3 d, float& t, float& u, float& v) {
    f3 pvec = vcross(d, T.e2);
    double det = (double)vdot(T.e1, pvec);
    if (det > (double)-K_EPS && det < (double)K_EPS) return false;
    double inv_det = 1.0 / det;
    f3 tvec = vsub(o, T.v0);
    float uf = (float)((double)vdot(tvec, pvec) * inv_det);
    if (uf < 0.f || uf > 1.f) return false;
    f3 qvec = vcross(tvec, T.e1);
    float vf = (float)((double)vdot(d, qvec) * inv_det);
    if (vf < 0.f || (double)(uf + vf) > 1.0) return false;
    t = (float)((double)vdot(T.e2, qvec) * inv_det);
    u = uf;
    v = vf;
    return true;
}
// dTriangle::shadow_hit (CRT/dTriangle.cu:110-138)
__device__ __forceinline__ bool mt_shadow(const Tri& T, f3 o, f3 d, float& t) {
    f3 pvec = vcross(d, T.e2);
    double det = (double)vdot(T.e1, pvec);
    if (det > (double)-K_EPS && det < (double)K_EPS) return false;
    double inv_det = 1.0 / det;
    f3 tvec = vsub(o, T.v0);
    double u = (double)vdot(tvec, pvec) * inv_det;
    if (u < 0.0 || u > 1.0) return false;
    f3 qvec = vcross(tvec, T.e1);
    double v = (double)vdot(d, qvec) * inv_det;
    if (v < 0.0 || u + v > 1.0) return false;
    float tf = (float)((double)vdot(T.e2, qvec) * inv_det);
    if (tf < 0.f) return false;
    t = tf;
    return true;
}

// Traversal stack: the first `lds_entries` entries of each lane live in LDS
// ([depth][lane], conflict-free), deeper entries in a per-lane global
// overflow area ([depth - lds_entries][grid thread]).
typedef __attribute__((address_space(3))) int lds_int;
typedef __attribute__((address_space(3))) uint32_t lds_u32;
typedef __attribute__((address_space(1))) int glb_int;
// Traversal stack: LDS entries first (ds_read / ds_write), then the lane's
// column of the global overflow area.  The pointers carry their address
// spaces so no access goes through a generic (flat) pointer.
struct Stack {
    lds_int* lds;      // &smem[threadIdx.x]
    glb_int* ovf;      // &overflow[grid thread]
    uint32_t lds_stride, ovf_stride;
    int lds_entries;
    int sp;
    __device__ __forceinline__ void push(int v) {
        if (sp < lds_entries) lds[sp * lds_stride] = v;
        else ovf[(size_t)(sp - lds_entries) * ovf_stride] = v;
        sp++;
    }
    __device__ __forceinline__ int pop() {
        sp--;
        int v;
        if (sp < lds_entries) v = lds[sp * lds_stride];
        else v = ovf[(size_t)(sp - lds_entries) * ovf_stride];
        return v;
    }
};

// The stack of a ray that four lanes share: its entries lie in the 64 LDS
// columns of the wave (BS columns to a row), 16 rays side by side.
template <int BS>
struct QuadStack {
    lds_int* col;  // &smem[first column of the wave + ray]
    int sp;
    __device__ __forceinline__ lds_int* at(int e) const { return col + (e >> 2) * BS + (e & 3) * 16; }
    __device__ __forceinline__ void push(int v) { *at(sp++) = v; }
    __device__ __forceinline__ int pop() { return *at(--sp); }
};

struct Hit { float t, u, v; int id; };
// pruning limit of the current closest hit
__device__ __forceinline__ float prune_lim(float t) { return t + t * PRUNE_REL + PRUNE_ABS; }

// Device BVH: the reference's binary tree (same nodes, same order) stored as
// 64-byte two-child records so one fetch tests both children's boxes:
//   a = (c0.lo.xyz, c0.hi.x)  b = (c0.hi.yz, c1.lo.xy)  c = (c1.lo.z, c1.hi.xyz)
//   m = (ref0, ref1, axis, -)
// ref >= 0: interior record index; ref < 0: leaf, ~ref = first slot << 4 |
// count (count 15 = read leaf_count[first slot]).  The root box is tested
// first, as the reference tests node 0.
struct Bvh {
    const float4* nodes;   // two-child records
    const float4* nodes4;  // 4-wide records (same tree, collapsed)
    const int32_t* leaf_count;
    const float* root;  // lo.xyz, hi.xyz, ref (int bits)
};

__device__ __forceinline__ void leaf_range(const Bvh& B, int ref, int& off, int& cnt) {
    int e = ~ref;
    off = e >> 4;
    cnt = e & 15;
    if (cnt == 15) cnt = ldg(B.leaf_count + off);
}

// Per-lane traversal state: the ray, its reciprocal direction and octant,
// and the next node reference to visit.
struct TravRay {
    f3 o, d, inv;
    bool nx, ny, nz;
    uint32_t negm;  // nx | ny << 1 | nz << 2 | XNAN_RAY
    int ref;
};

// Tests the root box (the reference tests node 0 first); false when the ray
// misses the scene or the scene lies wholly behind the origin.
__device__ __forceinline__ bool trav_begin(const Bvh& B, f3 o, f3 d, TravRay& R, Stack& st,
                                           uint32_t& cnt_nodes) {
    R.o = o;
    R.d = d;
    R.inv = V3(1.f / d.x, 1.f / d.y, 1.f / d.z);
    R.nx = R.inv.x < 0;
    R.ny = R.inv.y < 0;
    R.nz = R.inv.z < 0;
    R.negm = (R.nx ? 1u : 0u) | (R.ny ? 2u : 0u) | (R.nz ? 4u : 0u) |
             ((isfinite(R.inv.x) && isfinite(o.x)) ? 0u : XNAN_RAY);
    float tn, tf;
    cnt_nodes++;
    float4 r0 = ldg4((const float4*)B.root), r1 = ldg4((const float4*)B.root + 1);
    if (!slab(r0.x, r0.y, r0.z, r0.w, r1.x, r1.y, o, R.inv, R.nx, R.ny, R.nz, tn, tf) || tf < -PRUNE_BEHIND)
        return false;
    R.ref = __float_as_int(r1.z);
    st.sp = 0;
    return true;
}

// One interior record: both child boxes are tested; the near child (by
// dirIsNeg[axis]) is visited next and the far one pushed when both are hit.
// Returns false when neither child is entered (the caller pops).
template <bool PRUNE>
__device__ __forceinline__ bool visit_interior(const Bvh& B, TravRay& R, float lim, Stack& st,
                                               uint32_t& cnt_nodes) {
    // 32-bit byte offset (records < 2^26, checked at scene creation): the
    // load adds it to the base without 64-bit address arithmetic
    const float4* n = (const float4*)((const char*)B.nodes + ((uint32_t)R.ref << 6));
    float4 a = ldg4(n), b = ldg4(n + 1), c = ldg4(n + 2);
    int4 m = ldg4i((const int4*)(n + 3));
    cnt_nodes += 2;
    float tn0, tf0, tn1, tf1;
    bool h0, h1;
    if (__ballot((R.negm & XNAN_RAY) != 0) == 0) {  // wave-uniform: no lane can see a NaN x distance
        h0 = slab_box(a.x, a.y, a.z, a.w, b.x, b.y, R.o, R.inv, R.nx, R.ny, R.nz, tn0, tf0);
        h1 = slab_box(b.z, b.w, c.x, c.y, c.z, c.w, R.o, R.inv, R.nx, R.ny, R.nz, tn1, tf1);
    } else {
        h0 = slab(a.x, a.y, a.z, a.w, b.x, b.y, R.o, R.inv, R.nx, R.ny, R.nz, tn0, tf0);
        h1 = slab(b.z, b.w, c.x, c.y, c.z, c.w, R.o, R.inv, R.nx, R.ny, R.nz, tn1, tf1);
    }
    if (PRUNE) {
        h0 = h0 && !(tn0 > lim || tf0 < -PRUNE_BEHIND);
        h1 = h1 && !(tn1 > lim || tf1 < -PRUNE_BEHIND);
    } else {
        h0 = h0 && !(tf0 < -PRUNE_BEHIND);
        h1 = h1 && !(tf1 < -PRUNE_BEHIND);
    }
    // both hit: the near child (by dirIsNeg[axis]) next, the far one pushed;
    // one hit: that one next (no direction test needed)
    if (h0 && h1) {
        bool neg = ((R.negm >> (uint32_t)m.z) & 1u) != 0;  // dirIsNeg[axis]
        st.push(neg ? m.x : m.y);
        R.ref = neg ? m.y : m.x;
        return true;
    }
    if (h0 || h1) {
        R.ref = h0 ? m.x : m.y;
        return true;
    }
    return false;
}

// One 4-wide record: the four grandchild boxes are tested at once and the
// hit ones are visited in the binary tree's near-first order (side by the
// parent's split axis, then each side by its own axis): the first is entered,
// the others pushed so that they pop in order.  Leaves are visited in the
// order the binary walk visits them, so the closest hit (ties included) is
// unchanged.  Empty slots (box +inf..-inf) never hit.
__device__ __forceinline__ float sel4(const float4& v, int k) {
    return k == 0 ? v.x : (k == 1 ? v.y : (k == 2 ? v.z : v.w));
}
__device__ __forceinline__ int sel4i(const int4& v, int k) {
    return k == 0 ? v.x : (k == 1 ? v.y : (k == 2 ? v.z : v.w));
}
template <bool PRUNE>
__device__ __forceinline__ bool visit_interior4(const Bvh& B, TravRay& R, float lim, Stack& st,
                                                uint32_t& cnt_nodes) {
    const float4* n = (const float4*)((const char*)B.nodes4 + ((uint64_t)(uint32_t)R.ref << 7));
    float4 lx = ldg4(n), ly = ldg4(n + 1), lz = ldg4(n + 2);
    float4 hx = ldg4(n + 3), hy = ldg4(n + 4), hz = ldg4(n + 5);
    int4 rf = ldg4i((const int4*)(n + 6)), ax = ldg4i((const int4*)(n + 7));
    bool hit[4];
#pragma unroll
    for (int k = 0; k < 4; k++) {
        float tn, tf;
        bool h = slab(sel4(lx, k), sel4(ly, k), sel4(lz, k), sel4(hx, k), sel4(hy, k), sel4(hz, k), R.o, R.inv,
                      R.nx, R.ny, R.nz, tn, tf);
        hit[k] = PRUNE ? (h && !(tn > lim || tf < -PRUNE_BEHIND)) : (h && !(tf < -PRUNE_BEHIND));
    }
    cnt_nodes += (rf.x != -1 ? 1u : 0u) + (rf.y != -1 ? 1u : 0u) + (rf.z != -1 ? 1u : 0u) + (rf.w != -1 ? 1u : 0u);
    bool negN = ((R.negm >> (uint32_t)ax.x) & 1u) != 0;
    bool negA = ((R.negm >> (uint32_t)ax.y) & 1u) != 0;
    bool negB = ((R.negm >> (uint32_t)ax.z) & 1u) != 0;
    int s0 = negN ? 2 : 0, s1 = negN ? 0 : 2;
    bool f0 = negN ? negB : negA, f1 = negN ? negA : negB;
    int o0 = s0 + (f0 ? 1 : 0), o1 = s0 + (f0 ? 0 : 1), o2 = s1 + (f1 ? 1 : 0), o3 = s1 + (f1 ? 0 : 1);
    bool h0 = o0 == 0 ? hit[0] : (o0 == 1 ? hit[1] : (o0 == 2 ? hit[2] : hit[3]));
    bool h1 = o1 == 0 ? hit[0] : (o1 == 1 ? hit[1] : (o1 == 2 ? hit[2] : hit[3]));
    bool h2 = o2 == 0 ? hit[0] : (o2 == 1 ? hit[1] : (o2 == 2 ? hit[2] : hit[3]));
    bool h3 = o3 == 0 ? hit[0] : (o3 == 1 ? hit[1] : (o3 == 2 ? hit[2] : hit[3]));
    int r0 = sel4i(rf, o0), r1 = sel4i(rf, o1), r2 = sel4i(rf, o2), r3 = sel4i(rf, o3);
    if (h3 && (h0 || h1 || h2)) st.push(r3);
    if (h2 && (h0 || h1)) st.push(r2);
    if (h1 && h0) st.push(r1);
    if (h0) { R.ref = r0; return true; }
    if (h1) { R.ref = r1; return true; }
    if (h2) { R.ref = r2; return true; }
    if (h3) { R.ref = r3; return true; }
    return false;
}
template <bool WIDE, bool PRUNE>
__device__ __forceinline__ bool visit_node(const Bvh& B, TravRay& R, float lim, Stack& st, uint32_t& cnt_nodes) {
    return WIDE ? visit_interior4<PRUNE>(B, R, lim, st, cnt_nodes)
                : visit_interior<PRUNE>(B, R, lim, st, cnt_nodes);
}

// The closest hit of a persistent traversal lane: t in a register (every
// test reads it), u, v and the triangle slot in three LDS words of the lane
// (written only when a closer hit is found, read once at the end), which
// keeps the closest-hit kernels at 8 waves per SIMD.
typedef __attribute__((address_space(3))) float lds_float;
struct HitSlots {
    lds_float* u;
    lds_float* v;
    lds_int* id;
    lds_float* redo;  // wide walk: smallest t whose outcome the reference's order decides
};
__device__ __forceinline__ void leaf_closest_slots(const Bvh& B, const float* __restrict__ tris, const TravRay& R,
                                                   float& t_hit, const HitSlots& hs, bool two_sided,
                                                   uint32_t& cnt_tris) {
    int off, np;
    leaf_range(B, R.ref, off, np);
    for (int i = 0; i < np; i++) {
        Tri T = load_tri(tris, off + i);
        cnt_tris++;
        float t = 0.f, u = 0.f, v = 0.f;
        bool ok = two_sided ? mt_two(T, R.o, R.d, t, u, v) : mt_cull(T, R.o, R.d, t, u, v);
        if (ok && !(t < 0.f) && t < t_hit) {
            t_hit = t;
            *hs.u = u;
            *hs.v = v;
            *hs.id = off + i;
        }
    }
}
// any-hit test of the leaf R.ref's triangles
__device__ __forceinline__ bool leaf_any(const Bvh& B, const float* __restrict__ tris, const TravRay& R,
                                         uint32_t& cnt_tris) {
    int off, np;
    leaf_range(B, R.ref, off, np);
    for (int i = 0; i < np; i++) {
        Tri T = load_tri(tris, off + i);
        cnt_tris++;
        float t = 0.f;
        if (mt_shadow(T, R.o, R.d, t) && t < K_HUGE) return true;
    }
    return false;
}

__device__ __forceinline__ Hit no_hit() {
    Hit h;
    h.t = K_HUGE; h.u = 0.f; h.v = 0.f; h.id = -1;
    return h;
}

// intersect_shadows with tmin = K_HUGE (CRT/dTriangle.cu:215-259,
// CRT/dEnvironmentLight.cu:60-64), one step.  Returns 0 while work remains,
// 1 when a triangle with 0 <= t < 1e32 is found, 2 when the ray is unoccluded.
template <bool WIDE = false>
__device__ __forceinline__ int any_step(const Bvh& B, const float* __restrict__ tris, TravRay& R, Stack& st,
                                        uint32_t& cnt_nodes, uint32_t& cnt_tris) {
    if (R.ref >= 0) {
        if (visit_node<WIDE, false>(B, R, 0.f, st, cnt_nodes)) return 0;
    } else if (leaf_any(B, tris, R, cnt_tris)) {
        return 1;
    }
    if (st.sp == 0) return 2;
    R.ref = st.pop();
    return 0;
}

// ------------------------------------------------- compressed wide walk --
// The records the renders and the ray queries walk (built by ff_pack.hip from
// the reference's binary tree): groups of four 64-byte records, one group per
// wide node, holding its up to four children.  A child is another wide node or
// one triangle.  A child reference is (record index | interior children of its
// group << 29); groups are 4-aligned and interior children come first, so a
// reference names a triangle exactly when (ref & 3) >= ref >> 29.
//   node:     (org.xyz, reference of the child group)
//             (lox01, lox23, loy01, loy23) (loz01, loz23, hix01, hix23)
//             (hiy01, hiy23, hiz01, hiz23)
//             child planes relative to org, two bfloat16 a word, rounded
//             outwards; an empty child has the box (+inf, -inf)
//   triangle: v0, e1, e2 (9 floats), slot, then the box of the reference's leaf
//             that holds the triangle (6 floats, exact)
// Which triangles the reference tests depends on leaf boxes alone: slab
// distances are monotone in the planes, so a leaf whose own box passes has
// ancestors that all pass.  The walk therefore may use any boxes that hold the
// leaf boxes, and a triangle that is hit counts only if its leaf's exact box
// passes the reference's test.  The closest hit is the smallest t, whatever
// the visit order; where two triangles share it exactly, or a box plane
// distance is NaN (0 * inf), the ray is traced again in the reference's order.
//
// Early hits: the t of a grazing hit is rounded so coarsely that it can lie
// before the entry into its own leaf's box, beyond the pruning's slack (a
// triangle 4.4 long met at an angle of 3e-6: t 20.4, entry 21.2).  Whether such
// a triangle is reached depends on the hits found before it, so it is no
// candidate and lowers no pruning limit; every triangle that is one is then
// reached whatever the order.  A ray with an early hit nearer than its closest
// candidate is traced again in the reference's order, which decides.  (An early
// hit is missed only where the walk in that order tests its leaf's box before it
// has a hit nearer than that box, and this walk after: 4 of 500000 grazing rays
// through random slivers.  With pruning that walk itself misses 3 of the hits
// that the same rays have without.)
#define WREF_INDEX 0x1fffffffu
#define WREF_ROOT (4u << 29)  // record 0, an interior child
// Slack of the conservative plane distances: a distance is fma(plane, inv, b)
// with b = (org - o) * inv.  Against the reference's (lo - o) * inv the two
// differ by at most 2.5 * 2^-23 |b| + 1.5 * 2^-23 |plane * inv|; the first is
// covered here, the second by the planes' padding (2^-16 of their value).
constexpr float WIDE_SLACK = 0x1p-21f;
constexpr float WIDE_INV_MAX = 0x1p80f;  // |1/d| used for boxes (a zero direction component stays finite)

struct WideRay {
    f3 o, d, inv;  // inv: 1 / d, clamped to +-WIDE_INV_MAX
    bool nx, ny, nz;
    uint32_t fl;   // XNAN_RAY, WINV_CLAMPED
};
constexpr uint32_t WINV_CLAMPED = 16u;

__device__ __forceinline__ void wide_begin(f3 o, f3 d, WideRay& R) {
    R.o = o;
    R.d = d;
    f3 inv = V3(1.f / d.x, 1.f / d.y, 1.f / d.z);
    R.nx = inv.x < 0;
    R.ny = inv.y < 0;
    R.nz = inv.z < 0;
    R.inv = V3(fminf(fmaxf(inv.x, -WIDE_INV_MAX), WIDE_INV_MAX), fminf(fmaxf(inv.y, -WIDE_INV_MAX), WIDE_INV_MAX),
               fminf(fmaxf(inv.z, -WIDE_INV_MAX), WIDE_INV_MAX));
    R.fl = ((isfinite(inv.x) && isfinite(o.x)) ? 0u : XNAN_RAY) |
           ((R.inv.x == inv.x && R.inv.y == inv.y && R.inv.z == inv.z) ? 0u : WINV_CLAMPED);
}

__device__ __forceinline__ const float4* wide_rec(const float4* rec, uint32_t ref) {
    return (const float4*)((const char*)rec + ((uint64_t)(ref & WREF_INDEX) << 6));
}
__device__ __forceinline__ bool wide_is_leaf(uint32_t ref) { return (ref & 3u) >= (ref >> 29); }

__device__ __forceinline__ int imin(int a, int b) { return a < b ? a : b; }
__device__ __forceinline__ int imax(int a, int b) { return a > b ? a : b; }
constexpr int WKEY_MISS = 0x7fffffff;

// One wide node: the entry and exit distances of the four child boxes (entry
// at least -PRUNE_BEHIND, exit at most lim); returns the child group's
// reference.  Child k may be entered unless tn[k] > tf[k].
template <bool PRUNE>
__device__ __forceinline__ uint32_t visit_wide(const float4* rec, uint32_t ref, const WideRay& R, float lim,
                                               float tn[4], float tf[4]) {
    const float4* p = wide_rec(rec, ref);
    float4 n0 = ldg4(p);
    int4 n1 = ldg4i((const int4*)(p + 1)), n2 = ldg4i((const int4*)(p + 2)), n3 = ldg4i((const int4*)(p + 3));
    float bx = (n0.x - R.o.x) * R.inv.x, by = (n0.y - R.o.y) * R.inv.y, bz = (n0.z - R.o.z) * R.inv.z;
    float bnx = __builtin_fmaf(-WIDE_SLACK, fabsf(bx), bx), bfx = __builtin_fmaf(WIDE_SLACK, fabsf(bx), bx);
    float bny = __builtin_fmaf(-WIDE_SLACK, fabsf(by), by), bfy = __builtin_fmaf(WIDE_SLACK, fabsf(by), by);
    float bnz = __builtin_fmaf(-WIDE_SLACK, fabsf(bz), bz), bfz = __builtin_fmaf(WIDE_SLACK, fabsf(bz), bz);
    const int lx[2] = {n1.x, n1.y}, ly[2] = {n1.z, n1.w}, lz[2] = {n2.x, n2.y};
    const int hx[2] = {n2.z, n2.w}, hy[2] = {n3.x, n3.y}, hz[2] = {n3.z, n3.w};
#pragma unroll
    for (int h = 0; h < 2; h++) {
        int ax = R.nx ? hx[h] : lx[h], ay = R.ny ? hy[h] : ly[h], az = R.nz ? hz[h] : lz[h];
        int cx = R.nx ? lx[h] : hx[h], cy = R.ny ? ly[h] : hy[h], cz = R.nz ? lz[h] : hz[h];
#pragma unroll
        for (int q = 0; q < 2; q++) {
            auto plane = [&](int w) {
                return __int_as_float(q ? (int)((uint32_t)w & 0xffff0000u) : (int)((uint32_t)w << 16));
            };
            float x0 = __builtin_fmaf(plane(ax), R.inv.x, bnx), x1 = __builtin_fmaf(plane(cx), R.inv.x, bfx);
            float y0 = __builtin_fmaf(plane(ay), R.inv.y, bny), y1 = __builtin_fmaf(plane(cy), R.inv.y, bfy);
            float z0 = __builtin_fmaf(plane(az), R.inv.z, bnz), z1 = __builtin_fmaf(plane(cz), R.inv.z, bfz);
            tn[2 * h + q] = fmaxf(fmaxf(x0, y0), fmaxf(z0, -PRUNE_BEHIND));
            tf[2 * h + q] = PRUNE ? fminf(fminf(x1, y1), fminf(z1, lim)) : fminf(fminf(x1, y1), z1);
        }
    }
    return __float_as_uint(n0.w);
}
// The children that may be entered, in order of entry distance: distance bits
// with the child number in the low two (WKEY_MISS: not entered).  Distances
// below zero (at least -PRUNE_BEHIND) order before every positive one.
__device__ __forceinline__ void wide_order(const float tn[4], const float tf[4], int key[4]) {
#pragma unroll
    for (int k = 0; k < 4; k++) key[k] = !(tn[k] > tf[k]) ? ((__float_as_int(tn[k]) & ~3) | k) : WKEY_MISS;
    int a = imin(key[0], key[1]), b = imax(key[0], key[1]), c = imin(key[2], key[3]), d = imax(key[2], key[3]);
    int m1 = imax(a, c), m2 = imin(b, d);
    key[0] = imin(a, c);
    key[3] = imax(b, d);
    key[1] = imin(m1, m2);
    key[2] = imax(m1, m2);
}

// One child box by one lane: the lanes 4q .. 4q + 3 of a wave share a ray and
// take a child each (k = lane & 3).
template <bool PRUNE>
__device__ __forceinline__ uint32_t visit_quad(const float4* rec, uint32_t ref, const WideRay& R, float lim, uint32_t k,
                                               float& tn, float& tf) {
    const float4* p = wide_rec(rec, ref);
    const int* w = (const int*)p + 4 + (k >> 1);  // the lane's pair of children
    float4 n0 = ldg4(p);
    int lx = ldg(w), ly = ldg(w + 2), lz = ldg(w + 4), hx = ldg(w + 6), hy = ldg(w + 8), hz = ldg(w + 10);
    float bx = (n0.x - R.o.x) * R.inv.x, by = (n0.y - R.o.y) * R.inv.y, bz = (n0.z - R.o.z) * R.inv.z;
    float bnx = __builtin_fmaf(-WIDE_SLACK, fabsf(bx), bx), bfx = __builtin_fmaf(WIDE_SLACK, fabsf(bx), bx);
    float bny = __builtin_fmaf(-WIDE_SLACK, fabsf(by), by), bfy = __builtin_fmaf(WIDE_SLACK, fabsf(by), by);
    float bnz = __builtin_fmaf(-WIDE_SLACK, fabsf(bz), bz), bfz = __builtin_fmaf(WIDE_SLACK, fabsf(bz), bz);
    const uint32_t sh = (k & 1u) ? 0u : 16u;
    auto plane = [&](int v) { return __uint_as_float(((uint32_t)v << sh) & 0xffff0000u); };
    float ax = plane(R.nx ? hx : lx), ay = plane(R.ny ? hy : ly), az = plane(R.nz ? hz : lz);
    float cx = plane(R.nx ? lx : hx), cy = plane(R.ny ? ly : hy), cz = plane(R.nz ? lz : hz);
    float x0 = __builtin_fmaf(ax, R.inv.x, bnx), x1 = __builtin_fmaf(cx, R.inv.x, bfx);
    float y0 = __builtin_fmaf(ay, R.inv.y, bny), y1 = __builtin_fmaf(cy, R.inv.y, bfy);
    float z0 = __builtin_fmaf(az, R.inv.z, bnz), z1 = __builtin_fmaf(cz, R.inv.z, bfz);
    tn = fmaxf(fmaxf(x0, y0), fmaxf(z0, -PRUNE_BEHIND));
    tf = PRUNE ? fminf(fminf(x1, y1), fminf(z1, lim)) : fminf(fminf(x1, y1), z1);
    return __float_as_uint(n0.w);
}
// values of the quad's other lanes (lane ^ X)
template <int X>
__device__ __forceinline__ int quad_xor(int v) {
    return __builtin_amdgcn_mov_dpp(v, X == 1 ? 0xB1 : (X == 2 ? 0x4E : 0x1B), 0xf, 0xf, true);
}
template <int X>
__device__ __forceinline__ float quad_xor(float v) {
    return __int_as_float(quad_xor<X>(__float_as_int(v)));
}

// A triangle record
struct WideTri {
    Tri T;
    int slot;
    f3 lo, hi;  // the reference leaf's box
};
__device__ __forceinline__ WideTri load_wide_tri(const float4* rec, uint32_t ref) {
    const float4* p = wide_rec(rec, ref);
    float4 a = ldg4(p), b = ldg4(p + 1), c = ldg4(p + 2), d = ldg4(p + 3);
    WideTri w;
    w.T.v0 = V3(a.x, a.y, a.z);
    w.T.e1 = V3(a.w, b.x, b.y);
    w.T.e2 = V3(b.z, b.w, c.x);
    w.slot = __float_as_int(c.y);
    w.lo = V3(c.z, c.w, d.x);
    w.hi = V3(d.y, d.z, d.w);
    return w;
}
// The reference's test of the triangle's leaf box, as its walk makes it; tn:
// the entry.  nanx: an x plane distance is NaN there, so ancestors may not follow.
__device__ __forceinline__ bool wide_leaf_box(const WideTri& w, const WideRay& R, bool& nanx, float& tn) {
    f3 inv = R.inv;
    float tf;
    nanx = false;
    if (__ballot(R.fl != 0u) == 0)
        return slab_box(w.lo.x, w.lo.y, w.lo.z, w.hi.x, w.hi.y, w.hi.z, R.o, inv, R.nx, R.ny, R.nz, tn, tf) &&
               !(tf < -PRUNE_BEHIND);
    if (R.fl & WINV_CLAMPED) inv = V3(1.f / R.d.x, 1.f / R.d.y, 1.f / R.d.z);
    nanx = (R.fl & XNAN_RAY) != 0u && (!isfinite(R.o.x) || R.o.x == w.lo.x || R.o.x == w.hi.x);
    return slab(w.lo.x, w.lo.y, w.lo.z, w.hi.x, w.hi.y, w.hi.z, R.o, inv, R.nx, R.ny, R.nz, tn, tf) &&
           !(tf < -PRUNE_BEHIND);
}
// an early hit: the leaf is entered (tn) beyond the pruning limit of the hit's own t
__device__ __forceinline__ bool early_hit(float t, float tn) { return tn > prune_lim(t); }
__device__ __forceinline__ void wide_leaf_closest(const float4* rec, uint32_t ref, const WideRay& R, float& t_hit,
                                                  const HitSlots& hs, bool two_sided) {
    WideTri w = load_wide_tri(rec, ref);
    float t = 0.f, u = 0.f, v = 0.f;
    bool ok = two_sided ? mt_two(w.T, R.o, R.d, t, u, v) : mt_cull(w.T, R.o, R.d, t, u, v);
    if (ok && !(t < 0.f) && t <= t_hit) {
        bool nanx;
        float tn;
        if (wide_leaf_box(w, R, nanx, tn)) {
            const bool early = early_hit(t, tn);
            if (early || nanx || t == t_hit) *hs.redo = fminf(*hs.redo, t);
            if (!early && t < t_hit) {
                t_hit = t;
                *hs.u = u;
                *hs.v = v;
                *hs.id = w.slot;
            }
        }
    }
}
// 0: no hit, 1: occluded, 2: to be traced again in the reference's order
__device__ __forceinline__ int wide_leaf_any(const float4* rec, uint32_t ref, const WideRay& R) {
    WideTri w = load_wide_tri(rec, ref);
    float t = 0.f;
    if (!(mt_shadow(w.T, R.o, R.d, t) && t < K_HUGE)) return 0;
    bool nanx;
    float tn;
    if (!wide_leaf_box(w, R, nanx, tn)) return 0;
    return nanx ? 2 : 1;
}

__device__ __forceinline__ void lds_count(lds_u32* word, uint32_t n) {
    __hip_atomic_fetch_add(word, n, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
// One ray in the reference's order over the binary records (the rare rays
// above), one box or triangle in registers at a time, so that it adds no
// registers to the kernels that hold it: the boxes and triangles it tests are
// added to two words in LDS (again, or null), which add_tested() hands on.  (In
// registers they took the seven-wave form from 44 spills to 81; in the lane's
// stack to 60, and a 1021x577 8-sample render from 4.03 to 4.09 ms.)
template <bool ANY, class S>
__device__ __forceinline__ Hit reference_walk(const Bvh& B, const float* __restrict__ tris, f3 o, f3 d, bool two_sided,
                                              S& st, lds_u32* again) {
    Hit h = no_hit();
    const f3 inv = V3(1.f / d.x, 1.f / d.y, 1.f / d.z);
    const bool nx = inv.x < 0, ny = inv.y < 0, nz = inv.z < 0;
    float tn, tf;
    int ref = __float_as_int(ldg(B.root + 6));
    if (again) lds_count(again, 1u);
    if (!slab(ldg(B.root), ldg(B.root + 1), ldg(B.root + 2), ldg(B.root + 3), ldg(B.root + 4), ldg(B.root + 5), o, inv,
              nx, ny, nz, tn, tf) ||
        tf < -PRUNE_BEHIND)
        return h;
    st.sp = 0;
    for (;;) {
        bool down = false;
        if (ref >= 0) {
            const float* n = (const float*)((const char*)B.nodes + ((uint64_t)(uint32_t)ref << 6));
            bool hit[2];
            if (again) lds_count(again, 2u);
#pragma unroll 1
            for (int c = 0; c < 2; c++) {
                const float* b = n + 6 * c;
                bool in = slab(ldg(b), ldg(b + 1), ldg(b + 2), ldg(b + 3), ldg(b + 4), ldg(b + 5), o, inv, nx, ny, nz,
                               tn, tf) &&
                          !(tf < -PRUNE_BEHIND) && (ANY || !(tn > prune_lim(h.t)));
                if (c == 0) hit[0] = in;
                else hit[1] = in;
            }
            const int axis = __float_as_int(ldg(n + 14));
            const bool neg = axis == 0 ? nx : (axis == 1 ? ny : nz);
            const int r0 = __float_as_int(ldg(n + 12)), r1 = __float_as_int(ldg(n + 13));
            if (hit[0] && hit[1]) st.push(neg ? r0 : r1);
            down = hit[0] || hit[1];
            if (down) ref = hit[0] && hit[1] ? (neg ? r1 : r0) : (hit[0] ? r0 : r1);
        } else {
            int off, np;
            leaf_range(B, ref, off, np);
#pragma unroll 1
            for (int i = off; i < off + np; i++) {
                Tri T = load_tri(tris, i);
                float t = 0.f, u = 0.f, v = 0.f;
                if (again) lds_count(again + 1, 1u);
                if (ANY) {
                    if (mt_shadow(T, o, d, t) && t < K_HUGE) {
                        h.id = i;
                        return h;
                    }
                } else {
                    bool ok = two_sided ? mt_two(T, o, d, t, u, v) : mt_cull(T, o, d, t, u, v);
                    if (ok && !(t < 0.f) && t < h.t) { h.t = t; h.u = u; h.v = v; h.id = i; }
                }
            }
        }
        if (!down) {
            if (st.sp == 0) return h;
            ref = st.pop();
        }
    }
}

// At a wave's end (one lane): the records and triangles it tested and, of the
// workgroup's rays traced again, what has been counted since the last wave's
// end (every wave counts its own before, so the last one takes the rest).
__device__ __forceinline__ void add_tested(unsigned long long* cnt, uint32_t records, uint32_t tris, lds_u32* again) {
    const uint32_t b = __hip_atomic_exchange(again, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    const uint32_t t = __hip_atomic_exchange(again + 1, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    atomicAdd(&cnt[0], 4ull * records + b);
    atomicAdd(&cnt[1], (unsigned long long)tris + t);
}

// ----------------------------------------------------- wave64 utilities --
// Sum of a per-lane value over a full wave, added once per wave.  Must be
// called with every lane of the wave active (after the grid-stride loop).
__device__ __forceinline__ void wave_sum_add(unsigned long long* counter, uint32_t v) {
    unsigned long long s = v;
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off);
    if (__lane_id() == 0) atomicAdd(counter, s);
}

// Queue appends staged in LDS.  A device-scope atomic on one address costs
// about 11 ns at the memory side however many workgroups issue it, so one
// atomic per queue per 256-path tile (a pass over 133 M paths: 520 k of them
// on each counter) bounds a kernel at several milliseconds.  A workgroup
// instead collects the entries of several tiles in LDS and appends each
// queue's run with one atomic when fewer than BS free places remain (and at
// the end): CAP / BS times fewer atomics, and the runs are written coalesced.
// Each lane adds at most one entry per add(), so the staged count grows by at
// most BS per add(): flush_if_full(..., adds) makes room for the next `adds`
// calls of add() (a workgroup that stages two entries per thread per tile
// passes 2).  Every thread of the workgroup calls add(), flush_if_full() and
// flush() the same number of times.
template <int BS, int NQ, int CAP>
struct QStage {
    static constexpr int NW = BS / 64;
    static_assert(CAP >= 4 * BS && NQ < BS && NQ <= 16, "staging room for several adds");
    uint32_t val[CAP];       // entry values
    uint32_t pos[CAP];       // queue << 28 | rank in the queue's run
    uint32_t wtot[NQ][NW];   // this add's entries per queue and wave
    uint32_t fill[NQ];       // entries staged per queue
    uint32_t base[NQ];       // first queue place of each run (flush)
    uint32_t total;          // entries staged

    __device__ __forceinline__ void init() {
        if (threadIdx.x < NQ) fill[threadIdx.x] = 0u;
        if (threadIdx.x == 0) total = 0u;
        __syncthreads();
    }
    // q: the lane's queue (-1: no entry), v: the entry
    __device__ __forceinline__ void add(int q, uint32_t v) {
        const uint32_t w = threadIdx.x >> 6;
        uint32_t rank_q = 0u;
#pragma unroll
        for (int k = 0; k < NQ; k++) {
            uint64_t b = __ballot(q == k);
            uint32_t r = __builtin_amdgcn_mbcnt_hi((uint32_t)(b >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)b, 0u));
            if (q == k) rank_q = r;
            if (__lane_id() == 0) wtot[k][w] = (uint32_t)__popcll(b);
        }
        uint64_t ball = __ballot(q >= 0);
        uint32_t rank_all = __builtin_amdgcn_mbcnt_hi((uint32_t)(ball >> 32),
                                                      __builtin_amdgcn_mbcnt_lo((uint32_t)ball, 0u));
        __syncthreads();
        if (q >= 0) {
            uint32_t off_all = 0u, off_q = 0u;
            for (uint32_t ww = 0; ww < w; ww++) {
#pragma unroll
                for (int k = 0; k < NQ; k++) off_all += wtot[k][ww];
                off_q += wtot[q][ww];
            }
            uint32_t slot = total + off_all + rank_all;
            val[slot] = v;
            pos[slot] = ((uint32_t)q << 28) | (fill[q] + off_q + rank_q);
        }
        __syncthreads();
        if (threadIdx.x <= (unsigned)NQ) {
            uint32_t t = 0u;
            if (threadIdx.x < (unsigned)NQ) {
                for (int ww = 0; ww < NW; ww++) t += wtot[threadIdx.x][ww];
                fill[threadIdx.x] += t;
            } else {
                for (int k = 0; k < NQ; k++)
                    for (int ww = 0; ww < NW; ww++) t += wtot[k][ww];
                total += t;
            }
        }
        __syncthreads();
    }
    // appends every staged run: queue q's entries go to queues[q] from the
    // place an atomic on counters[qidx[q]] returns
    __device__ __forceinline__ void flush(uint32_t* counters, const int* qidx, uint32_t* const* queues) {
        if (threadIdx.x < (unsigned)NQ) {
            uint32_t f = fill[threadIdx.x];
            base[threadIdx.x] = f ? atomicAdd(&counters[qidx[threadIdx.x]], f) : 0u;
        }
        __syncthreads();
        const uint32_t T = total;
        for (uint32_t k = threadIdx.x; k < T; k += BS) {
            uint32_t p = pos[k];
            uint32_t q = p >> 28;
            uint32_t* dst = queues[0];
#pragma unroll
            for (int j = 1; j < NQ; j++)
                if (q == (uint32_t)j) dst = queues[j];
            dst[base[q] + (p & 0x0fffffffu)] = val[k];
        }
        __syncthreads();
        if (threadIdx.x < (unsigned)NQ) fill[threadIdx.x] = 0u;
        if (threadIdx.x == 0) total = 0u;
        __syncthreads();
    }
    __device__ __forceinline__ void flush_if_full(uint32_t* counters, const int* qidx, uint32_t* const* queues,
                                                  uint32_t adds = 1u) {
        // total is the same for every thread; afterwards total + adds * BS <= CAP
        if (total + adds * BS > CAP) flush(counters, qidx, queues);
    }
};

// The work counters in device memory (SegFetch): lane 0 claims; lane k reads
// counter k with a device-coherent load, one round trip for all.
static_assert(FETCH_SEGS == 64, "one segment per lane of the scan");
struct DevCounters {
    uint32_t* ctr;  // FETCH_SEGS counters, FETCH_STRIDE words apart
    __device__ __forceinline__ uint32_t claim(uint32_t seg, uint32_t want) const {
        uint32_t base = 0;
        if (__lane_id() == 0) base = atomicAdd(ctr + (size_t)seg * FETCH_STRIDE, want);
        return __shfl(base, 0);
    }
    template <class F>
    __device__ __forceinline__ uint64_t open(const F& f) const {
        const uint32_t k = __lane_id();
        const uint32_t lk = f.seg_size(k);
        const uint32_t v = lk ? __hip_atomic_load(ctr + (size_t)k * FETCH_STRIDE, __ATOMIC_RELAXED,
                                                  __HIP_MEMORY_SCOPE_AGENT)
                              : 0u;
        return __ballot(lk > 0 && v < lk);
    }
    __device__ __forceinline__ uint32_t uniform(uint32_t v) const {
        return (uint32_t)__builtin_amdgcn_readfirstlane((int)v);
    }
};

}  // namespace ffd
