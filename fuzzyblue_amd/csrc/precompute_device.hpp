// precompute_device.hpp — what the precompute passes' translation units
// share: the density quadrature's direction tables, nu profiles in LDS,
// batch tiles and block order.
#pragma once

#include <math.h>
#include <algorithm>

#include "atmo_device.hpp"
#include "kernels.hpp"

// The constant address space (read-only for the whole kernel): loads through
// it are scalar when uniform, and addresses loaded from it are known to
// point to global memory.  The host pass only parses device code, without
// address spaces.
#if defined(__HIP_DEVICE_COMPILE__)
#define FB_CONSTANT_AS __attribute__((address_space(4)))
#else
#define FB_CONSTANT_AS
#endif

namespace fbk {

// Direction tables of the density quadrature, computed once on the host in
// binary32 exactly as the reference evaluates them (scattering_density.comp:
// 34-66), and in binary64 for the precision mode's geometry: l = 0..15
// (theta), m = 0..31 (phi), dtheta = dphi = pi/16.  One symbol, so that a
// builder uploads it with one copy, in each translation unit that reads it.
struct DensityTables {
    float4 dir[kDenTheta * kDenPhi];     // (cos phi sin t, sin phi sin t, cos t, domega)
    float2 phi[kDenPhi / 2];             // cos phi, sin phi of the half turn m < 16
    float cx[kDenTheta * kDenPhi / 2];   // dir's x of the half turn
    float cos[kDenTheta], sin[kDenTheta];
    double cos_d[kDenTheta];

    static DensityTables make() {
        DensityTables t;
        const float PI = 3.14159265358979323846f;
        const float dphi = PI / float(16), dtheta = PI / float(16);
        const double dtheta_d = M_PI / 16.0;
        for (int l = 0; l < kDenTheta; ++l) {
            const float theta = (float(l) + 0.5f) * dtheta;
            const float ct = cosf(theta), st = sinf(theta);
            t.cos[l] = ct;
            t.sin[l] = st;
            t.cos_d[l] = ::cos((double(l) + 0.5) * dtheta_d);
            for (int m = 0; m < kDenPhi; ++m) {
                const float phi = (float(m) + 0.5f) * dphi;
                const float domega = dtheta * dphi * sinf(theta);
                t.dir[l * kDenPhi + m] = make_float4(cosf(phi) * st, sinf(phi) * st, ct, domega);
                if (m < kDenPhi / 2) {
                    t.phi[m] = make_float2(cosf(phi), sinf(phi));
                    t.cx[l * kDenPhi / 2 + m] = t.dir[l * kDenPhi + m].x;
                }
            }
        }
        return t;
    }
};
static __constant__ DensityTables c_den;

static hipError_t upload_density_tables() {
    static const DensityTables t = DensityTables::make();
    return hipMemcpyToSymbol(HIP_SYMBOL(c_den), &t, sizeof(t));
}

template <typename G>
__device__ __forceinline__ G den_cos(int l);
template <>
__device__ __forceinline__ float den_cos<float>(int l) { return c_den.cos[l]; }
template <>
__device__ __forceinline__ double den_cos<double>(int l) { return c_den.cos_d[l]; }

// ------------------------------------------------------------ nu profiles
template <typename G>
__device__ __forceinline__ Taps slice_taps(const DevParams& P, int slice, G u_mu_s) {
    G x = (G(slice) + u_mu_s) / G(P.s_nu);
    return linear_taps<G>(x, P.s_nu * P.s_mus);
}

// H: the texture is binary16 (FB_FLAG_F16_STORAGE).
template <bool H>
__device__ __forceinline__ float4 trilinear_taps_t(const DevParams& P,
                                                   const float4* __restrict__ tex, const Taps& tx,
                                                   const Taps& ty, const Taps& tz) {
    const int W = P.s_nu * P.s_mus;
    const size_t p00 = (size_t(tz.i0) * P.s_mu + ty.i0) * W;
    const size_t p01 = (size_t(tz.i0) * P.s_mu + ty.i1) * W;
    const size_t p10 = (size_t(tz.i1) * P.s_mu + ty.i0) * W;
    const size_t p11 = (size_t(tz.i1) * P.s_mu + ty.i1) * W;
    auto at = [&](size_t row, int x) { return ld_tex(tex, row + x, H); };
    return lerp4(lerp4(lerp4(at(p00, tx.i0), at(p00, tx.i1), tx.w),
                       lerp4(at(p01, tx.i0), at(p01, tx.i1), tx.w), ty.w),
                 lerp4(lerp4(at(p10, tx.i0), at(p10, tx.i1), tx.w),
                       lerp4(at(p11, tx.i0), at(p11, tx.i1), tx.w), ty.w),
                 tz.w);
}

// A profile entry: the value at slot k (rgb) and the difference to slot
// k+1, so a lerp is one fma per channel.  32-byte stride; a lookup reads
// 24 bytes (one b128 and one b64 LDS load).
struct ProfEntry {
    float4 a;  // v.r, v.g, v.b, d.r
    float2 b;  // d.g, d.b
    float2 pad;
};

// Linear filtering at texel coordinate t over entries e = k+1, k in
// [-1, kmax]: entry 0 holds the clamped left edge and entry kmax+1 the
// clamped right edge, which reproduces CLAMP_TO_EDGE.  Callers pass a
// finite t (their inputs are clamped unit vectors); the med3 clamp keeps
// the entry index inside [0, kmax+1].
__device__ __forceinline__ float3 prof_lerp(const ProfEntry* __restrict__ prof, float t,
                                            float kmax) {
    float k = floorf(t);
    float f = t - k;
    k = __builtin_amdgcn_fmed3f(k, -1.0f, kmax);
    const ProfEntry* e = prof + (int(k) + 1);
    float4 a = e->a;
    float2 b = e->b;
    return make_float3(fmaf(a.w, f, a.x), fmaf(b.x, f, a.y), fmaf(b.y, f, a.z));
}

// 1/x^1.5 for x >= (1-|g|)^2 > 0: the raw v_rsq_f32 (no denormal rescaling
// is needed for this range).
__device__ __forceinline__ float rsqrt_cubed(float x) {
    float r = __builtin_amdgcn_rsqf(x);
    return r * r * r;
}

__device__ __forceinline__ ProfEntry make_entry(float4 v, float4 w) {
    ProfEntry e;
    e.a = make_float4(v.x, v.y, v.z, w.x - v.x);
    e.b = make_float2(w.y - v.y, w.z - v.z);
    e.pad = make_float2(0.0f, 0.0f);
    return e;
}

// Order 2 (single scattering as incident radiance): the Rayleigh and Mie
// profile entries of one slot side by side, so that one lookup reads both
// with three b128 LDS reads instead of two b128 + b64 pairs.
struct PairEntry {
    float4 a;  // R: v.r, v.g, v.b, d.r
    float4 b;  // R: d.g, d.b; M: v.r, v.g
    float4 c;  // M: v.b, d.r, d.g, d.b
};

// Dynamic LDS of a density block: the raw profiles (float4 per texture,
// theta row and nu slot), whose space the irradiance entries reuse once the
// profile entries are built; the entries (PairEntry at order 2, ProfEntry
// after); the x taps of the NU + 2 slots.  Kept small: at order 2 it sets
// how many blocks share a CU.
inline size_t density_lds_bytes(int nu, int i_mus, bool single) {
    const int ntex = single ? 2 : 1;
    const size_t raw = sizeof(float4) * size_t(ntex) * kDenTheta * (nu + 2);
    const size_t erow = sizeof(ProfEntry) * size_t(i_mus + 1);
    const size_t ent = (single ? sizeof(PairEntry) : sizeof(ProfEntry)) * kDenTheta * (nu + 1);
    return std::max(raw, erow) + ent + sizeof(Taps) * size_t(nu + 2);
}

// -------------------------------------------------------- tiles and blocks
__device__ __forceinline__ void decode_tile(uint32_t t, int& atm, int& local) {
    atm = int(t >> 24);
    local = int(t & 0xffffffu);
}
// Batched kernels read the LUT addresses from memory.  Read through the
// constant address space (the arrays are written by the host before the
// launch and only read here), the loaded addresses are known to point to
// global memory, so the compiler emits global rather than flat accesses
// (flat ones also count against the LDS wait counter, serialising LDS and
// memory waits).
typedef FB_CONSTANT_AS const LutPtrs ConstLutPtrs;
__device__ __forceinline__ LutPtrs lut_ptrs(const LutPtrs* L, int atm) {
    return ((ConstLutPtrs*)L)[atm];
}
// Workgroups go to the 8 XCDs round-robin by linear id, and each XCD has
// its own L2.  With `remap` set, XCD k instead runs the k-th contiguous
// share of the logical blocks, so blocks of neighbouring rows / tiles, which
// read overlapping LUT rows, share an L2.  A bijection on [0, N).
constexpr unsigned kXcds = 8;
__device__ __forceinline__ unsigned xcd_remap(unsigned L, unsigned N) {
    const unsigned xcd = L % kXcds, local = L / kXcds;
    const unsigned per = N / kXcds, rem = N % kXcds;
    return xcd * per + min(xcd, rem) + local;
}
__device__ __forceinline__ unsigned logical_block(bool remap) {
    const unsigned L = blockIdx.x + gridDim.x * (blockIdx.y + gridDim.y * blockIdx.z);
    return remap ? xcd_remap(L, gridDim.x * gridDim.y * gridDim.z) : L;
}

static inline unsigned cdiv(size_t a, size_t b) { return unsigned((a + b - 1) / b); }

}  // namespace fbk
