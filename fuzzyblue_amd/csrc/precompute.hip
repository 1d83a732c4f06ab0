// precompute.hip — the six precompute passes of the reference as CDNA4
// kernels (shaders/transmittance.comp, direct_irradiance.comp,
// single_scattering.comp, scattering_density.comp, indirect_irradiance.comp,
// multiple_scattering.comp), plus the irradiance clear.  The scattering
// density's kernels are in density.hpp, compiled by density_f32.hip and
// density_f64.hip.
//
// Every LUT is a row-major float4 array in HBM (x fastest).  Launch
// wrappers at the bottom take a DevParams by value and raw device pointers;
// the host runtime (runtime.hip) owns allocation and ordering.
#include <math.h>
#include <type_traits>

#include "precompute_device.hpp"

namespace fbk {

// ------------------------------------------------------------------ tables
// Direction tables of the irradiance quadrature, as the density's
// (precompute_device.hpp): j = 0..15 (theta), i = 0..63 (phi), dtheta = dphi
// = pi/32 (indirect_irradiance.comp:20-33).
struct IrradianceTables {
    float4 dir[kIndTheta * kIndPhi];
    float cos[kIndTheta];
    double cos_d[kIndTheta];

    static IrradianceTables make() {
        IrradianceTables t;
        const float PI = 3.14159265358979323846f;
        const float dphi = PI / float(32), dtheta = PI / float(32);
        const double dtheta_d = M_PI / 32.0;
        for (int j = 0; j < kIndTheta; ++j) {
            const float theta = (float(j) + 0.5f) * dtheta;
            t.cos[j] = cosf(theta);
            t.cos_d[j] = ::cos((double(j) + 0.5) * dtheta_d);
            for (int i = 0; i < kIndPhi; ++i) {
                const float phi = (float(i) + 0.5f) * dphi;
                const float domega = dtheta * dphi * sinf(theta);
                t.dir[j * kIndPhi + i] = make_float4(cosf(phi) * sinf(theta),
                                                     sinf(phi) * sinf(theta), cosf(theta), domega);
            }
        }
        return t;
    }
};
__constant__ IrradianceTables c_ind;

hipError_t upload_tables() {
    static const IrradianceTables t = IrradianceTables::make();
    hipError_t e = hipMemcpyToSymbol(HIP_SYMBOL(c_ind), &t, sizeof(t));
    if (e != hipSuccess) return e;
    // Each translation unit that reads the density tables has its own.
    if ((e = upload_density_tables()) != hipSuccess) return e;
    if ((e = DensityLaunch<float>::upload()) != hipSuccess) return e;
    return DensityLaunch<double>::upload();
}

template <typename G>
__device__ __forceinline__ G ind_cos(int j);
template <>
__device__ __forceinline__ float ind_cos<float>(int j) { return c_ind.cos[j]; }
template <>
__device__ __forceinline__ double ind_cos<double>(int j) { return c_ind.cos_d[j]; }

// Running sum with optional Neumaier compensation (precision mode).
template <bool COMP>
struct Sum {
    float s = 0.0f, c = 0.0f;
    __device__ __forceinline__ void add(float x) {
        if (COMP) {
            float t = s + x;
            if (fabsf(s) >= fabsf(x))
                c += (s - t) + x;
            else
                c += (x - t) + s;
            s = t;
        } else {
            s = s + x;
        }
    }
    __device__ __forceinline__ float value() const { return COMP ? s + c : s; }
};

// ============================================================ 1. transmittance
// transmittance.comp:8-46,71-80.  LANES lanes per texel: lane s sums the
// trapezoid samples k = s, s+LANES, ... of all three optical lengths (the
// reference recomputes r_i per profile with identical inputs), then the
// partial sums are combined with lane shuffles: the precision mode, 16
// lanes with compensated partial sums.  The FP32 mode keeps the reference's
// sequential summation order, so its rounding matches the reference's
// (transmittance_block_ordered below).
// T = exp(-(beta_R L_R + beta_M,ext L_M + beta_abs L_O)) (transmittance.comp:
// 34-46) for texel (i, j); with OD, also the optical depth itself, for
// transmittances below binary32's range (see log_transmittance_to_top).
__device__ __forceinline__ void store_transmittance(const DevParams& P, int i, int j, float LR,
                                                    float LM, float LO, float4* __restrict__ T,
                                                    float4* __restrict__ OD) {
    const float t0 = P.rayleigh_scattering[0] * LR + P.mie_extinction[0] * LM +
                     P.absorption_extinction[0] * LO;
    const float t1 = P.rayleigh_scattering[1] * LR + P.mie_extinction[1] * LM +
                     P.absorption_extinction[1] * LO;
    const float t2 = P.rayleigh_scattering[2] * LR + P.mie_extinction[2] * LM +
                     P.absorption_extinction[2] * LO;
    T[j * P.t_mu + i] = make_float4(expf(-t0), expf(-t1), expf(-t2), 1.0f);
    if (OD) OD[j * P.t_mu + i] = make_float4(t0, t1, t2, 0.0f);
}

template <typename G, bool COMP, int LANES>
__device__ __forceinline__ void transmittance_block(const DevParams& P, const int bx, const int by, const int bz, float4* __restrict__ T, float4* __restrict__ OD) {
    const int sub = threadIdx.x % LANES;
    const int texel = (bx * blockDim.x + threadIdx.x) / LANES;
    const int n = P.t_mu * P.t_r;
    const bool active = texel < n;
    const int i = active ? texel % P.t_mu : 0, j = active ? texel / P.t_mu : 0;
    G x_mu = G(i) / G(P.t_mu - 1);
    G x_r = G(j) / G(P.t_r - 1);
    G r, mu;
    rmu_from_transmittance_unit<G>(P, x_mu, x_r, r, mu);
    const int SAMPLE_COUNT = 500;
    G dx = distance_to_top<G>(P, r, mu) / G(SAMPLE_COUNT);
    float dxf = float(dx);
    Sum<COMP> lr, lm, lo;
    // Two samples per iteration: their square-root and exp chains overlap
    // (35-36 -> 32 us for 256x64 texels; the sums still add in k order).
#pragma unroll 2
    for (int k = sub; k <= SAMPLE_COUNT; k += LANES) {
        G d_i = G(k) * dx;
        // (r_i - bottom exactly as the oracle forms it: the density profile
        // switches layer at altitude 0, so a sample at the horizon ray's
        // tangent point must round the same way.)
        G r_i = sqrt(d_i * d_i + G(2) * r * mu * d_i + r * r);
        float alt = float(r_i - G(P.bottom));
        float w = (k == 0 || k == SAMPLE_COUNT) ? 0.5f : 1.0f;
        lr.add(profile_density(P.prof[0], alt) * w * dxf);
        lm.add(profile_density(P.prof[1], alt) * w * dxf);
        lo.add(profile_density(P.prof[2], alt) * w * dxf);
    }
    float LR = lr.value(), LM = lm.value(), LO = lo.value();
    for (int off = 1; off < LANES; off <<= 1) {
        LR += __shfl_xor(LR, off, 64);
        LM += __shfl_xor(LM, off, 64);
        LO += __shfl_xor(LO, off, 64);
    }
    if (!active || sub != 0) return;
    store_transmittance(P, i, j, LR, LM, LO, T, OD);
}

// Lanes per texel of the FP32-mode transmittance (a wavefront; the kernels
// pick transmittance_block_ordered for this lane count).
constexpr int kOrderedLanes = 64;

// FP32 mode: the reference's summation order — per profile, s = s + term
// for k = 0..500 in sequence (transmittance.comp:16-31) — with the terms
// computed by a wavefront's 64 lanes in parallel (each term by the same
// binary32 operations as in the sequential loop) and summed in order, one
// lane per profile.  Bit-identical to one lane doing all of it.
template <typename G>
__device__ __forceinline__ void transmittance_block_ordered(const DevParams& P, const int bx,
                                                            float4* __restrict__ T) {
    constexpr int SAMPLE_COUNT = 500;
    // Per wavefront of a 256-thread block; rows padded to 504 floats so that
    // each starts 16-byte aligned (read as float4 below).
    __shared__ __align__(16) float s_terms[4][3][504];
    const int wave = threadIdx.x / 64, lane = threadIdx.x % 64;
    const int texel = bx * int(blockDim.x / 64) + wave;
    const int n = P.t_mu * P.t_r;
    const bool active = texel < n;
    const int i = active ? texel % P.t_mu : 0, j = active ? texel / P.t_mu : 0;
    G x_mu = G(i) / G(P.t_mu - 1);
    G x_r = G(j) / G(P.t_r - 1);
    G r, mu;
    rmu_from_transmittance_unit<G>(P, x_mu, x_r, r, mu);
    G dx = distance_to_top<G>(P, r, mu) / G(SAMPLE_COUNT);
    float dxf = float(dx);
    for (int k = lane; k <= SAMPLE_COUNT; k += 64) {
        G d_i = G(k) * dx;
        G r_i = sqrt(d_i * d_i + G(2) * r * mu * d_i + r * r);
        float alt = float(r_i - G(P.bottom));
        float w = (k == 0 || k == SAMPLE_COUNT) ? 0.5f : 1.0f;
        s_terms[wave][0][k] = profile_density(P.prof[0], alt) * w * dxf;
        s_terms[wave][1][k] = profile_density(P.prof[1], alt) * w * dxf;
        s_terms[wave][2][k] = profile_density(P.prof[2], alt) * w * dxf;
    }
    // The first wavefront sums the block's four texels, one lane per texel and
    // profile: a quarter of the issue slots of each wavefront summing its own.
    __shared__ float s_len[12];
    __syncthreads();
    if (threadIdx.x < 12) {
        // Terms 0..499 four at a time (still added one by one, in order),
        // then term 500.
        const float* tp = s_terms[threadIdx.x / 3][threadIdx.x % 3];
        const float4* tp4 = reinterpret_cast<const float4*>(tp);
        float L = 0.0f;
#pragma unroll 5
        for (int q = 0; q < SAMPLE_COUNT / 4; ++q) {
            const float4 v = tp4[q];
            L = L + v.x;
            L = L + v.y;
            L = L + v.z;
            L = L + v.w;
        }
        s_len[threadIdx.x] = L + tp[SAMPLE_COUNT];
    }
    __syncthreads();
    if (!active || lane != 0) return;
    const float LR = s_len[3 * wave], LM = s_len[3 * wave + 1], LO = s_len[3 * wave + 2];
    store_transmittance(P, i, j, LR, LM, LO, T, nullptr);
}

// ====================================================== 2. direct irradiance
// direct_irradiance.comp:10-46
template <typename G>
__device__ __forceinline__ void direct_irradiance_block(const DevParams& P, const int bx, const int by, const int bz,
                                                           const float4* __restrict__ T,
                                                           float4* __restrict__ dE) {
    int i = bx * blockDim.x + threadIdx.x;
    int j = by;
    if (i >= P.i_mus || j >= P.i_r) return;
    G x_mu_s = G(i) / G(P.i_mus - 1);
    G x_r = G(j) / G(P.i_r - 1);
    G r, mu_s;
    rmus_from_irradiance_unit<G>(P, x_mu_s, x_r, r, mu_s);
    G alpha_s = G(P.sun_angular_radius);
    G avg = mu_s < -alpha_s
                ? G(0)
                : (mu_s > alpha_s ? mu_s : (mu_s + alpha_s) * (mu_s + alpha_s) / (G(4) * alpha_s));
    float a = float(avg);
    float3 t = transmittance_to_top<G>(P, T, r, mu_s);
    dE[j * P.i_mus + i] =
        make_float4(P.solar[0] * t.x * a, P.solar[1] * t.y * a, P.solar[2] * t.z * a, 0.0f);
}


// ===================================================== 3. single scattering
// single_scattering.comp:10-101.
//
// As for multiple scattering, the texels of one (r, mu) row share the view
// ray: for each of the 51 samples, d_i, r_d, the view transmittance
// T(r, mu, d_i), the densities at r_d and the transmittance-LUT row taps
// and horizon terms of r_d are computed once per row (row_geometry_block,
// in the per-set geometry pass) and read from the row table.  Each texel
// then evaluates only its sun transmittance T(r_d, mu_s_d) (one bilinear
// lookup) and accumulates.

// Multiple scattering interpolates each sample's value from four density
// rows, (r0, mu0), (r0, mu1), (r1, mu0), (r1, mu1).  Consecutive samples of
// a ray often share rows (the same cell, or the next one in mu or r: at
// default sizes 79 distinct rows serve the 204 taps of an (r, mu) row), so
// the kernel keeps four row "slots" in registers from sample to sample.
// Row (r index z, mu index y) always lives in slot 2*(z & 1) + (y & 1):
// the rows of one sample differ by at most one step in z and in y, so they
// never collide (clamped duplicates are the same row), and a row shared by
// consecutive samples stays where it is.  Per sample, the table gives the
// slots to load (a used slot is loaded unless the previous sample used it
// for the same row), the row offsets to load, and each slot's weight: the
// summed bilinear weights of its taps, 0 for an unused slot.
struct MsSlots {
    int mask;   // bit s: load slot s
    int4 load;  // row offset loaded into slot s (0 when not loaded)
    float4 w;   // slot weights
};
// i: this lane's sample; z[k], y[k], off[k], wt[k]: its taps (A, B, C, D).
// Every lane of the wavefront calls this (lane i holds sample i; lanes past
// the last sample repeat it).
__device__ __forceinline__ MsSlots ms_row_slots(int i, const int z[4], const int y[4],
                                                const int off[4], const float wt[4]) {
    int row[4] = {-1, -1, -1, -1};  // row offset held by each slot, -1 if unused
    float w[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const int s = ((z[k] & 1) << 1) | (y[k] & 1);
#pragma unroll
        for (int t = 0; t < 4; ++t)
            if (t == s) {
                row[t] = off[k];
                w[t] += wt[k];
            }
    }
    MsSlots r{0, make_int4(0, 0, 0, 0), make_float4(w[0], w[1], w[2], w[3])};
    int ld[4] = {0, 0, 0, 0};
#pragma unroll
    for (int t = 0; t < 4; ++t) {
        const int prev = __shfl_up(row[t], 1, 64);  // sample i - 1's slot t
        if (row[t] >= 0 && (i == 0 || prev != row[t])) {
            r.mask |= 1 << t;
            ld[t] = row[t];
        }
    }
    r.load = make_int4(ld[0], ld[1], ld[2], ld[3]);
    return r;
}

// The single- and multiple-scattering row tables of row (y, z): thread i
// computes sample i.  The multiple-scattering passes march the same 51
// samples (multiple_scattering.comp:16-47, the same dx and d_i).
template <typename G>
__device__ __forceinline__ void row_geometry_block(const DevParams& P, const int y, const int z,
                                                   const float4* __restrict__ T,
                                                   const float4* __restrict__ OD,
                                                   float4* __restrict__ SR,
                                                   float4* __restrict__ MR) {
    const int tid = threadIdx.x;
    const int MU = P.s_mu, W = P.s_nu * P.s_mus;
    const TexelCoord<G> rc = scattering_texel_coord<G>(P, 0u, unsigned(y), unsigned(z));
    const G r = rc.r, mu = rc.mu;
    const bool ground = rc.ground;
    const G dx = distance_to_nearest<G>(P, r, mu, ground) / G(kMsSamples - 1);
    // Lanes 51..63 evaluate sample 50 again and write nothing: every lane
    // takes part in the cross-lane reads of ms_row_slots.
    const int i = min(tid, kMsSamples - 1);
    const bool writer = tid < kMsSamples;
    const G d_i = G(i) * dx;
    const G r_d = clamp_radius<G>(P, sqrt(d_i * d_i + G(2) * r * mu * d_i + r * r));
    float3 tv;
    if constexpr (sizeof(G) == sizeof(double))
        tv = get_transmittance_precise(P, T, OD, r, mu, d_i, ground);
    else
        tv = get_transmittance<G>(P, T, r, mu, d_i, ground);
    const float w = (i == 0 || i == kMsSamples - 1) ? 0.5f : 1.0f;
    const float alt = float(r_d - G(P.bottom));
    const G sin_h = G(P.bottom) / r_d;
    const G cos_h = -sqrt(fmax(G(1) - sin_h * sin_h, G(0)));
    // transmittance.h:7-24 terms that depend on r_d only.
    const G H = sqrt(G(P.top) * G(P.top) - G(P.bottom) * G(P.bottom));
    const G rho = safe_sqrt<G>(r_d * r_d - G(P.bottom) * G(P.bottom));
    const G d_min = G(P.top) - r_d, d_max = rho + H;
    const Taps tr = linear_taps<G>(tex_from_unit<G>(rho / H, P.t_r), P.t_r);
    if (writer) {
        float4* o = SR + (size_t(z) * MU + y) * kSsRowFloat4s;
        o[i] = make_float4(tv.x * w, tv.y * w, tv.z * w, float(d_i));
        o[kMsSamples + i] = make_float4(float(r_d), profile_density(P.prof[0], alt),
                                        profile_density(P.prof[1], alt), float(sin_h));
        o[2 * kMsSamples + i] =
            make_float4(float(cos_h), float(d_min), float(d_max - d_min), tr.w);
        o[3 * kMsSamples + i] =
            make_float4(float(G(1) / r_d), float(G(1) / (d_max - d_min)),
                        float(fmax(G(P.top) * G(P.top) - r_d * r_d, G(0))),
                        float(G(1) / (G(2) * sin_h * G(P.sun_angular_radius))));
        o[4 * kMsSamples + i] = make_float4(__int_as_float(tr.i0 * P.t_mu),
                                            __int_as_float(tr.i1 * P.t_mu), float(dx), 0.0f);
    }
    // Multiple scattering: T(r, mu, d_i) x dx x weight, then the (mu, r)
    // taps of the sample point (r_i, mu_i).
    const G mu_i = clamp_cosine<G>((r * mu + d_i) / r_d);
    const Taps ty = linear_taps<G>(scattering_u_mu<G>(P, r_d, mu_i, ground), MU);
    const Taps tz = linear_taps<G>(scattering_u_r<G>(P, r_d), P.s_r);
    const float f = float(dx) * w;
    float4* m = MR + (size_t(z) * MU + y) * kMsRowFloat4s;
    // The four density rows of the sample, (r0, mu0), (r0, mu1), (r1, mu0),
    // (r1, mu1), as offsets into J, and their bilinear weights.
    const int tz4[4] = {tz.i0, tz.i0, tz.i1, tz.i1}, ty4[4] = {ty.i0, ty.i1, ty.i0, ty.i1};
    int off[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) off[k] = (tz4[k] * MU + ty4[k]) * W;
    const G wy = G(ty.w), wz = G(tz.w);
    const float wt[4] = {float((G(1) - wy) * (G(1) - wz)), float(wy * (G(1) - wz)),
                         float((G(1) - wy) * wz), float(wy * wz)};
    const MsSlots sl = ms_row_slots(i, tz4, ty4, off, wt);
    if (!writer) return;
    m[i] = make_float4(tv.x * f, tv.y * f, tv.z * f, float(d_i));
    m[kMsSamples + i] =
        make_float4(float(r / r_d), __int_as_float(sl.mask), float(d_i / r_d), 0.0f);
    reinterpret_cast<int4*>(m + 2 * kMsSamples)[i] = sl.load;
    m[3 * kMsSamples + i] = sl.w;
}

// A raw buffer resource over `bytes` bytes at p (descriptor word 3 for
// untyped 32-bit loads on gfx9-family parts); loads past the end return 0.
// Offsets are 32-bit, so the tap addresses need no 64-bit arithmetic.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t buffer_rsrc(const void* p, int bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), short(0), bytes, 0x00020000);
}
__device__ __forceinline__ float3 buffer_rgb(__amdgpu_buffer_rsrc_t r, int byte_offset) {
    const auto v = __builtin_amdgcn_raw_buffer_load_b96(r, byte_offset, 0, 0);
    return make_float3(__uint_as_float(v[0]), __uint_as_float(v[1]), __uint_as_float(v[2]));
}
__device__ __forceinline__ float3 lerp3(float3 a, float3 b, float w) {
    return make_float3(fmaf(w, b.x - a.x, a.x), fmaf(w, b.y - a.y, a.y), fmaf(w, b.z - a.z, a.z));
}

// The sun-direction coordinate of sample (tv, gq, lq, iv) of texel
// (mu_s, nu): mu_s_d, the texel coordinate t of T(r_d, mu_s_d) along the
// LUT's mu axis (clamped to [0, TMU-1]) and the smoothstep sun-disc factor
// (transmittance.h:26-33, 63-74).
template <bool PRECISE>
__device__ __forceinline__ void ss_sun_coord(float rf, float mu_s, float nu, float4 tv, float4 gq,
                                             float4 lq, float4 iv, float top2, int TMU,
                                             float& t, float& sm) {
    const float r_d = gq.x, d_i = tv.w;
    const float tmax = float(TMU - 1);
    float mu_s_d;
    if constexpr (PRECISE) {
        // Sun-ray distance to the top boundary without cancellation: for
        // mu_s_d > 0 the root is (top^2 - r_d^2) / (r_d mu_s_d + sqrt(disc)),
        // with top^2 - r_d^2 from the FP64 set-up.  Reciprocals of the
        // per-sample divisors come from FP64 too.
        mu_s_d = __builtin_amdgcn_fmed3f(fmaf(rf, mu_s, d_i * nu) * iv.x, -1.0f, 1.0f);
        const float rm = r_d * mu_s_d;
        const float sq = __builtin_amdgcn_sqrtf(fmaf(rm, rm, iv.z));
        const float d = mu_s_d > 0.0f ? iv.z * __builtin_amdgcn_rcpf(rm + sq) : sq - rm;
        // tex_from_unit then linear_taps: texel coordinate x_mu*(N-1).
        t = __builtin_amdgcn_fmed3f((d - lq.y) * iv.y * tmax, 0.0f, tmax);
    } else {
        // (The table's reciprocals are IEEE ones here: the quotients' bits are
        // the divisions'.)
        mu_s_d = clamp_cosine<float>(div_markstein(rf * mu_s + d_i * nu, r_d, iv.x));
        float disc = r_d * r_d * (mu_s_d * mu_s_d - 1.0f) + top2;
        float d = clamp_distance<float>(-r_d * mu_s_d + safe_sqrt<float>(disc));
        float x_mu = div_markstein(d - lq.y, lq.z, iv.y);
        // linear_taps of tex_from_unit(x_mu): u*N - 0.5 = x_mu*(N-1), clamped.
        const float u = tex_from_unit<float>(x_mu, TMU);
        t = fminf(fmaxf(u * float(TMU) - 0.5f, 0.0f), tmax);
    }
    // smoothstep(-sin_h alpha, sin_h alpha, mu_s_d - cos_h) with the
    // divisor's reciprocal from the table.
    const float u = __builtin_amdgcn_fmed3f(fmaf(mu_s_d - lq.x, iv.w, 0.5f), 0.0f, 1.0f);
    sm = u * u * (3.0f - 2.0f * u);
}


// STAGED (texels per thread): per sample, the block first interpolates the
// sample's two transmittance rows (its r taps) into one row in LDS (double
// buffered, one barrier per sample) and each texel interpolates that row in
// mu: all texels of the (r, mu) row look up the same two LUT rows, so this
// replaces four scattered loads per texel and sample by coalesced loads of the
// rows.  0 (transmittance LUTs wider than kSsMaxStagedMu): each texel reads its
// four taps itself.
//
// Staged it is bound by the chain of a sample and its LDS taps, which scatter
// over the row (half of the LDS cycles are bank conflicts).  With the rows
// loaded and staged before the evaluation, registers for four texels in every
// thread and IEEE divisions in FP32 mode: default 0.125 ms, now 0.120 (FP32
// mode 0.177, now 0.151), double 1.16, now 1.09, 27x64x26x18 0.093, now 0.087.
template <typename G, bool COMP, bool H, int STAGED>
__device__ __forceinline__ void single_scattering_block(const DevParams& P, const int bx, const int by, const int bz,
                                                           const float4* __restrict__ T,
                                                           const float4* __restrict__ SR,
                                                           float4* __restrict__ dR,
                                                           float4* __restrict__ dM,
                                                           float4* __restrict__ S) {
    // The row table (read-only here, every read block-uniform: scalar loads
    // through the constant address space).
    typedef FB_CONSTANT_AS const float4 CF4;
    CF4* row = (CF4*)(SR + (size_t(by) * P.s_mu + bx) * kSsRowFloat4s);
    CF4* s_tv = row;                    // T(r,mu,d_i) * weight (rgb), d_i
    CF4* s_geo = row + kMsSamples;      // r_d, rho_rayleigh, rho_mie, sin_theta_h
    CF4* s_lut = row + 2 * kMsSamples;  // cos_theta_h, d_min, d_max - d_min, T-row weight
    CF4* s_inv = row + 3 * kMsSamples;  // 1/r_d, 1/(d_max - d_min), top^2 - r_d^2, 1/(2 sin_theta_h alpha)
    CF4* s_trw = row + 4 * kMsSamples;  // T-row offsets (int bits), dx
    constexpr bool kPrecise = sizeof(G) == sizeof(double);
    const int NU = P.s_nu, MUS = P.s_mus, MU = P.s_mu;
    const int W = NU * MUS;
    const int y = bx, z = by;
    const int tid = threadIdx.x, nt = blockDim.x;
    const G r = scattering_texel_coord<G>(P, 0u, unsigned(y), unsigned(z)).r;
    const float rf = float(r);
    const float top2 = P.top * P.top;
    const int TMU = P.t_mu;
    const float dxf = s_trw[0].z;
    auto store = [&](int x, const Sum<COMP>* rs, const Sum<COMP>* ms) {
        float3 ray = make_float3(rs[0].value() * dxf * P.solar[0] * P.rayleigh_scattering[0],
                                 rs[1].value() * dxf * P.solar[1] * P.rayleigh_scattering[1],
                                 rs[2].value() * dxf * P.solar[2] * P.rayleigh_scattering[2]);
        float3 mie = make_float3(ms[0].value() * dxf * P.solar[0] * P.mie_scattering[0],
                                 ms[1].value() * dxf * P.solar[1] * P.mie_scattering[1],
                                 ms[2].value() * dxf * P.solar[2] * P.mie_scattering[2]);
        const size_t idx = (size_t(z) * MU + y) * W + x;
        st_tex(dR, idx, make_float4(ray.x, ray.y, ray.z, 0.0f), H);
        st_tex(dM, idx, make_float4(mie.x, mie.y, mie.z, 0.0f), H);
        st_tex(S, idx, make_float4(ray.x, ray.y, ray.z, mie.x), H);
    };
    // One sample's contribution: transmittances and densities.
    auto accumulate = [&](Sum<COMP>* rs, Sum<COMP>* ms, float4 tv, float4 gq, float3 ts,
                          float sm) {
        float t0 = tv.x * (ts.x * sm), t1 = tv.y * (ts.y * sm), t2 = tv.z * (ts.z * sm);
        if constexpr (kPrecise && !COMP) {
            rs[0].s = fmaf(t0, gq.y, rs[0].s);
            rs[1].s = fmaf(t1, gq.y, rs[1].s);
            rs[2].s = fmaf(t2, gq.y, rs[2].s);
            ms[0].s = fmaf(t0, gq.z, ms[0].s);
            ms[1].s = fmaf(t1, gq.z, ms[1].s);
            ms[2].s = fmaf(t2, gq.z, ms[2].s);
            return;
        }
        rs[0].add(t0 * gq.y);
        rs[1].add(t1 * gq.y);
        rs[2].add(t2 * gq.y);
        ms[0].add(t0 * gq.z);
        ms[1].add(t1 * gq.z);
        ms[2].add(t2 * gq.z);
    };
    if constexpr (STAGED != 0) {
        extern __shared__ float4 s_trow[];  // [2][TMU]
        float tmu_s[STAGED], tnu[STAGED];
        Sum<COMP> rs[STAGED][3], ms[STAGED][3];
#pragma unroll
        for (int q = 0; q < STAGED; ++q) {
            const int x = tid + q * nt;
            tmu_s[q] = 0.0f;
            tnu[q] = 0.0f;
            if (x < W) {
                TexelCoord<G> c =
                    scattering_texel_coord<G>(P, unsigned(x), unsigned(y), unsigned(z));
                tmu_s[q] = float(c.mu_s);
                tnu[q] = float(c.nu);
            }
        }
        // Sample i's two T rows, lerped in r with the row weight, into a staged
        // row.  The first kAhead columns of a thread are loaded before the
        // evaluation of the sample before and written after it, so that their
        // latency is hidden; further ones at once.
        constexpr int kAhead = 2;
        float3 ta[kAhead], tb[kAhead];
        auto load = [&](int i) {
            const float4 tr4 = s_trw[i];
            const float4* t0 = T + __float_as_int(tr4.x);
            const float4* t1 = T + __float_as_int(tr4.y);
#pragma unroll
            for (int c = 0; c < kAhead; ++c) {
                const int j = tid + c * nt;
                if (j < TMU) {
                    ta[c] = *reinterpret_cast<const float3*>(t0 + j);
                    tb[c] = *reinterpret_cast<const float3*>(t1 + j);
                }
            }
        };
        auto put = [&](int i, float4* dst) {
            const float w = s_lut[i].w;
#pragma unroll
            for (int c = 0; c < kAhead; ++c) {
                const int j = tid + c * nt;
                if (j < TMU) {
                    const float3 v = lerp3(ta[c], tb[c], w);
                    dst[j] = make_float4(v.x, v.y, v.z, 0.0f);
                }
            }
            if (kAhead * nt < TMU) {
                const float4 tr4 = s_trw[i];
                const float4* t0 = T + __float_as_int(tr4.x);
                const float4* t1 = T + __float_as_int(tr4.y);
                for (int j = tid + kAhead * nt; j < TMU; j += nt) {
                    const float4 a = ldg4(t0 + j), b = ldg4(t1 + j);
                    dst[j] = make_float4(fmaf(w, b.x - a.x, a.x), fmaf(w, b.y - a.y, a.y),
                                         fmaf(w, b.z - a.z, a.z), 0.0f);
                }
            }
        };
        load(0);
        put(0, s_trow);
        __syncthreads();
        for (int i = 0; i < kMsSamples; ++i) {
            const float4* cur = s_trow + (i & 1) * TMU;
            const bool next = i + 1 < kMsSamples;
            if (next) load(i + 1);
            const float4 tv = s_tv[i], gq = s_geo[i], lq = s_lut[i], iv = s_inv[i];
#pragma unroll
            for (int q = 0; q < STAGED; ++q) {
                if (tid + q * nt >= W) continue;
                float t, sm;
                ss_sun_coord<kPrecise>(rf, tmu_s[q], tnu[q], tv, gq, lq, iv, top2, TMU, t, sm);
                const int i0 = int(t);  // t >= 0: truncation is floor
                const int i1 = min(i0 + 1, TMU - 1);
                const float f = t - float(i0);
                const float4 a = cur[i0], b = cur[i1];
                const float3 ts = make_float3(fmaf(f, b.x - a.x, a.x), fmaf(f, b.y - a.y, a.y),
                                              fmaf(f, b.z - a.z, a.z));
                accumulate(rs[q], ms[q], tv, gq, ts, sm);
            }
            if (next) put(i + 1, s_trow + ((i + 1) & 1) * TMU);
            __syncthreads();
        }
#pragma unroll
        for (int q = 0; q < STAGED; ++q)
            if (tid + q * nt < W) store(tid + q * nt, rs[q], ms[q]);
    } else {
        for (int x = tid; x < W; x += nt) {
            TexelCoord<G> c = scattering_texel_coord<G>(P, unsigned(x), unsigned(y), unsigned(z));
            const float mu_s = float(c.mu_s), nu = float(c.nu);
            Sum<COMP> rs[3], ms[3];
            // The row table's entries of sample i+1 are loaded while sample i
            // is evaluated (scalar loads, waited for at their first use).
            float4 tv_n = s_tv[0], gq_n = s_geo[0], lq_n = s_lut[0], iv_n = s_inv[0];
            float4 tr4_n = s_trw[0];
            for (int i = 0; i < kMsSamples; ++i) {
                const float4 tv = tv_n, gq = gq_n, lq = lq_n, iv = iv_n, tr4 = tr4_n;
                const int in = i + 1 < kMsSamples ? i + 1 : i;
                tv_n = s_tv[in];
                gq_n = s_geo[in];
                lq_n = s_lut[in];
                iv_n = s_inv[in];
                tr4_n = s_trw[in];
                // The sample's two T rows (r taps) as one buffer: row 0 at byte
                // 0, row 1 at `drow` (0 when both taps are the same row).
                const int row0 = __float_as_int(tr4.x),
                          drow = (__float_as_int(tr4.y) - row0) * 16;
                const __amdgpu_buffer_rsrc_t tb = buffer_rsrc(T + row0, drow + TMU * 16);
                float t, sm;
                ss_sun_coord<kPrecise>(rf, mu_s, nu, tv, gq, lq, iv, top2, TMU, t, sm);
                const int i0 = int(t);
                const int o0 = i0 * 16, o1 = min(i0 + 1, TMU - 1) * 16;
                const float f = t - float(i0);
                const float3 ts =
                    lerp3(lerp3(buffer_rgb(tb, o0), buffer_rgb(tb, o1), f),
                          lerp3(buffer_rgb(tb, drow + o0), buffer_rgb(tb, drow + o1), f), lq.w);
                accumulate(rs, ms, tv, gq, ts, sm);
            }
            store(x, rs, ms);
        }
    }
}

// Rows of at most kSsChunkMaxW texels on the direct-lookup path
// (ss_chunked): the block's ss_chunks(P) groups of W threads each integrate
// a contiguous chunk of the row's samples -- per sample, the arithmetic of
// single_scattering_block's direct path -- and the chunk sums are added in
// chunk order.  The row table's reads depend on the group's sample: vector
// loads.
template <typename G, bool H>
__device__ __forceinline__ void single_scattering_block_chunked(
    const DevParams& P, const int y, const int z, const float4* __restrict__ T,
    const float4* __restrict__ SR, float4* __restrict__ dR, float4* __restrict__ dM,
    float4* __restrict__ S) {
    extern __shared__ float s_ssp[];  // [chunk][W][6]: Rayleigh rgb, Mie rgb
    const float4* row = SR + (size_t(z) * P.s_mu + y) * kSsRowFloat4s;
    const float4* s_tv = row;
    const float4* s_geo = row + kMsSamples;
    const float4* s_lut = row + 2 * kMsSamples;
    const float4* s_inv = row + 3 * kMsSamples;
    const float4* s_trw = row + 4 * kMsSamples;
    constexpr bool kPrecise = sizeof(G) == sizeof(double);
    const int NU = P.s_nu, MUS = P.s_mus, MU = P.s_mu;
    const int W = NU * MUS;
    const int CH = ss_chunks(P);
    const int tid = threadIdx.x;
    const int g = tid / W, x = tid - g * W;
    const bool in_chunk = g < CH;
    const G r = scattering_texel_coord<G>(P, 0u, unsigned(y), unsigned(z)).r;
    const float rf = float(r);
    const float top2 = P.top * P.top;
    const int TMU = P.t_mu;
    if (in_chunk) {
        const int i0 = g * kMsSamples / CH, i1 = (g + 1) * kMsSamples / CH;
        TexelCoord<G> c = scattering_texel_coord<G>(P, unsigned(x), unsigned(y), unsigned(z));
        const float mu_s = float(c.mu_s), nu = float(c.nu);
        float rs0 = 0.0f, rs1 = 0.0f, rs2 = 0.0f, ms0 = 0.0f, ms1 = 0.0f, ms2 = 0.0f;
        for (int i = i0; i < i1; ++i) {
            const float4 tv = s_tv[i], gq = s_geo[i], lq = s_lut[i], iv = s_inv[i],
                         tr4 = s_trw[i];
            const int row0 = __float_as_int(tr4.x), drow = (__float_as_int(tr4.y) - row0) * 16;
            const __amdgpu_buffer_rsrc_t tb = buffer_rsrc(T + row0, drow + TMU * 16);
            float t, sm;
            ss_sun_coord<kPrecise>(rf, mu_s, nu, tv, gq, lq, iv, top2, TMU, t, sm);
            const int k0 = int(t);
            const int o0 = k0 * 16, o1 = min(k0 + 1, TMU - 1) * 16;
            const float f = t - float(k0);
            const float3 ts =
                lerp3(lerp3(buffer_rgb(tb, o0), buffer_rgb(tb, o1), f),
                      lerp3(buffer_rgb(tb, drow + o0), buffer_rgb(tb, drow + o1), f), lq.w);
            const float t0 = tv.x * (ts.x * sm), t1 = tv.y * (ts.y * sm), t2 = tv.z * (ts.z * sm);
            rs0 = rs0 + t0 * gq.y;
            rs1 = rs1 + t1 * gq.y;
            rs2 = rs2 + t2 * gq.y;
            ms0 = ms0 + t0 * gq.z;
            ms1 = ms1 + t1 * gq.z;
            ms2 = ms2 + t2 * gq.z;
        }
        float* p = s_ssp + size_t(g * W + x) * 6;
        p[0] = rs0;
        p[1] = rs1;
        p[2] = rs2;
        p[3] = ms0;
        p[4] = ms1;
        p[5] = ms2;
    }
    __syncthreads();
    if (g == 0) {
        float v[6];
#pragma unroll
        for (int k = 0; k < 6; ++k) v[k] = s_ssp[size_t(x) * 6 + k];
        for (int cg = 1; cg < CH; ++cg)
#pragma unroll
            for (int k = 0; k < 6; ++k) v[k] = v[k] + s_ssp[size_t(cg * W + x) * 6 + k];
        const float dxf = s_trw[0].z;
        const float3 ray = make_float3(v[0] * dxf * P.solar[0] * P.rayleigh_scattering[0],
                                       v[1] * dxf * P.solar[1] * P.rayleigh_scattering[1],
                                       v[2] * dxf * P.solar[2] * P.rayleigh_scattering[2]);
        const float3 mie = make_float3(v[3] * dxf * P.solar[0] * P.mie_scattering[0],
                                       v[4] * dxf * P.solar[1] * P.mie_scattering[1],
                                       v[5] * dxf * P.solar[2] * P.mie_scattering[2]);
        const size_t idx = (size_t(z) * MU + y) * W + x;
        st_tex(dR, idx, make_float4(ray.x, ray.y, ray.z, 0.0f), H);
        st_tex(dM, idx, make_float4(mie.x, mie.y, mie.z, 0.0f), H);
        st_tex(S, idx, make_float4(ray.x, ray.y, ray.z, mie.x), H);
    }
}

// ============================================ 4. scattering density: geometry
// The kernels are in density.hpp.
//
// The density geometry table (dg_row / dg_x) of one LUT set; block b < R
// fills the rows of r index b, block R + j the x taps of mu_s index j.
// scattering_density.comp:34-66 for the directions, :45-60 for the ground
// term; the taps are GetScatteringTextureUvwzFromRMuMuSNu's (scattering.h
// :7-60) for r = r(z), mu = cos(theta_l), mu_s = mu_s(j).
template <typename G>
__device__ __forceinline__ void density_geometry_block(const DevParams& P, const int b,
                                                       const float4* __restrict__ T,
                                                       const float4* __restrict__ OD,
                                                       float4* __restrict__ DG) {
    const int tid = threadIdx.x;
    const int R = P.s_r, NU = P.s_nu;
    if (b < R) {
        const int z = b;
        const G r = scattering_texel_coord<G>(P, 0u, 0u, unsigned(z)).r;
        float4* row = DG + dg_row(z);
        if (tid < kDenTheta) {
            const int l = tid;
            const G ct = den_cos<G>(l);
            const bool g_l = ray_intersects_ground<G>(P, r, ct);
            const Taps ty = linear_taps<G>(scattering_u_mu<G>(P, r, ct, g_l), P.s_mu);
            float4 gv = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
            float ginv = 0.0f;
            if (g_l) {
                const G dg = distance_to_bottom<G>(P, r, ct);
                float3 tg;
                if constexpr (sizeof(G) == sizeof(double))
                    tg = get_transmittance_precise(P, T, OD, r, ct, dg, true);
                else
                    tg = get_transmittance<G>(P, T, r, ct, dg, true);
                gv = make_float4(tg.x * P.albedo[0] * (1.0f / kPi),
                                 tg.y * P.albedo[1] * (1.0f / kPi),
                                 tg.z * P.albedo[2] * (1.0f / kPi), float(dg));
                // The ground normal's length does not depend on phi.
                const float4 o = c_den.dir[l * kDenPhi];
                const G st2 = G(o.x) * G(o.x) + G(o.y) * G(o.y);
                const G gz = r + ct * dg;
                ginv = float(G(1) / sqrt(st2 * dg * dg + gz * gz));
            }
            row[l] = gv;
            row[kDenTheta + l] =
                make_float4(__int_as_float(ty.i0), __int_as_float(ty.i1), ty.w, ginv);
        } else if (tid == kDenTheta) {
            const Taps tz = linear_taps<G>(scattering_u_r<G>(P, r), P.s_r);
            row[2 * kDenTheta] =
                make_float4(__int_as_float(tz.i0), __int_as_float(tz.i1), tz.w, 0.0f);
        }
    } else {
        const int j = b - R;
        if (tid < NU + 2) {
            const G mu_s = scattering_texel_coord<G>(P, unsigned(j), 0u, 0u).mu_s;
            const Taps tx = slice_taps<G>(P, tid - 1, scattering_u_mu_s<G>(P, mu_s));
            DG[dg_x(R, j, NU) + tid] =
                make_float4(__int_as_float(tx.i0), __int_as_float(tx.i1), tx.w, 0.0f);
        }
    }
}

// =================================================== 5. indirect irradiance
// indirect_irradiance.comp:10-74.  One wavefront per irradiance texel: lane
// i takes phi_i (64 lanes = the 64 phi samples), loops the 16 theta rows,
// and the wave reduces.  As in the density pass, the lookups of one theta
// row share (u_r, u_mu, u_mu_s), so each wave first builds its 16 nu
// profiles in LDS.
constexpr int kIndWaves = 4;  // waves per block (fewer when LDS would exceed 64 KiB)

__host__ __device__ inline size_t indirect_lds_bytes_per_wave(int nu, bool single) {
    const int ntex = single ? 2 : 1;
    return sizeof(float4) * size_t(ntex) * kIndTheta * (nu + 2) +
           sizeof(ProfEntry) * size_t(ntex) * kIndTheta * (nu + 1);
}

template <typename G, bool SINGLE, bool H>
__device__ __forceinline__ void indirect_irradiance_block(const DevParams& P, const int bx, const int by, const int bz, const float4* __restrict__ dR, const float4* __restrict__ dM,
    const float4* __restrict__ dMS, float4* __restrict__ dE, float4* __restrict__ E) {
    extern __shared__ float4 s_dyn[];
    constexpr int NTEX = SINGLE ? 2 : 1;
    const int waves = blockDim.x / 64;
    const int wave = threadIdx.x / 64, lane = threadIdx.x % 64;
    const int texel = bx * waves + wave;
    const int n = P.i_mus * P.i_r;
    const bool active = texel < n;
    const int ti = active ? texel % P.i_mus : 0, tj = active ? texel / P.i_mus : 0;
    const int NU = P.s_nu, nslots = NU + 2, nent = NU + 1;
    const size_t per_wave = indirect_lds_bytes_per_wave(NU, SINGLE);
    float4* s_raw = reinterpret_cast<float4*>(reinterpret_cast<char*>(s_dyn) + wave * per_wave);
    ProfEntry* s_prof = reinterpret_cast<ProfEntry*>(s_raw + NTEX * kIndTheta * nslots);

    G x_mu_s = G(ti) / G(P.i_mus - 1);
    G x_r = G(tj) / G(P.i_r - 1);
    G r, mu_s;
    rmus_from_irradiance_unit<G>(P, x_mu_s, x_r, r, mu_s);
    const G u_mu_s = scattering_u_mu_s<G>(P, mu_s);
    const Taps tz = linear_taps<G>(scattering_u_r<G>(P, r), P.s_r);
    for (int e = lane; e < NTEX * kIndTheta * nslots; e += 64) {
        int tex_sel = e / (kIndTheta * nslots);
        int rem = e % (kIndTheta * nslots);
        int jj = rem / nslots, slot = rem % nslots;
        G ct = ind_cos<G>(jj);
        Taps ty = linear_taps<G>(scattering_u_mu<G>(P, r, ct, false), P.s_mu);
        const float4* tex = SINGLE ? (tex_sel == 0 ? dR : dM) : dMS;
        s_raw[e] = trilinear_taps_t<H>(P, tex, slice_taps<G>(P, slot - 1, u_mu_s), ty, tz);
    }
    __syncthreads();
    for (int e = lane; e < NTEX * kIndTheta * nent; e += 64) {
        int row = e / nent, k = e % nent;
        s_prof[e] = make_entry(s_raw[row * nslots + k], s_raw[row * nslots + k + 1]);
    }
    __syncthreads();
    if (!active) return;

    const float osx = float(sqrt(G(1) - mu_s * mu_s)), osz = float(mu_s);
    const float g = P.g;
    const float kR = 3.0f / (16.0f * kPi);
    const float kM = 3.0f / (8.0f * kPi) * (1.0f - g * g) / (2.0f + g * g);
    const float g1 = 1.0f + g * g, g2 = -2.0f * g;
    const float hnu = 0.5f * float(NU - 1);
    const int kmax = NU - 1;
    float a0 = 0.0f, a1 = 0.0f, a2 = 0.0f;
    for (int jj = 0; jj < kIndTheta; ++jj) {
        const float4 om = c_ind.dir[jj * kIndPhi + lane];
        const float nu = fmaf(om.x, osx, om.z * osz);
        const float t = fmaf(nu, hnu, hnu);
        float3 v = prof_lerp(s_prof + jj * nent, t, kmax);
        if (SINGLE) {
            float3 m = prof_lerp(s_prof + (kIndTheta + jj) * nent, t, kmax);
            float q = fmaf(nu, nu, 1.0f);
            float rs = rsqrtf(fmaf(g2, nu, g1));
            float pR = kR * q, pM = kM * q * (rs * rs * rs);
            v = make_float3(fmaf(m.x, pM, v.x * pR), fmaf(m.y, pM, v.y * pR),
                            fmaf(m.z, pM, v.z * pR));
        }
        const float w = om.z * om.w;
        a0 = fmaf(v.x, w, a0);
        a1 = fmaf(v.y, w, a1);
        a2 = fmaf(v.z, w, a2);
    }
    for (int off = 32; off > 0; off >>= 1) {
        a0 += __shfl_xor(a0, off, 64);
        a1 += __shfl_xor(a1, off, 64);
        a2 += __shfl_xor(a2, off, 64);
    }
    if (lane == 0) {
        int o = tj * P.i_mus + ti;
        dE[o] = make_float4(a0, a1, a2, 0.0f);
        float4 prev = E[o];
        E[o] = make_float4(a0 + prev.x, a1 + prev.y, a2 + prev.z, 0.0f + prev.w);
    }
}

// =================================================== 6. multiple scattering
// multiple_scattering.comp:9-93.
//
// All texels of one (r, mu) row (x = nu*MUS + mu_s varies) march the same
// ray: d_i, r_i, mu_i, the view transmittance T(r, mu, d_i) and the
// (u_mu, u_r) taps of every sample are shared, only mu_s_i (and the fixed
// nu slice) differ per texel.  A block owns one row: for each sample it
// stages the (mu, r)-bilinear row of the density LUT in LDS (double buffered,
// one barrier per sample), and each texel lerps its mu_s taps from LDS: two
// in its own nu slice, and two in the next where its nu falls between slices
// (MsTexel).
//
// Where the density LUT fits the L2s it is bound by the chain of a sample
// (coordinate, LDS taps, staging, barrier), else by the latency of the row
// loads that miss the L2 (10 GB from beyond it per launch at double).  With
// four taps for every texel and the coordinate after the barrier a launch took
// 0.118 ms at default and 0.149 at 27x64x26x18, now 0.097 and 0.087; at double
// 2.35, now 2.21.  Loads two samples ahead (24 more VGPRs): 2.48 at double,
// 0.123 at default.
constexpr int kMsTexelsPerThread = 4;
// Threads per block of the multiple-scattering kernels: up to one per
// texel of the widest row (NU * MUS <= 1024).
constexpr int kMsMaxThreads = 1024;
// Staged density rows per block (sample i is evaluated from one while
// sample i+1 is staged into the other).
constexpr int kMsStagedRows = 2;

// A staged density value: rgb only (12 bytes, 4-byte aligned), so the
// four taps of a sample cost 48 bytes of LDS reads, not 64.
struct Rgb {
    float x, y, z;
};

__device__ __forceinline__ Rgb to_rgb(const Rgb& v) { return v; }
__device__ __forceinline__ Rgb to_rgb(const Half4& v) {
    return Rgb{float(v.x), float(v.y), float(v.z)};
}

// GetScatteringTextureUvwzFromRMuMuSNu's mu_s coordinate (scattering.h:
// 48-56) of a sample, (1 - a/A) / (1 + a) (MUS-1), as the texel coordinate
// within a nu slice.  a = (d - d_min) / (d_max - d_min), d the distance from
// the ground to the top boundary at mu_s, d / H = sqrt(c^2 mu_s^2 + 1) - c
// mu_s, c = bottom / H.  With u = sqrt(c^2 mu_s^2 + 1) + c |mu_s|, which has
// no cancellation, d / H is u for mu_s < 0 and 1 / u otherwise, and the
// coordinate is a quotient of two linear functions of it: three times closer
// to the exact coordinate than the difference of two terms of bottom's size.
// Kept in [0, MUS-1] (a >= 0 up to rounding, and the reference clamps 1 - a/A
// at 0).  FP32 mode takes the reference's expression.
template <typename G>
struct MsCoord {
    MsCoordConst k;
    float top;
    __device__ explicit MsCoord(const DevParams& P) : k(P.ms), top(float(P.s_mus - 1)) {}
    // mu_s at the sample (multiple_scattering.comp:38): (r mu_s + d_i nu) / r_i.
    __device__ float operator()(float mu_s, float nu, float r_ri, float d_ri) const {
        const float m = fmaf(r_ri, mu_s, d_ri * nu);
        const float u = fmaf(k.c, fabsf(m), __builtin_amdgcn_sqrtf(fmaf(k.c2, m * m, 1.0f)));
        const float s = m < 0.0f ? u : 1.0f, t = m < 0.0f ? 1.0f : u;
        return __builtin_amdgcn_fmed3f(
            fmaf(k.p1, s, k.p0 * t) * __builtin_amdgcn_rcpf(fmaf(k.q0, t, s)), 0.0f, top);
    }
};
template <>
struct MsCoord<float> {
    float b, b2, h2, d_min, inv, inv_a, top;
    __device__ explicit MsCoord(const DevParams& P) {
        b = P.bottom;
        b2 = b * b;
        h2 = P.top * P.top - b2;
        d_min = P.top - b;
        inv = 1.0f / (sqrtf(h2) - d_min);
        inv_a = 1.0f / (-2.0f * P.mu_s_min * b * inv);
        top = float(P.s_mus - 1);
    }
    __device__ float operator()(float mu_s, float nu, float r_ri, float d_ri) const {
        const float m = __builtin_amdgcn_fmed3f(fmaf(r_ri, mu_s, d_ri * nu), -1.0f, 1.0f);
        const float d =
            fmaxf(fmaf(-b, m, __builtin_amdgcn_sqrtf(fmaf(b2, m * m, h2))), 0.0f);
        const float a = (d - d_min) * inv;
        return top * __builtin_amdgcn_fmed3f(
                         fmaf(-a, inv_a, 1.0f) * __builtin_amdgcn_rcpf(1.0f + a), 0.0f, 1.0f);
    }
};

// A row's texels in thread order.  Position x of the row is nu slot x / MUS:
// nu index 0, NU-1, 1, 2, ..., NU-2, so that the outer texels come first.
__device__ __forceinline__ int ms_nu_index(int slot, int NU) {
    return slot == 0 ? 0 : (slot == 1 ? NU - 1 : slot - 1);
}

// A texel of a multiple-scattering row.  nu is constant along the ray, so an
// inner texel, whose nu is its slice's, reads that slice only (lerp 0); where
// nu is clamped (scattering.h:132-134) it falls between slices.  An inner
// index with a clamped nu has the nu, mu_s and so the value of the outer texel
// on its side: its thread copies that one's sum (`copy`: 1 + 0 for index 0's,
// 1 + 1 for NU-1's, 0 if the texel has a value of its own).  FP32 mode, where
// mu_s depends on the nu index by its rounding, evaluates it like an outer one.
struct MsTexel {
    float mu_s, nu, lerp;
    int x, entry, copy;  // x: texel in the row; entry: slice's first staged entry
    bool two;            // reads two slices
};
template <typename G>
__device__ __forceinline__ MsTexel ms_texel(const DevParams& P, int slot, int j, int y, int z) {
    const int NU = P.s_nu, k = ms_nu_index(slot, NU);
    MsTexel t;
    t.x = k * P.s_mus + j;
    const TexelCoord<G> c = scattering_texel_coord<G>(P, unsigned(t.x), unsigned(y), unsigned(z));
    t.mu_s = float(c.mu_s);
    t.nu = float(c.nu);
    const G knot = clamp_cosine<G>(G(k) / G(NU - 1) * G(2) - G(1));  // as in the texel map
    const float tc = (t.nu + 1.0f) / 2.0f * float(NU - 1);
    float slice = floorf(tc);
    t.lerp = tc - slice;
    t.copy = 0;
    t.two = slot < 2 || (c.nu != knot && sizeof(G) == sizeof(float));
    if (!t.two) {
        slice = float(k);
        t.lerp = 0.0f;
        if (c.nu != knot) t.copy = c.nu > knot ? 1 : 2;
    }
    t.entry = int(slice) * (P.s_mus + 1);
    return t;
}

// H: the density LUT J, the delta and the scattering LUT are binary16
// (FB_FLAG_F16_STORAGE); the density rows then stay binary16 in the slots
// until put() widens them.
template <typename G, int TPT, bool H>
__device__ __forceinline__ void multiple_scattering_block(const DevParams& P, const int bx, const int by, const int bz,
                                                             const float4* __restrict__ MR,
                                                             const float4* __restrict__ J,
                                                             float4* __restrict__ dMS,
                                                             float4* __restrict__ S) {
    extern __shared__ Rgb s_row[];              // [2][(NU + 1) * (MUS + 1)]: staged density rows
    const int NU = P.s_nu, MUS = P.s_mus, MU = P.s_mu;
    const int W = NU * MUS;
    const int y = bx, z = by;
    const int tid = threadIdx.x, nt = blockDim.x;

    // Row geometry: the 51 samples' terms, written by the geometry pass (the
    // same samples, single_scattering.comp:30-65).  Every read of it is
    // block-uniform, and the table is read-only here: read through the
    // constant address space, the reads are scalar loads.
    typedef FB_CONSTANT_AS const float4 CF4;
    typedef FB_CONSTANT_AS const int4 CI4;
    CF4* desc = (CF4*)(MR + (size_t(z) * MU + y) * kMsRowFloat4s);
    auto d_tw = [&](int i) { return desc[i]; };  // T(r,mu,d_i)*dx*weight (rgb), d_i
    auto d_geo = [&](int i) { return desc[kMsSamples + i]; };  // r/r_i, slot load mask, d_i/r_i
    auto d_off = [&](int i) { return ((CI4*)(desc + 2 * kMsSamples))[i]; };  // slot rows
    auto d_wt = [&](int i) { return desc[3 * kMsSamples + i]; };  // slot weights

    // Per-texel constants: thread tid's texels are positions tid + q*nt.
    MsTexel tx[TPT];
    bool inner[TPT];  // every texel of the wavefront reads one slice (wave-uniform)
    int spos[TPT];    // the texel's entry in a staged row
    float acc0[TPT], acc1[TPT], acc2[TPT];
#pragma unroll
    for (int q = 0; q < TPT; ++q) {
        const int x = tid + q * nt;
        tx[q] = MsTexel{0.0f, 0.0f, 0.0f, 0, 0, 0, false};
        if (x < W) tx[q] = ms_texel<G>(P, x / MUS, x % MUS, y, z);
        inner[q] = __builtin_amdgcn_ballot_w64(tx[q].two) == 0;
        spos[q] = tx[q].x + tx[q].x / MUS;
        acc0[q] = acc1[q] = acc2[q] = 0.0f;
    }
    __syncthreads();

    const MsCoord<G> coord(P);
    const int SS = MUS + 1;  // staged entries per nu slice

    // The four density-row slots of this thread's texels, carried from sample
    // to sample (ms_row_slots): each sample loads only the rows it does not
    // share with the previous one.
    typedef typename std::conditional<H, Half4, Rgb>::type Slot;
    Slot slot[TPT][4];
#pragma unroll
    for (int q = 0; q < TPT; ++q)
#pragma unroll
        for (int k = 0; k < 4; ++k) slot[q][k] = Slot{};
    // Row loads as buffer loads: the row start (block-uniform) goes in the
    // scalar offset and the texel's byte offset in a loop-invariant vector
    // offset, so no address arithmetic writes a register between the loads
    // and each load lands directly in its slot.  (Positions past the row load
    // texel 0 and never use it.)
    constexpr int TB = H ? 8 : 16;  // bytes per texel of J
    const __amdgpu_buffer_rsrc_t jb = buffer_rsrc(J, int(size_t(P.s_r) * MU * W * TB));
    int xoff[TPT];
#pragma unroll
    for (int q = 0; q < TPT; ++q) xoff[q] = tx[q].x * TB;
    auto ld = [&](int o, int q) {
        if constexpr (H) {
            return __builtin_bit_cast(Half4,
                                      __builtin_amdgcn_raw_buffer_load_b64(jb, xoff[q], o * TB, 0));
        } else {
            const auto v = __builtin_amdgcn_raw_buffer_load_b96(jb, xoff[q], o * TB, 0);
            return Rgb{__uint_as_float(v[0]), __uint_as_float(v[1]), __uint_as_float(v[2])};
        }
    };
    // Issue the loads of the sample whose slot mask and row offsets are
    // (mask, o); they stay in flight until put() reads them.
    auto advance = [&](int mask, int4 o) {
#pragma unroll
        for (int q = 0; q < TPT; ++q) {
            if (mask & 1) slot[q][0] = ld(o.x, q);
            if (mask & 2) slot[q][1] = ld(o.y, q);
            if (mask & 4) slot[q][2] = ld(o.z, q);
            if (mask & 8) slot[q][3] = ld(o.w, q);
        }
    };
    // Row layout: nu slice k (k = 0..NU-1) at entries k*SS .. k*SS+MUS-1,
    // then one pad entry; then a zero slice NU.  Pads and the zero slice are
    // read only with weight 0 (the mu_s tap after a slice's last entry has
    // weight 0, and so has the nu slice above the last one), so every tap
    // index goes unclamped.  The pad entry shifts consecutive slices by one
    // LDS bank (taps of neighbouring slices at the same mu_s would otherwise
    // share banks).
    const int WP = (NU + 1) * SS;
    for (int e = tid; e < NU + 1 + MUS; e += nt) {
        const int k = e < NU ? e * SS + MUS : NU * SS + (e - NU);  // pads, then the zero slice
#pragma unroll
        for (int b = 0; b < kMsStagedRows; ++b) s_row[b * WP + k] = Rgb{0.0f, 0.0f, 0.0f};
    }
    // The (mu, r)-bilinear density value of sample i at texel x (the slot
    // weights are the bilinear weights), into the staged row dst.
    auto put = [&](int i, const Slot* s, Rgb* dst, int x) {
        const float4 w = d_wt(i);
        const Rgb t[4] = {to_rgb(s[0]), to_rgb(s[1]), to_rgb(s[2]), to_rgb(s[3])};
        const Rgb v{fmaf(w.w, t[3].x, fmaf(w.z, t[2].x, fmaf(w.y, t[1].x, w.x * t[0].x))),
                    fmaf(w.w, t[3].y, fmaf(w.z, t[2].y, fmaf(w.y, t[1].y, w.x * t[0].y))),
                    fmaf(w.w, t[3].z, fmaf(w.z, t[2].z, fmaf(w.y, t[1].z, w.x * t[0].z)))};
        dst[x] = v;
    };
    auto put_all = [&](int i, Rgb* dst) {
#pragma unroll
        for (int q = 0; q < TPT; ++q)
            if (tid + q * nt < W) put(i, slot[q], dst, spos[q]);
    };
    // A texel's mu_s coordinate at sample i, and sample i of every texel of
    // this thread from the staged row `cur`: the coordinates of sample i+1
    // are computed while the taps of sample i are on their way from LDS.
    float xt[TPT];
    auto locate = [&](float4 geo, int q) {
        return coord(tx[q].mu_s, tx[q].nu, geo.x, geo.z);
    };
    auto eval = [&](float4 tw, float4 geo_next, const Rgb* __restrict__ cur) {
#pragma unroll
        for (int q = 0; q < TPT; ++q) {
            if (tid + q * nt < W) {
                // 0 <= xt <= MUS - 1 and 0 <= entry <= (NU - 1) SS: the taps
                // i0, i0+1, i0+SS, i0+SS+1 stay inside the padded row (see the
                // layout above).
                const float w = __builtin_amdgcn_fractf(xt[q]);
                const Rgb* p = cur + (tx[q].entry + int(xt[q]));
                const Rgb p0 = p[0], p1 = p[1];
                xt[q] = locate(geo_next, q);
                float v0 = fmaf(w, p1.x - p0.x, p0.x), v1 = fmaf(w, p1.y - p0.y, p0.y),
                      v2 = fmaf(w, p1.z - p0.z, p0.z);
                if (!inner[q]) {
                    const Rgb p2 = p[SS], p3 = p[SS + 1];
                    const float u0 = fmaf(w, p3.x - p2.x, p2.x), u1 = fmaf(w, p3.y - p2.y, p2.y),
                                u2 = fmaf(w, p3.z - p2.z, p2.z);
                    const float l = tx[q].lerp;
                    v0 = fmaf(l, u0 - v0, v0);
                    v1 = fmaf(l, u1 - v1, v1);
                    v2 = fmaf(l, u2 - v2, v2);
                }
                acc0[q] = fmaf(v0, tw.x, acc0[q]);
                acc1[q] = fmaf(v1, tw.y, acc1[q]);
                acc2[q] = fmaf(v2, tw.z, acc2[q]);
            }
        }
    };
    // (Each thread stages exactly its own texels: W <= TPT*nt.)
    float4 geo = d_geo(0);
    advance(__float_as_int(geo.y), d_off(0));
    put_all(0, s_row);
#pragma unroll
    for (int q = 0; q < TPT; ++q) xt[q] = locate(geo, q);
    __syncthreads();
    // The descriptors of the sample after next are read (scalar loads) one
    // iteration ahead of their use.
    geo = d_geo(1);
    int4 off = d_off(1);
    for (int i = 0; i < kMsSamples; ++i) {
        const Rgb* cur = s_row + (i & 1) * WP;
        Rgb* nxt = s_row + ((i + 1) & 1) * WP;
        const bool next = i + 1 < kMsSamples;
        // The loads of sample i+1 are issued first, so that their latency
        // overlaps the evaluation of sample i.
        if (next) advance(__float_as_int(geo.y), off);
        const int i2 = i + 2 < kMsSamples ? i + 2 : kMsSamples - 1;
        const float4 geo2 = d_geo(i2);
        off = d_off(i2);
        eval(d_tw(i), geo, cur);
        if (next) put_all(i + 1, nxt);
        __syncthreads();
        geo = geo2;
    }
    // The outer texels' sums (positions 0..2 MUS-1), for the threads that
    // copy them.
#pragma unroll
    for (int q = 0; q < TPT; ++q)
        if (tid + q * nt < 2 * MUS) s_row[tid + q * nt] = Rgb{acc0[q], acc1[q], acc2[q]};
    __syncthreads();
#pragma unroll
    for (int q = 0; q < TPT; ++q) {
        if (tid + q * nt < W) {
            const size_t idx = (size_t(z) * MU + y) * W + tx[q].x;
            float m0 = acc0[q], m1 = acc1[q], m2 = acc2[q];
            if (tx[q].copy) {
                const Rgb o = s_row[(tx[q].copy - 1) * MUS + tx[q].x % MUS];
                m0 = o.x;
                m1 = o.y;
                m2 = o.z;
            }
            st_tex(dMS, idx, make_float4(m0, m1, m2, 0.0f), H);
            float pr = phase_rayleigh(tx[q].nu);
            float4 prev = ld_tex(S, idx, H);
            st_tex(S, idx,
                   make_float4(m0 / pr + prev.x, m1 / pr + prev.y, m2 / pr + prev.z,
                               0.0f + prev.w),
                   H);
        }
    }
}


// Rows of at most kMsChunkMaxW texels (ms_chunked): the block's
// ms_chunks(P) groups of W threads each integrate a contiguous chunk of the
// row's samples -- per sample, the arithmetic of multiple_scattering_block
// with TPT = 1, on the group's own staged rows and row slots -- and the
// chunk sums are added in chunk order.  The row's table is staged in LDS
// (its reads depend on the group's sample).
template <typename G, bool H>
__device__ __forceinline__ void multiple_scattering_block_chunked(
    const DevParams& P, const int y, const int z, const float4* __restrict__ MR,
    const float4* __restrict__ J, float4* __restrict__ dMS, float4* __restrict__ S) {
    // The row table [kMsRowFloat4s] and the slots' rows at each sample
    // [kMsSamples], then [chunk][2][(NU + 1) * (MUS + 1)] staged rows, then
    // [chunk][W] sums.
    extern __shared__ float4 s_ms[];
    float4* s_desc = s_ms;
    int4* s_held = reinterpret_cast<int4*>(s_ms + kMsRowFloat4s);
    Rgb* s_row = reinterpret_cast<Rgb*>(s_ms + kMsRowFloat4s + kMsSamples);
    const int NU = P.s_nu, MUS = P.s_mus, MU = P.s_mu;
    const int W = NU * MUS;
    const int CH = ms_chunks(P);
    const int tid = threadIdx.x, nt = blockDim.x;
    const int g = tid / W, x = tid - g * W;
    const bool in_chunk = g < CH;  // threads past CH * W only take the barriers
    const int i0 = in_chunk ? g * kMsSamples / CH : 0;
    const int i1 = in_chunk ? (g + 1) * kMsSamples / CH : 0;
    const int steps = (kMsSamples + CH - 1) / CH;  // the longest chunk

    const float4* desc = MR + (size_t(z) * MU + y) * kMsRowFloat4s;
    for (int e = tid; e < kMsRowFloat4s; e += nt) s_desc[e] = desc[e];
    auto d_tw = [&](int i) { return s_desc[i]; };
    auto d_geo = [&](int i) { return s_desc[kMsSamples + i]; };
    auto d_off = [&](int i) { return reinterpret_cast<const int4*>(s_desc + 2 * kMsSamples)[i]; };
    auto d_wt = [&](int i) { return s_desc[3 * kMsSamples + i]; };

    float tmu_s = 0.0f, tnu = 0.0f, tslice = 0.0f, tlerp = 0.0f;
    if (in_chunk) {
        TexelCoord<G> c = scattering_texel_coord<G>(P, unsigned(x), unsigned(y), unsigned(z));
        tmu_s = float(c.mu_s);
        tnu = float(c.nu);
        float u_nu = (tnu + 1.0f) / 2.0f;
        float tcx = u_nu * float(NU - 1);
        tslice = floorf(tcx);
        tlerp = tcx - tslice;
    }
    const int spos = x + x / MUS;

    const MsCoord<G> coord(P);
    const int SS = MUS + 1;
    const int entry = int(tslice) * SS;

    typedef typename std::conditional<H, Half4, Rgb>::type Slot;
    Slot slot[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) slot[k] = Slot{};
    constexpr int TB = H ? 8 : 16;
    const __amdgpu_buffer_rsrc_t jb = buffer_rsrc(J, int(size_t(P.s_r) * MU * W * TB));
    const int xoff = x * TB;
    auto ld = [&](int o) {
        if constexpr (H) {
            return __builtin_bit_cast(Half4, __builtin_amdgcn_raw_buffer_load_b64(jb, xoff, o * TB, 0));
        } else {
            const auto v = __builtin_amdgcn_raw_buffer_load_b96(jb, xoff, o * TB, 0);
            return Rgb{__uint_as_float(v[0]), __uint_as_float(v[1]), __uint_as_float(v[2])};
        }
    };
    auto advance = [&](int mask, int4 o) {
        if (mask & 1) slot[0] = ld(o.x);
        if (mask & 2) slot[1] = ld(o.y);
        if (mask & 4) slot[2] = ld(o.z);
        if (mask & 8) slot[3] = ld(o.w);
    };
    // Each chunk's two staged rows, laid out as in multiple_scattering_block
    // (pad entry per nu slice, zero slice NU).
    const int WP = (NU + 1) * SS;
    const int PADS = NU + 1 + MUS;
    for (int e = tid; e < CH * PADS; e += nt) {
        const int cg = e / PADS, e0 = e - cg * PADS;
        const int k = e0 < NU ? e0 * SS + MUS : NU * SS + (e0 - NU);
        s_row[(2 * cg) * WP + k] = Rgb{0.0f, 0.0f, 0.0f};
        s_row[(2 * cg + 1) * WP + k] = Rgb{0.0f, 0.0f, 0.0f};
    }
    Rgb* rows = s_row + 2 * (in_chunk ? g : 0) * WP;
    auto put = [&](int i, Rgb* dst) {
        const float4 w = d_wt(i);
        const Rgb t[4] = {to_rgb(slot[0]), to_rgb(slot[1]), to_rgb(slot[2]), to_rgb(slot[3])};
        dst[spos] = Rgb{fmaf(w.w, t[3].x, fmaf(w.z, t[2].x, fmaf(w.y, t[1].x, w.x * t[0].x))),
                        fmaf(w.w, t[3].y, fmaf(w.z, t[2].y, fmaf(w.y, t[1].y, w.x * t[0].y))),
                        fmaf(w.w, t[3].z, fmaf(w.z, t[2].z, fmaf(w.y, t[1].z, w.x * t[0].z)))};
    };
    float a0 = 0.0f, a1 = 0.0f, a2 = 0.0f;
    auto eval = [&](int i, const Rgb* __restrict__ cur) {
        const float4 tw = d_tw(i), geo = d_geo(i);
        const float xt = coord(tmu_s, tnu, geo.x, geo.z);
        const float w = __builtin_amdgcn_fractf(xt);
        const int k0 = entry + int(xt);
        const Rgb p0 = cur[k0], p1 = cur[k0 + 1], p2 = cur[k0 + SS], p3 = cur[k0 + SS + 1];
        float l = tlerp;
        float v0 = fmaf(w, p1.x - p0.x, p0.x), v1 = fmaf(w, p1.y - p0.y, p0.y),
              v2 = fmaf(w, p1.z - p0.z, p0.z);
        float u0 = fmaf(w, p3.x - p2.x, p2.x), u1 = fmaf(w, p3.y - p2.y, p2.y),
              u2 = fmaf(w, p3.z - p2.z, p2.z);
        a0 = fmaf(fmaf(l, u0 - v0, v0), tw.x, a0);
        a1 = fmaf(fmaf(l, u1 - v1, v1), tw.y, a1);
        a2 = fmaf(fmaf(l, u2 - v2, v2), tw.z, a2);
    };
    __syncthreads();  // the table and the rows' pads
    // The rows the four slots hold at each sample: a slot that a sample uses
    // without loading it holds the row it was last loaded with (the table's
    // offset is 0 for slots a sample does not load).  Lane j of the first
    // wavefront takes sample j: per slot, the last sample <= j that loads
    // it, by a prefix maximum over the lanes.
    if (tid < 64) {
        const int j = tid;
        const int m = j < kMsSamples ? __float_as_int(d_geo(j).y) : 0;
        int last[4];
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            int v = (m >> t) & 1 ? j : -1;
#pragma unroll
            for (int k = 1; k < 64; k <<= 1) {
                const int u = __shfl_up(v, k, 64);
                if (j >= k) v = max(v, u);
            }
            last[t] = v;
        }
        if (j < kMsSamples)
            s_held[j] = make_int4(last[0] >= 0 ? d_off(last[0]).x : 0,
                                  last[1] >= 0 ? d_off(last[1]).y : 0,
                                  last[2] >= 0 ? d_off(last[2]).z : 0,
                                  last[3] >= 0 ? d_off(last[3]).w : 0);
    }
    __syncthreads();
    if (in_chunk) {
        advance(15, s_held[i0]);
        put(i0, rows);
    }
    __syncthreads();
    for (int s = 0; s < steps; ++s) {
        const int i = i0 + s;
        const bool has = in_chunk && i < i1;
        const bool next = in_chunk && i + 1 < i1;
        if (next) advance(__float_as_int(d_geo(i + 1).y), d_off(i + 1));
        if (has) eval(i, rows + (s & 1) * WP);
        if (next) put(i + 1, rows + ((s + 1) & 1) * WP);
        __syncthreads();
    }
    Rgb* part = s_row + 2 * CH * WP;
    if (in_chunk) part[g * W + x] = Rgb{a0, a1, a2};
    __syncthreads();
    if (g == 0) {
        float m0 = part[x].x, m1 = part[x].y, m2 = part[x].z;
        for (int c = 1; c < CH; ++c) {
            const Rgb q = part[c * W + x];
            m0 = m0 + q.x;
            m1 = m1 + q.y;
            m2 = m2 + q.z;
        }
        const size_t idx = (size_t(z) * MU + y) * W + x;
        st_tex(dMS, idx, make_float4(m0, m1, m2, 0.0f), H);
        float pr = phase_rayleigh(tnu);
        float4 prev = ld_tex(S, idx, H);
        st_tex(S, idx,
               make_float4(m0 / pr + prev.x, m1 / pr + prev.y, m2 / pr + prev.z, 0.0f + prev.w),
               H);
    }
}

// ================================================== kernel entry points
// Plain kernels: one atmosphere, block coordinates from blockIdx, the
// parameters as a kernel argument.  Batched kernels (kb_*): one launch over
// many atmospheres; each block reads a 32-bit tile word (atmosphere slot in
// the top 8 bits, block index within that atmosphere's grid in the low 24)
// and the atmosphere's parameters and LUT pointers from HBM arrays.
template <typename G, bool COMP, int LANES>
__global__ __launch_bounds__(256) void k_transmittance(DevParams P, float4* __restrict__ T,
                                                       float4* __restrict__ OD) {
    if constexpr (LANES == kOrderedLanes)
        transmittance_block_ordered<G>(P, blockIdx.x, T);
    else
        transmittance_block<G, COMP, LANES>(P, blockIdx.x, 0, 0, T, OD);
}
template <typename G, bool COMP, int LANES>
__global__ __launch_bounds__(256) void kb_transmittance(const DevParams* __restrict__ Ps,
                                                        const LutPtrs* __restrict__ L,
                                                        const uint32_t* __restrict__ tiles, unsigned ntiles) {
    // Persistent when the grid is smaller than the tile list: the block
    // takes tiles blockIdx.x, +gridDim.x, ...; the barrier keeps one
    // tile's LDS reads apart from the next tile's writes.
    for (unsigned t = blockIdx.x; t < ntiles; t += gridDim.x) {
        if (t != blockIdx.x) __syncthreads();
        int atm, local;
        decode_tile(tiles[t], atm, local);
        const LutPtrs l = lut_ptrs(L, atm);
        if constexpr (LANES == kOrderedLanes)
            transmittance_block_ordered<G>(Ps[atm], local, l.T);
        else
            transmittance_block<G, COMP, LANES>(Ps[atm], local, 0, 0, l.T, l.OD);
    }
}

template <typename G>
__global__ __launch_bounds__(256) void k_direct_irradiance(DevParams P, const float4* __restrict__ T,
                                                           float4* __restrict__ dE) {
    direct_irradiance_block<G>(P, blockIdx.x, blockIdx.y, 0, T, dE);
}
template <typename G>
__global__ __launch_bounds__(256) void kb_direct_irradiance(const DevParams* __restrict__ Ps,
                                                            const LutPtrs* __restrict__ L,
                                                            const uint32_t* __restrict__ tiles, unsigned ntiles) {
    // Persistent when the grid is smaller than the tile list: the block
    // takes tiles blockIdx.x, +gridDim.x, ...; the barrier keeps one
    // tile's LDS reads apart from the next tile's writes.
    for (unsigned t = blockIdx.x; t < ntiles; t += gridDim.x) {
        if (t != blockIdx.x) __syncthreads();
        int atm, local;
        decode_tile(tiles[t], atm, local);
        const DevParams& P = Ps[atm];
        const int gx = (P.i_mus + 63) / 64;
        const LutPtrs l = lut_ptrs(L, atm);
        direct_irradiance_block<G>(P, local % gx, local / gx, 0, l.T, l.dE);
    }
}

template <typename G, bool COMP, bool H, int STAGED>
__global__ __launch_bounds__(256) void k_single_scattering(DevParams P, const float4* __restrict__ T,
                                                           const float4* __restrict__ SR,
                                                           float4* __restrict__ dR,
                                                           float4* __restrict__ dM,
                                                           float4* __restrict__ S,
                                                           unsigned remap) {
    const unsigned b = logical_block(remap);
    single_scattering_block<G, COMP, H, STAGED>(P, b % P.s_mu, b / P.s_mu, 0, T, SR, dR, dM, S);
}
template <typename G, bool COMP, bool H, int STAGED>
__global__ __launch_bounds__(256) void kb_single_scattering(const DevParams* __restrict__ Ps,
                                                            const LutPtrs* __restrict__ L,
                                                            const uint32_t* __restrict__ tiles, unsigned ntiles) {
    // Persistent when the grid is smaller than the tile list: the block
    // takes tiles blockIdx.x, +gridDim.x, ...; the barrier keeps one
    // tile's LDS reads apart from the next tile's writes.
    for (unsigned t = blockIdx.x; t < ntiles; t += gridDim.x) {
        if (t != blockIdx.x) __syncthreads();
        int atm, local;
        decode_tile(tiles[t], atm, local);
        const DevParams& P = Ps[atm];
        const LutPtrs l = lut_ptrs(L, atm);
        single_scattering_block<G, COMP, H, STAGED>(P, local % P.s_mu, local / P.s_mu, 0, l.T,
                                                    l.SR, l.dR, l.dM, l.S);
    }
}

template <typename G, bool H>
__global__ __launch_bounds__(kSsChunkThreads) void k_single_scattering_chunked(
    DevParams P, const float4* __restrict__ T, const float4* __restrict__ SR,
    float4* __restrict__ dR, float4* __restrict__ dM, float4* __restrict__ S, unsigned remap) {
    const unsigned b = logical_block(remap);
    single_scattering_block_chunked<G, H>(P, b % P.s_mu, b / P.s_mu, T, SR, dR, dM, S);
}
template <typename G, bool H>
__global__ __launch_bounds__(kSsChunkThreads) void kb_single_scattering_chunked(
    const DevParams* __restrict__ Ps, const LutPtrs* __restrict__ L,
    const uint32_t* __restrict__ tiles, unsigned ntiles) {
    for (unsigned t = blockIdx.x; t < ntiles; t += gridDim.x) {
        if (t != blockIdx.x) __syncthreads();
        int atm, local;
        decode_tile(tiles[t], atm, local);
        const DevParams& P = Ps[atm];
        const LutPtrs l = lut_ptrs(L, atm);
        single_scattering_block_chunked<G, H>(P, local % P.s_mu, local / P.s_mu, l.T, l.SR, l.dR,
                                              l.dM, l.S);
    }
}

// Per-set geometry: blocks [0, R + MUS) fill the density geometry table,
// the next MU * R blocks the single- and multiple-scattering row tables.
template <typename G>
__device__ __forceinline__ void geometry_block(const DevParams& P, const int b,
                                               const float4* __restrict__ T,
                                               const float4* __restrict__ OD,
                                               float4* __restrict__ DG, float4* __restrict__ SR,
                                               float4* __restrict__ MR) {
    const int nd = P.s_r + P.s_mus;
    if (b < nd) {
        density_geometry_block<G>(P, b, T, OD, DG);
    } else {
        const int rb = b - nd;
        row_geometry_block<G>(P, rb % P.s_mu, rb / P.s_mu, T, OD, SR, MR);
    }
}
template <typename G>
__global__ __launch_bounds__(64) void k_geometry(DevParams P, const float4* __restrict__ T,
                                                 const float4* __restrict__ OD,
                                                 float4* __restrict__ DG, float4* __restrict__ SR,
                                                 float4* __restrict__ MR) {
    geometry_block<G>(P, blockIdx.x, T, OD, DG, SR, MR);
}
template <typename G>
__global__ __launch_bounds__(64) void kb_geometry(const DevParams* __restrict__ Ps,
                                                  const LutPtrs* __restrict__ L,
                                                  const uint32_t* __restrict__ tiles,
                                                  unsigned ntiles) {
    for (unsigned t = blockIdx.x; t < ntiles; t += gridDim.x) {
        int atm, local;
        decode_tile(tiles[t], atm, local);
        const LutPtrs l = lut_ptrs(L, atm);
        geometry_block<G>(Ps[atm], local, l.T, l.OD, l.DG, l.SR, l.MR);
    }
}
template <typename G, bool SINGLE, bool H>
__global__ __launch_bounds__(64 * kIndWaves) void k_indirect_irradiance(
    DevParams P, const float4* __restrict__ dR, const float4* __restrict__ dM,
    const float4* __restrict__ dMS, float4* __restrict__ dE, float4* __restrict__ E) {
    indirect_irradiance_block<G, SINGLE, H>(P, blockIdx.x, 0, 0, dR, dM, dMS, dE, E);
}
template <typename G, bool SINGLE, bool H>
__global__ __launch_bounds__(64 * kIndWaves) void kb_indirect_irradiance(
    const DevParams* __restrict__ Ps, const LutPtrs* __restrict__ L,
    const uint32_t* __restrict__ tiles, unsigned ntiles) {
    // Persistent when the grid is smaller than the tile list: the block
    // takes tiles blockIdx.x, +gridDim.x, ...; the barrier keeps one
    // tile's LDS reads apart from the next tile's writes.
    for (unsigned t = blockIdx.x; t < ntiles; t += gridDim.x) {
        if (t != blockIdx.x) __syncthreads();
        int atm, local;
        decode_tile(tiles[t], atm, local);
        const LutPtrs l = lut_ptrs(L, atm);
        indirect_irradiance_block<G, SINGLE, H>(Ps[atm], local, 0, 0, l.dR, l.dM, l.dMS, l.dE,
                                                l.E);
    }
}

template <typename G, int TPT, bool H>
__global__ __launch_bounds__(kMsMaxThreads) void k_multiple_scattering(DevParams P,
                                                             const float4* __restrict__ MR,
                                                             const float4* __restrict__ J,
                                                             float4* __restrict__ dMS,
                                                             float4* __restrict__ S,
                                                             unsigned remap) {
    const unsigned b = logical_block(remap);
    multiple_scattering_block<G, TPT, H>(P, b % P.s_mu, b / P.s_mu, 0, MR, J, dMS, S);
}
template <typename G, int TPT, bool H>
__global__ __launch_bounds__(kMsMaxThreads) void kb_multiple_scattering(const DevParams* __restrict__ Ps,
                                                              const LutPtrs* __restrict__ L,
                                                              const uint32_t* __restrict__ tiles, unsigned ntiles) {
    // Persistent when the grid is smaller than the tile list: the block
    // takes tiles blockIdx.x, +gridDim.x, ...; the barrier keeps one
    // tile's LDS reads apart from the next tile's writes.
    for (unsigned t = blockIdx.x; t < ntiles; t += gridDim.x) {
        if (t != blockIdx.x) __syncthreads();
        int atm, local;
        decode_tile(tiles[t], atm, local);
        const DevParams& P = Ps[atm];
        const LutPtrs l = lut_ptrs(L, atm);
        multiple_scattering_block<G, TPT, H>(P, local % P.s_mu, local / P.s_mu, 0, l.MR,
                                                   l.J, l.dMS, l.S);
    }
}

template <typename G, bool H>
__global__ __launch_bounds__(kMsChunkMaxThreads) void k_multiple_scattering_chunked(
    DevParams P, const float4* __restrict__ MR, const float4* __restrict__ J,
    float4* __restrict__ dMS, float4* __restrict__ S, unsigned remap) {
    const unsigned b = logical_block(remap);
    multiple_scattering_block_chunked<G, H>(P, b % P.s_mu, b / P.s_mu, MR, J, dMS, S);
}
template <typename G, bool H>
__global__ __launch_bounds__(kMsChunkMaxThreads) void kb_multiple_scattering_chunked(
    const DevParams* __restrict__ Ps, const LutPtrs* __restrict__ L,
    const uint32_t* __restrict__ tiles, unsigned ntiles) {
    for (unsigned t = blockIdx.x; t < ntiles; t += gridDim.x) {
        if (t != blockIdx.x) __syncthreads();
        int atm, local;
        decode_tile(tiles[t], atm, local);
        const DevParams& P = Ps[atm];
        const LutPtrs l = lut_ptrs(L, atm);
        multiple_scattering_block_chunked<G, H>(P, local % P.s_mu, local / P.s_mu, l.MR, l.J,
                                                l.dMS, l.S);
    }
}

// ================================================================== clear
__global__ void k_fill_zero(float4* __restrict__ p, size_t n) {
    size_t i = size_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i < n) p[i] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
}
// Clear every atmosphere's irradiance LUT (src/precompute.rs:1802-1816).
__global__ void kb_clear_irradiance(const DevParams* __restrict__ Ps,
                                    const LutPtrs* __restrict__ L,
                                    const uint32_t* __restrict__ tiles, unsigned ntiles) {
    // Persistent when the grid is smaller than the tile list: the block
    // takes tiles blockIdx.x, +gridDim.x, ...; the barrier keeps one
    // tile's LDS reads apart from the next tile's writes.
    for (unsigned t = blockIdx.x; t < ntiles; t += gridDim.x) {
        if (t != blockIdx.x) __syncthreads();
        int atm, local;
        decode_tile(tiles[t], atm, local);
        const size_t n = size_t(Ps[atm].i_mus) * Ps[atm].i_r;
        const size_t i = size_t(local) * blockDim.x + threadIdx.x;
        if (i < n) lut_ptrs(L, atm).E[i] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    }
}

// ========================================================== launch wrappers
hipError_t launch_transmittance(const DevParams& P, float4* T, float4* OD, hipStream_t s) {
    size_t texels = size_t(P.t_mu) * P.t_r;
    if (P.flags & 1)
        k_transmittance<double, true, 16><<<cdiv(texels * 16, 256), 256, 0, s>>>(P, T, OD);
    else
        k_transmittance<float, false, kOrderedLanes>
            <<<cdiv(texels * kOrderedLanes, 256), 256, 0, s>>>(P, T, nullptr);
    return hipGetLastError();
}

hipError_t launch_direct_irradiance(const DevParams& P, const float4* T, float4* dE,
                                    hipStream_t s) {
    dim3 grid(cdiv(P.i_mus, 64), P.i_r);
    if (P.flags & 1)
        k_direct_irradiance<double><<<grid, 64, 0, s>>>(P, T, dE);
    else
        k_direct_irradiance<float><<<grid, 64, 0, s>>>(P, T, dE);
    return hipGetLastError();
}

hipError_t launch_geometry(const DevParams& P, const float4* T, const float4* OD, float4* DG,
                           float4* SR, float4* MR, hipStream_t s) {
    const unsigned blocks = unsigned(P.s_r + P.s_mus + P.s_mu * P.s_r);
    if (P.flags & 1)
        k_geometry<double><<<blocks, 64, 0, s>>>(P, T, OD, DG, SR, MR);
    else
        k_geometry<float><<<blocks, 64, 0, s>>>(P, T, OD, DG, SR, MR);
    return hipGetLastError();
}

template <bool H>
static hipError_t launch_single_scattering_h(const DevParams& P, const float4* T,
                                             const float4* SR, float4* dR, float4* dM, float4* S,
                                             const Tuning& tu, hipStream_t s) {
    const unsigned threads = tuned_threads(P, kPassSingle, 2, tu);
    const unsigned remap = (tu.remap >> kPassSingle) & 1u;
    dim3 grid(P.s_mu, P.s_r);
    if (ss_chunked(P)) {
        const size_t lds = ss_chunked_lds_bytes(P);
        if (P.flags & 1)
            k_single_scattering_chunked<double, H>
                <<<grid, kSsChunkThreads, lds, s>>>(P, T, SR, dR, dM, S, remap);
        else
            k_single_scattering_chunked<float, H>
                <<<grid, kSsChunkThreads, lds, s>>>(P, T, SR, dR, dM, S, remap);
    } else if (ss_staged(P)) {
        const size_t lds = ss_staged_lds_bytes(P.t_mu);
        const unsigned tpt = ss_tpt(P, threads);
#define FB_SS(G, X) \
    k_single_scattering<G, false, H, X><<<grid, threads, lds, s>>>(P, T, SR, dR, dM, S, remap)
        if (P.flags & 1)
            tpt == 1 ? FB_SS(double, 1) : tpt == 2 ? FB_SS(double, 2) : FB_SS(double, 4);
        else
            tpt == 1 ? FB_SS(float, 1) : tpt == 2 ? FB_SS(float, 2) : FB_SS(float, 4);
#undef FB_SS
    } else if (P.flags & 1) {
        k_single_scattering<double, false, H, 0><<<grid, threads, 0, s>>>(P, T, SR, dR, dM, S, remap);
    } else {
        k_single_scattering<float, false, H, 0><<<grid, threads, 0, s>>>(P, T, SR, dR, dM, S, remap);
    }
    return hipGetLastError();
}
hipError_t launch_single_scattering(const DevParams& P, const float4* T, const float4* SR,
                                    float4* dR, float4* dM, float4* S, const Tuning& tu,
                                    hipStream_t s) {
    return (P.flags & kFlagF16Storage)
               ? launch_single_scattering_h<true>(P, T, SR, dR, dM, S, tu, s)
               : launch_single_scattering_h<false>(P, T, SR, dR, dM, S, tu, s);
}

hipError_t launch_scattering_density(const DevParams& P, int order, const float4* DG,
                                     const float4* dR, const float4* dM, const float4* dMS,
                                     const float4* dE, float4* J, const Tuning& tu,
                                     hipStream_t s) {
    const unsigned threads = tuned_threads(P, kPassDensity, order, tu);
    const unsigned remap = (tu.remap >> kPassDensity) & 1u;
    return (P.flags & 1)
               ? DensityLaunch<double>::plain(P, order, DG, dR, dM, dMS, dE, J, threads, remap, s)
               : DensityLaunch<float>::plain(P, order, DG, dR, dM, dMS, dE, J, threads, remap, s);
}

template <bool H>
static hipError_t launch_indirect_irradiance_h(const DevParams& P, int order, const float4* dR,
                                               const float4* dM, const float4* dMS, float4* dE,
                                               float4* E, const Tuning& tu, hipStream_t s) {
    size_t n = size_t(P.i_mus) * P.i_r;
    const bool single = order == 1;
    size_t per_wave = indirect_lds_bytes_per_wave(P.s_nu, single);
    const int waves = int(tuned_threads(P, kPassIndirect, order + 1, tu) / 64);
    size_t lds = per_wave * waves;
    dim3 grid(cdiv(n, waves)), block(64 * waves);
    const bool precise = P.flags & 1;
    if (precise && single)
        k_indirect_irradiance<double, true, H><<<grid, block, lds, s>>>(P, dR, dM, dMS, dE, E);
    else if (precise)
        k_indirect_irradiance<double, false, H><<<grid, block, lds, s>>>(P, dR, dM, dMS, dE, E);
    else if (single)
        k_indirect_irradiance<float, true, H><<<grid, block, lds, s>>>(P, dR, dM, dMS, dE, E);
    else
        k_indirect_irradiance<float, false, H><<<grid, block, lds, s>>>(P, dR, dM, dMS, dE, E);
    return hipGetLastError();
}
hipError_t launch_indirect_irradiance(const DevParams& P, int order, const float4* dR,
                                      const float4* dM, const float4* dMS, float4* dE, float4* E,
                                      const Tuning& tu, hipStream_t s) {
    return (P.flags & kFlagF16Storage)
               ? launch_indirect_irradiance_h<true>(P, order, dR, dM, dMS, dE, E, tu, s)
               : launch_indirect_irradiance_h<false>(P, order, dR, dM, dMS, dE, E, tu, s);
}

template <bool H>
static hipError_t launch_multiple_scattering_h(const DevParams& P, const float4* MR,
                                               const float4* J, float4* dMS, float4* S,
                                               const Tuning& tu, hipStream_t s) {
    const int W = P.s_nu * P.s_mus;
    const int threads = int(tuned_threads(P, kPassMultiple, 2, tu));
    const unsigned remap = (tu.remap >> kPassMultiple) & 1u;
    dim3 grid(P.s_mu, P.s_r);
    if (ms_chunked(P)) {
        const size_t lds = ms_chunked_lds_bytes(P);
        const unsigned ct = ms_chunk_threads(P);
        if (P.flags & 1)
            k_multiple_scattering_chunked<double, H><<<grid, ct, lds, s>>>(P, MR, J, dMS, S,
                                                                          remap);
        else
            k_multiple_scattering_chunked<float, H><<<grid, ct, lds, s>>>(P, MR, J, dMS, S,
                                                                         remap);
        return hipGetLastError();
    }
    if (W > threads * kMsTexelsPerThread) return hipErrorInvalidValue;
    size_t lds = sizeof(Rgb) * kMsStagedRows * size_t(P.s_nu + 1) * (P.s_mus + 1);
    // Texels per thread: 1 up to 256 texels per row, else 2 or 4.  The
    // arithmetic of a texel does not depend on it.
    const int tpt = W <= threads ? 1 : (W <= 2 * threads ? 2 : 4);
    const bool precise = P.flags & 1;
#define FB_MS(G, TPT) \
    k_multiple_scattering<G, TPT, H><<<grid, threads, lds, s>>>(P, MR, J, dMS, S, remap)
    if (precise)
        tpt == 1 ? FB_MS(double, 1) : tpt == 2 ? FB_MS(double, 2) : FB_MS(double, 4);
    else
        tpt == 1 ? FB_MS(float, 1) : tpt == 2 ? FB_MS(float, 2) : FB_MS(float, 4);
#undef FB_MS
    return hipGetLastError();
}
hipError_t launch_multiple_scattering(const DevParams& P, const float4* MR, const float4* J,
                                      float4* dMS, float4* S, const Tuning& tu, hipStream_t s) {
    return (P.flags & kFlagF16Storage)
               ? launch_multiple_scattering_h<true>(P, MR, J, dMS, S, tu, s)
               : launch_multiple_scattering_h<false>(P, MR, J, dMS, S, tu, s);
}

// ------------------------------------------------------------ tuning
// Default and tuned block sizes.  `order` is the launch's scattering order
// (density n, the indirect pass of the order-n loop iteration, multiple n).
unsigned default_threads(const DevParams& P, int pass, int order) {
    const unsigned W = unsigned(P.s_nu * P.s_mus);
    const unsigned row = (W + 63) / 64 * 64;
    switch (pass) {
        case kPassSingle:
            return std::min(256u, row);
        case kPassMultiple:  // one texel per thread
            return std::min(unsigned(kMsMaxThreads), row);
        case kPassDensity:  // 256, or the tile's threads (in 256-thread blocks, half of them
                            // idle, a 64x64x32x8 FP32 launch takes 0.235 ms, not 0.176; a
                            // larger tile cut evenly, 3 x 192 for 256 + 256 + 64, is slower:
                            // 0.171 instead of 0.154 ms at 27x64x26x18)
            return std::min(256u, cdiv(unsigned(DenLayout(P, den_tpx(P)).total), 64) * 64);
        case kPassIndirect: {
            const size_t per_wave = indirect_lds_bytes_per_wave(P.s_nu, (order - 1) == 1);
            size_t waves = 65536 / per_wave;
            waves = waves < 1 ? 1 : (waves > size_t(kIndWaves) ? size_t(kIndWaves) : waves);
            return unsigned(64 * waves);
        }
    }
    return 256;
}

unsigned tuned_threads(const DevParams& P, int pass, int order, const Tuning& tu) {
    unsigned t = 0;
    switch (pass) {
        case kPassSingle: t = tu.single; break;
        case kPassDensity: t = order == 2 ? tu.density2 : tu.density; break;
        case kPassIndirect: t = 64 * (order == 2 ? tu.indirect1 : tu.indirect); break;
        case kPassMultiple: t = tu.multiple; break;
    }
    return (t != 0 && tuning_valid(P, pass, order, t)) ? t : default_threads(P, pass, order);
}

bool tuning_valid(const DevParams& P, int pass, int order, unsigned threads) {
    if (threads == 0 || threads % 64 != 0) return false;
    const unsigned W = unsigned(P.s_nu * P.s_mus);
    if (pass == kPassMultiple)  // above 256 threads, at most one wavefront more than the row
        return threads <= unsigned(kMsMaxThreads) && (threads <= 256 || threads < W + 64) &&
               W <= threads * unsigned(kMsTexelsPerThread);
    if (threads > 256) return false;
    switch (pass) {
        case kPassSingle:  // the staged kernel holds at most 4 texels per thread
            return !ss_staged(P) || W <= threads * unsigned(kSsTexelsPerThread);
        case kPassDensity:
            return true;
        case kPassIndirect:
            return indirect_lds_bytes_per_wave(P.s_nu, (order - 1) == 1) * (threads / 64) <=
                   65536;
    }
    return false;
}

// ------------------------------------------------------------ batched
PassShape batch_pass_shape(const DevParams& P, int pass, int order, unsigned threads) {
    const size_t ni = size_t(P.i_mus) * P.i_r;
    const bool precise = P.flags & 1;
    switch (pass) {
        case kPassTransmittance: {
            const size_t lanes = precise ? 16 : kOrderedLanes;
            return {cdiv(size_t(P.t_mu) * P.t_r * lanes, 256), 256, 0};
        }
        case kPassDirect:
            return {cdiv(P.i_mus, 64) * unsigned(P.i_r), 64, 0};
        case kPassSingle:
            if (ss_chunked(P))
                return {unsigned(P.s_mu) * unsigned(P.s_r), kSsChunkThreads,
                        ss_chunked_lds_bytes(P)};
            return {unsigned(P.s_mu) * unsigned(P.s_r), threads,
                    ss_staged(P) ? ss_staged_lds_bytes(P.t_mu) : 0};
        case kPassClear:
            return {cdiv(ni, 256), 256, 0};
        case kPassGeometry:
            return {unsigned(P.s_r + P.s_mus + P.s_mu * P.s_r), 64, 0};
        case kPassDensity:
            return {cdiv(size_t(DenLayout(P, den_tpx(P)).total), threads) * unsigned(P.s_mus) *
                        unsigned(P.s_r),
                    threads, density_lds_bytes(P.s_nu, P.i_mus, (order - 1) == 1)};
        case kPassIndirect: {  // one wave per texel
            const unsigned waves = threads / 64;
            return {cdiv(ni, waves), threads,
                    indirect_lds_bytes_per_wave(P.s_nu, (order - 1) == 1) * waves};
        }
        case kPassMultiple:
            if (ms_chunked(P))
                return {unsigned(P.s_mu) * unsigned(P.s_r), ms_chunk_threads(P),
                        ms_chunked_lds_bytes(P)};
            return {unsigned(P.s_mu) * unsigned(P.s_r), threads,
                    sizeof(Rgb) * kMsStagedRows * size_t(P.s_nu + 1) * (P.s_mus + 1)};
    }
    return {0, 0, 0};
}

template <bool H>
static hipError_t launch_batch_h(int pass, int order, bool precise, const DevParams* Ps,
                                 const LutPtrs* L, const uint32_t* tiles, unsigned ntiles,
                                 unsigned threads, size_t lds, unsigned grid_blocks, unsigned tpt,
                                 hipStream_t s) {
    if (ntiles == 0) return hipSuccess;
    const dim3 grid(grid_blocks && grid_blocks < ntiles ? grid_blocks : ntiles), block(threads);
    const bool single = (order - 1) == 1;
    switch (pass) {
        case kPassTransmittance:
            if (precise)
                kb_transmittance<double, true, 16><<<grid, block, 0, s>>>(Ps, L, tiles, ntiles);
            else
                kb_transmittance<float, false, kOrderedLanes>
                    <<<grid, block, 0, s>>>(Ps, L, tiles, ntiles);
            break;
        case kPassDirect:
            if (precise)
                kb_direct_irradiance<double><<<grid, block, 0, s>>>(Ps, L, tiles, ntiles);
            else
                kb_direct_irradiance<float><<<grid, block, 0, s>>>(Ps, L, tiles, ntiles);
            break;
        case kPassSingle:  // tpt: staged texels per thread, kSsDirect or kSsChunked
#define FB_KBSS(G, X) kb_single_scattering<G, false, H, X><<<grid, block, lds, s>>>(Ps, L, tiles, ntiles)
            if (tpt == kSsChunked) {
                if (precise)
                    kb_single_scattering_chunked<double, H><<<grid, block, lds, s>>>(Ps, L, tiles, ntiles);
                else
                    kb_single_scattering_chunked<float, H><<<grid, block, lds, s>>>(Ps, L, tiles, ntiles);
            } else if (precise) {
                tpt == 4   ? FB_KBSS(double, 4)
                : tpt == 2 ? FB_KBSS(double, 2)
                : tpt == 1 ? FB_KBSS(double, 1)
                           : FB_KBSS(double, 0);
            } else {
                tpt == 4   ? FB_KBSS(float, 4)
                : tpt == 2 ? FB_KBSS(float, 2)
                : tpt == 1 ? FB_KBSS(float, 1)
                           : FB_KBSS(float, 0);
            }
#undef FB_KBSS
            break;
        case kPassClear:
            kb_clear_irradiance<<<grid, block, 0, s>>>(Ps, L, tiles, ntiles);
            break;
        case kPassGeometry:
            if (precise)
                kb_geometry<double><<<grid, block, 0, s>>>(Ps, L, tiles, ntiles);
            else
                kb_geometry<float><<<grid, block, 0, s>>>(Ps, L, tiles, ntiles);
            break;
        case kPassDensity:  // tpt: texels per thread (den_tpx)
            if (precise)
                DensityLaunch<double>::batch(single, H, tpt, Ps, L, tiles, ntiles, grid, block, lds, s);
            else
                DensityLaunch<float>::batch(single, H, tpt, Ps, L, tiles, ntiles, grid, block, lds, s);
            break;
        case kPassIndirect:
            if (precise && single)
                kb_indirect_irradiance<double, true, H><<<grid, block, lds, s>>>(Ps, L, tiles, ntiles);
            else if (precise)
                kb_indirect_irradiance<double, false, H><<<grid, block, lds, s>>>(Ps, L, tiles, ntiles);
            else if (single)
                kb_indirect_irradiance<float, true, H><<<grid, block, lds, s>>>(Ps, L, tiles, ntiles);
            else
                kb_indirect_irradiance<float, false, H><<<grid, block, lds, s>>>(Ps, L, tiles, ntiles);
            break;
        case kPassMultiple:
#define FB_KBMS(G, T) kb_multiple_scattering<G, T, H><<<grid, block, lds, s>>>(Ps, L, tiles, ntiles)
            if (tpt == kMsChunkedTpt) {
                if (precise)
                    kb_multiple_scattering_chunked<double, H><<<grid, block, lds, s>>>(Ps, L, tiles, ntiles);
                else
                    kb_multiple_scattering_chunked<float, H><<<grid, block, lds, s>>>(Ps, L, tiles, ntiles);
            } else if (precise)
                tpt == 1 ? FB_KBMS(double, 1) : tpt == 2 ? FB_KBMS(double, 2) : FB_KBMS(double, 4);
            else
                tpt == 1 ? FB_KBMS(float, 1) : tpt == 2 ? FB_KBMS(float, 2) : FB_KBMS(float, 4);
#undef FB_KBMS
            break;
        default:
            return hipErrorInvalidValue;
    }
    return hipGetLastError();
}
hipError_t launch_batch(int pass, int order, bool precise, bool f16, const DevParams* Ps,
                        const LutPtrs* L, const uint32_t* tiles, unsigned ntiles,
                        unsigned threads, size_t lds, unsigned grid_blocks, unsigned tpt,
                        hipStream_t s) {
    return f16 ? launch_batch_h<true>(pass, order, precise, Ps, L, tiles, ntiles, threads, lds,
                                      grid_blocks, tpt, s)
               : launch_batch_h<false>(pass, order, precise, Ps, L, tiles, ntiles, threads, lds,
                                       grid_blocks, tpt, s);
}

// Blocks of one batched launch that fit on the device at once (per-CU
// occupancy of the launch's kernel x CUs); 0 if it cannot be determined.
template <bool H>
static unsigned batch_resident_blocks_h(int pass, int order, bool precise, unsigned threads,
                                        size_t lds, unsigned tpt) {
    const bool single = (order - 1) == 1;
    const void* fn = nullptr;
    switch (pass) {
        case kPassTransmittance:
            fn = precise ? (const void*)kb_transmittance<double, true, 16>
                         : (const void*)kb_transmittance<float, false, kOrderedLanes>;
            break;
        case kPassDirect:
            fn = precise ? (const void*)kb_direct_irradiance<double>
                         : (const void*)kb_direct_irradiance<float>;
            break;
        case kPassSingle:
            if (tpt == kSsChunked)
                fn = precise ? (const void*)kb_single_scattering_chunked<double, H>
                             : (const void*)kb_single_scattering_chunked<float, H>;
            else
#define FB_KBSS(X)                                                        \
    (precise ? (const void*)kb_single_scattering<double, false, H, X>     \
             : (const void*)kb_single_scattering<float, false, H, X>)
                fn = tpt == 4   ? FB_KBSS(4)
                     : tpt == 2 ? FB_KBSS(2)
                     : tpt == 1 ? FB_KBSS(1)
                                : FB_KBSS(0);
#undef FB_KBSS
            break;
        case kPassClear:
            fn = (const void*)kb_clear_irradiance;
            break;
        case kPassGeometry:
            fn = precise ? (const void*)kb_geometry<double> : (const void*)kb_geometry<float>;
            break;
        case kPassDensity:
            fn = precise ? DensityLaunch<double>::batch_kernel(single, H, tpt)
                         : DensityLaunch<float>::batch_kernel(single, H, tpt);
            break;
        case kPassIndirect:
            fn = precise ? (single ? (const void*)kb_indirect_irradiance<double, true, H>
                                   : (const void*)kb_indirect_irradiance<double, false, H>)
                         : (single ? (const void*)kb_indirect_irradiance<float, true, H>
                                   : (const void*)kb_indirect_irradiance<float, false, H>);
            break;
        case kPassMultiple:
            if (tpt == kMsChunkedTpt)
                fn = precise ? (const void*)kb_multiple_scattering_chunked<double, H>
                             : (const void*)kb_multiple_scattering_chunked<float, H>;
            else if (tpt == 1)
                fn = precise ? (const void*)kb_multiple_scattering<double, 1, H>
                             : (const void*)kb_multiple_scattering<float, 1, H>;
            else if (tpt == 2)
                fn = precise ? (const void*)kb_multiple_scattering<double, 2, H>
                             : (const void*)kb_multiple_scattering<float, 2, H>;
            else
                fn = precise ? (const void*)kb_multiple_scattering<double, 4, H>
                             : (const void*)kb_multiple_scattering<float, 4, H>;
            break;
    }
    int per_cu = 0, dev = 0, cus = 0;
    if (!fn || hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, fn, int(threads), lds) !=
                   hipSuccess ||
        hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess) {
        (void)hipGetLastError();
        return 0;
    }
    return unsigned(per_cu) * unsigned(cus);
}
unsigned batch_resident_blocks(int pass, int order, bool precise, bool f16, unsigned threads,
                               size_t lds, unsigned tpt) {
    return f16 ? batch_resident_blocks_h<true>(pass, order, precise, threads, lds, tpt)
               : batch_resident_blocks_h<false>(pass, order, precise, threads, lds, tpt);
}

hipError_t launch_fill_zero(float4* p, size_t n, hipStream_t s) {
    if (n == 0) return hipSuccess;
    k_fill_zero<<<cdiv(n, 256), 256, 0, s>>>(p, n);
    return hipGetLastError();
}

}  // namespace fbk
