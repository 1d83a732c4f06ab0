// density.hpp — the scattering density pass (shaders/scattering_density.comp)
// of geometry type G, compiled by density_f32.hip and density_f64.hip.
#pragma once

#include <type_traits>

#include "precompute_device.hpp"

namespace fbk {

// ===================================================== 4. scattering density
// scattering_density.comp:10-155.
//
// For a texel (r, mu, mu_s, nu) every incident-radiance lookup of the
// 16x32-direction quadrature is GetScattering(r, cos(theta_l), mu_s, nu1),
// so its (u_r, u_mu, u_mu_s) coordinates depend only on the texel's r and
// mu_s and on theta_l; only u_nu varies with phi.  All MU*NU texels that
// share (r, mu_s) therefore read the same 16 "nu profiles": for each theta
// row, the trilinear (mu_s, mu, r) sample of every nu slice k = -1..NU
// (slices -1 and NU reproduce CLAMP_TO_EDGE at the LUT's x edges).  A block
// builds those profiles in LDS once; each sample is then a 1D lerp between
// two LDS entries — the same value the reference's two trilinear texture
// fetches produce, with 8x-64x fewer gathers.
//
// Grid: (ceil(DenLayout.total/threads), MUS, R); each block serves one (r,
// mu_s) tile.

__device__ __forceinline__ PairEntry make_pair_entry(float4 rv, float4 rw, float4 mv, float4 mw) {
    PairEntry e;
    e.a = make_float4(rv.x, rv.y, rv.z, rw.x - rv.x);
    e.b = make_float4(rw.y - rv.y, rw.z - rv.z, mv.x, mv.y);
    e.c = make_float4(mv.z, mw.x - mv.x, mw.y - mv.y, mw.z - mv.z);
    return e;
}

// Per-texel constants of the density quadrature.  Order 2 works in nu1 =
// omega_i.omega_s, higher orders in the profile's entry coordinate
// x = (nu1 + 1) (NU-1)/2 + 1: (sx, sy) are omega_s.x, .y in those units.
struct DenTexel {
    float omx, omz;  // omega = (omx, 0, omz)
    float sx, sy;
};
// Per-row constants (of one mu).
template <typename G>
struct DenRow {
    float c;              // nu1 (order 2) or x (order >= 3) at the row's centre, nu1 =
                          // cos(theta) mu_s: a lookup is at c + sin(theta)
                          // (cos(phi) sx +- sin(phi) sy)
    float omzc, st;       // cos(theta) omega.z, sin(theta)
    float omx;            // omega.x, in FP32 mode sin(theta) omega.x
    const float* cx;      // sin(theta) cos(phi) of the row's directions
    const ProfEntry* pr;  // nu profile of multiple scattering (order n-1 >= 2)
    const PairEntry* pp;  // nu profiles of single Rayleigh and Mie (order 1)

    // nu2 = omega.omega_i of the directions phi_m and phi_{31-m}.  Near the Mie
    // peak an ulp of it counts: rounding sin(theta) omega.x once for the whole
    // row, as FP32 mode does, raises a g = 0.95 density's error by 14%.
    __device__ __forceinline__ float nu2(int m) const {
        return fmaf(sizeof(G) == sizeof(double) ? cx[m] : c_den.phi[m].x, omx, omzc);
    }
};
// Block constants of the quadrature.
struct DenConst {
    float g1, g2;     // 1 + g^2, -2g
    float hnu, hnu1;  // (NU-1)/2, (NU-1)/2 + 1
    float3 rho;       // Mie / Rayleigh coefficient at r, per channel
};
// The phase weight of a direction at a texel's mu, in units of the Rayleigh
// coefficient: (1 + nu2^2) (1 + rho x^-1.5), x = 1 + g^2 - 2 g nu2.
__device__ __forceinline__ float3 den_phase(const DenConst& k, float nu2, float& q, float& qw) {
    q = fmaf(nu2, nu2, 1.0f);
    qw = q * rsqrt_cubed(fmaf(k.g2, nu2, k.g1));
    return make_float3(fmaf(k.rho.x, qw, q), fmaf(k.rho.y, qw, q), fmaf(k.rho.z, qw, q));
}

// Linear filtering at texel coordinate t, given as e = t + 1: entry k + 1
// holds slot k, so floor(e) is the entry and fract(e) the weight, as
// prof_lerp computes for t >= -1.  Coordinates come from unit vectors, so
// rounding puts t at most a few ulp outside [0, kmax]: for t in (-1, 0), e
// is in (0, 1) and lerps slots -1 and 0, as the reference's two fetches do
// for a nu coordinate just below its range; just above kmax, int(e) is still
// the last entry and the weight of its delta a few ulp.  With e > 0,
// truncation is floor: the entry and weight take one conversion and one
// fract, and no clamp.  The +1 is folded into the per-texel and per-row
// terms the callers add anyway.
__device__ __forceinline__ float3 prof_lerp_i(const ProfEntry* __restrict__ prof, float e1) {
    const int k = int(e1);
    const float f = __builtin_amdgcn_fractf(e1);
    const ProfEntry* e = prof + k;
    float4 a = e->a;
    float2 b = e->b;
    return make_float3(fmaf(a.w, f, a.x), fmaf(b.x, f, a.y), fmaf(b.y, f, a.z));
}
// The same for a Rayleigh / Mie pair of profiles.
__device__ __forceinline__ void pair_lerp_i(const PairEntry* __restrict__ prof, float e1,
                                            float3& R, float3& M) {
    const int k = int(e1);
    const float f = __builtin_amdgcn_fractf(e1);
    const PairEntry* e = prof + k;
    const float4 a = e->a, b = e->b, c = e->c;
    R = make_float3(fmaf(a.w, f, a.x), fmaf(b.x, f, a.y), fmaf(b.y, f, a.z));
    M = make_float3(fmaf(c.y, f, b.z), fmaf(c.z, f, b.w), fmaf(c.w, f, c.x));
}

// The incident radiance at nu1 (order 2): Rayleigh and Mie profiles (which
// carry the phase constants) times their phase functions.
__device__ __forceinline__ float3 den_single(const DenConst& k, const PairEntry* pp, float nu1,
                                             float& q) {
    float3 R, M;
    pair_lerp_i(pp, fmaf(nu1, k.hnu, k.hnu1), R, M);
    q = fmaf(nu1, nu1, 1.0f);
    const float w = rsqrt_cubed(fmaf(k.g2, nu1, k.g1));
    return make_float3(fmaf(M.x, w, R.x), fmaf(M.y, w, R.y), fmaf(M.z, w, R.z));
}

// The 16 direction pairs (phi_m, phi_{31-m}) of one theta row, for N texels
// of one mu (one thread).  Both members of a pair share cos(phi), hence nu2
// = omega.omega_i and the phase weight, which depends on mu and the
// direction only, so the N texels share it too; the members' sin(phi) terms
// have opposite signs.  MOM: also the phase weights' sum and first cos(phi)
// moment (the caller's ground term at order 2).
template <bool SINGLE, bool MOM, int N, typename G>
__device__ __forceinline__ void density_row(const DenConst& k, const DenTexel* dt,
                                            const DenRow<G>& row, float3* a, float3& m0,
                                            float3& m1) {
    float sx[N], sy[N];
#pragma unroll
    for (int u = 0; u < N; ++u) {
        sx[u] = row.st * dt[u].sx;
        sy[u] = row.st * dt[u].sy;
    }
#pragma unroll
    for (int m = 0; m < kDenPhi / 2; ++m) {
        const float cp = c_den.phi[m].x, sp = c_den.phi[m].y;
        float q, qw;
        const float3 p = den_phase(k, row.nu2(m), q, qw);
        if (MOM) {
            m0 = make_float3(m0.x + p.x, m0.y + p.y, m0.z + p.z);
            m1 = make_float3(fmaf(cp, p.x, m1.x), fmaf(cp, p.y, m1.y), fmaf(cp, p.z, m1.z));
        }
#pragma unroll
        for (int u = 0; u < N; ++u) {
            const float base = fmaf(cp, sx[u], row.c);
            const float ca = fmaf(sp, sy[u], base), cb = fmaf(-sp, sy[u], base);
            float3 S;
            if (SINGLE) {
                float qa, qb;
                const float3 A = den_single(k, row.pp, ca, qa), B = den_single(k, row.pp, cb, qb);
                S = make_float3(fmaf(qb, B.x, qa * A.x), fmaf(qb, B.y, qa * A.y),
                                fmaf(qb, B.z, qa * A.z));
            } else {
                const float3 A = prof_lerp_i(row.pr, ca), B = prof_lerp_i(row.pr, cb);
                S = make_float3(A.x + B.x, A.y + B.y, A.z + B.z);
            }
            a[u].x = fmaf(p.x, S.x, a[u].x);
            a[u].y = fmaf(p.y, S.y, a[u].y);
            a[u].z = fmaf(p.z, S.z, a[u].z);
        }
    }
}

// The ground's share of a theta row whose irradiance lookups span one knot
// of the irradiance LUT, beyond the affine part: kappa x max(0, coordinate -
// knot), summed with the phase weights (coordinates in the units of row.c).
template <int N, typename G>
__device__ __forceinline__ void density_kink(const DenConst& k, const DenTexel* dt,
                                             const DenRow<G>& row, float4 kink, float3* a) {
    float sq[N] = {}, sw[N] = {}, sx[N], sy[N];
#pragma unroll
    for (int u = 0; u < N; ++u) {
        sx[u] = row.st * dt[u].sx;
        sy[u] = row.st * dt[u].sy;
    }
    const float c = row.c - kink.w;
#pragma unroll 4
    for (int m = 0; m < kDenPhi / 2; ++m) {
        const float cp = c_den.phi[m].x, sp = c_den.phi[m].y;
        float q, qw;
        (void)den_phase(k, row.nu2(m), q, qw);
#pragma unroll
        for (int u = 0; u < N; ++u) {
            const float base = fmaf(cp, sx[u], c);
            const float s = fmaxf(fmaf(sp, sy[u], base), 0.0f) +
                            fmaxf(fmaf(-sp, sy[u], base), 0.0f);
            sq[u] = fmaf(q, s, sq[u]);
            sw[u] = fmaf(qw, s, sw[u]);
        }
    }
#pragma unroll
    for (int u = 0; u < N; ++u) {
        a[u].x = fmaf(kink.x, fmaf(k.rho.x, sw[u], sq[u]), a[u].x);
        a[u].y = fmaf(kink.y, fmaf(k.rho.y, sw[u], sq[u]), a[u].y);
        a[u].z = fmaf(kink.z, fmaf(k.rho.z, sw[u], sq[u]), a[u].z);
    }
}

// The ground's share of a theta row whose irradiance lookups span more than
// one knot: an irradiance lookup per direction.  The entry coordinate is
// ec at the row's centre and changes by e1 per unit of row.c's coordinate.
template <int N, typename G>
__device__ __forceinline__ void density_ground(const DenConst& k, const DenTexel* dt,
                                               const DenRow<G>& row, const ProfEntry* erow, float ec,
                                               float e1, float3 gv, float3* a) {
    float3 s[N];
    float sx[N], sy[N];
#pragma unroll
    for (int u = 0; u < N; ++u) {
        s[u] = make_float3(0.0f, 0.0f, 0.0f);
        sx[u] = e1 * row.st * dt[u].sx;
        sy[u] = e1 * row.st * dt[u].sy;
    }
#pragma unroll 4
    for (int m = 0; m < kDenPhi / 2; ++m) {
        const float cp = c_den.phi[m].x, sp = c_den.phi[m].y;
        float q, qw;
        const float3 p = den_phase(k, row.nu2(m), q, qw);
#pragma unroll
        for (int u = 0; u < N; ++u) {
            const float base = fmaf(cp, sx[u], ec);
            const float3 A = prof_lerp_i(erow, fmaf(sp, sy[u], base)),
                         B = prof_lerp_i(erow, fmaf(-sp, sy[u], base));
            s[u].x = fmaf(p.x, A.x + B.x, s[u].x);
            s[u].y = fmaf(p.y, A.y + B.y, s[u].y);
            s[u].z = fmaf(p.z, A.z + B.z, s[u].z);
        }
    }
#pragma unroll
    for (int u = 0; u < N; ++u)
        a[u] = make_float3(fmaf(gv.x, s[u].x, a[u].x), fmaf(gv.y, s[u].y, a[u].y),
                           fmaf(gv.z, s[u].z, a[u].z));
}

// One (r, mu_s) tile's share of the density LUT.  DenLayout (kernels.hpp)
// maps the tile's threads to texels: the inner ones, TPX per thread, then,
// from a wavefront boundary, the outer ones.
//
// Outer texels (nu index 0 and NU-1, precision mode).  Their nu is clamped to mu mu_s -+
// sin sin_s (scattering.h:132-134): omega_s lies in omega's meridian plane,
// at azimuth pi or 0 for every mu.  So the incident radiance of direction
// (theta_l, phi_m) is the same for all mu of the tile: the block evaluates it
// once (s_outer, 16 x 16 directions, phi_m and phi_{31-m} being equal), and
// a thread only weighs it with its mu's phases: at azimuth 0 the value of
// direction m, at azimuth pi that of 15 - m.
//
// Bound by instruction issue (about 26 VALU slots per direction pair and
// inner texel at seven texels per thread, 33 at one, 10 per outer texel; 0.6
// of the 2.4 GHz issue peak at double).  ms per order >= 3 launch / order 2,
// with a ground lookup per direction on ground rows, every texel on the
// general path and two texels per thread before: default 0.236 -> 0.186 /
// 0.393 -> 0.321, double 3.48 -> 2.08 / 6.11 -> 4.35, half resolution 0.066 ->
// 0.041 / 0.085 -> 0.063.
template <typename G, bool SINGLE, bool H, int TPX = 1>
__device__ __forceinline__ void scattering_density_block(const DevParams& P, const int bx, const int by, const int bz, const float4* __restrict__ DG, const float4* __restrict__ dR,
    const float4* __restrict__ dM, const float4* __restrict__ dMS, const float4* __restrict__ dE,
    float4* __restrict__ J) {
    extern __shared__ float4 s_dyn[];
    __shared__ Taps s_ty[kDenTheta];      // mu taps of each theta row
    __shared__ Taps s_tz;                 // r taps of the tile
    // The ground term of each theta row (zero where the row misses the
    // ground), as a function of nu1 (see 0. below).
    __shared__ float4 s_gv[kDenTheta];    // T_g * albedo / pi (rgb), entry coordinate at centre
    __shared__ float4 s_glin[kDenTheta];  // affine part: value at centre (rgb), e per nu1
    __shared__ float4 s_gslope[kDenTheta];  // affine part: slope per nu1 (rgb)
    __shared__ float4 s_kink[kDenTheta];  // slope change per nu1 (rgb) at nu1 = w
    __shared__ int s_masks[3];            // rows with an affine part, one knot, more knots
    __shared__ float4 s_outer[kDenTheta][kDenOuterStride];  // incident radiance (outer texels)

    constexpr int NTEX = SINGLE ? 2 : 1;
    constexpr bool OUTER = sizeof(G) == sizeof(double);  // den_outer
    const int NU = P.s_nu, MUS = P.s_mus, MU = P.s_mu, NE = P.i_mus;
    const int W = NU * MUS;
    const int nslots = NU + 2, nent = NU + 1;
    const int j = by;  // mu_s index within a nu slice
    const int z = bz;  // r index
    const int tid = threadIdx.x;
    const int raw_f4 = NTEX * kDenTheta * nslots;
    float4* s_raw = s_dyn;                                   // [NTEX][16][nslots]
    ProfEntry* s_erow = reinterpret_cast<ProfEntry*>(s_dyn);  // [NE+1], after step 2
    float4* s_ent = s_dyn + max(raw_f4, 2 * (NE + 1));
    ProfEntry* s_prof = reinterpret_cast<ProfEntry*>(s_ent);  // [16][nent] (order >= 3)
    PairEntry* s_pair = reinterpret_cast<PairEntry*>(s_ent);  // [16][nent] (order 2)
    Taps* s_tx = reinterpret_cast<Taps*>(SINGLE ? static_cast<void*>(s_pair + kDenTheta * nent)
                                                : static_cast<void*>(s_prof + kDenTheta * nent));

    const float g = P.g;
    const float kR = 3.0f / (16.0f * kPi);
    const float kM = 3.0f / (8.0f * kPi) * (1.0f - g * g) / (2.0f + g * g);
    const TexelCoord<G> ct0 = scattering_texel_coord<G>(P, unsigned(j), 0u, unsigned(z));
    const float rf = float(ct0.r), osz = float(ct0.mu_s);
    const float sin_s = float(sqrt(fmax(G(1) - ct0.mu_s * ct0.mu_s, G(0))));
    DenConst kc;
    kc.g1 = 1.0f + g * g;
    kc.g2 = -2.0f * g;
    kc.hnu = 0.5f * float(NU - 1);
    kc.hnu1 = kc.hnu + 1.0f;
    const float hE = 0.5f * float(NE - 1);
    // delta_irradiance at r = bottom (irradiance.h:20-30 with x_r = 0).
    const Taps te = linear_taps<G>(tex_from_unit<G>(G(0), P.i_r), P.i_r);
    auto er = [&](int x) {
        x = min(max(x, 0), NE - 1);
        return lerp4(ldg4(dE + te.i0 * NE + x), ldg4(dE + te.i1 * NE + x), te.w);
    };

    // 0. Tile geometry from the density geometry table: the mu taps and
    // ground terms of each theta row (they depend on r only), the r taps,
    // and the x taps of each nu slot (they depend on mu_s only).
    //
    // The ground seen in direction omega_i is lit under the angle n.omega_s =
    // (r mu_s + d_g nu1) / |r zenith + d_g omega_i|, affine in nu1, so a
    // row's ground radiance is a piecewise linear function of nu1 whose
    // knots are the irradiance LUT's texels.  Over the row's range of nu1,
    // cos(theta) mu_s +- sin(theta) sin_s, most rows of an Earth-like planet
    // meet no knot (3/4 of the ground rows at default sizes, one knot 1/5):
    // the affine part then needs no lookup of its own per direction.  With
    // it in the profile entries (order >= 3) or in two moments of the phase
    // weights (order 2), one knot by density_kink and more by
    // density_ground, the ground costs 2-3 instead of 22 instructions per
    // direction pair on half of the rows.
    const int S = TPX > 1 ? 1 : P.den_split;  // threads per texel group (see below)
    const int slot0 = int(blockDim.x) >= 64 + nslots ? 64 : kDenTheta;
    // Lane l of the block's last wavefront takes the ground term of row l;
    // its irradiance loads overlap the profile gathers of the others.
    const int gl0 = tid - (int(blockDim.x) - 64);
    const bool ground_lane = gl0 >= 0 && gl0 < kDenTheta;
    float4 gd = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    float ginv = 0.0f;
    if (ground_lane) {
        const float4* dgz = DG + dg_row(z);
        gd = dgz[gl0];
        ginv = dgz[kDenTheta + gl0].w;
    }
    if (tid < kDenTheta) {
        const float4 t = DG[dg_row(z) + kDenTheta + tid];
        s_ty[tid] = Taps{__float_as_int(t.x), __float_as_int(t.y), t.z};
    } else if (tid >= slot0 && tid < slot0 + nslots) {
        const float4 x = DG[dg_x(P.s_r, j, NU) + (tid - slot0)];
        s_tx[tid - slot0] = Taps{__float_as_int(x.x), __float_as_int(x.y), x.z};
        if (tid == slot0) {
            const float4 c = DG[dg_row(z) + 2 * kDenTheta];
            s_tz = Taps{__float_as_int(c.x), __float_as_int(c.y), c.z};
        }
    }
    __syncthreads();
    if (ground_lane) {
        const float ct = c_den.cos[gl0];
        const float C = ct * osz;
        // Entry coordinate of the lookup (slot k at entry k + 1): ec + e1 (nu1 - C).
        const float ec = fmaf((rf + ct * gd.w) * ginv * osz, hE, hE + 1.0f);
        const float e1 = gd.w * ginv * hE;
        const float e_half = e1 * c_den.sin[gl0] * sin_s;
        int knots = -1;
        float4 lin = make_float4(0.0f, 0.0f, 0.0f, e1), slope = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        float4 kink = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        if (ginv != 0.0f) {
            const float lo = floorf(ec - e_half);
            knots = int(floorf(ec + e_half) - lo);
            // Theta-split lanes run their rows' loops one after the other
            // where they differ: one kind of loop for rows with knots.
            if (S > 1 && knots == 1) knots = 2;
            if (knots <= 1) {
                const int e = int(lo);  // entry e: slots e - 1 and e
                const float4 v0 = er(e - 1), v1 = er(e), v2 = er(e + 1);
                const float3 d = make_float3(v1.x - v0.x, v1.y - v0.y, v1.z - v0.z);
                lin.x = gd.x * fmaf(d.x, ec - lo, v0.x);
                lin.y = gd.y * fmaf(d.y, ec - lo, v0.y);
                lin.z = gd.z * fmaf(d.z, ec - lo, v0.z);
                slope = make_float4(gd.x * d.x * e1, gd.y * d.y * e1, gd.z * d.z * e1, 0.0f);
                if (knots == 1)
                    kink = make_float4(gd.x * ((v2.x - v1.x) - d.x) * e1,
                                       gd.y * ((v2.y - v1.y) - d.y) * e1,
                                       gd.z * ((v2.z - v1.z) - d.z) * e1,
                                       C + (lo + 1.0f - ec) / e1);
            }
        }
        s_gv[gl0] = make_float4(gd.x, gd.y, gd.z, ec);
        s_glin[gl0] = lin;
        s_gslope[gl0] = slope;
        s_kink[gl0] = kink;
        const unsigned long long b0 = __ballot(knots == 0 || knots == 1);
        const unsigned long long b1 = __ballot(knots == 1), b2 = __ballot(knots > 1);
        if (gl0 == 0) {
            s_masks[0] = int(b0 & 0xffffull);
            s_masks[1] = int(b1 & 0xffffull);
            s_masks[2] = int(b2 & 0xffffull);
        }
    }
    // 1. Raw profiles: 16 theta rows x (NU+2) nu slots (-1..NU) per texture.
    {
        const Taps tz = s_tz;
        for (int e = tid; e < NTEX * kDenTheta * nslots; e += blockDim.x) {
            int tex_sel = e / (kDenTheta * nslots);
            int rem = e % (kDenTheta * nslots);
            int l = rem / nslots, slot = rem % nslots;
            const float4* tex = SINGLE ? (tex_sel == 0 ? dR : dM) : dMS;
            s_raw[e] = trilinear_taps_t<H>(P, tex, s_tx[slot], s_ty[l], tz);
        }
    }
    __syncthreads();
    const int lin_mask = __builtin_amdgcn_readfirstlane(s_masks[0]);
    const int kink_mask = __builtin_amdgcn_readfirstlane(s_masks[1]);
    const int many_mask = __builtin_amdgcn_readfirstlane(s_masks[2]);
    // 2. Entries.  Order 1 (single scattering): (value, delta) times the phase
    // constants, rayleigh x 3/(16 pi), mie x 3/(8 pi)(1-g^2)/(2+g^2) (util.h:
    // 26-34).  Later orders: (value, delta), the affine part of the ground term
    // included.
    for (int e = tid; e < kDenTheta * nent; e += blockDim.x) {
        const int row = e / nent, k = e % nent;  // entry k holds slot k-1
        const float4 v = s_raw[row * nslots + k], w = s_raw[row * nslots + k + 1];
        if (SINGLE) {
            const float4 mv = s_raw[(kDenTheta + row) * nslots + k],
                         mw = s_raw[(kDenTheta + row) * nslots + k + 1];
            auto scaled = [](float4 x, float s) {
                return make_float4(x.x * s, x.y * s, x.z * s, 0.0f);
            };
            s_pair[e] = make_pair_entry(scaled(v, kR), scaled(w, kR), scaled(mv, kM),
                                        scaled(mw, kM));
        } else {
            const float4 gl = s_glin[row], gs = s_gslope[row];
            const float h = 1.0f / kc.hnu;
            const float dn = fmaf(float(k) - kc.hnu1, h, -c_den.cos[row] * osz);  // nu1 - centre
            const float3 d = make_float3(fmaf(gs.x, h, w.x - v.x), fmaf(gs.y, h, w.y - v.y),
                                         fmaf(gs.z, h, w.z - v.z));
            ProfEntry p;
            p.a = make_float4(v.x + fmaf(gs.x, dn, gl.x), v.y + fmaf(gs.y, dn, gl.y),
                              v.z + fmaf(gs.z, dn, gl.z), d.x);
            p.b = make_float2(d.y, d.z);
            p.pad = make_float2(0.0f, 0.0f);
            s_prof[e] = p;
        }
    }
    __syncthreads();
    // 3. The irradiance as (value, delta) entries, in the raw profiles' space,
    // for tiles with rows that look it up per direction.
    if (many_mask) {
        for (int e = tid; e <= NE; e += blockDim.x) s_erow[e] = make_entry(er(e - 1), er(e));
        __syncthreads();
    }

    // Coordinates are nu1 at order 2, else the entry coordinate nu1 hnu + hnu1.
    const float unit = SINGLE ? 1.0f : kc.hnu, per_unit = 1.0f / unit;
    auto make_row = [&](int l, float ct, float omx, float omz) {
        DenRow<G> row;
        row.c = SINGLE ? ct * osz : fmaf(ct * osz, kc.hnu, kc.hnu1);
        row.omzc = ct * omz;
        row.st = c_den.sin[l];
        row.omx = OUTER ? omx : row.st * omx;
        row.cx = c_den.cx + l * kDenPhi / 2;
        row.pr = s_prof + l * nent;
        row.pp = s_pair + l * nent;
        return row;
    };
    auto row_kink = [&](int l) {
        const float4 k = s_kink[l];
        return make_float4(k.x * per_unit, k.y * per_unit, k.z * per_unit,
                           SINGLE ? k.w : fmaf(k.w, kc.hnu, kc.hnu1));
    };

    const DenLayout lay(P, TPX);
    // 4. The outer texels' incident radiance, in the blocks that hold some.
    if (OUTER && (bx + 1) * int(blockDim.x) > lay.inner) {
        for (int e = tid; e < kDenTheta * kDenPhi / 2; e += blockDim.x) {
            const int l = e / (kDenPhi / 2), m = e % (kDenPhi / 2);
            const float4 o = c_den.dir[l * kDenPhi + m];
            const DenRow<G> row = make_row(l, o.z, 0.0f, 0.0f);
            const float dn = o.x * sin_s;  // nu1 - centre
            float3 L;
            if (SINGLE) {
                float q;
                L = den_single(kc, row.pp, row.c + dn, q);
                const float4 gl = s_glin[l], gs = s_gslope[l];
                L = make_float3(fmaf(q, L.x, fmaf(gs.x, dn, gl.x)),
                                fmaf(q, L.y, fmaf(gs.y, dn, gl.y)),
                                fmaf(q, L.z, fmaf(gs.z, dn, gl.z)));
            } else {
                L = prof_lerp_i(row.pr, fmaf(dn, kc.hnu, row.c));
            }
            if ((kink_mask >> l) & 1) {
                const float4 k = s_kink[l];
                const float t = fmaxf(fmaf(o.z, osz, dn) - k.w, 0.0f);
                L = make_float3(fmaf(k.x, t, L.x), fmaf(k.y, t, L.y), fmaf(k.z, t, L.z));
            }
            if ((many_mask >> l) & 1) {
                const float4 gv = s_gv[l];
                const float3 E = prof_lerp_i(s_erow, fmaf(s_glin[l].w, dn, gv.w));
                L = make_float3(fmaf(gv.x, E.x, L.x), fmaf(gv.y, E.y, L.y),
                                fmaf(gv.z, E.z, L.z));
            }
            s_outer[l][m] = make_float4(L.x, L.y, L.z, 0.0f);
        }
        __syncthreads();
    }

    // The phase functions' constants and the coefficients at r, per channel:
    // Rayleigh, and Mie in units of Rayleigh (of 1e-8 of Mie where there is
    // less Rayleigh than that).
    const float alt = float(ct0.r - G(P.bottom));
    const float rho_r = profile_density(P.prof[0], alt), rho_m = profile_density(P.prof[1], alt);
    float3 cr;
    {
        auto coef = [&](int c, float& rho) {
            const float cm = kM * P.mie_scattering[c] * rho_m;
            const float r = fmaxf(kR * P.rayleigh_scattering[c] * rho_r, 1e-8f * cm);
            rho = r > 0.0f ? cm / r : 0.0f;
            return r;
        };
        cr.x = coef(0, kc.rho.x);
        cr.y = coef(1, kc.rho.y);
        cr.z = coef(2, kc.rho.z);
    }
    // omega, omega_s of texel (nu index k, mu index y) (scattering_density.
    // comp:28-32), built in G.
    auto texel_setup = [&](int k, int y, DenTexel& dt) {
        const TexelCoord<G> c =
            scattering_texel_coord<G>(P, unsigned(k * MUS + j), unsigned(y), unsigned(z));
        G om_x = sqrt(G(1) - c.mu * c.mu);
        G sdx = om_x == G(0) ? G(0) : (c.nu - c.mu * c.mu_s) / om_x;
        G sdy = sqrt(fmax(G(1) - sdx * sdx - c.mu_s * c.mu_s, G(0)));
        dt.omx = float(om_x);
        dt.omz = float(c.mu);
        // Unit-vector components, clamped so every lookup coordinate is finite.
        dt.sx = fminf(fmaxf(float(sdx), -1.0f), 1.0f) * unit;
        dt.sy = fminf(fmaxf(float(sdy), -1.0f), 1.0f) * unit;
    };
    auto store = [&](int k, int y, float3 a) {
        st_tex(J, (size_t(z) * MU + y) * W + size_t(k * MUS + j),
               make_float4(cr.x * a.x, cr.y * a.y, cr.z * a.z, 0.0f), H);
    };
    // S consecutive lanes per thread group, lane l0 taking theta rows l0, l0 +
    // S, ... (S = 1: one thread walks all 16 rows), summed by a tree.
    auto reduce = [&](float3& a) {
        if (TPX > 1) return;
        for (int o = S / 2; o > 0; o >>= 1) {
            a.x += __shfl_xor(a.x, o);
            a.y += __shfl_xor(a.y, o);
            a.z += __shfl_xor(a.z, o);
        }
    };
    const int p = bx * int(blockDim.x) + tid;
    if (OUTER && p >= lay.inner) {
        const int y = (p - lay.inner) / S, l0 = (p - lay.inner) % S;
        if (y >= MU) return;  // a whole group of S lanes
        DenTexel dt;
        texel_setup(0, y, dt);
        float3 lo = make_float3(0.0f, 0.0f, 0.0f), hi = lo;  // azimuth pi, 0
        for (int l = l0; l < kDenTheta; l += S) {
            const float4 d0 = c_den.dir[l * kDenPhi];
            const DenRow<G> row = make_row(l, d0.z, dt.omx, dt.omz);
            float3 a = make_float3(0.0f, 0.0f, 0.0f), b = a;
#pragma unroll
            for (int m = 0; m < kDenPhi / 2; ++m) {
                float q, qw;
                const float3 w = den_phase(kc, row.nu2(m), q, qw);
                const float4 u = s_outer[l][m], v = s_outer[l][kDenPhi / 2 - 1 - m];
                a = make_float3(fmaf(w.x, u.x, a.x), fmaf(w.y, u.y, a.y), fmaf(w.z, u.z, a.z));
                b = make_float3(fmaf(w.x, v.x, b.x), fmaf(w.y, v.y, b.y), fmaf(w.z, v.z, b.z));
            }
            const float dom = 2.0f * d0.w;  // phi_m and phi_{31-m}
            hi = make_float3(fmaf(dom, a.x, hi.x), fmaf(dom, a.y, hi.y), fmaf(dom, a.z, hi.z));
            lo = make_float3(fmaf(dom, b.x, lo.x), fmaf(dom, b.y, lo.y), fmaf(dom, b.z, lo.z));
        }
        reduce(lo);
        reduce(hi);
        if (l0 != 0) return;
        store(0, y, lo);
        store(NU - 1, y, hi);
        return;
    }
    const int t = p / S, l0 = p % S;
    if (t >= lay.groups) return;  // a whole group of S lanes
    // Consecutive lanes take consecutive mu: their lookups lie close together.
    const int y = t % MU, k0 = lay.first + t / MU * TPX;
    DenTexel dt[TPX];
#pragma unroll
    for (int u = 0; u < TPX; ++u) texel_setup(k0 + u, y, dt[u]);
    float3 acc[TPX];
#pragma unroll
    for (int u = 0; u < TPX; ++u) acc[u] = make_float3(0.0f, 0.0f, 0.0f);
    for (int l = l0; l < kDenTheta; l += S) {
        const float4 d0 = c_den.dir[l * kDenPhi];
        const float ct = d0.z, dom = d0.w;
        const DenRow<G> row = make_row(l, ct, dt[0].omx, dt[0].omz);
        float3 a[TPX], m0 = make_float3(0.0f, 0.0f, 0.0f), m1 = m0;
#pragma unroll
        for (int u = 0; u < TPX; ++u) a[u] = m0;
        if (SINGLE && ((lin_mask >> l) & 1)) {
            density_row<SINGLE, true, TPX>(kc, dt, row, a, m0, m1);
            const float4 gl = s_glin[l], gs = s_gslope[l];
#pragma unroll
            for (int u = 0; u < TPX; ++u) {
                const float s = 2.0f * row.st * dt[u].sx;
                a[u].x = fmaf(2.0f * gl.x, m0.x, fmaf(s * gs.x, m1.x, a[u].x));
                a[u].y = fmaf(2.0f * gl.y, m0.y, fmaf(s * gs.y, m1.y, a[u].y));
                a[u].z = fmaf(2.0f * gl.z, m0.z, fmaf(s * gs.z, m1.z, a[u].z));
            }
        } else {
            density_row<SINGLE, false, TPX>(kc, dt, row, a, m0, m1);
        }
        if ((kink_mask >> l) & 1) density_kink<TPX>(kc, dt, row, row_kink(l), a);
        if ((many_mask >> l) & 1) {
            const float4 gv = s_gv[l];
            density_ground<TPX>(kc, dt, row, s_erow, gv.w, s_glin[l].w * per_unit,
                                make_float3(gv.x, gv.y, gv.z), a);
        }
#pragma unroll
        for (int u = 0; u < TPX; ++u)
            acc[u] = make_float3(fmaf(dom, a[u].x, acc[u].x), fmaf(dom, a[u].y, acc[u].y),
                                 fmaf(dom, a[u].z, acc[u].z));
    }
#pragma unroll
    for (int u = 0; u < TPX; ++u) reduce(acc[u]);
    if (l0 != 0) return;
#pragma unroll
    for (int u = 0; u < TPX; ++u) store(k0 + u, y, acc[u]);
}

// ------------------------------------------------------------------ kernels
template <typename G, bool SINGLE, bool H, int TPX = 1>
__global__ __launch_bounds__(256, den_occupancy(TPX, SINGLE)) void k_scattering_density(
    DevParams P, const float4* __restrict__ DG, const float4* __restrict__ dR,
    const float4* __restrict__ dM, const float4* __restrict__ dMS, const float4* __restrict__ dE,
    float4* __restrict__ J, unsigned remap) {
    const unsigned b = logical_block(remap), gx = gridDim.x;
    scattering_density_block<G, SINGLE, H, TPX>(P, b % gx, (b / gx) % P.s_mus,
                                                b / (gx * P.s_mus), DG, dR, dM, dMS, dE, J);
}

template <typename G, bool SINGLE, bool H, int TPX = 1>
__global__ __launch_bounds__(256, den_occupancy(TPX, SINGLE)) void kb_scattering_density(
    const DevParams* __restrict__ Ps, const LutPtrs* __restrict__ L,
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
        const int gx = (DenLayout(P, TPX).total + int(blockDim.x) - 1) / int(blockDim.x);
        scattering_density_block<G, SINGLE, H, TPX>(P, local % gx, (local / gx) % P.s_mus,
                                                    local / (gx * P.s_mus), l.DG, l.dR, l.dM,
                                                    l.dMS, l.dE, l.J);
    }
}

// -------------------------------------------------------- launch wrappers
// Calls f(order-2 flag, binary16 flag, texels per thread) as compile-time
// constants.
template <typename F>
static void den_dispatch(bool single, bool f16, int tpx, F f) {
    auto by_tpx = [&](auto sg, auto h) {
        switch (tpx) {
            case 7: f(sg, h, std::integral_constant<int, 7>{}); break;
            case 6: f(sg, h, std::integral_constant<int, 6>{}); break;
            case 4: f(sg, h, std::integral_constant<int, 4>{}); break;
            case 2: f(sg, h, std::integral_constant<int, 2>{}); break;
            default: f(sg, h, std::integral_constant<int, 1>{}); break;
        }
    };
    auto by_h = [&](auto sg) {
        f16 ? by_tpx(sg, std::true_type{}) : by_tpx(sg, std::false_type{});
    };
    single ? by_h(std::true_type{}) : by_h(std::false_type{});
}

template <typename G>
hipError_t DensityLaunch<G>::upload() {
    return upload_density_tables();
}

template <typename G>
hipError_t DensityLaunch<G>::plain(const DevParams& P, int order, const float4* DG,
                                   const float4* dR, const float4* dM, const float4* dMS,
                                   const float4* dE, float4* J, unsigned threads, unsigned remap,
                                   hipStream_t s) {
    const int tpx = den_tpx(P);
    const dim3 grid(cdiv(size_t(DenLayout(P, tpx).total), threads), P.s_mus, P.s_r);
    // The density of order n reads the scattering of order n-1; order 1 is
    // single Rayleigh + Mie (scattering.h:157-179).
    const bool single = (order - 1) == 1;
    const size_t lds = density_lds_bytes(P.s_nu, P.i_mus, single);
    den_dispatch(single, P.flags & kFlagF16Storage, tpx, [&](auto sg, auto h, auto x) {
        k_scattering_density<G, sg.value, h.value, x.value>
            <<<grid, threads, lds, s>>>(P, DG, dR, dM, dMS, dE, J, remap);
    });
    return hipGetLastError();
}

template <typename G>
void DensityLaunch<G>::batch(bool single, bool f16, unsigned tpx, const DevParams* Ps,
                             const LutPtrs* L, const uint32_t* tiles, unsigned ntiles, dim3 grid,
                             dim3 block, size_t lds, hipStream_t s) {
    den_dispatch(single, f16, int(tpx), [&](auto sg, auto h, auto x) {
        kb_scattering_density<G, sg.value, h.value, x.value>
            <<<grid, block, lds, s>>>(Ps, L, tiles, ntiles);
    });
}

template <typename G>
const void* DensityLaunch<G>::batch_kernel(bool single, bool f16, unsigned tpx) {
    const void* fn = nullptr;
    den_dispatch(single, f16, int(tpx), [&](auto sg, auto h, auto x) {
        fn = (const void*)kb_scattering_density<G, sg.value, h.value, x.value>;
    });
    return fn;
}

}  // namespace fbk
