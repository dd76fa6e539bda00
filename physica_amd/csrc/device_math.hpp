// Device-side vector math and SPH kernel functions for gfx950.
//
// Every function keeps the operand order of the reference's device helpers so
// that, compiled with -ffp-contract=off (no FMA formation) and HIP's default
// correctly rounded FP32 division and square root, each result is the IEEE
// value of the same expression. Reference: fluids/liquid/particle/
// domain/device.cuh:8-82, density/device.cuh:10-88, pbf/pbf.cu:18-71.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace phx {

constexpr float kPi = 3.14159265358979323846F;

struct Float3 {
    float x, y, z;
};

__device__ __forceinline__ Float3 make3(float x, float y, float z) { return Float3{x, y, z}; }
__device__ __forceinline__ Float3 add(Float3 a, Float3 b) { return {a.x + b.x, a.y + b.y, a.z + b.z}; }
__device__ __forceinline__ Float3 sub(Float3 a, Float3 b) { return {a.x - b.x, a.y - b.y, a.z - b.z}; }
__device__ __forceinline__ Float3 scale(Float3 v, float f) { return {f * v.x, f * v.y, f * v.z}; }
__device__ __forceinline__ float dot(Float3 a, Float3 b) { return a.x * b.x + a.y * b.y + a.z * b.z; }
__device__ __forceinline__ Float3 cross(Float3 a, Float3 b) {
    return {a.y * b.z - a.z * b.y, a.z * b.x - a.x * b.z, a.x * b.y - a.y * b.x};
}
__device__ __forceinline__ float length(Float3 a) { return sqrtf(dot(a, a)); }

// SoA field of three float arrays (domain/device.h:20-36).
struct Vec {
    float* x;
    float* y;
    float* z;
};
struct CVec {
    const float* x;
    const float* y;
    const float* z;
};

__device__ __forceinline__ Float3 load(CVec f, uint32_t i) { return {f.x[i], f.y[i], f.z[i]}; }
__device__ __forceinline__ Float3 load(Vec f, uint32_t i) { return {f.x[i], f.y[i], f.z[i]}; }
__device__ __forceinline__ void store(Vec f, uint32_t i, Float3 v) {
    f.x[i] = v.x;
    f.y[i] = v.y;
    f.z[i] = v.z;
}

// ---------------------------------------------------------------- kernels
// poly6, density/device.cuh:10-16
__device__ __forceinline__ float poly6(Float3 d, float h) {
    const float sq = dot(d, d);
    const float hr = h * h;
    if (sq >= hr) return 0.0F;
    const float diff = hr - sq;
    return 315.0F * diff * diff * diff / (64.0F * kPi * hr * hr * hr * h * h * h);
}

// poly6 gradient, density/device.cuh:18-24
__device__ __forceinline__ Float3 poly6_gradient(Float3 d, float h) {
    const float sq = dot(d, d);
    const float hr = h * h;
    if (sq >= hr) return {0.0F, 0.0F, 0.0F};
    const float diff = hr - sq;
    return scale(d, -945.0F * diff * diff / (32.0F * kPi * hr * hr * hr * h * h * h));
}

// cubic spline, density/device.cuh:26-34
__device__ __forceinline__ float cubic(Float3 d, float h) {
    const float dist = length(d);
    if (dist >= h) return 0.0F;
    const float q = dist / h;
    const float coef = 8.0F / (kPi * h * h * h);
    if (q <= 0.5F) return coef * (6.0F * q * q * q - 6.0F * q * q + 1.0F);
    const float diff = 1.0F - q;
    return coef * 2.0F * diff * diff * diff;
}

// cubic spline gradient, density/device.cuh:36-43
__device__ __forceinline__ Float3 cubic_gradient(Float3 d, float h) {
    const float dist = length(d);
    if (dist == 0.0F || dist >= h) return {0.0F, 0.0F, 0.0F};
    const float q = dist / h;
    const float coef = 8.0F / (kPi * h * h * h);
    const float deriv = q <= 0.5F ? 18.0F * q * q - 12.0F * q : -6.0F * (1.0F - q) * (1.0F - q);
    return scale(d, coef * deriv / (h * dist));
}

// Kernel constants evaluated once on the host with the reference's FP32
// expressions (density/device.cuh:30,40,75): cubic 8/(pi h^3) and the
// viscosity Laplacian's pi h^6.
struct KernelConstants {
    float h;
    float cubic;        // 8 / (pi h h h)
    float viscosity;    // pi h h h h h h
    float sqrt_support; // smallest float t with sqrtf(t) >= h
    float inv_h;        // RN(1 / h)
    float inv_viscosity; // RN(1 / viscosity)
    uint32_t plain;      // h lies outside [2^-20, 2^16], where div_in_range is not used: beyond 2^16.4 the gradient
                         // factors next to the support's edge are subnormal
};

// Correctly rounded x / b from inv_b = RN(1 / b), for b > 0: the estimate
// q0 = x inv_b is refined once, q1 = q0 + (x - b q0) inv_b, which leaves it
// within an ulp of x / b; the remainder x - b q1 is then exact and
// q1 + (x - b q1) inv_b rounds to RN(x / b) (P. Markstein, IBM J. Res. Dev.
// 34(1), 1990). Each step is one IEEE multiply or fused multiply-add, so the
// host and the device agree. Exact for x = 0 and for x >= 2^-100 while the
// quotient stays normal (below 2^-105 the remainders underflow and it can
// miss); the callers' arguments are distances, at least 2^-74.5 when
// nonzero, and multiples of them. Checked against x / b for every float x
// of two binades for many b and for every x in [2^-100, h) on the GPU.
__host__ __device__ inline float div_rn(float x, float b, float inv_b) {
    const float q0 = x * inv_b;
    const float r0 = fmaf(-q0, b, x);
    const float q1 = fmaf(r0, inv_b, q0);
    const float r1 = fmaf(-q1, b, x);
    return fmaf(r1, inv_b, q1);
}

// A particle's rest density as the divisor of its candidates' masses. With
// masses and rest densities in [2^-60, 2^60], whose quotients and remainders
// stay normal, the reciprocal is taken once (div_rn); otherwise, zeros and
// infinities included, each pair's quotient is the compiler's. The masses are
// checked as a step gathers them (Channels::flag), so that the choice does not
// change within a walk: a check of each candidate's mass made a PBF step of
// 32,768 particles 178 us for 168.
__device__ __forceinline__ bool outside_quick_range(float v) { return !(v >= 0x1p-60F && v <= 0x1p60F); }
struct RestDensity {
    float value, inverse;
    bool plain;
};
__device__ __forceinline__ RestDensity rest_density_of(float rest, bool unusual_masses) {
    return RestDensity{rest, 1.0F / rest, unusual_masses || outside_quick_range(rest)};
}
__device__ __forceinline__ float over_rest(float mass, const RestDensity& rest) {
    return rest.plain ? mass / rest.value : div_rn(mass, rest.value, rest.inverse);
}

// a / b for operands whose quotient, remainders and reciprocal stay normal:
// the compiler's own sequence of reciprocal estimate, one Newton step and two
// quotient refinements, hence its correctly rounded result, without the
// scaling and special cases around it (8 instructions for 11). With
// sqrt_rn it took PBF steps of 1,048,576 particles from 1,738 to 1,625 us.
__device__ __forceinline__ float div_in_range(float a, float b) {
    float r = __builtin_amdgcn_rcpf(b);
    r = fmaf(fmaf(-b, r, 1.0F), r, r);
    float q = a * r;
    q = fmaf(fmaf(-b, q, a), r, q);
    return fmaf(fmaf(-b, q, a), r, q);
}

// Correctly rounded square root of 0 <= x < 2^64 from the reciprocal square
// root s of y = x 2^64 (a normal number for every such x but 0): g = y s is
// within an ulp of sqrt(y), its residual y - g^2 is exact, and
// g + (y - g^2) s / 2 rounds correctly (checked on the GPU for every float
// below 2^64); the scale is undone exactly. x = 0 gives 0 without a branch,
// across which the compiler does not move a pair term's later loads
// (non-pressure pass of 4,194,304 particles 1,116 -> 1,003 us). From 2^64 on
// the result is +inf; NaN stays NaN.
__device__ __forceinline__ float sqrt_rn(float x) {
    const float y = x * 0x1p64F;
    const float s = __builtin_amdgcn_rsqf(__builtin_amdgcn_fmed3f(y, 0x1p-90F, 0x1.fffffep127F));
    const float g = __builtin_amdgcn_fmed3f(y, 0.0F, 0x1.fffffep127F) * s;
    return fmaf(fmaf(-g, g, y), 0.5F * s, g) * 0x1p-32F;
}

// length(d) of a neighbour pair (the same value; any |d| >= 2^32 gives +inf,
// which lies outside every support).
__device__ __forceinline__ float pair_distance(Float3 d) { return sqrt_rn(dot(d, d)); }

// cubic(d, h) as a function of dist = length(d), with the constants
// supplied: the same operations as cubic(), both branches evaluated and
// selected, so that a wave walking neighbours does not diverge.
__device__ __forceinline__ float cubic_value(float dist, const KernelConstants& k) {
    const float q = div_rn(dist, k.h, k.inv_h);
    const float near = k.cubic * (6.0F * q * q * q - 6.0F * q * q + 1.0F);
    const float diff = 1.0F - q;
    const float far = k.cubic * 2.0F * diff * diff * diff;
    const float w = q <= 0.5F ? near : far;
    return dist >= k.h ? 0.0F : w;
}

// The radial factor f of cubic_gradient(d, h) = f * d (zero outside the
// support and at d = 0), with the constants supplied; branch-free like
// cubic_value() but for the choice of the quotient with kQuick, which the
// derivative passes take. The forward passes, held by their gathers, lose more
// by the choice's branch at every pair than the shorter quotient saves (force
// pass of 4,194,304 particles 486 us, with it 503; of 1,048,576 87.5 and 88.3;
// WCSPH steps of 2,097,152 886 and 886); the derivatives, held by their
// arithmetic, gain (a DFSPH step of 35,805 particles with JVP and VJP 1,717 us,
// with it 1,691).
template <bool kQuick = false>
__device__ __forceinline__ float cubic_gradient_factor(float dist, const KernelConstants& k) {
    const float q = div_rn(dist, k.h, k.inv_h);
    const float near = 18.0F * q * q - 12.0F * q;
    const float diff = 1.0F - q;
    const float far = -6.0F * diff * diff;
    const float deriv = q <= 0.5F ? near : far;
    const float top = k.cubic * deriv;
    const float bottom = k.h * dist;
    const float f = !kQuick || k.plain != 0u ? top / bottom : div_in_range(top, bottom);
    return dist == 0.0F || dist >= k.h ? 0.0F : f;
}

__device__ __forceinline__ float viscosity_laplacian_c(Float3 d, const KernelConstants& k) {
    const float dist = pair_distance(d);
    const float l = div_rn(45.0F * (k.h - dist), k.viscosity, k.inv_viscosity);
    return dist >= k.h ? 0.0F : l;
}

// viscosity Laplacian, density/device.cuh:72-76
__device__ __forceinline__ float viscosity_laplacian(Float3 d, float h) {
    const float dist = length(d);
    if (dist >= h) return 0.0F;
    return 45.0F * (h - dist) / (kPi * h * h * h * h * h * h);
}

// spiky gradient, pbf.cu:26-32. The coefficient -45/(pi h^6) is computed once
// on the host (the reference evaluates the same powf per pair).
__device__ __forceinline__ Float3 spiky_gradient(Float3 d, float h, float coefficient) {
    const float dist = length(d);
    if (dist == 0.0F || dist >= h) return {0.0F, 0.0F, 0.0F};
    const float diff = h - dist;
    return scale(d, coefficient * diff * diff / dist);
}

// True when the artificial pressure -k (W(d) / W(dq))^n of a particle is the
// signed zero -k for every pair with W(d) > 0: k is +-0 and the power stays
// finite for every ratio up to W(0) / W(dq) (powf is non-decreasing in the
// base for n >= 0). `reference` is W(dq).
__device__ __forceinline__ bool artificial_vanishes(float h, float strength, float exponent, float reference) {
    if (strength != 0.0F || !(reference > 0.0F) || !(exponent >= 0.0F)) return false;
    const float largest = poly6(Float3{0.0F, 0.0F, 0.0F}, h) / reference;
    return powf(largest, exponent) < 1.0e37F;
}

// The PBF kernels' constants for one support radius, evaluated with the
// reference's FP32 expressions on the host: the poly6 denominator
// 64 pi h^9 scaled by a power of two into [1, 2) (poly6_value scales its
// numerator alike, so no remainder underflows), and the spiky coefficient.
struct PbfKernel {
    float h;
    float hr;           // h h
    float spiky;        // spiky_coefficient(h)
    float poly6;        // 64 pi hr hr hr h h h
    float poly6_scaled; // poly6 scale
    float inv_poly6;    // RN(1 / poly6_scaled)
    float scale;
    uint32_t plain;     // h lies outside [2^-11, 2^8], where the quotients below are taken by the compiler's division
};

// poly6(d, h) from d2 = dot(d, d).
__device__ __forceinline__ float poly6_value(float d2, const PbfKernel& k) {
    const float diff = k.hr - d2;
    const float top = 315.0F * diff * diff * diff;
    const float w = k.plain != 0u ? top / k.poly6 : div_rn(top * k.scale, k.poly6_scaled, k.inv_poly6);
    return d2 >= k.hr ? 0.0F : w;
}

// Whether poly6(d, h) is zero.
__device__ __forceinline__ bool poly6_vanishes(float d2, const PbfKernel& k) {
    return k.plain != 0u ? poly6_value(d2, k) == 0.0F : d2 >= k.hr;
}

// The factor f of spiky_gradient(d, h) = f d from d2 = dot(d, d); both sides
// of its condition are evaluated and selected, so that a wave does not
// diverge.
__device__ __forceinline__ float spiky_factor(float d2, const PbfKernel& k) {
    const float dist = sqrt_rn(d2);
    const float diff = k.h - dist;
    const float top = k.spiky * diff * diff;
    const float f = k.plain != 0u ? top / dist : div_in_range(top, dist);
    return dist == 0.0F || dist >= k.h ? 0.0F : f;
}

// artificial pressure value, pbf.cu:56-71 (value only), from d2 = dot(d, d).
// `reference` is poly6((radius,0,0), h) of the particle.
__device__ __forceinline__ float artificial_value(float d2, const PbfKernel& k, float strength, float exponent,
                                                  float reference) {
    const float kernel = poly6_value(d2, k);
    if (kernel == 0.0F) return 0.0F;
    return -strength * powf(kernel / reference, exponent);
}

// 1 / sqrt(x) for a positive normal x: the hardware estimate refined by two
// Newton steps, y <- y + y (1 - x y^2) / 2, to within a few units of the
// last place (the derivative passes compare with the FP64 oracle to 1e-10;
// the square root and the division they replace cost about 30 instructions).
__device__ __forceinline__ double inverse_sqrt(double x) {
    double y = __builtin_amdgcn_rsq(x);
#pragma unroll
    for (int step = 0; step < 2; ++step) {
        const double e = fma(-x * y, y, 1.0);
        y = fma(0.5 * y, e, y);
    }
    return y;
}

// min(C-1, max(0, floor(v))) with NaN and negatives mapped to 0, as the
// reference's __float2int_rd + clamp (neighborhood.cu:34-36).
__device__ __forceinline__ int cell_clamp(float v, uint32_t count) {
    const float f = floorf(v);
    if (!(f > 0.0F)) return 0;
    if (f >= static_cast<float>(count - 1u)) return static_cast<int>(count) - 1;
    return static_cast<int>(f);
}

// Collision box of the solvers (sph.cpp:21-35, pbf.cpp:17-31).
struct Box {
    float lo[3];
    float hi[3];
    float vel[3];
    uint32_t no_slip;
};

// Semi-implicit Euler with box clamp: integrate/predict body of
// sph/common.cu:302-320 and sph/dfsph.cu:26-44.
__device__ __forceinline__ void predict_clamped(const Box& box, float dt, Float3 x, Float3 v, Float3 a, Float3& out_x,
                                                Float3& out_v) {
    Float3 vel = add(v, scale(a, dt));
    Float3 pos = add(x, scale(vel, dt));
    const bool cx = pos.x < box.lo[0] || pos.x > box.hi[0];
    const bool cy = pos.y < box.lo[1] || pos.y > box.hi[1];
    const bool cz = pos.z < box.lo[2] || pos.z > box.hi[2];
    pos.x = fminf(box.hi[0], fmaxf(box.lo[0], pos.x));
    pos.y = fminf(box.hi[1], fmaxf(box.lo[1], pos.y));
    pos.z = fminf(box.hi[2], fmaxf(box.lo[2], pos.z));
    if (box.no_slip != 0u && (cx || cy || cz)) {
        vel = {box.vel[0], box.vel[1], box.vel[2]};
    } else {
        if (cx) vel.x = box.vel[0];
        if (cy) vel.y = box.vel[1];
        if (cz) vel.z = box.vel[2];
    }
    out_x = pos;
    out_v = vel;
}

// Box-collision bits (x: 1, y: 2, z: 4) of the unclamped prediction
// x + dt (v + dt a) of predict_clamped.
__device__ __forceinline__ uint32_t predict_collisions(const Box& box, float dt, Float3 x, Float3 v, Float3 a) {
    const Float3 pos = add(x, scale(add(v, scale(a, dt)), dt));
    return (pos.x < box.lo[0] || pos.x > box.hi[0] ? 1u : 0u) | (pos.y < box.lo[1] || pos.y > box.hi[1] ? 2u : 0u) |
           (pos.z < box.lo[2] || pos.z > box.hi[2] ? 4u : 0u);
}

// Uniform grid in sorted (cell-major) particle order: the cell range of cell c
// is [offsets[c], offsets[c+1]) of the sorted arrays.
struct SortedGrid {
    const uint32_t* offsets;
    uint32_t cx, cy, cz;
    float ox, oy, oz;
    float cell;
};

// particle_cell, neighborhood/device.cuh:44-48
__device__ __forceinline__ void particle_cell(const SortedGrid& g, Float3 p, int& x, int& y, int& z) {
    x = cell_clamp((p.x - g.ox) / g.cell, g.cx);
    y = cell_clamp((p.y - g.oy) / g.cell, g.cy);
    z = cell_clamp((p.z - g.oz) / g.cell, g.cz);
}

// Sorted boundary samples of a grid build, the boundary half of
// NeighborhoodView and BoundaryView (neighborhood/device.h:8-36): per cell
// the samples in ascending original index, each stored as its position at
// the step's time t, x0 + t v (boundary_position, neighborhood/device.cuh:
// 16-22), with its volume, and its velocity.
// Candidate records are read up to kScanPadding past the end of a cell
// (mark_members), so the arrays of records that are scanned are that longer.
constexpr uint32_t kScanPadding = 3;

struct BoundaryGrid {
    const uint32_t* offsets;  // C + 1 cell starts; null when the domain has no boundary samples
    const float4* x;          // position at t (xyz), volume (w)
    const float4* v;          // velocity (xyz)
};

// Calls cell(c) for the in-grid cells of the 27 around (cx, cy, cz) in the
// reference order: offset_x outer, offset_y, offset_z inner (cell_range,
// neighborhood/device.cuh:32-42, skips cells outside the grid).
template <class Cell>
__device__ __forceinline__ void for_each_cell(const SortedGrid& g, int cx, int cy, int cz, Cell&& cell) {
    // not unrolled: 27 inlined copies of a visitor cost registers (occupancy)
    // and instruction cache for no gain, the visit loop being dynamic anyway
#pragma unroll 1
    for (int ox = -1; ox <= 1; ++ox) {
        const int X = cx + ox;
        if (X < 0 || X >= static_cast<int>(g.cx)) continue;
#pragma unroll 1
        for (int oy = -1; oy <= 1; ++oy) {
            const int Y = cy + oy;
            if (Y < 0 || Y >= static_cast<int>(g.cy)) continue;
            const uint32_t row = (static_cast<uint32_t>(Y)) * g.cx + static_cast<uint32_t>(X);
#pragma unroll 1
            for (int oz = -1; oz <= 1; ++oz) {
                const int Z = cz + oz;
                if (Z < 0 || Z >= static_cast<int>(g.cz)) continue;
                cell(static_cast<uint32_t>(Z) * g.cy * g.cx + row);
            }
        }
    }
}

// Visits the sorted candidates of the 27 cells around (cx, cy, cz) in the
// reference order; ascending sorted position (= ascending original index)
// within a cell.
template <class Visit>
__device__ __forceinline__ void for_each_candidate(const SortedGrid& g, int cx, int cy, int cz, Visit&& visit) {
    for_each_cell(g, cx, cy, cz, [&](uint32_t c) {
        const uint32_t first = g.offsets[c];
        const uint32_t last = g.offsets[c + 1u];
        for (uint32_t s = first; s < last; ++s) visit(s);
    });
}

// The same walk with each cell's boundary samples visited after its
// particles, the order of every reference neighbour loop (e.g.
// density/density.cu:28-37).
template <class Visit, class VisitBoundary>
__device__ __forceinline__ void for_each_candidate(const SortedGrid& g, const BoundaryGrid& b, int cx, int cy, int cz,
                                                   Visit&& visit, VisitBoundary&& visit_boundary) {
    for_each_cell(g, cx, cy, cz, [&](uint32_t c) {
        const uint32_t first = g.offsets[c];
        const uint32_t last = g.offsets[c + 1u];
        for (uint32_t s = first; s < last; ++s) visit(s);
        const uint32_t bfirst = b.offsets[c];
        const uint32_t blast = b.offsets[c + 1u];
        for (uint32_t s = bfirst; s < blast; ++s) visit_boundary(s);
    });
}

}  // namespace phx
