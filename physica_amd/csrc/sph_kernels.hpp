// Neighbour-pass kernels shared by the SPH solvers (DFSPH, PCISPH, IISPH,
// WCSPH) in sorted (cell-major) particle order.
//
// Every per-particle sum runs in the reference order (27 cells, offset_x
// outer, ascending original index) over the precomputed neighbour masks, and
// every masked-out candidate contributes an exact zero in the reference, so
// results equal the reference expressions operation by operation. The kernels
// live in an unnamed namespace: each solver translation unit instantiates the
// ones it launches.
#pragma once

#include "engine.hpp"
#include "group_walk.hpp"
#include "neighbor_mask.hpp"
#include "profiler.hpp"

#include <type_traits>

namespace phx {
namespace {

__device__ __forceinline__ Float3 xyz(float4 q) { return Float3{q.x, q.y, q.z}; }

// Whether q can be within the support of p (a distance that is NaN can, as
// its terms are NaN); the kernels' values are exact zeros where it is not.
__device__ __forceinline__ bool within_support(const KernelConstants& k, Float3 p, Float3 q) {
    const Float3 d = sub(p, q);
    return !(dot(d, d) >= k.sqrt_support);
}

constexpr uint32_t kBlock = 256;
constexpr uint32_t kWaves = kBlock / 64;  // waves of a pass workgroup
// candidates a masked walk fetches ahead of the one it processes
constexpr int kWalkDepth = 2;
// Particle counts up to which 16 and 4 lanes share a particle. More lanes
// shorten a pass that does not fill the GPU and add work (listing the
// candidates, idle lanes in a particle's last trip) to one that does. DFSPH
// steps of 4 + 6 iterations, us, with 1 / 4 / 16 lanes: 2,000 particles
// 419 / 278 / 194, 16,000 476 / 303 / 270, 32,000 432 / 297 / 346, 64,000
// 458 / 370 / 501, 130,000 505 / 558 / 829, 260,000 710 / 897 / -; IISPH and
// PCISPH cross at the same counts. From 400,000 four lanes are 6 % faster on
// cubic lattices and 6 to 20 % slower on a dam break of 128 x 64 x 128. These
// scenes have no crowded cells, for which the rule has no term: a crowded lane
// of the one-lane passes evaluates every candidate of its stencil while its
// wave waits. On a lattice whose planes lie on cell borders, so that a few
// cells hold 17 or 18 particles, one lane takes 1,900 us and four take 924 at
// 103,823 particles (2,160 and 1,295 at 262,144; with the planes inside the
// cells 437 and 440, 635 and 770).
constexpr uint32_t kGroup16Particles = 20000;
constexpr uint32_t kGroup4Particles = 90000;

// Marks the 27 cells around (cx, cy, cz) with `stamp` (plain stores: every
// writer writes the same value).
__device__ __forceinline__ void taint_neighbour_cells(const SortedGrid& g, int cx, int cy, int cz, uint32_t* taint,
                                                      uint32_t stamp) {
    for (int z = max(cz - 1, 0); z <= min(cz + 1, static_cast<int>(g.cz) - 1); ++z)
        for (int y = max(cy - 1, 0); y <= min(cy + 1, static_cast<int>(g.cy) - 1); ++y)
            for (int x = max(cx - 1, 0); x <= min(cx + 1, static_cast<int>(g.cx) - 1); ++x)
                taint[cell_of(g, x, y, z)] = stamp;
}

// Per-cell displacement bound of a step: scale * the largest displacement
// of the previous step among the cell's particles (sorted order), plus
// `allowance`; 0 for an empty cell.
[[maybe_unused]] __global__ void __launch_bounds__(kBlock)
    cell_bound_kernel(uint32_t cells, const uint32_t* __restrict__ offsets, const float* __restrict__ moved,
                      float scale, float allowance, float* __restrict__ bound) {
    const uint32_t c = blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= cells) return;
    const uint32_t first = offsets[c];
    const uint32_t last = offsets[c + 1u];
    float largest = 0.0F;
    for (uint32_t s = first; s < last; ++s) largest = fmaxf(largest, moved[s]);
    bound[c] = first == last ? 0.0F : scale * largest + allowance;
}

struct MaskDensityArgs {
    uint32_t n;
    KernelConstants kc;
    float t_skin;
    SortedGrid grid;
    BoundaryGrid boundary;  // offsets null: no boundary samples
    const float4* xm;
    uint16_t* exact;
    uint16_t* skin;
    const float* p_div;  // optional: t_div = p_div / rho^2
    const float* p_den;  // optional: t_den = p_den / rho^2
    float* rho;
    float* t_div;
    float* t_den;
    // rho0 (boundary terms), and the equation of state (WCSPH): p = EOS(rho),
    // aux = (rho, p / rho^2, c, sigma)
    const float* rest_density;
    const float* tait_exponent;
    float* pressures;
    float4* aux;  // z (speed of sound) and w (surface tension) are inputs
    // per particle: set where a stencil cell holds more than kMaskBits
    // particles (that particle walks the full stencil in every pass)
    uint8_t* crowded;
    uint32_t* cell;  // out: the grid cell of each particle
    // per cell: a bound on how far its particles move this step; non-null:
    // the skin mask keeps a pair while d2 < (h + B_ci + B_cj)^2 (plus a
    // rounding margin) instead of d2 < t_skin
    const float* cell_bound = nullptr;
    // optional: (x, y, z, t_div) and (x, y, z, t_den) per particle, the
    // candidate records of the force passes that read these t
    float4* xt_div = nullptr;
    float4* xt_den = nullptr;
    // optional: the step's mass state (see ForceArgs::mass_state): [1] the
    // bits of sorted particle 0's mass; [0] set to mass_stamp by every
    // particle whose mass has other bits
    uint32_t* mass_state = nullptr;
    uint32_t mass_stamp = 0u;
    // masks of the cells' boundary samples, as exact and skin (a launch with
    // samples)
    uint16_t* exact_samples = nullptr;
    uint16_t* skin_samples = nullptr;
};

// What the mask pass writes for particle i at p with density `result`.
template <bool kEos>
__device__ __forceinline__ void write_density(const MaskDensityArgs& a, uint32_t i, Float3 p, float result) {
    a.rho[i] = result;
    if constexpr (kEos) {
        const float4 aux = a.aux[i];
        const float rest_density = a.rest_density[i];
        const float speed = aux.z;
        const float exponent = a.tait_exponent[i];
        const float ratio = result / rest_density;
        const float pressure = rest_density * speed * speed * (powf(ratio, exponent) - 1.0F) / exponent;
        a.pressures[i] = pressure;
        a.aux[i] = make_float4(result, pressure / (result * result), speed, aux.w);
    } else {
        if (a.p_div != nullptr) {
            const float t = a.p_div[i] / (result * result);
            a.t_div[i] = t;
            if (a.xt_div != nullptr) a.xt_div[i] = make_float4(p.x, p.y, p.z, t);
        }
        if (a.p_den != nullptr) {
            const float t = a.p_den[i] / (result * result);
            a.t_den[i] = t;
            if (a.xt_den != nullptr) a.xt_den[i] = make_float4(p.x, p.y, p.z, t);
        }
    }
}

// Notes particle i's mass in the step's mass state (MaskDensityArgs::mass_state).
__device__ __forceinline__ void note_mass(const MaskDensityArgs& a, uint32_t i, float mass) {
    if (a.mass_state == nullptr) return;
    const uint32_t bits = __float_as_uint(mass);
    if (i == 0u) a.mass_state[1] = bits;
    if (bits != __float_as_uint(a.xm[0].w)) a.mass_state[0] = a.mass_stamp;  // one value for every writer
}

// Mask build, then density_forward_kernel (density.cu:18-40, cubic kernel,
// topology = positions) over the exact mask and the first_term p/rho^2 of
// pressure_forward_kernel (common.cu:171) for the given pressures, or with
// kEos the Tait pressure of eos_forward_kernel (wcsph.cu:92-100) and its
// first_term. A particle with a stencil cell of more than kMaskBits
// particles is marked crowded and walks the full stencil here and in every
// later pass. The expanding threads build the masks, each for its own stencil
// slots, so a particle's 27 cells are scanned by G threads at once: one lane
// per particle scanned them in turn, a chain of loads that took 50 us however
// few the particles (3,315 particles: 49 -> 8 us with 16 lanes; 64,000:
// 50 -> 19 us with four; 1,048,576: 206 -> 181 us). With kSamples the cells'
// boundary samples get masks of their own (a sample moves with the step, not
// within it, so its skin covers the particle's displacement alone), and each
// cell's samples b add rho0_i V_b W after its particles (density.cu:34-37).
template <bool kEos, int G, bool kSamples>
__global__ void __launch_bounds__(kGroupBlock) mask_density_kernel(MaskDensityArgs a) {
    constexpr uint32_t kParticles = kGroupParticles<G>;
    constexpr uint32_t kSlots = kGroupSlots<G>;
    __shared__ GroupLds<G> lds;
    __shared__ uint32_t crowd[kParticles];
    const uint32_t base = xcd_block() * kParticles;
    const uint32_t expanded = threadIdx.x % kParticles;
    const uint32_t part = threadIdx.x / kParticles;
    const uint32_t i = base + expanded;
    const bool valid = i < a.n;
    if (threadIdx.x < kParticles) crowd[threadIdx.x] = 0u;
    __syncthreads();
    Float3 p{0.0F, 0.0F, 0.0F};
    uint32_t first[kSlots] = {}, last[kSlots] = {};
    [[maybe_unused]] uint32_t sample_first[kSlots] = {}, sample_last[kSlots] = {};
    float bound_i = 0.0F;
    float bound[kSlots] = {};
    if (valid) {
        const float4 self = a.xm[i];
        p = xyz(self);
        if (part == 0u) note_mass(a, i, self.w);
        int cx, cy, cz;
        particle_cell(a.grid, p, cx, cy, cz);
        const uint32_t center = cell_of(a.grid, cx, cy, cz);
        if (part == 0u) a.cell[i] = center;
        bool crowded = group_ranges<G>(a.grid, a.grid.offsets, cx, cy, cz, first, last);
        if constexpr (kSamples)
            crowded = group_ranges<G>(a.grid, a.boundary.offsets, cx, cy, cz, sample_first, sample_last) || crowded;
        if (a.cell_bound != nullptr) {
            bound_i = a.cell_bound[center];
#pragma unroll
            for (uint32_t j = 0; j < kSlots; ++j)
                if (last[j] != first[j]) bound[j] = a.cell_bound[center + slot_delta(a.grid, part * kSlots + j)];
        }
        if (crowded) crowd[expanded] = 1u;
    }
    // the exact mask of members from .. to - 1 at positions x[s], their skin
    // mask in `skin`; with the margin of exact_mask_threshold, as the FP64
    // derivatives take the distance of a pair at the very edge of the support
    // to be inside it where the FP32 passes do not. With samples a distance
    // that is NaN is kept, as its terms are (a particle at a NaN position and
    // its neighbours have NaN sums); without, such a particle has no neighbours.
    const float t_exact = a.kc.sqrt_support * (1.0F + 4e-6F);
    auto within = [](float d2, float bound) { return kSamples ? !(d2 >= bound) : d2 < bound; };
    auto mark = [&](const float4* x, uint32_t from, uint32_t to, float t_skin, uint32_t& skin) {
        uint32_t bits[2];
        mark_members<2>(x, from, to, bits, [&](Float3 q, bool (&marked)[2]) {
            const Float3 d = sub(p, q);
            const float d2 = dot(d, d);
            marked[0] = within(d2, t_exact);
            marked[1] = within(d2, t_skin);
        });
        skin = bits[1];
        return bits[0];
    };
    // the threshold of pairs within h after moving up to `reach` together
    // (the relative margin covers rounding), or the step's global one
    auto threshold = [&](float reach) {
        if (a.cell_bound == nullptr) return a.t_skin;
        const float radius = a.kc.h + reach;
        return radius * radius * (1.0F + 2e-5F);
    };
    auto slots = [&](uint32_t (&bits)[kSlots], uint32_t (&start)[kSlots]) {
#pragma unroll
        for (uint32_t j = 0; j < kSlots; ++j) {
            const uint32_t k = part * kSlots + j;
            start[j] = first[j];
            if (!valid || k >= static_cast<uint32_t>(kStencil)) continue;
            uint32_t skin;
            bits[j] = mark(a.xm, first[j], last[j], threshold(bound_i + bound[j]), skin);
            a.exact[static_cast<size_t>(k) * a.n + i] = static_cast<uint16_t>(bits[j]);
            a.skin[static_cast<size_t>(k) * a.n + i] = static_cast<uint16_t>(skin);
        }
    };
    auto sample_slots = [&](uint32_t (&bits)[kSlots], uint32_t (&start)[kSlots]) {
        if constexpr (kSamples) {
#pragma unroll
            for (uint32_t j = 0; j < kSlots; ++j) {
                const uint32_t k = part * kSlots + j;
                start[j] = sample_first[j];
                if (!valid || k >= static_cast<uint32_t>(kStencil)) continue;
                uint32_t skin;
                bits[j] = mark(a.boundary.x, sample_first[j], sample_last[j], threshold(bound_i), skin);
                a.exact_samples[static_cast<size_t>(k) * a.n + i] = static_cast<uint16_t>(bits[j]);
                a.skin_samples[static_cast<size_t>(k) * a.n + i] = static_cast<uint16_t>(skin);
            }
        }
    };
    const uint32_t walked = threadIdx.x / G;
    const uint32_t w = base + walked;
    const bool active = w < a.n;
    const float4 own = a.xm[active ? w : 0u];
    const float rest = kSamples && active ? a.rest_density[w] : 0.0F;
    float sum[1] = {0.0F};
    auto fetch = [&](uint32_t entry) {
        if constexpr (kSamples) {
            if ((entry & kSampleEntry) != 0u) return a.boundary.x[entry & ~kSampleEntry];
        }
        return a.xm[entry];
    };
    auto pair = [&](float4 q, uint32_t entry, float (&terms)[1]) {
        const float weight = cubic_value(pair_distance(sub(xyz(own), xyz(q))), a.kc);
        terms[0] = kSamples && (entry & kSampleEntry) != 0u ? rest * q.w * weight : q.w * weight;
    };
    auto fold = [&](const float (&terms)[1]) { group_add<G, 1>(sum, terms); };
    group_expand<G, kSamples>(lds, slots, sample_slots, [&](const uint32_t* row, uint32_t count) {
        if (active && crowd[walked] == 0u) group_walk_list<G, 1>(row, count, w, fetch, pair, fold);
    });
    if (valid && part == 0u) a.crowded[i] = static_cast<uint8_t>(crowd[expanded]);
    if (!active) return;
    if (crowd[walked] != 0u) {
        int cx, cy, cz;
        particle_cell(a.grid, xyz(own), cx, cy, cz);
        group_walk_stencil<G, 1>(
            a.grid, kSamples ? a.boundary.offsets : nullptr, cx, cy, cz, ~0u, w, group_row(lds),
            [&](uint32_t entry) { return within_support(a.kc, xyz(own), xyz(fetch(entry))); }, fetch, pair, fold);
    }
    if (threadIdx.x % G == 0u) write_density<kEos>(a, w, xyz(own), sum[0]);
}

// Tolerance mode: the convergence state of a pressure phase. The projection
// adds each wave's compression errors max(0, rho* - target) / rho0 in FP64
// (shuffles, no block barrier, so every wave retires as soon as its own walk
// ends) and stores the sum in partials[blockIdx.x * kWaves + wave];
// converge_kernel then
// marks the phase done at this iteration when the mean is within the
// tolerance or the iteration is the last allowed one. Every pass of the
// phase reads `done`: passes of later iterations (launched ahead by the
// host) then return at once, and the force pass of the marked iteration ends
// the phase.
struct Convergence {
    double* partials;      // null: fixed iteration counts; else one error sum per wave
    const uint32_t* done;  // iteration that ended the phase; 0 while it runs
    const float* rest;  // rho0, the scale of the error
};

// Block-wide FP64 sum reaching thread 0 (other threads get partial sums).
// The order of the additions is fixed, so the result is reproducible.
template <uint32_t kBlockSize>
__device__ __forceinline__ double block_sum(double value) {
    __shared__ double wave_sum[kBlockSize / 64];
    double v = value;
    for (int offset = 32; offset > 0; offset >>= 1) v += __shfl_xor(v, offset, 64);
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t wave = threadIdx.x >> 6;
    if (lane == 0u) wave_sum[wave] = v;
    __syncthreads();
    double total = 0.0;
    if (threadIdx.x == 0u)
        for (uint32_t w = 0; w < kBlockSize / 64; ++w) total += wave_sum[w];
    return total;
}

constexpr uint32_t kConvergeBlock = 1024;

// The value *done has after this iteration, for the host: a store to
// host-visible (pinned) memory at system scope.
__device__ __forceinline__ void publish_done(uint32_t* host_flag, uint32_t value) {
    __hip_atomic_store(host_flag, value, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

// Ends a tolerance-mode phase: sums the projection's per-wave error sums in
// a fixed order (thread t takes partials t, t + 1024, ...), and
// records the iteration in *done when the mean error is within the
// tolerance or the iteration is the last allowed. One workgroup; the kernel
// boundaries order it after the projection and before the force pass, so
// no atomics or fences are needed on the device. The resulting *done is also
// stored to the host's flag of this iteration (pinned memory mapped for the
// device), which the host reads once the iteration's event has completed,
// with no copy in between.
[[maybe_unused]] __global__ void __launch_bounds__(kConvergeBlock)
    converge_kernel(const double* partials, uint32_t count, uint32_t n, double tolerance, uint32_t iteration,
                    uint32_t max_iterations, uint32_t* done, uint32_t* host_flag) {
    const uint32_t ended = *done;
    if (ended != 0u) {  // the phase ended at an earlier iteration
        if (threadIdx.x == 0u) publish_done(host_flag, ended);
        return;
    }
    double sum = 0.0;
    for (uint32_t k = threadIdx.x; k < count; k += kConvergeBlock) sum += partials[k];
    const double total = block_sum<kConvergeBlock>(sum);
    if (threadIdx.x == 0u) {
        const double mean = total / static_cast<double>(n);
        const uint32_t now = mean <= tolerance || iteration >= max_iterations ? iteration : 0u;
        if (now != 0u) *done = now;
        publish_done(host_flag, now);
    }
}

struct ProjectionArgs {
    uint32_t n;
    KernelConstants kc;
    float dt;
    float gradient_norm;
    float limit2;  // largest squared displacement for which the skin mask is exact
    uint32_t slot;
    SortedGrid grid;
    const float4* xm;  // topology: state positions (+ masses)
    const float4* xs;  // predicted positions (+ masses)
    const uint16_t* skin;
    const uint32_t* flags;
    const float* rho;
    const float* volume_density;  // rho (DFSPH, IISPH) or rho0 (PCISPH) in V = m / density
    const float* target;
    const float* relaxation;
    const float* p_prev;  // pressures before the update (may equal p)
    float* p;
    float* t;
    float* rs_out;  // optional (recorded step): the predicted densities
    Convergence cv;
    BoundaryGrid boundary;     // offsets null: no boundary samples
    const float* rest_density;  // rho0, for the boundary terms
    const uint8_t* crowded;     // per particle: walks the full stencil
    const uint32_t* cell;       // MaskDensityArgs::cell
    // per-cell skins: the skin mask applies to particle i unless its cell
    // holds `stamp` (a particle of a neighbouring cell moved past its cell's
    // bound in the prediction this pass reads); null: the global rule
    // (every particle moved at most sqrt(limit2))
    const uint32_t* taint = nullptr;
    uint32_t stamp = 0u;
    float4* xt_out = nullptr;  // optional: (x, y, z, t) per particle, the force pass's candidate record
    const uint16_t* skin_samples = nullptr;  // MaskDensityArgs::skin_samples
};

// Whether the skin masks apply to particle i of cell `cell` in this pass.
__device__ __forceinline__ bool projection_masked(const ProjectionArgs& a, uint32_t i, uint32_t cell) {
    const bool moved_within = a.taint != nullptr
                                  ? a.taint[cell] != a.stamp
                                  : __uint_as_float(a.flags[kFlagDisplacement + a.slot]) <= a.limit2;
    return a.crowded[i] == 0u && moved_within;
}

// The pressure update of particle i from its predicted density rs; returns
// its compression error in tolerance mode.
__device__ __forceinline__ double update_pressure(const ProjectionArgs& a, uint32_t i, float4 topology, float mass,
                                                  float rs) {
    const float rho = a.rho[i];
    const float target = a.target[i];
    const float volume = mass / a.volume_density[i];
    const float delta_p = 1.0F / (2.0F * a.dt * a.dt * volume * volume * a.gradient_norm);
    const float pressure = fmaxf(0.0F, a.p_prev[i] + a.relaxation[i] * delta_p * (rs - target));
    a.p[i] = pressure;
    const float t = pressure / (rho * rho);
    a.t[i] = t;
    if (a.xt_out != nullptr) a.xt_out[i] = make_float4(topology.x, topology.y, topology.z, t);
    if (a.rs_out != nullptr) a.rs_out[i] = rs;
    if (a.cv.partials == nullptr) return 0.0;
    return fmax(0.0, static_cast<double>(rs) - static_cast<double>(target)) / static_cast<double>(a.cv.rest[i]);
}

// Adds the wave's errors and stores the sum; every lane of the wave calls it.
__device__ __forceinline__ void store_wave_error(const ProjectionArgs& a, double error) {
    double wave_error = error;
    for (int offset = 32; offset > 0; offset >>= 1) wave_error += __shfl_xor(wave_error, offset, 64);
    if ((threadIdx.x & 63u) == 0u) a.cv.partials[blockIdx.x * kWaves + (threadIdx.x >> 6)] = wave_error;
}

// The pressure phase a projection serves. The kernel is the same for both;
// the two instantiations only give profiles one kernel name per phase.
enum ProjectionPhase : int { kProjectDivergence = 0, kProjectDensity = 1 };

// density at predicted positions (density.cu:18-40 with topology = x,
// positions = x*) fused with the pressure update and the next pressure
// pass's first_term: projection_update_forward_kernel (dfsph.cu:104-110),
// pressure_update_forward_kernel (pcisph.cu:104-110) or
// jacobi_update_forward_kernel (iisph.cu:104-110), which differ only in the
// density of the volume V = m / density.
template <int kPhase>
__global__ void __launch_bounds__(kBlock) projection_kernel(ProjectionArgs a) {
    __shared__ uint16_t smask[kStencil * kBlock];
    __shared__ int delta[kStencil];
    fill_slot_deltas(a.grid, delta);
    __syncthreads();
    const bool tolerance = a.cv.partials != nullptr;
    if (tolerance && *a.cv.done != 0u) return;  // the phase ended at an earlier iteration
    const uint32_t i = xcd_block() * kBlock + threadIdx.x;
    double error = 0.0;
    if (i < a.n) {
        const float4 topology = a.xm[i];
        const uint32_t center = a.cell[i];
        const bool crowded = a.crowded[i] != 0u;
        const bool masked = projection_masked(a, i, center);
        const float4 self = a.xs[i];
        const Float3 ps = xyz(self);
        float rs = 0.0F;
        if (!crowded) {
            uint16_t* column = smask + threadIdx.x;
            uint32_t nonzero = 0u;
            if (masked) {
                nonzero = load_lane_column(a.skin, a.n, i, column, kBlock);
            } else {
                // moved past the skin: mark the candidates at the predicted
                // positions, then walk those (scan_stencil)
                int cx, cy, cz;
                cell_coordinates(a.grid, center, cx, cy, cz);
                scan_stencil(
                    a.grid, a.xs, cx, cy, cz, [&](Float3 q) { return within_support(a.kc, ps, q); },
                    [&](uint32_t k, uint32_t bits) {
                        column[k * kBlock] = static_cast<uint16_t>(bits);
                        nonzero |= bits != 0u ? 1u << k : 0u;
                    });
            }
            walk_masked_prefetch<kWalkDepth>(
                a.grid.offsets, center, delta, column, kBlock, nonzero, i,
                [&](uint32_t s) { return a.xs[s]; },
                [&](float4 q) { rs += q.w * cubic_value(pair_distance(sub(ps, xyz(q))), a.kc); });
        } else {
            int cx, cy, cz;
            cell_coordinates(a.grid, center, cx, cy, cz);
            for_each_candidate(a.grid, cx, cy, cz, [&](uint32_t s) {
                const float4 q = a.xs[s];
                rs += q.w * cubic_value(pair_distance(sub(ps, xyz(q))), a.kc);
            });
        }
        error = update_pressure(a, i, topology, self.w, rs);
    }
    if (tolerance) store_wave_error(a, error);  // every lane of the wave is here (no early return above)
}

// projection_kernel with a group of G lanes per particle; with kSamples each
// cell's boundary samples add rho0_i V_b W(x*_i - x_b) after its particles.
template <int kPhase, int G, bool kSamples>
__global__ void __launch_bounds__(kGroupBlock) projection_group_kernel(ProjectionArgs a) {
    constexpr uint32_t kParticles = kGroupParticles<G>;
    __shared__ GroupLds<G> lds;
    const bool tolerance = a.cv.partials != nullptr;
    if (tolerance && *a.cv.done != 0u) return;  // the phase ended at an earlier iteration
    const uint32_t base = xcd_block() * kParticles;
    const uint32_t i = base + threadIdx.x % kParticles;
    uint32_t center = 0u;
    bool listed = false, masked = false;
    Float3 expanded{0.0F, 0.0F, 0.0F};
    int cx = 0, cy = 0, cz = 0;
    if (i < a.n) {
        center = a.cell[i];
        listed = a.crowded[i] == 0u;
        masked = projection_masked(a, i, center);
        if (listed && !masked) {  // moved past the skin: marked at the predicted positions below
            expanded = xyz(a.xs[i]);
            cell_coordinates(a.grid, center, cx, cy, cz);
        }
    }
    const uint32_t w = base + threadIdx.x / G;
    const bool active = w < a.n;
    const float4 self = a.xs[active ? w : 0u];
    const float rest = kSamples && active ? a.rest_density[w] : 0.0F;
    float sum[1] = {0.0F};
    auto fetch = [&](uint32_t entry) {
        if constexpr (kSamples) {
            if ((entry & kSampleEntry) != 0u) return a.boundary.x[entry & ~kSampleEntry];
        }
        return a.xs[entry];
    };
    auto pair = [&](float4 q, uint32_t entry, float (&terms)[1]) {
        const float weight = cubic_value(pair_distance(sub(xyz(self), xyz(q))), a.kc);
        terms[0] = kSamples && (entry & kSampleEntry) != 0u ? rest * q.w * weight : q.w * weight;
    };
    auto fold = [&](const float (&terms)[1]) { group_add<G, 1>(sum, terms); };
    group_expand<G, kSamples>(
        lds,
        [&](auto& bits, auto& first) {
            if (masked) {
                stored_slots<G, false>(a.skin, a.grid, a.grid.offsets, a.n, i, center, bits, first);
            } else if (listed) {
                scanned_slots<G>(a.grid, a.grid.offsets, a.xs, cx, cy, cz, bits, first,
                                 [&](Float3 q) { return within_support(a.kc, expanded, q); });
            }
        },
        [&](auto& bits, auto& first) {
            if (masked) {
                stored_slots<G, false>(a.skin_samples, a.grid, a.boundary.offsets, a.n, i, center, bits, first);
            } else if (listed) {
                scanned_slots<G>(a.grid, a.boundary.offsets, a.boundary.x, cx, cy, cz, bits, first,
                                 [&](Float3 q) { return within_support(a.kc, expanded, q); });
            }
        },
        [&](const uint32_t* row, uint32_t count) {
            if (active) group_walk_list<G, 1>(row, count, w, fetch, pair, fold);
        });
    double error = 0.0;
    if (active) {
        if (a.crowded[w] != 0u) {
            cell_coordinates(a.grid, a.cell[w], cx, cy, cz);
            group_walk_stencil<G, 1>(
                a.grid, kSamples ? a.boundary.offsets : nullptr, cx, cy, cz, ~0u, w, group_row(lds),
                [&](uint32_t entry) { return within_support(a.kc, xyz(self), xyz(fetch(entry))); }, fetch, pair, fold);
        }
        if (threadIdx.x % G == 0u) error = update_pressure(a, w, a.xm[w], self.w, sum[0]);
    }
    if (tolerance) store_wave_error(a, error);
}

enum Epilogue : int {
    kDivPredict = 0,   // total = a_p(t1)
    kDivEnd = 1,       // a_div = a_p(t1); total = a_div + a_p(t2)
    kDenPredict = 2,   // total = a_div + a_p(t1)
    kInitPredict = 3,  // total = 0 (cleared pressure acceleration), no pressure pass
    kDivAuto = 4,      // tolerance mode: kDivEnd at the iteration that ends the phase, else kDivPredict
};

struct ForceArgs {
    uint32_t n;
    KernelConstants kc;
    float dt;
    SortedGrid grid;
    Box box;
    Float3 gravity;
    const float4* xm;
    const float4* vmu;  // velocity (+ viscosity)
    CVec u;
    const float* rho;
    const float* t1;
    const float* t2;
    const uint16_t* exact;
    uint32_t* flags;
    uint32_t slot;
    float4* anp;
    float4* adiv;
    float4* xs;
    uint8_t* collisions;  // optional (recorded step): box-collision bits of the prediction
    uint32_t final_step;
    const uint32_t* perm;
    Vec next_x, next_v;
    const float* p_div;
    float* warm_div_out;
    const float* p_den;
    float* warm_den_out;
    // tolerance mode: the phase's done word and this pass's iteration; a
    // pass of a later iteration than the one that ended the phase returns
    const uint32_t* done;
    uint32_t iteration;
    BoundaryGrid boundary;      // offsets null: no boundary samples
    const float* rest_density;  // rho0, for the boundary pressure terms
    const uint8_t* crowded;     // per particle: walks the full stencil
    const uint32_t* cell;       // MaskDensityArgs::cell
    // per-cell skins: a predicting pass marks the 27 cells around every
    // particle that moved farther than its cell's bound with `stamp`
    const float* cell_bound = nullptr;
    uint32_t* taint = nullptr;
    uint32_t stamp = 0u;
    // optional: |x_next - x| per particle (original order), written with the next state
    float* moved_out = nullptr;
    // optional: (x, y, z, t1) per particle and the step's mass state {
    // mass_stamp if some mass differs from particle 0's, particle 0's mass
    // bits} (written by the mask pass): with equal masses a candidate is one
    // 16-byte record instead of its position, mass and t1
    const float4* xt1 = nullptr;
    const uint32_t* mass_state = nullptr;
    uint32_t mass_stamp = 0u;
    const uint16_t* exact_samples = nullptr;  // MaskDensityArgs::exact_samples
};

// What a force pass does with particle i's non-pressure acceleration `acc`
// and pressure accelerations ap1, ap2 (the latter with `two`): the prediction
// or next state. Returns the squared displacement of a prediction.
template <bool kNonPressure, int kEpilogue>
__device__ __forceinline__ float finish_force(const ForceArgs& a, uint32_t i, float4 self, Float3 vel, bool two,
                                              uint32_t final_step, uint32_t cell, Float3 acc, Float3 ap1, Float3 ap2) {
    const Float3 p = xyz(self);
    if constexpr (kNonPressure) {
        a.anp[i] = make_float4(acc.x, acc.y, acc.z, 0.0F);
    } else {
        acc = xyz(a.anp[i]);
    }
    Float3 total;
    if constexpr (kEpilogue == kInitPredict) {
        total = Float3{0.0F, 0.0F, 0.0F};
    } else if constexpr (kEpilogue == kDenPredict) {
        total = add(xyz(a.adiv[i]), ap1);
    } else if (two) {
        a.adiv[i] = make_float4(ap1.x, ap1.y, ap1.z, 0.0F);
        total = add(ap1, ap2);
    } else {
        total = ap1;
    }
    Float3 nx, nv;
    const Float3 a_total = add(acc, total);
    predict_clamped(a.box, a.dt, p, vel, a_total, nx, nv);
    if (a.collisions != nullptr)
        a.collisions[i] = static_cast<uint8_t>(predict_collisions(a.box, a.dt, p, vel, a_total));
    if (two && a.warm_div_out != nullptr) a.warm_div_out[a.perm[i]] = a.p_div[i];
    const Float3 moved = sub(nx, p);
    if (final_step != 0u) {
        const uint32_t j = a.perm[i];
        store(a.next_x, j, nx);
        store(a.next_v, j, nv);
        if (a.warm_den_out != nullptr) a.warm_den_out[j] = a.p_den[i];
        if (a.moved_out != nullptr) a.moved_out[j] = sqrtf(dot(moved, moved));
        return 0.0F;
    }
    a.xs[i] = make_float4(nx.x, nx.y, nx.z, self.w);
    const float moved2 = dot(moved, moved);
    if (a.taint != nullptr) {
        const float bound = a.cell_bound[cell];
        if (moved2 > bound * bound) {
            int cx, cy, cz;
            cell_coordinates(a.grid, cell, cx, cy, cz);
            taint_neighbour_cells(a.grid, cx, cy, cz, a.taint, a.stamp);
        }
    }
    return moved2;
}

// Pressure acceleration (pressure_forward_kernel, common.cu:165-194),
// optionally fused with the non-pressure acceleration
// (non_pressure_forward_kernel, common.cu:14-47), then the predict of the
// next iteration (dfsph.cu:26-44) or, on the last pass, the next state.
// cubic_gradient(d, h) is evaluated as f * d with f its radial factor, the
// same operations as the reference's expression. Launches with boundary
// samples go to the group kernel.
template <bool kNonPressure, int kEpilogue>
__global__ void __launch_bounds__(kBlock) force_kernel(ForceArgs a) {
    constexpr bool kAuto = kEpilogue == kDivAuto;
    constexpr bool kPressure = kEpilogue != kInitPredict;
    __shared__ uint16_t smask[kStencil * kBlock];
    __shared__ int delta[kStencil];
    fill_slot_deltas(a.grid, delta);
    __syncthreads();
    // the iteration that ends its phase (tolerance mode), uniform over the grid
    const uint32_t ended = a.done != nullptr ? *a.done : 0u;
    if (ended != 0u && ended < a.iteration) return;
    const bool ends = ended != 0u && ended == a.iteration;
    // a second pressure field: the divergence phase's end
    const bool kTwo = kEpilogue == kDivEnd || (kAuto && ends);
    // tolerance mode: the iteration that ends the last phase writes the state
    const uint32_t final_step =
        a.final_step != 0u || ((kEpilogue == kDenPredict || kEpilogue == kDivPredict) && ends) ? 1u : 0u;
    const uint32_t i = xcd_block() * kBlock + threadIdx.x;
    const bool active = i < a.n;
    float moved2 = 0.0F;
    if (active) {
        const bool masked = a.crowded[i] == 0u;
        const float4 self = a.xm[i];
        const Float3 p = xyz(self);
        const float4 vm = a.vmu[i];
        const Float3 vel = xyz(vm);
        Float3 acc{0.0F, 0.0F, 0.0F};
        if constexpr (kNonPressure) acc = add(a.gravity, load(a.u, i));
        const float t1_i = kPressure ? a.t1[i] : 0.0F;
        float t2_i = 0.0F;
        if (kTwo) t2_i = a.t2[i];
        Float3 ap1{0.0F, 0.0F, 0.0F};
        Float3 ap2{0.0F, 0.0F, 0.0F};
        const uint32_t center = a.cell[i];
        // candidates as (x, y, z, t1) records with one mass (uniform over the launch)
        const bool packed = kPressure && a.xt1 != nullptr && a.mass_state[0] != a.mass_stamp;
        const float mass = packed ? __uint_as_float(a.mass_state[1]) : 0.0F;
        auto pair = [&](uint32_t s, float4 q, float t1_s, float t2_s, Float3 d, float f) {
            const float ms = q.w;
            if constexpr (kNonPressure) {
                const float4 vq = a.vmu[s];
                const float viscosity = 0.5F * (vm.w + vq.w);
                const float weight = viscosity * ms * viscosity_laplacian_c(d, a.kc) / a.rho[s];
                acc = add(acc, scale(sub(xyz(vq), vel), weight));
            }
            if constexpr (kPressure) {
                const Float3 gradient = scale(d, f);
                ap1 = add(ap1, scale(gradient, -ms * (t1_i + t1_s)));
                if (kTwo) ap2 = add(ap2, scale(gradient, -ms * (t2_i + t2_s)));
            }
        };
        if (masked) {
            uint16_t* column = smask + threadIdx.x;
            uint32_t nonzero = load_lane_column(a.exact, a.n, i, column, kBlock);
            nonzero = drop_self(i, a.grid.offsets[center], column, kBlock, nonzero);
            if (packed) {
                // equal masses: (x, y, z, t1) is the whole candidate but t2
                if constexpr (kNonPressure) {
                    walk_masked(a.grid.offsets, center, delta, column, kBlock, nonzero, [&](uint32_t s) {
                        const float4 r = a.xt1[s];
                        const float t2_s = kTwo ? a.t2[s] : 0.0F;
                        const Float3 d = sub(p, xyz(r));
                        pair(s, make_float4(r.x, r.y, r.z, mass), r.w, t2_s, d,
                             kPressure ? cubic_gradient_factor(pair_distance(d), a.kc) : 0.0F);
                    });
                } else {
                    struct Record {
                        float4 r;
                        float t2;
                    };
                    walk_masked_prefetch<kWalkDepth>(
                        a.grid.offsets, center, delta, column, kBlock, nonzero, i,
                        [&](uint32_t s) { return Record{a.xt1[s], kTwo ? a.t2[s] : 0.0F}; },
                        [&](const Record& c) {
                            const Float3 d = sub(p, xyz(c.r));
                            pair(0u, make_float4(c.r.x, c.r.y, c.r.z, mass), c.r.w, c.t2, d,
                                 cubic_gradient_factor(pair_distance(d), a.kc));
                        });
                }
            } else if constexpr (kNonPressure) {
                walk_masked(a.grid.offsets, center, delta, column, kBlock, nonzero, [&](uint32_t s) {
                    const float4 q = a.xm[s];
                    const float t1_s = kPressure ? a.t1[s] : 0.0F;
                    const float t2_s = kTwo ? a.t2[s] : 0.0F;
                    const Float3 d = sub(p, xyz(q));
                    pair(s, q, t1_s, t2_s, d, kPressure ? cubic_gradient_factor(pair_distance(d), a.kc) : 0.0F);
                });
            } else {
                struct Candidate {
                    float4 q;
                    float t1, t2;
                };
                walk_masked_prefetch<kWalkDepth>(
                    a.grid.offsets, center, delta, column, kBlock, nonzero, i,
                    [&](uint32_t s) { return Candidate{a.xm[s], a.t1[s], kTwo ? a.t2[s] : 0.0F}; },
                    [&](const Candidate& c) {
                        const Float3 d = sub(p, xyz(c.q));
                        pair(0u, c.q, c.t1, c.t2, d, cubic_gradient_factor(pair_distance(d), a.kc));
                    });
            }
        } else {
            auto visit = [&](uint32_t s) {
                if (s == i) return;
                const float4 q = a.xm[s];
                const float t1_s = kPressure ? a.t1[s] : 0.0F;
                const float t2_s = kTwo ? a.t2[s] : 0.0F;
                const Float3 d = sub(p, xyz(q));
                pair(s, q, t1_s, t2_s, d, kPressure ? cubic_gradient_factor(pair_distance(d), a.kc) : 0.0F);
            };
            int cx, cy, cz;
            cell_coordinates(a.grid, center, cx, cy, cz);
            for_each_candidate(a.grid, cx, cy, cz, visit);
        }
        moved2 = finish_force<kNonPressure, kEpilogue>(a, i, self, vel, kTwo, final_step, center, acc, ap1, ap2);
    }
    if (final_step == 0u) block_max_to<kBlock>(moved2, &a.flags[kFlagDisplacement + a.slot]);
}

// force_kernel with a group of G lanes per particle. With kSamples the
// boundary samples add, after each cell's particles, mu_i V_b lap W
// (v_b - v_i) (common.cu:38-43) and grad W (-rho0_i V_b p_i / rho_i^2)
// (common.cu:185-190).
template <bool kNonPressure, int kEpilogue, int G, bool kSamples>
__global__ void __launch_bounds__(kGroupBlock) force_group_kernel(ForceArgs a) {
    constexpr uint32_t kParticles = kGroupParticles<G>;
    constexpr bool kAuto = kEpilogue == kDivAuto;
    constexpr bool kPressure = kEpilogue != kInitPredict;
    constexpr bool kMayTwo = kEpilogue == kDivEnd || kAuto;
    // the sums: non-pressure, first pressure and second pressure acceleration
    constexpr int kFirst = kNonPressure ? 3 : 0;
    constexpr int kSecond = kFirst + (kPressure ? 3 : 0);
    constexpr int kSums = kSecond + (kMayTwo ? 3 : 0);
    __shared__ GroupLds<G> lds;
    // the iteration that ends its phase (tolerance mode), uniform over the grid
    const uint32_t ended = a.done != nullptr ? *a.done : 0u;
    if (ended != 0u && ended < a.iteration) return;
    const bool ends = ended != 0u && ended == a.iteration;
    const bool two = kEpilogue == kDivEnd || (kAuto && ends);
    const uint32_t final_step =
        a.final_step != 0u || ((kEpilogue == kDenPredict || kEpilogue == kDivPredict) && ends) ? 1u : 0u;
    const uint32_t base = xcd_block() * kParticles;
    const uint32_t i = base + threadIdx.x % kParticles;
    uint32_t center = 0u;
    bool listed = false;
    if (i < a.n) {
        center = a.cell[i];
        listed = a.crowded[i] == 0u;
    }
    const uint32_t w = base + threadIdx.x / G;
    const bool active = w < a.n;
    const uint32_t own = active ? w : 0u;
    const float4 self = a.xm[own];
    const Float3 p = xyz(self);
    const float4 vm = a.vmu[own];
    const Float3 vel = xyz(vm);
    const float t1_i = kPressure ? a.t1[own] : 0.0F;
    const float t2_i = kMayTwo && two ? a.t2[own] : 0.0F;
    const float rest = kSamples ? a.rest_density[own] : 0.0F;
    // candidates as (x, y, z, t1) records with one mass (uniform over the launch)
    const bool packed = kPressure && a.xt1 != nullptr && a.mass_state[0] != a.mass_stamp;
    const float mass = packed ? __uint_as_float(a.mass_state[1]) : 0.0F;
    float sum[kSums];
#pragma unroll
    for (int f = 0; f < kSums; ++f) sum[f] = 0.0F;
    if constexpr (kNonPressure) {
        const Float3 start = add(a.gravity, load(a.u, own));
        sum[0] = start.x;
        sum[1] = start.y;
        sum[2] = start.z;
    }
    struct Record {
        float4 q;  // position and mass, or a sample's volume
        float t1, t2;
        float4 v;  // velocity and viscosity
        float rho;
    };
    auto fetch = [&](uint32_t entry) {
        Record r{};
        if constexpr (kSamples) {
            if ((entry & kSampleEntry) != 0u) {
                const uint32_t b = entry & ~kSampleEntry;
                r.q = a.boundary.x[b];
                if constexpr (kNonPressure) r.v = a.boundary.v[b];
                return r;
            }
        }
        if (packed) {
            const float4 x = a.xt1[entry];
            r.q = make_float4(x.x, x.y, x.z, mass);
            r.t1 = x.w;
        } else {
            r.q = a.xm[entry];
            if constexpr (kPressure) r.t1 = a.t1[entry];
        }
        if constexpr (kMayTwo) {
            if (two) r.t2 = a.t2[entry];
        }
        if constexpr (kNonPressure) {
            r.v = a.vmu[entry];
            r.rho = a.rho[entry];
        }
        return r;
    };
    auto put = [](float* terms, Float3 v) {
        terms[0] = v.x;
        terms[1] = v.y;
        terms[2] = v.z;
    };
    auto pair = [&](const Record& r, uint32_t entry, float (&terms)[kSums]) {
        const Float3 d = sub(p, xyz(r.q));
        const bool sample = kSamples && (entry & kSampleEntry) != 0u;
        if constexpr (kNonPressure) {
            const float laplacian = viscosity_laplacian_c(d, a.kc);
            const float weight = sample ? vm.w * r.q.w * laplacian
                                        : 0.5F * (vm.w + r.v.w) * r.q.w * laplacian / r.rho;
            put(terms, scale(sub(xyz(r.v), vel), weight));
        }
        if constexpr (kPressure) {
            const Float3 gradient = scale(d, cubic_gradient_factor(pair_distance(d), a.kc));
            put(terms + kFirst, scale(gradient, sample ? -rest * r.q.w * t1_i : -r.q.w * (t1_i + r.t1)));
            if constexpr (kMayTwo) {
                if (two) put(terms + kSecond, scale(gradient, sample ? -rest * r.q.w * t2_i : -r.q.w * (t2_i + r.t2)));
            }
        }
    };
    auto fold = [&](const float (&terms)[kSums]) {
        group_add<G, kSums>(sum, terms);
    };
    group_expand<G, kSamples>(
        lds,
        [&](auto& bits, auto& first) {
            if (listed) stored_slots<G, true>(a.exact, a.grid, a.grid.offsets, a.n, i, center, bits, first);
        },
        [&](auto& bits, auto& first) {
            if (listed) stored_slots<G, false>(a.exact_samples, a.grid, a.boundary.offsets, a.n, i, center, bits, first);
        },
        [&](const uint32_t* row, uint32_t count) {
            if (active) group_walk_list<G, kSums>(row, count, w, fetch, pair, fold);
        });
    float moved2 = 0.0F;
    if (active) {
        const uint32_t cell = a.cell[w];
        if (a.crowded[w] != 0u) {
            int cx, cy, cz;
            cell_coordinates(a.grid, cell, cx, cy, cz);
            group_walk_stencil<G, kSums>(
                a.grid, kSamples ? a.boundary.offsets : nullptr, cx, cy, cz, w, w, group_row(lds),
                [&](uint32_t entry) {
                    const bool sample = kSamples && (entry & kSampleEntry) != 0u;
                    return within_support(a.kc, p, xyz(sample ? a.boundary.x[entry & ~kSampleEntry] : a.xm[entry]));
                },
                fetch, pair, fold);
        }
        if (threadIdx.x % G == 0u) {
            Float3 acc{0.0F, 0.0F, 0.0F}, ap1{0.0F, 0.0F, 0.0F}, ap2{0.0F, 0.0F, 0.0F};
            if constexpr (kNonPressure) acc = Float3{sum[0], sum[1], sum[2]};
            if constexpr (kPressure) ap1 = Float3{sum[kFirst], sum[kFirst + 1], sum[kFirst + 2]};
            if constexpr (kMayTwo) ap2 = Float3{sum[kSecond], sum[kSecond + 1], sum[kSecond + 2]};
            moved2 = finish_force<kNonPressure, kEpilogue>(a, w, self, vel, two, final_step, cell, acc, ap1, ap2);
        }
    }
    if (final_step == 0u) block_max_to<kGroupBlock>(moved2, &a.flags[kFlagDisplacement + a.slot]);
}

// Lanes per particle of a pass that always runs in groups.
inline int wide_group(uint32_t n) { return n <= kGroup16Particles ? 16 : 4; }

// Lanes per particle of a projection or force pass (1: the kernels without
// groups, which do not take boundary samples).
inline int pass_group(uint32_t n, bool samples) { return samples || n <= kGroup4Particles ? wide_group(n) : 1; }

// Whole workgroups of a launch with groups of `group` lanes, padded to a
// multiple of the XCD count.
inline uint32_t pass_blocks(uint32_t n, int group) {
    return (blocks_for(n, kBlock / static_cast<uint32_t>(group)) + 7u) / 8u * 8u;
}

// Calls launch(std::integral_constant<int, G>, std::bool_constant<samples>)
// for a launch with groups.
template <class Launch>
void with_group(int group, bool samples, Launch&& launch) {
    if (group == 16) {
        if (samples) {
            launch(std::integral_constant<int, 16>{}, std::true_type{});
        } else {
            launch(std::integral_constant<int, 16>{}, std::false_type{});
        }
    } else {
        if (samples) {
            launch(std::integral_constant<int, 4>{}, std::true_type{});
        } else {
            launch(std::integral_constant<int, 4>{}, std::false_type{});
        }
    }
}

template <bool kNonPressure, int kEpilogue>
void launch_force(PassProfiler& profiler, hipStream_t stream, int group, const ForceArgs& args, int pass) {
    PassScope scope(profiler, stream, pass);
    const uint32_t blocks = pass_blocks(args.n, group);
    if (group == 1) {
        force_kernel<kNonPressure, kEpilogue><<<blocks, kBlock, 0, stream>>>(args);
    } else {
        with_group(group, args.boundary.offsets != nullptr, [&](auto g, auto samples) {
            force_group_kernel<kNonPressure, kEpilogue, g(), samples()><<<blocks, kGroupBlock, 0, stream>>>(args);
        });
    }
    PHX_LAUNCH_CHECK();
}

template <int kPhase>
void launch_projection_phase(hipStream_t stream, int group, const ProjectionArgs& args) {
    const uint32_t blocks = pass_blocks(args.n, group);
    if (group == 1) {
        projection_kernel<kPhase><<<blocks, kBlock, 0, stream>>>(args);
    } else {
        with_group(group, args.boundary.offsets != nullptr, [&](auto g, auto samples) {
            projection_group_kernel<kPhase, g(), samples()><<<blocks, kGroupBlock, 0, stream>>>(args);
        });
    }
}

void launch_projection(PassProfiler& profiler, hipStream_t stream, int group, const ProjectionArgs& args, int pass,
                       ProjectionPhase phase) {
    PassScope scope(profiler, stream, pass);
    if (phase == kProjectDivergence) {
        launch_projection_phase<kProjectDivergence>(stream, group, args);
    } else {
        launch_projection_phase<kProjectDensity>(stream, group, args);
    }
    PHX_LAUNCH_CHECK();
}

template <bool kEos>
void launch_mask_density(PassProfiler& profiler, hipStream_t stream, const MaskDensityArgs& args, int pass) {
    PassScope scope(profiler, stream, pass);
    const int group = wide_group(args.n);
    with_group(group, args.boundary.offsets != nullptr, [&](auto g, auto samples) {
        mask_density_kernel<kEos, g(), samples()><<<pass_blocks(args.n, group), kGroupBlock, 0, stream>>>(args);
    });
    PHX_LAUNCH_CHECK();
}

}  // namespace
}  // namespace phx
