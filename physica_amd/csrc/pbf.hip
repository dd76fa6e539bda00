// PBF forward step for gfx950 in sorted (cell-major) particle order.
//
// Reference: PBF::forward_step (pbf/pbf.cpp:167-191) and pbf/pbf.cu. Fusion:
//   grid       predict x* fused into the cell-key pass (pbf.cu:73-78)
//   per iter   A: density + lambda in one neighbour loop (density.cu:18-40,
//                 pbf.cu:95-127; the two sums keep their own order)
//              B: correction + project (pbf.cu:254-288, 417-431), written to
//                 a second position buffer so neighbours read the old values;
//                 the last iteration also reconstructs v = (p - x)/dt
//   post       vorticity + magnitude (pbf.cu:476-497, 565-569)
//              normal + confinement (pbf.cu:571-593, 674-678)
//              XSPH + scatter of the next state (pbf.cu:700-721)
// A pass gives each particle a group of 4 or 16 lanes (group_walk.hpp). The
// first pass at a set of positions (lambda, vorticity) scans the 27 cells and
// writes the exact neighbour masks that the others at those positions walk.
// Candidates are fetched as 16-byte records (position and mass, or velocity):
// single floats kept the CU's address unit busy 80 % of the time, and a record
// costs it about as much as one of the three to five single floats it
// replaces (814,213 particles in 12 scenes: lambda 270 -> 176 us, correction
// 147 -> 122, vorticity 306 -> 170, normal 118 -> 92, XSPH 151 -> 89; with the
// pair arithmetic of device_math.hpp 172, 102, 174, 78 and 78).
// Per-particle sums run in the reference order, so each value is the IEEE
// result of the reference expression.
#include "pbf.hpp"

#include "group_walk.hpp"
#include "neighbor_mask.hpp"

#include <cmath>
#include <type_traits>

namespace phx {
namespace {

__device__ __forceinline__ Float3 xyz(float4 q) { return Float3{q.x, q.y, q.z}; }

constexpr uint32_t kBlock = 256;
// Particle counts up to which 16 lanes share a particle; above, 4. One lane
// per particle, over skin masks built once a step, is slower at every size.
// Steps, us, with 1 / 4 / 16 lanes before the candidates were records: 1,300
// particles 532 / 169 / 106, 16,000 514 / 174 / 136, 32,000 524 / 179 / 181
// (30 clumps 1,799 / 613 / 524), 64,000 517 / 239 / 289, 1,048,576 4,080 /
// 2,313 / 3,424; with records, 4 / 16 lanes: 32,000 165 / 168, 64,000 196 /
// 254, 1,048,576 1,590 / 2,865.
constexpr uint32_t kGroup16Particles = 32768;

// Workgroups with crowded particles that a pass starts before all others.
constexpr uint32_t kEarlyBlocks = 512;
// Particle count from which a single scene orders its workgroups so (a batch
// always does): below, a pass's workgroups all start at once anyway.
constexpr uint32_t kEarlyParticles = 100000;

// The order of a pass's workgroups. A workgroup with crowded particles can
// last many times as long as the others; started last, it runs on alone.
// pbf_cell_kernel lists such workgroups, and the first kEarlyBlocks blocks of
// a launch serve the listed ones; a listed workgroup's own block returns at
// once. 262,144 particles with 60
// clumps: 1,317 -> 1,057 us a step.
struct Schedule {
    uint32_t* count;   // workgroups listed (may exceed kEarlyBlocks: the rest are not served early)
    uint32_t* listed;  // [kEarlyBlocks] their ids
    uint32_t* place;   // per workgroup: its place in `listed` + 1; 0: not listed
    uint32_t* seen;    // per workgroup: non-zero once a crowded particle was found
    uint32_t early;    // kEarlyBlocks, or 0: workgroups in order
};

// The workgroup id a block serves; ~0u for none.
__device__ __forceinline__ uint32_t scheduled_block(const Schedule& s) {
    if (s.early == 0u) return xcd_block();
    if (blockIdx.x < s.early) return blockIdx.x < *s.count ? s.listed[blockIdx.x] : ~0u;
    const uint32_t per_xcd = (gridDim.x - s.early) / 8u;
    const uint32_t b = blockIdx.x - s.early;
    const uint32_t id = b % 8u * per_xcd + b / 8u;
    return s.place[id] - 1u < s.early ? ~0u : id;
}

// The particle, grid and collision box of a lane: one scene (kBatch false),
// or in a batch the scene of the workgroup's block, whose grid starts at
// the scene's cell base in the batch's offsets.
struct Lane {
    uint32_t i;
    bool valid;
    SortedGrid grid;
    Box box;
};

template <bool kBatch>
__device__ __forceinline__ Lane lane_of(uint32_t id, uint32_t n, const SortedGrid& grid, const Box& box,
                                        const BatchView& batch) {
    Lane l;
    if constexpr (kBatch) {
        const BatchBlock blk = batch.blocks[id];
        const BatchScene& sc = batch.scenes[blk.scene];
        l.i = blk.first + threadIdx.x;
        l.valid = threadIdx.x < blk.count;
        // the lookup origin min + t v_box and the collision box of the step
        // (neighborhood.cpp:83-88, pbf.cpp:17-31), as the host computes them
        const float t = batch.time;
        l.grid = SortedGrid{grid.offsets + sc.cell_base,
                            sc.res[0],
                            sc.res[1],
                            sc.res[2],
                            sc.minimum[0] + t * sc.velocity[0],
                            sc.minimum[1] + t * sc.velocity[1],
                            sc.minimum[2] + t * sc.velocity[2],
                            batch.h};
        const float rp = sc.particle_radius;
        for (int a = 0; a < 3; ++a) {
            l.box.lo[a] = sc.minimum[a] + t * sc.velocity[a] + rp;
            l.box.hi[a] = sc.maximum[a] + t * sc.velocity[a] - rp;
            l.box.vel[a] = sc.velocity[a];
        }
        l.box.no_slip = sc.no_slip;
    } else {
        l.i = id * kBlock + threadIdx.x;
        l.valid = l.i < n;
        l.grid = grid;
        l.box = box;
    }
    return l;
}

// The particles of workgroup `id` of a launch with groups of G lanes: base ..
// base + count - 1, of one scene.
struct GroupScene {
    uint32_t base, count;
    SortedGrid grid;
    Box box;
};

template <bool kBatch, int G>
__device__ __forceinline__ GroupScene group_scene(uint32_t id, uint32_t n, const SortedGrid& grid, const Box& box,
                                                  const BatchView& batch) {
    if constexpr (kBatch) {
        const BatchBlock blk = batch.blocks[id];
        const Lane l = lane_of<true>(id, n, grid, box, batch);
        return GroupScene{blk.first, blk.count, l.grid, l.box};
    } else {
        const uint32_t base = id * kGroupParticles<G>;
        return GroupScene{base, base < n ? min(n - base, kGroupParticles<G>) : 0u, grid, box};
    }
}

// The cell and crowded byte of each particle (a stencil cell holds more than
// kMaskBits particles, or boundary samples), and the workgroups (of `particles`
// particles each) that hold crowded ones.
template <bool kBatch>
__global__ void __launch_bounds__(kBlock) pbf_cell_kernel(uint32_t n, SortedGrid launch_grid,
                                                          const uint32_t* sample_offsets, const float4* xs,
                                                          uint32_t* cell, uint8_t* crowded, uint32_t particles,
                                                          Schedule schedule, BatchView batch) {
    const uint32_t id = xcd_block();
    const Lane lane = lane_of<kBatch>(id, n, launch_grid, Box{}, batch);
    if (!lane.valid) return;
    const SortedGrid& grid = lane.grid;
    int cx, cy, cz;
    particle_cell(grid, xyz(xs[lane.i]), cx, cy, cz);
    cell[lane.i] = cell_of(grid, cx, cy, cz);
    bool many = false;
    for_each_cell(grid, cx, cy, cz, [&](uint32_t c) {
        many = many || grid.offsets[c + 1u] - grid.offsets[c] > kMaskBits;
        if (sample_offsets != nullptr) many = many || sample_offsets[c + 1u] - sample_offsets[c] > kMaskBits;
    });
    crowded[lane.i] = many ? 1u : 0u;
    if (!many) return;
    const uint32_t first = kBatch ? batch.blocks[id].group_block : id * (kBlock / particles);
    const uint32_t group_block = first + threadIdx.x / particles;
    if (atomicExch(schedule.seen + group_block, 1u) != 0u) return;
    const uint32_t place = atomicAdd(schedule.count, 1u);
    if (place < kEarlyBlocks) schedule.listed[place] = group_block;
    schedule.place[group_block] = place + 1u;
}

struct LambdaArgs {
    uint32_t n;
    PbfKernel k;
    SortedGrid grid;
    const float4* pos;  // positions and masses
    const float* rho0;
    const float* eps;
    float* rho;
    float* lambda;
    float* den;  // optional (recorded step)
    Vec gsum;    // optional (recorded step)
    // exact masks of the positions read (pairs inside exact_mask_threshold),
    // for the correction pass and the derivatives (crowded particles walk the
    // full stencil instead)
    float t_exact;
    uint16_t* exact_out;
    BoundaryGrid boundary;  // offsets null: no boundary samples
    // the cell and crowded byte of each particle, written by the step's first
    // pass (first_pass != 0) and read by the others
    uint32_t* cell;
    uint8_t* crowded;
    uint32_t first_pass;
    const uint32_t* unusual_masses;  // rest_density_of
};

// The terms of one candidate in the density and lambda sums: the density,
// the gradient sum and the denominator.
struct LambdaTerms {
    float density;
    Float3 gradient;
    float square;
};
__device__ __forceinline__ LambdaTerms lambda_terms(const LambdaArgs& a, Float3 d, float ms, const RestDensity& rest) {
    const float d2 = dot(d, d);
    const Float3 g = scale(d, spiky_factor(d2, a.k));
    const float coefficient = over_rest(ms, rest);
    return LambdaTerms{ms * poly6_value(d2, a.k), scale(g, coefficient), coefficient * coefficient * dot(g, g)};
}

__device__ __forceinline__ void finish_lambda(const LambdaArgs& a, uint32_t i, float rest, float density,
                                              Float3 gradient_sum, float denominator) {
    denominator += dot(gradient_sum, gradient_sum);
    a.rho[i] = density;
    a.lambda[i] = -(density / rest - 1.0F) / denominator;
    if (a.den != nullptr) {
        a.den[i] = denominator;
        store(a.gsum, i, gradient_sum);
    }
}

// The position of a list entry, and its mass or a sample's volume.
template <bool kSamples>
__device__ __forceinline__ float4 entry_record(const float4* pos, const BoundaryGrid& samples, uint32_t entry) {
    if constexpr (kSamples) {
        if ((entry & kSampleEntry) != 0u) return samples.x[entry & ~kSampleEntry];
    }
    return pos[entry];
}

// What the first walk of a set of positions (lambda, vorticity) does: each
// expanding thread scans its stencil slots at the positions `pos` and writes
// their exact masks. A scan shared by G lanes takes little longer than
// reading masks would, so a step keeps no skin masks. `samples`, with kSamples, lists the boundary samples
// near the particle. pair and fold are group_walk_list's; sum is kept by the
// caller. Returns the walked particle, or ~0u for a lane without one.
template <int G, bool kSamples, int F, class Args, class Load, class Pair, class Fold>
__device__ __forceinline__ uint32_t group_first_walk(const Args& a, const GroupScene& scene, GroupLds<G>& lds,
                                                     uint32_t* crowd, const BoundaryGrid& samples, uint32_t skip,
                                                     Load&& load_record, Pair&& pair, Fold&& fold) {
    constexpr uint32_t kParticles = kGroupParticles<G>;
    constexpr uint32_t kSlots = kGroupSlots<G>;
    const uint32_t expanded = threadIdx.x % kParticles;
    const uint32_t part = threadIdx.x / kParticles;
    const uint32_t i = scene.base + expanded;
    const bool valid = expanded < scene.count;
    if (threadIdx.x < kParticles) crowd[threadIdx.x] = 0u;
    __syncthreads();
    Float3 p{0.0F, 0.0F, 0.0F};
    uint32_t first[kSlots] = {}, last[kSlots] = {};
    [[maybe_unused]] uint32_t sample_first[kSlots] = {}, sample_last[kSlots] = {};
    if (valid) {
        p = xyz(a.pos[i]);
        int cx, cy, cz;
        if (a.first_pass != 0u) {  // at x*, whose cells hold for the step
            particle_cell(scene.grid, p, cx, cy, cz);
            if (part == 0u) a.cell[i] = cell_of(scene.grid, cx, cy, cz);
        } else {
            cell_coordinates(scene.grid, a.cell[i], cx, cy, cz);
        }
        bool crowded = group_ranges<G>(scene.grid, scene.grid.offsets, cx, cy, cz, first, last);
        if constexpr (kSamples)
            crowded = group_ranges<G>(scene.grid, samples.offsets, cx, cy, cz, sample_first, sample_last) || crowded;
        if (crowded) crowd[expanded] = 1u;
    }
    auto near = [&](Float3 from, Float3 to) {
        const Float3 d = sub(from, to);
        return !(dot(d, d) >= a.t_exact);
    };
    const uint32_t walked = threadIdx.x / G;
    const uint32_t w = scene.base + walked;
    const bool active = walked < scene.count;
    group_expand<G, kSamples>(
        lds,
        [&](uint32_t (&bits)[kSlots], uint32_t (&start)[kSlots]) {
#pragma unroll
            for (uint32_t j = 0; j < kSlots; ++j) {
                const uint32_t k = part * kSlots + j;
                start[j] = first[j];
                if (!valid || k >= static_cast<uint32_t>(kStencil)) continue;
                bits[j] = mark_members(a.pos, first[j], last[j], [&](Float3 q) { return near(p, q); });
                a.exact_out[static_cast<size_t>(k) * a.n + i] = static_cast<uint16_t>(bits[j]);
            }
        },
        [&](uint32_t (&bits)[kSlots], uint32_t (&start)[kSlots]) {
#pragma unroll
            for (uint32_t j = 0; j < kSlots; ++j) {
                start[j] = sample_first[j];
                bits[j] = mark_members(samples.x, sample_first[j], sample_last[j],
                                       [&](Float3 q) { return near(p, q); });
            }
        },
        [&](const uint32_t* row, uint32_t count) {
            if (active && crowd[walked] == 0u) group_walk_list<G, F>(row, count, w, load_record, pair, fold);
        });
    if (a.first_pass != 0u && valid && part == 0u) a.crowded[i] = static_cast<uint8_t>(crowd[expanded]);
    if (!active) return ~0u;
    if (crowd[walked] != 0u) {
        const Float3 own = xyz(a.pos[w]);
        int cx, cy, cz;
        if (a.first_pass != 0u) {
            particle_cell(scene.grid, own, cx, cy, cz);
        } else {
            cell_coordinates(scene.grid, a.cell[w], cx, cy, cz);
        }
        group_walk_stencil<G, F>(
            scene.grid, kSamples ? samples.offsets : nullptr, cx, cy, cz, skip, w, group_row(lds),
            [&](uint32_t entry) { return near(own, xyz(entry_record<kSamples>(a.pos, samples, entry))); }, load_record,
            pair, fold);
    }
    return w;
}

// A later walk at the same positions, over the exact masks of the first one;
// the samples near the particle are scanned again. The particle itself is
// left out.
template <int G, bool kSamples, int F, class Args, class Load, class Pair, class Fold>
__device__ __forceinline__ uint32_t group_exact_walk(const Args& a, const GroupScene& scene, GroupLds<G>& lds,
                                                     const BoundaryGrid& samples, float t_exact, Load&& load_record,
                                                     Pair&& pair, Fold&& fold) {
    constexpr uint32_t kParticles = kGroupParticles<G>;
    const uint32_t expanded = threadIdx.x % kParticles;
    const uint32_t i = scene.base + expanded;
    bool listed = false;
    uint32_t center = 0u;
    [[maybe_unused]] Float3 p{0.0F, 0.0F, 0.0F};
    [[maybe_unused]] int x = 0, y = 0, z = 0;
    if (expanded < scene.count) {
        center = a.cell[i];
        listed = a.crowded[i] == 0u;
        if constexpr (kSamples) {
            p = xyz(a.pos[i]);
            cell_coordinates(scene.grid, center, x, y, z);
        }
    }
    const uint32_t walked = threadIdx.x / G;
    const uint32_t w = scene.base + walked;
    const bool active = walked < scene.count;
    group_expand<G, kSamples>(
        lds,
        [&](auto& bits, auto& first) {
            if (listed) stored_slots<G, true>(a.exact, scene.grid, scene.grid.offsets, a.n, i, center, bits, first);
        },
        [&](auto& bits, auto& first) {
            if (!listed) return;
            scanned_slots<G>(scene.grid, samples.offsets, samples.x, x, y, z, bits, first, [&](Float3 q) {
                const Float3 d = sub(p, q);
                return !(dot(d, d) >= t_exact);
            });
        },
        [&](const uint32_t* row, uint32_t count) {
            if (active) group_walk_list<G, F>(row, count, w, load_record, pair, fold);
        });
    if (!active) return ~0u;
    if (a.crowded[w] != 0u) {
        int cx, cy, cz;
        cell_coordinates(scene.grid, a.cell[w], cx, cy, cz);
        const Float3 own = xyz(a.pos[w]);
        group_walk_stencil<G, F>(
            scene.grid, kSamples ? samples.offsets : nullptr, cx, cy, cz, w, w, group_row(lds),
            [&](uint32_t entry) {
                const Float3 d = sub(own, xyz(entry_record<kSamples>(a.pos, samples, entry)));
                return !(dot(d, d) >= t_exact);
            },
            load_record, pair, fold);
    }
    return w;
}

__device__ __forceinline__ void put(float* terms, Float3 v) {
    terms[0] = v.x;
    terms[1] = v.y;
    terms[2] = v.z;
}

// density_forward_kernel (density.cu:18-40, poly6) and lambda_forward_kernel
// (pbf.cu:95-127). With kSamples each cell's boundary samples b add, after
// its particles, rho0_i V_b W to the density and V_b grad W to the gradient
// sum (pbf.cu:118-121).
template <bool kBatch, int G, bool kSamples>
__global__ void __launch_bounds__(kGroupBlock) pbf_lambda_kernel(LambdaArgs a, Schedule schedule, BatchView batch) {
    constexpr int kSums = 5;
    __shared__ GroupLds<G> lds;
    __shared__ uint32_t crowd[kGroupParticles<G>];
    const uint32_t id = scheduled_block(schedule);
    if (id == ~0u) return;
    const GroupScene scene = group_scene<kBatch, G>(id, a.n, a.grid, Box{}, batch);
    const uint32_t own = threadIdx.x / G < scene.count ? scene.base + threadIdx.x / G : 0u;
    const Float3 p = xyz(a.pos[own]);
    const RestDensity rest = rest_density_of(a.rho0[own], *a.unusual_masses != 0u);
    float sum[kSums] = {0.0F, 0.0F, 0.0F, 0.0F, a.eps[own]};
    const uint32_t w = group_first_walk<G, kSamples, kSums>(
        a, scene, lds, crowd, a.boundary, ~0u,
        [&](uint32_t entry) { return entry_record<kSamples>(a.pos, a.boundary, entry); },
        [&](float4 c, uint32_t entry, float (&terms)[kSums]) {
            const Float3 d = sub(p, xyz(c));
            if (kSamples && (entry & kSampleEntry) != 0u) {
                const float d2 = dot(d, d);
                terms[0] = rest.value * c.w * poly6_value(d2, a.k);
                put(terms + 1, scale(scale(d, spiky_factor(d2, a.k)), c.w));
                return;
            }
            const LambdaTerms t = lambda_terms(a, d, c.w, rest);
            terms[0] = t.density;
            if (entry != own) {
                put(terms + 1, t.gradient);
                terms[4] = t.square;
            }
        },
        [&](const float (&terms)[kSums]) { group_add<G, kSums>(sum, terms); });
    if (w != ~0u && threadIdx.x % G == 0u)
        finish_lambda(a, w, rest.value, sum[0], Float3{sum[1], sum[2], sum[3]}, sum[4]);
}

// Candidate records.
struct PointLambda {
    float4 x;
    float lambda;
};
struct PointVector {
    float4 x, v;
};

// v as particle i's record, and in a recorded step as its recorded value.
__device__ __forceinline__ void store_both(float4* records, Vec recorded, uint32_t i, Float3 v) {
    records[i] = make_float4(v.x, v.y, v.z, 0.0F);
    if (recorded.x != nullptr) store(recorded, i, v);
}

struct CorrectionArgs {
    uint32_t n;
    PbfKernel k;
    SortedGrid grid;
    Box box;
    const float4* pos;  // positions and masses
    const float* rho0;
    const float* lambda;
    const float* strength;
    const float* exponent;
    const float* radius;
    float4* out;        // the corrected positions, and the masses
    Vec out_recorded;   // optional (recorded step): the positions
    uint8_t* mask;  // optional (recorded step): box-collision bits of the projection
    uint32_t reconstruct;
    CVec x0;
    float inv_dt;
    float4* vel;       // xyz used
    Vec vel_recorded;  // optional (recorded step)
    const uint16_t* exact;  // exact masks of the positions read
    BoundaryGrid boundary;  // offsets null: no boundary samples
    const uint32_t* cell;   // LambdaArgs::cell and crowded
    const uint8_t* crowded;
    float t_exact;
    const uint32_t* unusual_masses;
};

// The artificial pressure of a particle, as its correction pass evaluates it.
struct ArtificialPressure {
    float strength, exponent, reference;
    bool vanishes;  // with k = +-0 the term is -k wherever W(d) > 0 (no powf per pair)
};
__device__ __forceinline__ ArtificialPressure artificial_of(const CorrectionArgs& a, uint32_t i) {
    ArtificialPressure s{a.strength[i], a.exponent[i], poly6(Float3{a.radius[i], 0.0F, 0.0F}, a.k.h), false};
    s.vanishes = artificial_vanishes(a.k.h, s.strength, s.exponent, s.reference);
    return s;
}
__device__ __forceinline__ float artificial_at(const CorrectionArgs& a, const ArtificialPressure& s, float d2) {
    return s.vanishes ? (poly6_vanishes(d2, a.k) ? 0.0F : -s.strength)
                      : artificial_value(d2, a.k, s.strength, s.exponent, s.reference);
}

// project_forward_kernel (pbf.cu:417-431) of particle i at p with its
// correction.
__device__ __forceinline__ void finish_correction(const CorrectionArgs& a, const Box& box, uint32_t i, float4 self,
                                                  Float3 correction) {
    const Float3 candidate = add(xyz(self), correction);
    if (a.mask != nullptr) {
        uint32_t bits = 0u;
        if (candidate.x < box.lo[0] || candidate.x > box.hi[0]) bits |= 1u;
        if (candidate.y < box.lo[1] || candidate.y > box.hi[1]) bits |= 2u;
        if (candidate.z < box.lo[2] || candidate.z > box.hi[2]) bits |= 4u;
        a.mask[i] = static_cast<uint8_t>(bits);
    }
    const Float3 projected{fminf(box.hi[0], fmaxf(box.lo[0], candidate.x)),
                           fminf(box.hi[1], fmaxf(box.lo[1], candidate.y)),
                           fminf(box.hi[2], fmaxf(box.lo[2], candidate.z))};
    a.out[i] = make_float4(projected.x, projected.y, projected.z, self.w);
    if (a.out_recorded.x != nullptr) store(a.out_recorded, i, projected);
    if (a.reconstruct != 0u) store_both(a.vel, a.vel_recorded, i, scale(sub(projected, load(a.x0, i)), a.inv_dt));
}

// correction_forward_kernel (pbf.cu:254-288) and project_forward_kernel. With
// kSamples a boundary sample b adds V_b (lambda_i + s_corr(d)) grad W after
// each cell's particles (pbf.cu:278-284).
template <bool kBatch, int G, bool kSamples>
__global__ void __launch_bounds__(kGroupBlock) pbf_correction_kernel(CorrectionArgs a, Schedule schedule, BatchView batch) {
    constexpr int kSums = 3;
    __shared__ GroupLds<G> lds;
    const uint32_t id = scheduled_block(schedule);
    if (id == ~0u) return;
    const GroupScene scene = group_scene<kBatch, G>(id, a.n, a.grid, a.box, batch);
    const uint32_t own = threadIdx.x / G < scene.count ? scene.base + threadIdx.x / G : 0u;
    const float4 self = a.pos[own];
    const Float3 p = xyz(self);
    const RestDensity rest = rest_density_of(a.rho0[own], *a.unusual_masses != 0u);
    const float lambda_i = a.lambda[own];
    const ArtificialPressure pressure = artificial_of(a, own);
    float sum[kSums] = {0.0F, 0.0F, 0.0F};
    const uint32_t w = group_exact_walk<G, kSamples, kSums>(
        a, scene, lds, a.boundary, a.t_exact,
        [&](uint32_t entry) {
            const bool sample = kSamples && (entry & kSampleEntry) != 0u;
            return PointLambda{entry_record<kSamples>(a.pos, a.boundary, entry), sample ? 0.0F : a.lambda[entry]};
        },
        [&](const PointLambda& c, uint32_t entry, float (&terms)[kSums]) {
            const Float3 d = sub(p, xyz(c.x));
            const float d2 = dot(d, d);
            const float artificial = artificial_at(a, pressure, d2);
            const float factor = kSamples && (entry & kSampleEntry) != 0u
                                     ? c.x.w * (lambda_i + artificial)
                                     : over_rest(c.x.w, rest) * (lambda_i + c.lambda + artificial);
            put(terms, scale(scale(d, spiky_factor(d2, a.k)), factor));
        },
        [&](const float (&terms)[kSums]) { group_add<G, kSums>(sum, terms); });
    if (w != ~0u && threadIdx.x % G == 0u)
        finish_correction(a, scene.box, w, self, Float3{sum[0], sum[1], sum[2]});
}

__global__ void __launch_bounds__(kBlock) pbf_reconstruct_kernel(uint32_t n, const float4* pos, CVec x0, float inv_dt,
                                                                 float4* vel, Vec recorded) {
    const uint32_t i = xcd_block() * kBlock + threadIdx.x;
    if (i >= n) return;
    store_both(vel, recorded, i, scale(sub(xyz(pos[i]), load(x0, i)), inv_dt));
}

struct PostArgs {
    uint32_t n;
    PbfKernel k;
    float dt;
    SortedGrid grid;
    const float4* pos;  // positions and masses
    const float4* vel;  // xyz used
    Vec vort;
    float* magnitude;
    float4* pos_magnitude;  // the normal pass's candidate records: position and |omega|
    const float* confinement;
    float4* vc;        // xyz used
    Vec vc_recorded;   // optional (recorded step)
    Vec normals;         // optional (recorded step)
    float* normalizers;  // optional (recorded step)
    const float* xsph;
    const uint32_t* perm;
    Vec next_x, next_v;
    // exact masks of the final positions: written by the vorticity pass and
    // walked by the normal and XSPH passes
    float t_exact;
    uint16_t* exact_out;
    const uint16_t* exact;
    // LambdaArgs::cell, crowded and first_pass
    uint32_t* cell;
    uint8_t* crowded;
    uint32_t first_pass;
};

__device__ __forceinline__ void finish_vorticity(const PostArgs& a, uint32_t i, Float3 p, Float3 w) {
    store(a.vort, i, w);
    const float magnitude = length(w);
    a.magnitude[i] = magnitude;
    a.pos_magnitude[i] = make_float4(p.x, p.y, p.z, magnitude);
}

__device__ __forceinline__ void finish_normal(const PostArgs& a, uint32_t i, Float3 g) {
    const float normalizer = length(g);
    const Float3 normal = normalizer > 0.0F ? scale(g, 1.0F / normalizer) : Float3{0.0F, 0.0F, 0.0F};
    if (a.normalizers != nullptr) {
        a.normalizers[i] = normalizer;
        store(a.normals, i, normal);
    }
    const Float3 w = load(CVec{a.vort.x, a.vort.y, a.vort.z}, i);
    store_both(a.vc, a.vc_recorded, i, add(xyz(a.vel[i]), scale(cross(normal, w), a.dt * a.confinement[i])));
}

__device__ __forceinline__ void finish_xsph(const PostArgs& a, uint32_t i, Float3 p, Float3 v, Float3 smoothing) {
    const uint32_t j = a.perm[i];
    store(a.next_v, j, add(v, scale(smoothing, a.xsph[i])));
    store(a.next_x, j, p);
}

template <bool kBatch, int G>
__global__ void __launch_bounds__(kGroupBlock) pbf_vorticity_kernel(PostArgs a, Schedule schedule, BatchView batch) {
    constexpr int kSums = 3;
    __shared__ GroupLds<G> lds;
    __shared__ uint32_t crowd[kGroupParticles<G>];
    const uint32_t id = scheduled_block(schedule);
    if (id == ~0u) return;
    const GroupScene scene = group_scene<kBatch, G>(id, a.n, a.grid, Box{}, batch);
    const uint32_t own = threadIdx.x / G < scene.count ? scene.base + threadIdx.x / G : 0u;
    const Float3 p = xyz(a.pos[own]);
    const Float3 v = xyz(a.vel[own]);
    float sum[kSums] = {0.0F, 0.0F, 0.0F};
    const uint32_t w = group_first_walk<G, false, kSums>(
        a, scene, lds, crowd, BoundaryGrid{}, own,
        [&](uint32_t s) { return PointVector{a.pos[s], a.vel[s]}; },
        [&](const PointVector& c, uint32_t s, float (&terms)[kSums]) {
            const Float3 d = sub(p, xyz(c.x));
            if (s != own) put(terms, cross(sub(xyz(c.v), v), scale(d, spiky_factor(dot(d, d), a.k))));
        },
        [&](const float (&terms)[kSums]) { group_add<G, kSums>(sum, terms); });
    if (w != ~0u && threadIdx.x % G == 0u) finish_vorticity(a, w, p, Float3{sum[0], sum[1], sum[2]});
}

template <bool kBatch, int G>
__global__ void __launch_bounds__(kGroupBlock) pbf_normal_kernel(PostArgs a, Schedule schedule, BatchView batch) {
    constexpr int kSums = 3;
    __shared__ GroupLds<G> lds;
    const uint32_t id = scheduled_block(schedule);
    if (id == ~0u) return;
    const GroupScene scene = group_scene<kBatch, G>(id, a.n, a.grid, Box{}, batch);
    const uint32_t own = threadIdx.x / G < scene.count ? scene.base + threadIdx.x / G : 0u;
    const float4 self = a.pos_magnitude[own];
    const Float3 p = xyz(self);
    const float mag_i = self.w;
    float sum[kSums] = {0.0F, 0.0F, 0.0F};
    const uint32_t w = group_exact_walk<G, false, kSums>(
        a, scene, lds, BoundaryGrid{}, a.t_exact,
        [&](uint32_t s) { return a.pos_magnitude[s]; },
        [&](float4 c, uint32_t, float (&terms)[kSums]) {
            const Float3 d = sub(p, xyz(c));
            put(terms, scale(scale(d, spiky_factor(dot(d, d), a.k)), c.w - mag_i));
        },
        [&](const float (&terms)[kSums]) { group_add<G, kSums>(sum, terms); });
    if (w != ~0u && threadIdx.x % G == 0u) finish_normal(a, w, Float3{sum[0], sum[1], sum[2]});
}

template <bool kBatch, int G>
__global__ void __launch_bounds__(kGroupBlock) pbf_xsph_kernel(PostArgs a, Schedule schedule, BatchView batch) {
    constexpr int kSums = 3;
    __shared__ GroupLds<G> lds;
    const uint32_t id = scheduled_block(schedule);
    if (id == ~0u) return;
    const GroupScene scene = group_scene<kBatch, G>(id, a.n, a.grid, Box{}, batch);
    const uint32_t own = threadIdx.x / G < scene.count ? scene.base + threadIdx.x / G : 0u;
    const Float3 p = xyz(a.pos[own]);
    const Float3 v = xyz(a.vc[own]);
    float sum[kSums] = {0.0F, 0.0F, 0.0F};
    const uint32_t w = group_exact_walk<G, false, kSums>(
        a, scene, lds, BoundaryGrid{}, a.t_exact,
        [&](uint32_t s) { return PointVector{a.pos[s], a.vc[s]}; },
        [&](const PointVector& c, uint32_t, float (&terms)[kSums]) {
            const Float3 d = sub(p, xyz(c.x));
            put(terms, scale(sub(xyz(c.v), v), poly6_value(dot(d, d), a.k)));
        },
        [&](const float (&terms)[kSums]) { group_add<G, kSums>(sum, terms); });
    if (w != ~0u && threadIdx.x % G == 0u) finish_xsph(a, w, p, v, Float3{sum[0], sum[1], sum[2]});
}

// Lanes per particle of a step's passes.
inline int pbf_group(uint32_t n) { return n <= kGroup16Particles ? 16 : 4; }

// Workgroups of a pass over n particles, padded to a multiple of the XCD count.
inline uint32_t pbf_blocks(uint32_t n, int group) {
    return (blocks_for(n, kBlock / static_cast<uint32_t>(group)) + 7u) / 8u * 8u;
}

// The launches of a step's passes with `group` lanes per particle over
// `blocks` blocks (the schedule's early ones included).
template <bool kBatch>
struct PassLauncher {
    int group;
    uint32_t blocks;
    hipStream_t stream;
    Schedule schedule;
    BatchView batch;

    // launch(std::integral_constant<int, G>) with G the launch's group
    template <class Launch>
    void with_group(Launch&& launch) const {
        if (group == 16) {
            launch(std::integral_constant<int, 16>{});
        } else {
            launch(std::integral_constant<int, 4>{});
        }
        PHX_LAUNCH_CHECK();
    }
    void lambda(const LambdaArgs& a) const {
        with_group([&](auto g) {
            if constexpr (!kBatch) {
                if (a.boundary.offsets != nullptr) {
                    pbf_lambda_kernel<false, g(), true><<<blocks, kGroupBlock, 0, stream>>>(a, schedule, batch);
                    return;
                }
            }
            pbf_lambda_kernel<kBatch, g(), false><<<blocks, kGroupBlock, 0, stream>>>(a, schedule, batch);
        });
    }
    void correction(const CorrectionArgs& a) const {
        with_group([&](auto g) {
            if constexpr (!kBatch) {
                if (a.boundary.offsets != nullptr) {
                    pbf_correction_kernel<false, g(), true><<<blocks, kGroupBlock, 0, stream>>>(a, schedule, batch);
                    return;
                }
            }
            pbf_correction_kernel<kBatch, g(), false><<<blocks, kGroupBlock, 0, stream>>>(a, schedule, batch);
        });
    }
    void vorticity(const PostArgs& a) const {
        with_group([&](auto g) { pbf_vorticity_kernel<kBatch, g()><<<blocks, kGroupBlock, 0, stream>>>(a, schedule, batch); });
    }
    void normal(const PostArgs& a) const {
        with_group([&](auto g) { pbf_normal_kernel<kBatch, g()><<<blocks, kGroupBlock, 0, stream>>>(a, schedule, batch); });
    }
    void xsph(const PostArgs& a) const {
        with_group([&](auto g) { pbf_xsph_kernel<kBatch, g()><<<blocks, kGroupBlock, 0, stream>>>(a, schedule, batch); });
    }
};

}  // namespace

const char* pbf_pass_name(int pass) {
    static const char* names[kPbfPassCount] = {"grid",      "mask",               "density_lambda",
                                               "correction_project", "vorticity", "normal_confinement",
                                               "xsph",      "jvp",                "vjp"};
    return pass >= 0 && pass < kPbfPassCount ? names[pass] : "unknown";
}

double pbf_pass_bytes(int pass, uint32_t particles, uint32_t cells) {
    const double offsets = particles > 0 ? 4.0 * (static_cast<double>(cells) + 1.0) / particles : 0.0;
    switch (pass) {
        case kPbfGrid:  // x, v, u in, x* out (original order); x*, x + 8 parameters gathered; permutation
            return 36.0 + 12.0 + 2.0 * (24.0 + 32.0) + 4.0 + 2.0 * offsets;
        case kPbfMask:  // x* in (the masks are an acceleration structure)
            return 12.0 + offsets;
        case kPbfLambda:  // x*, p, m, rho0, eps in; rho, lambda out
            return 36.0 + 8.0 + offsets;
        case kPbfCorrection:  // x*, p, m, rho0, lambda, s_corr k, n, dq in; p' out (+ x in, v out on the last)
            return 48.0 + 12.0 + offsets;
        case kPbfVorticity:  // x*, p, v in; omega, |omega| out
            return 36.0 + 16.0 + offsets;
        case kPbfNormal:  // x*, p, |omega|, omega, v, confinement in; v_c out
            return 56.0 + 12.0 + offsets;
        case kPbfXsph:  // x*, p, v_c, xsph in; next x, v out + permutation
            return 40.0 + 24.0 + 4.0 + offsets;
        case kPbfJvp:  // whole-step passes, not a single roofline figure
        case kPbfVjp:
            return 0.0;
        default:
            return 0.0;
    }
}

PbfKernel pbf_kernel(float h) {
    PbfKernel k{};
    k.h = h;
    k.hr = h * h;
    k.spiky = spiky_coefficient(h);
    k.poly6 = 64.0F * kPi * k.hr * k.hr * k.hr * h * h * h;
    k.plain = h >= 0x1p-11F && h <= 0x1p8F ? 0u : 1u;
    if (k.plain == 0u) {
        int exponent = 0;
        (void)std::frexp(k.poly6, &exponent);
        k.scale = std::ldexp(1.0F, 1 - exponent);
        k.poly6_scaled = k.poly6 * k.scale;
        k.inv_poly6 = 1.0F / k.poly6_scaled;
    }
    return k;
}

void PbfCache::allocate(uint32_t n, uint32_t cells, uint32_t pressure_iterations) {
    neighborhood.allocate(n, cells);
    predicted.resize(n);
    densities.resize(n);
    lambdas.resize(n);
    magnitudes.resize(n);  // StepCache::vorticity_magnitudes (pbf/pbf.ixx:67)
    if (!record) return;
    const size_t per = static_cast<size_t>(pressure_iterations) * n;
    for (VecBuffer* b : {&xs, &x0, &velocities, &vorticities, &normals, &confined}) b->resize(n);
    positions.resize(n, pressure_iterations);
    gradient_sums.resize(n, pressure_iterations);
    rho.resize(per);
    lambda.resize(per);
    den.resize(per);
    masks.resize(per);
    normalizers.resize(n);
    crowded.resize(n);
    exact_masks.resize(static_cast<size_t>(pressure_iterations + 1u) * kStencil * n);
}

PbfSolver::PbfSolver(const phx_domain_configuration* domain, const phx_pbf_configuration* configuration,
                     phx_execution_mode mode, hipStream_t stream)
    : domain_(make_domain(domain)), mode_(mode), stream_(stream) {
    require(configuration != nullptr, PHX_ERROR_INVALID_ARGUMENT, "null PBF configuration");

    config_ = *configuration;
    require(config_.checkpoint_interval > 0u, PHX_ERROR_INVALID_ARGUMENT, "checkpoint_interval must be positive");
    require(mode == PHX_MODE_FORWARD || mode == PHX_MODE_DIFFERENTIABLE, PHX_ERROR_INVALID_ARGUMENT,
            "unknown execution mode");
    boundary_.upload(domain_.config);
    domain_.config.boundary_particles = nullptr;  // the caller's host array is not kept
    spiky_ = spiky_coefficient(domain_.config.support_radius);
    kernel_ = pbf_kernel(domain_.config.support_radius);
    const uint32_t n = domain_.config.particle_count;
    for (VecBuffer* b : {&x0_, &vort_}) b->resize(n);
    for (DeviceBuffer<float4>* b : {&vel_, &vc_, &pos_magnitude_}) b->resize(n);
    for (DeviceBuffer<float4>* b : {&xs_, &pa_, &pb_}) b->resize(n + static_cast<size_t>(kScanPadding));
    for (DeviceBuffer<float>* b : {&rho0_, &eps_, &strength_, &exponent_, &radius_, &xsph_, &confinement_})
        b->resize(n);
    exact_.resize(static_cast<size_t>(kStencil) * n);
    crowded_.resize(n);
    mass_flag_.resize(1u);
    cells_.resize(n);
    if (n >= kEarlyParticles)
        schedule_.resize(1u + kEarlyBlocks + 2u * static_cast<size_t>(pbf_blocks(n, pbf_group(n))));
}

void PbfSolver::forward_step(const phx_pbf_state& state, const phx_control& control,
                             const phx_pbf_parameters& parameters, phx_pbf_state& next, PbfCache& cache) {
    const auto& c = domain_.config;
    const uint32_t n = c.particle_count;
    const uint64_t step = state.particles.step_index;
    if (n == 0) {
        next.particles.step_index = step + 1u;
        return;
    }
    require_vec(state.particles.positions, "state positions");
    require_vec(state.particles.velocities, "state velocities");
    require_vec(control.external_accelerations, "control");
    require_vec(next.particles.positions, "next positions");
    require_vec(next.particles.velocities, "next velocities");
    const auto& pp = parameters.particles;
    require(pp.masses && pp.rest_densities, PHX_ERROR_INVALID_ARGUMENT, "null particle parameters");
    require(parameters.relaxation && parameters.artificial_pressure_strength && parameters.artificial_pressure_exponent &&
                parameters.artificial_pressure_radius && parameters.xsph_viscosity && parameters.vorticity_confinement,
            PHX_ERROR_INVALID_ARGUMENT, "null PBF parameters");
    cache.record = mode_ == PHX_MODE_DIFFERENTIABLE;
    cache.recorded = false;
    cache.allocate(n, domain_.cells, config_.pressure_iterations);
    const bool rec = cache.record;
    // recorded quantities live in the cache, the others in the workspace
    VecBuffer& x0 = rec ? cache.x0 : x0_;
    VecBuffer& vort = rec ? cache.vorticities : vort_;
    float* magnitude = cache.magnitudes.data();

    // predict (pbf.cu:73-78) fused into the key pass of build(step + 1, x*)
    PredictInput predict{};
    predict.velocities = cvec(state.particles.velocities);
    predict.controls = cvec(control.external_accelerations);
    predict.gravity = Float3{c.gravity.x, c.gravity.y, c.gravity.z};
    predict.dt = c.time_step;
    predict.predicted = cache.predicted.view();
    predict.mass_flag = mass_flag_.data();
    ChannelList gather;
    gather.check_masses(pp.masses, mass_flag_.data());
    gather.add(cache.predicted.cview(), xs_.data());
    gather.add(pp.masses, xs_.data(), 3);
    if (rec) gather.add(cache.predicted.cview(), cache.xs.view());
    gather.add(cvec(state.particles.positions), x0.view());
    gather.add(pp.rest_densities, rho0_.data());
    gather.add(parameters.relaxation, eps_.data());
    gather.add(parameters.artificial_pressure_strength, strength_.data());
    gather.add(parameters.artificial_pressure_exponent, exponent_.data());
    gather.add(parameters.artificial_pressure_radius, radius_.data());
    gather.add(parameters.xsph_viscosity, xsph_.data());
    gather.add(parameters.vorticity_confinement, confinement_.data());
    {
        PassScope scope(profiler_, stream_, kPbfGrid);
        cache.neighborhood.build(stream_, domain_, step + 1u, cvec(state.particles.positions), &predict,
                                 gather.get(), &boundary_);
    }

    const SortedGrid grid = cache.neighborhood.grid();
    const BoundaryGrid boundary = cache.neighborhood.boundary();
    const int group = pbf_group(n);
    // a large scene serves workgroups with crowded particles first; its cells
    // are then found by a launch of their own
    const bool ordered = n >= kEarlyParticles;
    const uint32_t group_blocks = pbf_blocks(n, group);
    Schedule schedule{};
    if (ordered) {
        schedule = Schedule{schedule_.data(), schedule_.data() + 1u, schedule_.data() + 1u + kEarlyBlocks,
                            schedule_.data() + 1u + kEarlyBlocks + group_blocks, kEarlyBlocks};
    }
    const PassLauncher<false> launch{group, group_blocks + schedule.early, stream_, schedule, BatchView{}};
    const float h = c.support_radius;
    const float inv_dt = 1.0F / c.time_step;
    // a recorded step keeps its exact masks for its derivative passes
    uint8_t* crowded = rec ? cache.crowded.data() : crowded_.data();
    if (ordered) {
        PassScope scope(profiler_, stream_, kPbfMask);
        fill_u32(stream_, schedule_.data(), schedule_.size(), 0u);
        pbf_cell_kernel<false><<<pbf_blocks(n, 1), kBlock, 0, stream_>>>(
            n, grid, boundary.offsets, xs_.data(), cells_.data(), crowded, kBlock / static_cast<uint32_t>(group),
            schedule, BatchView{});
        PHX_LAUNCH_CHECK();
    }
    // exact masks of position set k (iterate k, the final positions last):
    // written by the pass that first walks those positions, walked by the
    // later passes at them; a recorded step keeps every set
    const float t_exact = exact_mask_threshold(h);
    const uint32_t sets = config_.pressure_iterations + 1u;
    auto exact_set = [&](uint32_t k) {
        require(k < sets, PHX_ERROR_INVALID_ARGUMENT, "exact mask set out of range");
        return rec ? cache.exact_masks.data() + static_cast<size_t>(k) * kStencil * n : exact_.data();
    };

    LambdaArgs la{n,           kernel_,     grid,
                  xs_.data(),  rho0_.data(), eps_.data(),
                  cache.densities.data(), cache.lambdas.data()};
    la.t_exact = t_exact;
    la.unusual_masses = mass_flag_.data();
    la.boundary = boundary;
    la.cell = cells_.data();
    la.crowded = crowded;
    CorrectionArgs ca{};
    ca.n = n;
    ca.k = kernel_;
    ca.grid = grid;
    ca.box = collision_box(c, step + 1u);
    ca.rho0 = rho0_.data();
    ca.lambda = cache.lambdas.data();
    ca.strength = strength_.data();
    ca.exponent = exponent_.data();
    ca.radius = radius_.data();
    ca.x0 = x0.cview();
    ca.inv_dt = inv_dt;
    ca.vel = vel_.data();
    if (rec) ca.vel_recorded = cache.velocities.view();
    ca.boundary = boundary;
    ca.cell = cells_.data();
    ca.crowded = crowded;
    ca.t_exact = t_exact;
    ca.unusual_masses = mass_flag_.data();

    // positions start at x* (pbf.cpp:171) and ping-pong between two buffers
    // (a recorded step keeps every iterate)
    const float4* current = xs_.data();
    DeviceBuffer<float4>* targets[2] = {&pa_, &pb_};
    const uint32_t iterations = config_.pressure_iterations;
    for (uint32_t it = 0; it < iterations; ++it) {
        la.pos = current;
        la.first_pass = it == 0u && !ordered ? 1u : 0u;
        la.exact_out = exact_set(it);
        ca.exact = exact_set(it);
        if (rec) {
            const size_t off = static_cast<size_t>(it) * n;
            la.rho = cache.rho.data() + off;
            la.lambda = cache.lambda.data() + off;
            la.den = cache.den.data() + off;
            la.gsum = cache.gradient_sums.view(it);
            ca.lambda = la.lambda;
            ca.mask = cache.masks.data() + off;
        }
        {
            PassScope scope(profiler_, stream_, kPbfLambda);
            launch.lambda(la);
        }
        float4* target = targets[it & 1u]->data();
        ca.pos = current;
        ca.out = target;
        if (rec) ca.out_recorded = cache.positions.view(it);
        ca.reconstruct = it + 1u == iterations ? 1u : 0u;
        {
            PassScope scope(profiler_, stream_, kPbfCorrection);
            launch.correction(ca);
        }
        current = target;
    }
    if (rec && iterations > 0u) {
        // the cache's densities and lambdas are those of the last iteration
        const size_t off = static_cast<size_t>(iterations - 1u) * n;
        PHX_HIP(hipMemcpyAsync(cache.densities.data(), cache.rho.data() + off, sizeof(float) * n,
                               hipMemcpyDeviceToDevice, stream_));
        PHX_HIP(hipMemcpyAsync(cache.lambdas.data(), cache.lambda.data() + off, sizeof(float) * n,
                               hipMemcpyDeviceToDevice, stream_));
    }
    if (iterations == 0u) {
        pbf_reconstruct_kernel<<<pbf_blocks(n, 1), kBlock, 0, stream_>>>(n, current, x0.cview(), inv_dt, vel_.data(),
                                                                             rec ? cache.velocities.view() : Vec{});
        PHX_LAUNCH_CHECK();
    }

    PostArgs post{};
    post.n = n;
    post.k = kernel_;
    post.dt = c.time_step;
    post.grid = grid;
    post.pos = current;
    post.vel = vel_.data();
    post.pos_magnitude = pos_magnitude_.data();
    post.vort = vort.view();
    post.magnitude = magnitude;
    post.confinement = confinement_.data();
    post.vc = vc_.data();
    if (rec) {
        post.vc_recorded = cache.confined.view();
        post.normals = cache.normals.view();
        post.normalizers = cache.normalizers.data();
    }
    post.xsph = xsph_.data();
    post.perm = cache.neighborhood.perm.data();
    post.t_exact = t_exact;
    post.exact_out = exact_set(iterations);
    post.exact = exact_set(iterations);
    post.cell = cells_.data();
    post.crowded = crowded;
    post.first_pass = iterations == 0u && !ordered ? 1u : 0u;
    post.next_x = vec(next.particles.positions);
    post.next_v = vec(next.particles.velocities);
    {
        PassScope scope(profiler_, stream_, kPbfVorticity);
        launch.vorticity(post);
    }
    {
        PassScope scope(profiler_, stream_, kPbfNormal);
        launch.normal(post);
    }
    {
        PassScope scope(profiler_, stream_, kPbfXsph);
        launch.xsph(post);
    }
    if (rec) {
        cache.recorded = true;
        cache.iterations = iterations;
        cache.step_index = step;
    }
    next.particles.step_index = step + 1u;
}

}  // namespace phx

namespace phx {

// ------------------------------------------------------------------ batch
PbfBatch::PbfBatch(const phx_domain_configuration* domains, uint32_t scene_count,
                   const phx_pbf_configuration* configuration, const phx_pbf_batch_configuration* batch_configuration,
                   hipStream_t stream)
    : caller_(stream) {
    require(domains != nullptr && scene_count > 0u, PHX_ERROR_INVALID_ARGUMENT, "a batch needs at least one scene");
    require(configuration != nullptr, PHX_ERROR_INVALID_ARGUMENT, "null PBF configuration");
    config_ = *configuration;
    require(config_.pressure_iterations < 1024u, PHX_ERROR_INVALID_ARGUMENT, "too many pressure iterations");
    if (batch_configuration != nullptr) {
        // accepted as before; the passes keep no skin masks that it would size
        const float skin = batch_configuration->mask_skin;
        require(skin == 0.0F || (skin >= 0.01F && skin <= 1.0F), PHX_ERROR_INVALID_ARGUMENT,
                "mask_skin must be 0 (default) or in [0.01, 1]");
        use_graph_ = batch_configuration->use_graph != 0u;
    }
    uint64_t particles = 0, cells = 0;
    offsets_.push_back(0u);
    for (uint32_t k = 0; k < scene_count; ++k) {
        const Domain d = make_domain(&domains[k]);
        const auto& c = d.config;
        require(c.boundary_particle_count == 0u, PHX_ERROR_UNSUPPORTED, "batched scenes take no boundary particles");
        if (k == 0u) {
            h_ = c.support_radius;
            dt_ = c.time_step;
        }
        require(c.support_radius == h_ && c.time_step == dt_, PHX_ERROR_INVALID_ARGUMENT,
                "the scenes of a batch share the support radius and time step");
        BatchScene s{};
        s.cell_base = static_cast<uint32_t>(cells);
        for (int a = 0; a < 3; ++a) s.res[a] = d.resolution[a];
        s.minimum[0] = c.boundary.minimum.x;
        s.minimum[1] = c.boundary.minimum.y;
        s.minimum[2] = c.boundary.minimum.z;
        s.maximum[0] = c.boundary.maximum.x;
        s.maximum[1] = c.boundary.maximum.y;
        s.maximum[2] = c.boundary.maximum.z;
        s.velocity[0] = c.boundary.velocity.x;
        s.velocity[1] = c.boundary.velocity.y;
        s.velocity[2] = c.boundary.velocity.z;
        s.particle_radius = c.particle_radius;
        s.gravity[0] = c.gravity.x;
        s.gravity[1] = c.gravity.y;
        s.gravity[2] = c.gravity.z;
        s.no_slip = c.boundary.no_slip != 0u ? 1u : 0u;
        if (s.velocity[0] != 0.0F || s.velocity[1] != 0.0F || s.velocity[2] != 0.0F) static_boxes_ = false;
        scenes_.push_back(s);
        cells += d.cells;
        particles += c.particle_count;
        offsets_.push_back(particles);
    }
    require(particles < (1ull << 31) && cells < (1ull << 31), PHX_ERROR_CAPACITY, "batch too large");
    n_ = static_cast<uint32_t>(particles);
    cells_ = static_cast<uint32_t>(cells);
    // a captured substep bakes in the step time, which moving boxes change
    use_graph_ = use_graph_ && static_boxes_;
    kernel_ = pbf_kernel(h_);

    // workgroup tables: each scene's particles in blocks of kBlock (the grid
    // build) and of the passes' workgroups, padded to a multiple of the XCD count
    group_ = pbf_group(n_);
    const uint32_t group_particles = kBlock / static_cast<uint32_t>(group_);
    auto build_table = [&](uint32_t size, DeviceBuffer<BatchBlock>& device) {
        std::vector<BatchBlock> table;
        uint32_t scene_block = 0u;  // the scene's first workgroup of the passes
        for (uint32_t k = 0; k < scene_count; ++k) {
            for (uint64_t first = offsets_[k]; first < offsets_[k + 1]; first += size) {
                const uint64_t count = std::min<uint64_t>(size, offsets_[k + 1] - first);
                const auto within = static_cast<uint32_t>((first - offsets_[k]) / group_particles);
                table.push_back(
                    BatchBlock{k, static_cast<uint32_t>(first), static_cast<uint32_t>(count), scene_block + within});
            }
            scene_block += blocks_for(offsets_[k + 1] - offsets_[k], group_particles);
        }
        while (table.empty() || table.size() % 8u != 0u) table.push_back(BatchBlock{0u, 0u, 0u, 0u});
        device.resize(table.size());
        PHX_HIP(hipMemcpy(device.data(), table.data(), sizeof(BatchBlock) * table.size(), hipMemcpyHostToDevice));
        return static_cast<uint32_t>(table.size());
    };
    blocks_ = build_table(kBlock, block_table_);
    pass_blocks_ = build_table(group_particles, pass_table_);
    schedule_.resize(1u + kEarlyBlocks);
    for (DeviceBuffer<uint32_t>* b : {&schedule_place_, &schedule_seen_}) b->resize(pass_blocks_);
    scene_table_.resize(scenes_.size());
    PHX_HIP(hipMemcpy(scene_table_.data(), scenes_.data(), sizeof(BatchScene) * scenes_.size(),
                      hipMemcpyHostToDevice));

    const uint32_t n = n_;
    grid_.allocate(n, cells_);
    for (VecBuffer* b :
         {&positions_[0], &positions_[1], &velocities_[0], &velocities_[1], &predicted_, &x0_, &vort_})
        b->resize(n);
    for (DeviceBuffer<float4>* b : {&vel_, &vc_, &pos_magnitude_}) b->resize(n);
    for (DeviceBuffer<float4>* b : {&xs_, &pa_, &pb_}) b->resize(n + static_cast<size_t>(kScanPadding));
    for (DeviceBuffer<float>* b :
         {&rho0_, &eps_, &strength_, &exponent_, &radius_, &xsph_, &confinement_, &rho_, &lambda_, &magnitude_})
        b->resize(n);
    exact_.resize(static_cast<size_t>(kStencil) * n);
    crowded_.resize(n);
    mass_flag_.resize(1u);
    cell_index_.resize(n);
    // grid build 9, schedule fills 3, cells 1, two per iteration, three post passes
    const uint32_t it = config_.pressure_iterations;
    kernels_per_step_ = 9u + 3u + 1u + 2u * it + (it == 0u ? 1u : 0u) + 3u;
    PHX_HIP(hipStreamCreateWithFlags(&stream_, hipStreamNonBlocking));
    PHX_HIP(hipEventCreateWithFlags(&ready_, hipEventDisableTiming));
    PHX_HIP(hipEventCreateWithFlags(&done_, hipEventDisableTiming));
}

PbfBatch::~PbfBatch() {
    if (stream_ != nullptr) (void)hipStreamSynchronize(stream_);
    release_graphs();
    if (ready_ != nullptr) (void)hipEventDestroy(ready_);
    if (done_ != nullptr) (void)hipEventDestroy(done_);
    if (stream_ != nullptr) (void)hipStreamDestroy(stream_);
}

void PbfBatch::release_graphs() {
    for (hipGraphExec_t& g : graph_) {
        if (g != nullptr) (void)hipGraphExecDestroy(g);
        g = nullptr;
    }
    captured_inputs_.clear();
}

// One forward step of every scene from state_[from] into state_[1 - from]:
// the pass sequence of PbfSolver::forward_step in forward mode, each pass
// one launch over the batch's workgroup table.
void PbfBatch::substep(uint32_t from, uint64_t step, const phx_control& control,
                       const phx_pbf_parameters& parameters) {
    const uint32_t n = n_;
    const hipStream_t s = stream_;
    const VecBuffer& x = positions_[from];
    const VecBuffer& v = velocities_[from];
    VecBuffer& next_x = positions_[1u - from];
    VecBuffer& next_v = velocities_[1u - from];
    const auto& pp = parameters.particles;
    BatchView bv{block_table_.data(), scene_table_.data(), static_cast<float>(step + 1u) * dt_, h_};
    kernels_per_step_ = 0u;

    PredictInput predict{};
    predict.velocities = v.cview();
    predict.controls = cvec(control.external_accelerations);
    predict.dt = dt_;
    predict.predicted = predicted_.view();
    predict.mass_flag = mass_flag_.data();
    ChannelList gather;
    gather.check_masses(pp.masses, mass_flag_.data());
    gather.add(predicted_.cview(), xs_.data());
    gather.add(pp.masses, xs_.data(), 3);
    gather.add(x.cview(), x0_.view());
    gather.add(pp.rest_densities, rho0_.data());
    gather.add(parameters.relaxation, eps_.data());
    gather.add(parameters.artificial_pressure_strength, strength_.data());
    gather.add(parameters.artificial_pressure_exponent, exponent_.data());
    gather.add(parameters.artificial_pressure_radius, radius_.data());
    gather.add(parameters.xsph_viscosity, xsph_.data());
    gather.add(parameters.vorticity_confinement, confinement_.data());
    build_batch_grid(s, n, cells_, blocks_, bv, x.cview(), predict, gather.get(), grid_.scratch, grid_.perm.data(),
                     grid_.offsets.data());
    kernels_per_step_ += 9u;  // counts fill, key, three scan kernels, scatter, rank, big-cell sort, gather
    const Schedule schedule{schedule_.data(), schedule_.data() + 1u, schedule_place_.data(), schedule_seen_.data(),
                            kEarlyBlocks};
    const PassLauncher<true> launch{group_, pass_blocks_ + kEarlyBlocks, s, schedule,
                                    BatchView{pass_table_.data(), scene_table_.data(), bv.time, h_}};
    fill_u32(s, schedule_.data(), schedule_.size(), 0u);
    fill_u32(s, schedule_place_.data(), pass_blocks_, 0u);
    fill_u32(s, schedule_seen_.data(), pass_blocks_, 0u);
    kernels_per_step_ += 3u;
    // the batch's offsets; each lane's grid starts at its scene's cell base
    const SortedGrid grid{grid_.offsets.data(), 0u, 0u, 0u, 0.0F, 0.0F, 0.0F, h_};
    pbf_cell_kernel<true><<<blocks_, kBlock, 0, s>>>(n, grid, nullptr, xs_.data(), cell_index_.data(), crowded_.data(),
                                                     kBlock / static_cast<uint32_t>(group_), schedule, bv);
    PHX_LAUNCH_CHECK();
    ++kernels_per_step_;
    const float t_exact = exact_mask_threshold(h_);

    LambdaArgs la{n,           kernel_,     grid, xs_.data(), rho0_.data(),
                  eps_.data(), rho_.data(), lambda_.data()};
    la.t_exact = t_exact;
    la.unusual_masses = mass_flag_.data();
    la.exact_out = exact_.data();
    la.cell = cell_index_.data();
    la.crowded = crowded_.data();
    CorrectionArgs ca{};
    ca.n = n;
    ca.k = kernel_;
    ca.grid = grid;
    ca.rho0 = rho0_.data();
    ca.lambda = lambda_.data();
    ca.strength = strength_.data();
    ca.exponent = exponent_.data();
    ca.radius = radius_.data();
    ca.x0 = x0_.cview();
    ca.inv_dt = 1.0F / dt_;
    ca.vel = vel_.data();
    ca.exact = exact_.data();
    ca.cell = cell_index_.data();
    ca.crowded = crowded_.data();
    ca.t_exact = t_exact;
    ca.unusual_masses = mass_flag_.data();
    // the exact masks of each set of positions are rebuilt by the pass that
    // first walks them, so one buffer serves every set in forward mode
    const float4* current = xs_.data();
    DeviceBuffer<float4>* targets[2] = {&pa_, &pb_};
    const uint32_t iterations = config_.pressure_iterations;
    for (uint32_t it = 0; it < iterations; ++it) {
        la.pos = current;
        launch.lambda(la);
        float4* target = targets[it & 1u]->data();
        ca.pos = current;
        ca.out = target;
        ca.reconstruct = it + 1u == iterations ? 1u : 0u;
        launch.correction(ca);
        kernels_per_step_ += 2u;
        current = target;
    }
    if (iterations == 0u) {
        pbf_reconstruct_kernel<<<pbf_blocks(n, 1), kBlock, 0, s>>>(n, current, x0_.cview(), 1.0F / dt_, vel_.data(),
                                                                   Vec{});
        PHX_LAUNCH_CHECK();
        ++kernels_per_step_;
    }
    PostArgs post{};
    post.n = n;
    post.k = kernel_;
    post.dt = dt_;
    post.grid = grid;
    post.pos = current;
    post.vel = vel_.data();
    post.pos_magnitude = pos_magnitude_.data();
    post.vort = vort_.view();
    post.magnitude = magnitude_.data();
    post.confinement = confinement_.data();
    post.vc = vc_.data();
    post.xsph = xsph_.data();
    post.perm = grid_.perm.data();
    post.t_exact = t_exact;
    post.exact_out = exact_.data();
    post.exact = exact_.data();
    post.cell = cell_index_.data();
    post.crowded = crowded_.data();
    post.next_x = next_x.view();
    post.next_v = next_v.view();
    launch.vorticity(post);
    launch.normal(post);
    launch.xsph(post);
    kernels_per_step_ += 3u;
}
}  // namespace phx

namespace phx {

void PbfBatch::capture(const phx_control& control, const phx_pbf_parameters& parameters) {
    release_graphs();
    // one eager substep first, so every kernel is loaded before the capture
    // (it writes only the batch's own state buffers, which the replays overwrite)
    substep(0u, 0u, control, parameters);
    for (uint32_t from = 0; from < 2u; ++from) {
        hipGraph_t graph = nullptr;
        PHX_HIP(hipStreamBeginCapture(stream_, hipStreamCaptureModeThreadLocal));
        try {
            substep(from, 0u, control, parameters);
        } catch (...) {
            (void)hipStreamEndCapture(stream_, &graph);
            if (graph != nullptr) (void)hipGraphDestroy(graph);
            throw;
        }
        PHX_HIP(hipStreamEndCapture(stream_, &graph));
        hipGraphExec_t exec = nullptr;
        const hipError_t status = hipGraphInstantiate(&exec, graph, nullptr, nullptr, 0);
        (void)hipGraphDestroy(graph);
        PHX_HIP(status);
        graph_[from] = exec;
    }
}

void PbfBatch::run(phx_pbf_state& state, const phx_control& control, const phx_pbf_parameters& parameters,
                   uint32_t steps) {
    require_vec(state.particles.positions, "state positions");
    require_vec(state.particles.velocities, "state velocities");
    require_vec(control.external_accelerations, "control");
    const auto& pp = parameters.particles;
    require(pp.masses && pp.rest_densities, PHX_ERROR_INVALID_ARGUMENT, "null particle parameters");
    require(parameters.relaxation && parameters.artificial_pressure_strength && parameters.artificial_pressure_exponent &&
                parameters.artificial_pressure_radius && parameters.xsph_viscosity && parameters.vorticity_confinement,
            PHX_ERROR_INVALID_ARGUMENT, "null PBF parameters");
    if (steps == 0u || n_ == 0u) {
        state.particles.step_index += steps;
        return;
    }
    const size_t bytes = sizeof(float) * n_;
    // the batch's stream follows the caller's work on the state and inputs
    PHX_HIP(hipEventRecord(ready_, caller_));
    PHX_HIP(hipStreamWaitEvent(stream_, ready_, 0));
    const float* in[6] = {state.particles.positions.x,  state.particles.positions.y,  state.particles.positions.z,
                          state.particles.velocities.x, state.particles.velocities.y, state.particles.velocities.z};
    float* first[6] = {positions_[0].x.data(),  positions_[0].y.data(),  positions_[0].z.data(),
                       velocities_[0].x.data(), velocities_[0].y.data(), velocities_[0].z.data()};
    for (int k = 0; k < 6; ++k) PHX_HIP(hipMemcpyAsync(first[k], in[k], bytes, hipMemcpyDeviceToDevice, stream_));
    if (use_graph_) {
        // a captured substep reads the control and parameter arrays it was captured with
        const std::vector<const void*> inputs = {
            control.external_accelerations.x, control.external_accelerations.y, control.external_accelerations.z,
            pp.masses, pp.rest_densities, parameters.relaxation, parameters.artificial_pressure_strength,
            parameters.artificial_pressure_exponent, parameters.artificial_pressure_radius,
            parameters.xsph_viscosity, parameters.vorticity_confinement};
        if (graph_[0] == nullptr || inputs != captured_inputs_) {
            capture(control, parameters);
            captured_inputs_ = inputs;
        }
    }
    const uint64_t step = state.particles.step_index;
    uint32_t from = 0u;
    for (uint32_t k = 0; k < steps; ++k) {
        if (use_graph_) {
            PHX_HIP(hipGraphLaunch(graph_[from], stream_));
        } else {
            substep(from, step + k, control, parameters);
        }
        from = 1u - from;
    }
    float* out[6] = {state.particles.positions.x,  state.particles.positions.y,  state.particles.positions.z,
                     state.particles.velocities.x, state.particles.velocities.y, state.particles.velocities.z};
    const float* last[6] = {positions_[from].x.data(),  positions_[from].y.data(),  positions_[from].z.data(),
                            velocities_[from].x.data(), velocities_[from].y.data(), velocities_[from].z.data()};
    for (int k = 0; k < 6; ++k) PHX_HIP(hipMemcpyAsync(out[k], last[k], bytes, hipMemcpyDeviceToDevice, stream_));
    PHX_HIP(hipEventRecord(done_, stream_));
    PHX_HIP(hipStreamWaitEvent(caller_, done_, 0));
    state.particles.step_index = step + steps;
}

}  // namespace phx
