// Neighbour sums with a group of G lanes per particle.
//
// One lane per particle leaves most of the GPU idle below about 100,000
// particles (1,024 SIMDs of 64 lanes), and a pass then lasts as long as one
// lane's chain of some 40 candidates. Here G lanes (4 or 16) share a
// particle: each evaluates the pair terms of every G-th candidate, and the
// terms are then added one after the other, in the candidates' order, by
// every lane of the group through DPP broadcasts. The additions are the same
// as one lane's, in the same order, so the sums are equal bit for bit.
//
// A workgroup of kGroupBlock threads serves kGroupBlock / G particles in two
// mappings:
//   expand  thread t turns ceil(27 / G) stencil slots of particle t % P into
//           sorted candidate indices in the particle's LDS list (P particles
//           per workgroup); the slots of the G threads follow each other, so
//           the list is in the reference order
//   walk    lane t % G of particle t / G takes every G-th entry of that list
#pragma once

#include "neighbor_mask.hpp"

namespace phx {

constexpr uint32_t kGroupBlock = 256;
// candidates listed at a time; a particle with more is served in rounds
constexpr uint32_t kGroupList = 64;
// list entries with this bit are boundary samples (the launch has fewer
// particles and samples than that)
constexpr uint32_t kSampleEntry = 0x80000000u;

template <int G>
constexpr uint32_t kGroupParticles = kGroupBlock / G;
// stencil slots an expanding thread serves
template <int G>
constexpr uint32_t kGroupSlots = (static_cast<uint32_t>(kStencil) + G - 1u) / G;

template <int G>
struct GroupLds {
    // the row stride puts the entries that a wave reads together in distinct banks
    static constexpr uint32_t kStride = kGroupList + G;
    uint32_t list[kGroupParticles<G> * kStride];
    uint32_t counts[kGroupBlock];
    uint32_t totals[kGroupParticles<G>];
};

// The list of the particle the caller walks.
template <int G>
__device__ __forceinline__ uint32_t* group_row(GroupLds<G>& lds) {
    return lds.list + threadIdx.x / G * GroupLds<G>::kStride;
}

// The value lane k of the caller's group holds.
template <int G, int k>
__device__ __forceinline__ float group_broadcast(float v) {
    static_assert(G == 4 || G == 16, "groups are DPP quads or rows");
    constexpr int control = G == 4 ? k * 0x55 : 0x150 + k;  // quad_perm:[k,k,k,k], row_newbcast:k
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), control, 0xf, 0xf, true));
}

// sum[f] + terms[f] of lane 0, then of lane 1, ... of the group.
template <int G, int F, int k = 0>
__device__ __forceinline__ void group_add(float (&sum)[F], const float (&terms)[F]) {
#pragma unroll
    for (int f = 0; f < F; ++f) sum[f] = sum[f] + group_broadcast<G, k>(terms[f]);
    if constexpr (k + 1 < G) group_add<G, F, k + 1>(sum, terms);
}

// Walks entries 0 .. count - 1 of a group's list. load(entry) fetches an
// entry's record (it must accept `fallback`), pair(record, entry, terms)
// writes its terms, and fold(terms) adds every lane's to the sums (group_add);
// -0, which adds nothing to any value, stands in where the last trip has no
// entry. Records are fetched one trip ahead. The whole group calls this
// together.
template <int G, int F, class Load, class Pair, class Fold>
__device__ __forceinline__ void group_walk_list(const uint32_t* row, uint32_t count, uint32_t fallback, Load&& load,
                                                Pair&& pair, Fold&& fold) {
    const uint32_t lane = threadIdx.x % G;
    uint32_t entry = lane < count ? row[lane] : fallback;
    auto record = load(entry);
    for (uint32_t k = lane; k < count + lane; k += G) {
        const uint32_t ahead = k + G < count ? row[k + G] : fallback;
        const auto fetched = load(ahead);
        asm volatile("" ::: "memory");
        float terms[F];
#pragma unroll
        for (int f = 0; f < F; ++f) terms[f] = -0.0F;
        if (k < count) pair(record, entry, terms);
        fold(terms);
        entry = ahead;
        record = fetched;
    }
}

// Visits entries 0 .. count - 1 of a group's list for sums whose order is
// free: each lane takes its own entries, pair(load(entry), entry), fetching one
// ahead, and keeps partial sums (group_total).
template <int G, class Load, class Pair>
__device__ __forceinline__ void group_visit_list(const uint32_t* row, uint32_t count, Load&& load, Pair&& pair) {
    uint32_t k = threadIdx.x % G;
    if (k >= count) return;
    uint32_t entry = row[k];
    auto record = load(entry);
    while (true) {
        k += G;
        uint32_t ahead = entry;
        auto fetched = record;
        if (k < count) {
            ahead = row[k];
            fetched = load(ahead);
        }
        asm volatile("" ::: "memory");
        pair(record, entry);
        if (k >= count) return;
        entry = ahead;
        record = fetched;
    }
}

// v of the lane that DPP `control` reads for this one.
template <int control>
__device__ __forceinline__ double group_other(double v) {
    const long long bits = __double_as_longlong(v);
    const int low = __builtin_amdgcn_update_dpp(0, static_cast<int>(bits), control, 0xf, 0xf, true);
    const int high = __builtin_amdgcn_update_dpp(0, static_cast<int>(bits >> 32), control, 0xf, 0xf, true);
    return __longlong_as_double((static_cast<long long>(high) << 32) | static_cast<unsigned int>(low));
}

// The sum of the group's values, in every lane of the group.
template <int G>
__device__ __forceinline__ double group_total(double v) {
    static_assert(G == 4 || G == 16, "groups are DPP quads or rows");
    v += group_other<0xB1>(v);  // quad_perm:[1,0,3,2]
    v += group_other<0x4E>(v);  // quad_perm:[2,3,0,1]
    if constexpr (G == 16) {
        v += group_other<0x124>(v);  // row_ror:4
        v += group_other<0x128>(v);  // row_ror:8
    }
    return v;
}

// Walks the particles of the 27 cells around (cx, cy, cz), and with
// sample_offsets each cell's boundary samples after its particles: the walk of
// a particle with a crowded cell, whose candidates have no masks. The group
// tests G candidates at a time with near(entry), which is false only where the
// terms are exact zeros, and collects the others in its list `row`; a full
// list is walked on the way with run(row, count). Of the candidates of a
// crowded neighbourhood a sixth to a half are kept, and each one walked is
// dear. Entry `skip` is left out.
template <int G, class Near, class Run>
__device__ __forceinline__ void group_near_stencil(const SortedGrid& g, const uint32_t* sample_offsets, int cx, int cy,
                                                   int cz, uint32_t skip, uint32_t* row, Near&& near, Run&& walk) {
    const uint32_t lane = threadIdx.x % G;
    const uint32_t group_shift = __lane_id() - lane;
    uint32_t count = 0u;
    auto empty = [&] {
        // the list is written and read by this group alone, within its wave
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        walk(row, count);
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        count = 0u;
    };
    auto run = [&](uint32_t first, uint32_t last, uint32_t flag) {
        for (uint32_t base = first; base < last; base += G) {
            const uint32_t s = base + lane;
            const uint32_t entry = (s < last ? s : base) | flag;
            const bool kept = near(entry) && s < last && entry != skip;
            const uint32_t members =
                static_cast<uint32_t>(__ballot(kept) >> group_shift) & ((1u << static_cast<uint32_t>(G)) - 1u);
            if (kept) row[count + static_cast<uint32_t>(__popc(members & ((1u << lane) - 1u)))] = entry;
            count += static_cast<uint32_t>(__popc(members));
            if (count > kGroupList - G) empty();
        }
    };
    for_each_cell(g, cx, cy, cz, [&](uint32_t c) {
        run(g.offsets[c], g.offsets[c + 1u], 0u);
        if (sample_offsets != nullptr) run(sample_offsets[c], sample_offsets[c + 1u], kSampleEntry);
    });
    empty();
}

// group_near_stencil with the walks of group_walk_list.
template <int G, int F, class Near, class Load, class Pair, class Fold>
__device__ __forceinline__ void group_walk_stencil(const SortedGrid& g, const uint32_t* sample_offsets, int cx, int cy,
                                                   int cz, uint32_t skip, uint32_t fallback, uint32_t* row,
                                                   Near&& near, Load&& load, Pair&& pair, Fold&& fold) {
    group_near_stencil<G>(g, sample_offsets, cx, cy, cz, skip, row, near, [&](const uint32_t* list, uint32_t count) {
        group_walk_list<G, F>(list, count, fallback, load, pair, fold);
    });
}

// Lists the candidates of a workgroup's particles and walks them.
// slots(bits, first) sets, for each stencil slot k = part * kGroupSlots<G> + j
// of the expanding thread, bits[j] to the mask of its particle in that slot
// (empty for a particle that is not listed) and first[j] to the sorted index
// of that cell's first particle; with kSamples, sample_slots does the same
// for the cells' boundary samples.
// run(row, count) walks a list; it is called once for each round of
// kGroupList candidates. Every thread of the workgroup calls this together.
template <int G, bool kSamples, class Slots, class SampleSlots, class Run>
__device__ __forceinline__ void group_expand(GroupLds<G>& lds, Slots&& slots, SampleSlots&& sample_slots, Run&& run) {
    constexpr uint32_t kParticles = kGroupParticles<G>;
    constexpr uint32_t kSlots = kGroupSlots<G>;
    const uint32_t particle = threadIdx.x % kParticles;
    const uint32_t part = threadIdx.x / kParticles;
    uint32_t bits[kSlots] = {}, first[kSlots] = {};
    [[maybe_unused]] uint32_t sample_bits[kSlots] = {}, sample_first[kSlots] = {};
    slots(bits, first);
    if constexpr (kSamples) sample_slots(sample_bits, sample_first);
    uint32_t mine = 0u;
#pragma unroll
    for (uint32_t j = 0; j < kSlots; ++j) {
        mine += static_cast<uint32_t>(__popc(bits[j]));
        if constexpr (kSamples) mine += static_cast<uint32_t>(__popc(sample_bits[j]));
    }
    lds.counts[threadIdx.x] = mine;
    __syncthreads();
    uint32_t start = 0u, total = 0u;
#pragma unroll
    for (uint32_t v = 0; v < static_cast<uint32_t>(G); ++v) {
        const uint32_t c = lds.counts[v * kParticles + particle];
        start += v < part ? c : 0u;
        total += c;
    }
    uint32_t* list = lds.list + particle * GroupLds<G>::kStride;
    const uint32_t walked = threadIdx.x / G;
    const uint32_t* row = lds.list + walked * GroupLds<G>::kStride;
    for (uint32_t low = 0u;; low += kGroupList) {
        uint32_t place = start - low;  // wraps below the round's first entry
#pragma unroll
        for (uint32_t j = 0; j < kSlots; ++j) {
            for (uint32_t m = bits[j]; m != 0u; m &= m - 1u, ++place)
                if (place < kGroupList) list[place] = first[j] + static_cast<uint32_t>(__builtin_ctz(m));
            if constexpr (kSamples) {
                for (uint32_t m = sample_bits[j]; m != 0u; m &= m - 1u, ++place)
                    if (place < kGroupList)
                        list[place] = (sample_first[j] + static_cast<uint32_t>(__builtin_ctz(m))) | kSampleEntry;
            }
        }
        if (part == 0u) lds.totals[particle] = total;
        __syncthreads();
        const uint32_t all = lds.totals[walked];
        run(row, min(all > low ? all - low : 0u, kGroupList));
        if (__syncthreads_or(total > low + kGroupList ? 1 : 0) == 0) break;
    }
}

// Cell-index offset of stencil slot k (fill_slot_deltas).
__device__ __forceinline__ uint32_t slot_delta(const SortedGrid& g, uint32_t k) {
    const int ox = static_cast<int>(k / 9u) - 1;
    const int oy = static_cast<int>((k / 3u) % 3u) - 1;
    const int oz = static_cast<int>(k % 3u) - 1;
    return static_cast<uint32_t>(ox + (oz * static_cast<int>(g.cy) + oy) * static_cast<int>(g.cx));
}

// The expanding thread's slots from particle i's stored masks, for
// group_expand: with kDropSelf the particle's own bit is cleared. Every mask
// and every cell start is fetched at once, whether or not the mask turns out
// empty (a cell outside the grid has an empty mask; its start is read from
// the nearest cell index): a thread that waits for each mask before it
// fetches the cell start runs through G / 2 dependent pairs of loads.
template <int G, bool kDropSelf>
__device__ __forceinline__ void stored_slots(const uint16_t* __restrict__ masks, const SortedGrid& g,
                                             const uint32_t* __restrict__ offsets, uint32_t n, uint32_t i,
                                             uint32_t center, uint32_t (&bits)[kGroupSlots<G>],
                                             uint32_t (&first)[kGroupSlots<G>]) {
    constexpr uint32_t kSlots = kGroupSlots<G>;
    const uint32_t part = threadIdx.x / kGroupParticles<G>;
    const int last_cell = static_cast<int>(g.cx * g.cy * g.cz) - 1;
#pragma unroll
    for (uint32_t j = 0; j < kSlots; ++j) {
        const uint32_t k = min(part * kSlots + j, static_cast<uint32_t>(kStencil) - 1u);
        bits[j] = masks[static_cast<size_t>(k) * n + i];
        const int c = static_cast<int>(center + slot_delta(g, k));
        first[j] = offsets[min(max(c, 0), last_cell)];
    }
#pragma unroll
    for (uint32_t j = 0; j < kSlots; ++j) {
        const uint32_t k = part * kSlots + j;
        if (k >= static_cast<uint32_t>(kStencil)) bits[j] = 0u;
        if (kDropSelf && k == 13u) {
            const uint32_t own = i - first[j];
            bits[j] &= ~(own < kMaskBits ? 1u << own : 0u);
        }
    }
}

// The ranges [first, last) of the expanding thread's stencil slots of the cell
// (x, y, z), empty outside the grid; returns whether one holds more than
// kMaskBits. Fetched together, ahead of the members.
template <int G>
__device__ __forceinline__ bool group_ranges(const SortedGrid& g, const uint32_t* offsets, int x, int y, int z,
                                             uint32_t (&first)[kGroupSlots<G>],
                                             uint32_t (&last)[kGroupSlots<G>]) {
    constexpr uint32_t kSlots = kGroupSlots<G>;
    const uint32_t part = threadIdx.x / kGroupParticles<G>;
#pragma unroll
    for (uint32_t j = 0; j < kSlots; ++j) {
        first[j] = last[j] = 0u;
        const uint32_t k = part * kSlots + j;
        const int X = x + static_cast<int>(k / 9u) - 1;
        const int Y = y + static_cast<int>((k / 3u) % 3u) - 1;
        const int Z = z + static_cast<int>(k % 3u) - 1;
        if (k >= static_cast<uint32_t>(kStencil) || X < 0 || X >= static_cast<int>(g.cx) || Y < 0 ||
            Y >= static_cast<int>(g.cy) || Z < 0 || Z >= static_cast<int>(g.cz))
            continue;
        const uint32_t c = cell_of(g, X, Y, Z);
        first[j] = offsets[c];
        last[j] = offsets[c + 1u];
    }
    bool many = false;
#pragma unroll
    for (uint32_t j = 0; j < kSlots; ++j) many = many || last[j] - first[j] > kMaskBits;
    return many;
}

// The expanding thread's slots of a particle of cell (x, y, z) that is not
// crowded and whose stored masks do not apply: the members with near(position).
template <int G, class Near>
__device__ __forceinline__ void scanned_slots(const SortedGrid& g, const uint32_t* offsets, const float4* records,
                                              int x, int y, int z, uint32_t (&bits)[kGroupSlots<G>], uint32_t (&first)[kGroupSlots<G>],
                                              Near&& near) {
    uint32_t last[kGroupSlots<G>];
    (void)group_ranges<G>(g, offsets, x, y, z, first, last);
#pragma unroll
    for (uint32_t j = 0; j < kGroupSlots<G>; ++j) bits[j] = mark_members(records, first[j], last[j], near);
}

}  // namespace phx
