// Per-particle neighbour masks over the 27-cell stencil.
//
// For particle i and stencil slot k (offset_x outer, offset_z inner), bit b
// of mask[k * N + i] marks the b-th particle (in sorted order) of that cell
// as a neighbour. Walking slots in order and bits in ascending order visits
// the marked candidates in exactly the reference's summation order (27 cells,
// ascending original index), so a sum over the marked candidates equals the
// full-stencil sum whenever every unmarked candidate contributes an exact
// zero. Cells with more than kMaskBits particles cannot be encoded: a particle
// with such a cell among its 27 is marked crowded by the pass that builds the
// step's masks, and every pass walks the full stencil for that particle alone.
#pragma once

#include <cstdint>

#include "device_math.hpp"

namespace phx {

constexpr int kStencil = 27;
constexpr uint32_t kMaskBits = 16;

// Device flags of a step: [0] raised in the copy that a recorded step keeps
// where its masks do not serve its derivatives (boundary samples, which have
// masks of their own in the forward passes only); [1 + k] largest squared
// displacement |x* - x|^2 (float bits) written by the k-th predicting pass.
constexpr uint32_t kFlagOverflow = 0;
constexpr uint32_t kFlagDisplacement = 1;

// Linear index of cell (x, y, z), x fastest.
__device__ __forceinline__ uint32_t cell_of(const SortedGrid& g, int x, int y, int z) {
    return (static_cast<uint32_t>(z) * g.cy + static_cast<uint32_t>(y)) * g.cx + static_cast<uint32_t>(x);
}

// The coordinates of cell c.
__device__ __forceinline__ void cell_coordinates(const SortedGrid& g, uint32_t c, int& x, int& y, int& z) {
    const uint32_t row = c / g.cx;
    x = static_cast<int>(c - row * g.cx);
    z = static_cast<int>(row / g.cy);
    y = static_cast<int>(row - static_cast<uint32_t>(z) * g.cy);
}

// Cell-index offset of each stencil slot k = (ox + 1) * 9 + (oy + 1) * 3 +
// (oz + 1): ox + oy Cx + oz Cx Cy (two's complement). Filled by the first 27
// threads of the block; callers synchronise before use.
__device__ __forceinline__ void fill_slot_deltas(const SortedGrid& g, int* delta) {
    const uint32_t k = threadIdx.x;
    if (k < static_cast<uint32_t>(kStencil)) {
        const int ox = static_cast<int>(k) / 9 - 1;
        const int oy = (static_cast<int>(k) / 3) % 3 - 1;
        const int oz = static_cast<int>(k) % 3 - 1;
        delta[k] = ox + oy * static_cast<int>(g.cx) + oz * static_cast<int>(g.cx) * static_cast<int>(g.cy);
    }
}

// Copies the 27 masks of particle i into its LDS column and returns the
// bitmap of slots with a non-empty mask.
__device__ __forceinline__ uint32_t load_lane_column(const uint16_t* __restrict__ masks, uint32_t n, uint32_t i,
                                                     uint16_t* column, uint32_t stride) {
    uint32_t nonzero = 0u;
#pragma unroll
    for (int k = 0; k < kStencil; ++k) {
        const uint16_t m = masks[static_cast<size_t>(k) * n + i];
        column[static_cast<uint32_t>(k) * stride] = m;
        nonzero |= m != 0u ? 1u << k : 0u;
    }
    return nonzero;
}

// Marked candidates of one lane in the reference order, one candidate per
// loop trip; `nonzero` lists the slots to visit, `center` is the lane's cell.
// visit() should not branch on its candidate: a wave then runs one trip per
// candidate of its busiest lane with no other divergence.
template <class Visit>
__device__ __forceinline__ void walk_masked(const uint32_t* __restrict__ offsets, uint32_t center, const int* delta,
                                            const uint16_t* column, uint32_t stride, uint32_t nonzero, Visit&& visit) {
    uint32_t m = 0u;
    uint32_t base = 0u;
    while ((m | nonzero) != 0u) {
        if (m == 0u) {
            const uint32_t k = static_cast<uint32_t>(__builtin_ctz(nonzero));
            nonzero &= nonzero - 1u;
            m = column[k * stride];
            base = offsets[center + static_cast<uint32_t>(delta[k])];
        }
        const uint32_t b = static_cast<uint32_t>(__builtin_ctz(m));
        m &= m - 1u;
        visit(base + b);
    }
}

// walk_masked with the memory latency of each step taken off the critical
// path: the base index of the next non-empty slot (slot_base(k): the sorted
// index of the first particle of stencil cell k, or its place in a staged
// copy) is fetched when the current slot starts, and the data of the next
// kDepth candidates (load(s), which returns a value) is fetched before the
// current one is processed (process(value)), in the same order as
// walk_masked visits them. load() must be safe to call with any index the
// bases give (lanes without a next candidate load `fallback`, a valid index,
// and discard it).
template <int kDepth, class SlotBase, class Load, class Process>
__device__ __forceinline__ void walk_slots_prefetch(SlotBase&& slot_base, const uint16_t* column, uint32_t stride,
                                                    uint32_t nonzero, uint32_t fallback, Load&& load,
                                                    Process&& process) {
    auto fetch = [&](uint32_t& mask, uint32_t& base) {
        mask = 0u;
        if (nonzero != 0u) {
            const uint32_t k = static_cast<uint32_t>(__builtin_ctz(nonzero));
            nonzero &= nonzero - 1u;
            mask = column[k * stride];
            base = slot_base(k);
        }
    };
    uint32_t m = 0u, base = 0u, m_next = 0u, base_next = 0u;
    fetch(m, base);
    fetch(m_next, base_next);
    // the next candidate in the reference order, or fallback when none is left
    auto next = [&](bool& have) -> uint32_t {
        if (m == 0u) {
            m = m_next;
            base = base_next;
            fetch(m_next, base_next);
        }
        have = m != 0u;
        const uint32_t s = base + static_cast<uint32_t>(__builtin_ctz(m));
        m &= m - 1u;
        return have ? s : fallback;
    };
    using Data = decltype(load(0u));
    Data data[kDepth];
    bool have[kDepth];
#pragma unroll
    for (int d = 0; d < kDepth; ++d) data[d] = load(next(have[d]));
    // candidates arrive in order, so a lane is done at its first empty slot;
    // the ring is unrolled, so every data[d] stays in registers
    for (;;) {
#pragma unroll
        for (int d = 0; d < kDepth; ++d) {
            if (!have[d]) return;
            const Data current = data[d];
            data[d] = load(next(have[d]));
            // keeps the loads issued ahead of this candidate's arithmetic
            // (the compiler would otherwise sink them to their use)
            asm volatile("" ::: "memory");
            process(current);
        }
    }
}

// walk_slots_prefetch over the grid's cell offsets.
template <int kDepth = 1, class Load, class Process>
__device__ __forceinline__ void walk_masked_prefetch(const uint32_t* __restrict__ offsets, uint32_t center,
                                                     const int* delta, const uint16_t* column, uint32_t stride,
                                                     uint32_t nonzero, uint32_t fallback, Load&& load,
                                                     Process&& process) {
    walk_slots_prefetch<kDepth>([&](uint32_t k) { return offsets[center + static_cast<uint32_t>(delta[k])]; },
                                column, stride, nonzero, fallback, load, process);
}

// Clears particle i's own bit from its LDS column (slot 13, its own cell,
// whose first sorted particle is cell_first) for the sums that skip j == i;
// returns the bitmap of non-empty slots without slot 13 if that empties it.
__device__ __forceinline__ uint32_t drop_self(uint32_t i, uint32_t cell_first, uint16_t* column, uint32_t stride,
                                              uint32_t nonzero) {
    constexpr uint32_t kCenter = 13u;
    const uint32_t bit = i - cell_first;
    const uint32_t m = column[kCenter * stride] & ~(bit < kMaskBits ? 1u << bit : 0u);
    column[kCenter * stride] = static_cast<uint16_t>(m);
    return m == 0u ? nonzero & ~(1u << kCenter) : nonzero;
}

// Workgroup index with consecutive ranges of indices on one XCD (MI355X
// dispatches workgroup b to XCD b % 8). gridDim.x must be a multiple of 8.
__device__ __forceinline__ uint32_t xcd_block() {
    const uint32_t per_xcd = gridDim.x / 8u;
    return (blockIdx.x % 8u) * per_xcd + blockIdx.x / 8u;
}

// Masks of n particles, [kStencil][n].
struct MaskView {
    const uint16_t* masks;
    uint32_t n;
};

// The masks of members from .. to - 1 (the first kMaskBits of them) of the
// records x: test(position, marked) sets the bits of a member in the M masks.
// Four members are fetched together, past the end of a cell those of the next
// one or of the array's padding, whose bits are dropped at the end: fetching
// the last member again instead costs index arithmetic, a comparison and
// selects per member, as much as the test itself (PBF steps of 1,048,576
// particles 1,623 -> 1,590 us, of 260,000 496 -> 489; WCSPH 460 -> 453).
template <int M, class Test>
__device__ __forceinline__ void mark_members(const float4* x, uint32_t from, uint32_t to, uint32_t (&masks)[M],
                                             Test&& test) {
    const uint32_t count = min(to - from, kMaskBits);
    const float4* member = x + from;
#pragma unroll
    for (int m = 0; m < M; ++m) masks[m] = 0u;
    for (uint32_t s = 0u; s < count; s += kScanPadding + 1u, member += kScanPadding + 1u) {
        uint32_t four[M] = {};
#pragma unroll
        for (uint32_t u = 0; u < kScanPadding + 1u; ++u) {
            const float4 q = member[u];
            bool marked[M];
            test(Float3{q.x, q.y, q.z}, marked);
#pragma unroll
            for (int m = 0; m < M; ++m) four[m] |= marked[m] ? 1u << u : 0u;
        }
#pragma unroll
        for (int m = 0; m < M; ++m) masks[m] |= four[m] << s;
    }
#pragma unroll
    for (int m = 0; m < M; ++m) masks[m] &= (1u << count) - 1u;
}

// mark_members with one mask: the members with near(position).
template <class Near>
__device__ __forceinline__ uint32_t mark_members(const float4* x, uint32_t from, uint32_t to, Near&& near) {
    uint32_t masks[1];
    mark_members<1>(x, from, to, masks, [&](Float3 q, bool (&marked)[1]) { marked[0] = near(q); });
    return masks[0];
}

// Marks the members of the 27 cells around (cx, cy, cz) with near(position):
// emit(k, bits) takes stencil slot k's mask (every slot, in order; the first
// kMaskBits of a cell's members). The ranges of three cells are fetched
// together: with few waves in flight the scan is a chain of loads.
template <class Near, class Emit>
__device__ __forceinline__ void scan_stencil(const SortedGrid& g, const float4* records, int cx, int cy, int cz,
                                             Near&& near, Emit&& emit) {
    uint32_t k = 0u;
#pragma unroll 1
    for (int ox = -1; ox <= 1; ++ox) {
#pragma unroll 1
        for (int oy = -1; oy <= 1; ++oy, k += 3u) {
            const int X = cx + ox, Y = cy + oy;
            const bool row = X >= 0 && X < static_cast<int>(g.cx) && Y >= 0 && Y < static_cast<int>(g.cy);
            uint32_t first[3] = {0u, 0u, 0u}, last[3] = {0u, 0u, 0u};
            if (row) {
#pragma unroll
                for (int z = 0; z < 3; ++z) {
                    const int Z = cz + z - 1;
                    const bool inside = Z >= 0 && Z < static_cast<int>(g.cz);
                    const uint32_t c = cell_of(g, X, Y, inside ? Z : cz);
                    first[z] = g.offsets[c];
                    last[z] = inside ? g.offsets[c + 1u] : first[z];
                }
            }
#pragma unroll
            for (int z = 0; z < 3; ++z)
                emit(k + static_cast<uint32_t>(z), mark_members(records, first[z], last[z], near));
        }
    }
}

// Visits the candidates of particle i in the reference order: the marked
// ones of its masks (copied to its LDS column) or every particle of the 27
// cells around (cx, cy, cz).
template <class Visit>
__device__ __forceinline__ void visit_candidates(const SortedGrid& g, const MaskView& m, bool masked, uint32_t i, int cx,
                                                 int cy, int cz, const int* delta, uint16_t* column, uint32_t stride,
                                                 Visit&& visit) {
    if (masked) {
        const uint32_t nonzero = load_lane_column(m.masks, m.n, i, column, stride);
        walk_masked(g.offsets, cell_of(g, cx, cy, cz), delta, column, stride, nonzero, visit);
    } else {
        for_each_candidate(g, cx, cy, cz, visit);
    }
}

// Block-wide maximum of a non-negative float, folded into *target
// (non-negative IEEE floats order like their bit patterns). *target only
// grows, so a block whose maximum it already holds skips the atomic: one from
// each of 16,384 blocks to the same word took as long as the pass itself
// (force pass of 1,048,576 particles with four lanes each: 202 -> 150 us).
template <uint32_t kBlockSize>
__device__ __forceinline__ void block_max_to(float value, uint32_t* target) {
    __shared__ float wave_max[kBlockSize / 64];
    float v = value;
    for (int offset = 32; offset > 0; offset >>= 1) v = fmaxf(v, __shfl_xor(v, offset, 64));
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t wave = threadIdx.x >> 6;
    if (lane == 0u) wave_max[wave] = v;
    __syncthreads();
    if (threadIdx.x == 0u) {
        float m = wave_max[0];
        for (uint32_t w = 1; w < kBlockSize / 64; ++w) m = fmaxf(m, wave_max[w]);
        const uint32_t bits = __float_as_uint(m);
        if (bits > __hip_atomic_load(target, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) atomicMax(target, bits);
    }
}

}  // namespace phx
