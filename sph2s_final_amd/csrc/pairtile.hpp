// pairtile.hpp -- one wave walks the neighbours of 32 consecutive targets,
// with the matrix cores as the range filter.
//
// A wave owns a group of 32 targets, two lanes each (lane l and l + 32 share
// target l & 31 and take its even and its odd candidates).  The group's
// candidates are the particles of every grid row that the group's x-window
// reaches.  They pass through a ring of four words of 60 in the wave's own LDS
// tile, so there are no block barriers and no per-row phases, and a lane may be
// up to three words ahead of another.  For each word two
// V_MFMA_F32_32X32X16_F16 products form
//   |x_j - o|^2 - 2 (x_i - o).(x_j - o) + |x_i - o|^2 - h^2 - margin
// (o: a point among the targets) for all 32 targets in FP16, whose sign bits are
// the lanes' hit masks: one VALU instruction per 64 pairs instead of the seven
// of a distance test.  The margin covers the rounding of that form (its bound is
// at group_margin), so the masks hold every pair in range; a lane then takes
// its set bits in order and evaluates each pair from the staged global
// coordinates with the exact test, so the pairs summed and their values are
// those of a direct scan.
//
// A word holds fours of candidates from all over the group's list, so that each
// word has its share of every target's neighbours and the lanes stay even, and a
// four is 64 bytes of memory (single candidates touched 60 cache lines a word:
// the force pass spent half its time on them).  Takes per lane, modelled at 8 / 24
// particles per h^3, where a lane has 16 / 49 neighbours: 24 / 60 with the ring, 30 / 71
// with the list in parts of 320 that all lanes finish before the next, and three words
// or eight instead of four make it 25 / 61 and 24 / 59.
//
// Groups spread over many cells (spray, films), targets a million h from the origin or
// not finite, and targets whose sums are not finite are scanned directly instead: each
// lane walks every other row of its target's stencil (walk_targets, walk_direct).
//
// The index of a candidate in the group's list decides the lane that takes it
// and its place in the order, and the way a group is taken depends on its targets and
// their cells, so a target's sums depend on its group alone: not on the block size or
// the grid.
#pragma once

#include "neighbors.hpp"

namespace sph {

constexpr uint32_t kGroupTargets = 32;
typedef float v2f __attribute__((ext_vector_type(2)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef uint32_t v2u __attribute__((ext_vector_type(2)));
typedef float v16f __attribute__((ext_vector_type(16)));
typedef __fp16 v2h __attribute__((ext_vector_type(2)));
typedef _Float16 v8h __attribute__((ext_vector_type(8)));

// LDS by byte address.  16-byte elements are read whole (keep4): the 12-byte
// form that the compiler narrows an unused component to is markedly slower.
template <class T>
__device__ __forceinline__ T lds_read(uint32_t at) {
    return *reinterpret_cast<const __attribute__((address_space(3))) T*>(at);
}
template <class T>
__device__ __forceinline__ void lds_write(uint32_t at, const T& v) {
    *reinterpret_cast<__attribute__((address_space(3))) T*>(at) = v;
}
__device__ __forceinline__ uint32_t lds_address(const void* p) {
    return static_cast<uint32_t>(
        reinterpret_cast<size_t>((const __attribute__((address_space(3))) void*)(p)));
}
__device__ __forceinline__ void keep4(const v4f& q) { asm volatile("" ::"v"(q.w)); }

// Orders the wave's LDS writes before its later LDS reads (a wave's DS
// instructions execute in order; this stops the compiler moving them).
__device__ __forceinline__ void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Targets of one group: lane l holds target l & 31 (both halves the same).
struct GroupTargets {
    float4 x;        // position (any w)
    uint32_t key;    // cell of the grid's own cell array (cell_offset taken off)
    bool active;
};

// One group of targets: slots [start, end) of the internal order, all of one
// scene.  Single scenes are cut every 32 slots; a batch
// starts anew at each scene (its table of groups), so a scene's groups, and
// with them its sums, are those of the scene alone.
struct GroupRange {
    uint32_t start, end, scene, index;
};

template <bool kBatched>
__device__ __forceinline__ GroupRange group_range(uint32_t group, uint32_t n,
                                                  const uint4* __restrict__ groups,
                                                  uint32_t n_groups) {
    GroupRange r{0u, 0u, 0u, group};
    if (kBatched) {
        if (group < n_groups) {
            const uint4 v = groups[group];
            r.start = uniform_u32(v.x);
            r.end = min(uniform_u32(v.y), n);
            r.scene = uniform_u32(v.z);
        }
    } else if (group < n_groups) {
        r.start = group * kGroupTargets;
        r.end = min(r.start + kGroupTargets, n);
    }
    return r;
}

// The sum of both lane halves' partial sums of a target.
__device__ __forceinline__ double both_halves(double v) { return v + __shfl_xor(v, 32); }
__device__ __forceinline__ float both_halves(float v) { return v + __shfl_xor(v, 32); }

// The group's targets: positions, and cells from the sorted keys (a cell's
// slots are the same in the sorted and the internal order).
__device__ __forceinline__ GroupTargets load_targets(const GridView& g, const GroupRange& r,
                                                     const float4* __restrict__ tpos,
                                                     const uint32_t* __restrict__ skeys,
                                                     uint32_t& s) {
    GroupTargets t;
    s = r.start + (threadIdx.x & 31u);
    t.active = s < r.end;
    const uint32_t at = t.active ? s : r.start;
    t.x = tpos[at];
    t.key = skeys[at] - g.cell_offset;
    return t;
}

// A subgroup: the targets of a group that share a grid row and span at most
// g.span cells along it.
struct Subgroup {
    bool member;          // this lane's target
    int cy, cz;           // the row
    float x0, x1;         // first and last x offset from the grid origin (clamped into it)
    float ox, oy, oz;     // origin of the filter's coordinates: near the targets
    int y0, z0, ny, nz;   // rows reached: ny x nz from (y0, z0), inside the grid
    bool far;             // the filter's coordinates do not hold the targets
};

// The next subgroup of the targets in `rem` (a mask of 32 targets), which
// loses its members.  Targets are ordered by x inside each cell.
__device__ __forceinline__ Subgroup next_subgroup(const GridView& g, const GroupTargets& t,
                                                  uint32_t& rem) {
    Subgroup s;
    const int first = __builtin_ctz(rem);
    const float xf = lane_f32(t.x.x, first);
    s.oy = lane_f32(t.x.y, first);
    s.oz = lane_f32(t.x.z, first);
    // From a million h from the origin on (or at a NaN): there the rounding of
    // o / h is h / 16 and more, then the words' fill is no longer out of range,
    // and beyond 2^31 h a target would miss itself.
    auto size = [](float x) { return __float_as_uint(x) & 0x7FFFFFFFu; };
    s.far = max(size(xf), max(size(s.oy), size(s.oz))) >= __float_as_uint(g.filter_max);
    const uint32_t key = min(lane_u32(t.key, first), 0x7FFFFFFFu);
    const uint32_t line = static_cast<uint32_t>((static_cast<uint64_t>(key) * g.mx) >> (31u + g.lx));
    const uint32_t row = line * static_cast<uint32_t>(g.dx);
    const uint32_t plane = static_cast<uint32_t>((static_cast<uint64_t>(line) * g.my) >> (31u + g.ly));
    s.cy = static_cast<int>(line - plane * static_cast<uint32_t>(g.dy));
    s.cz = static_cast<int>(plane);
    const uint32_t c0 = key - row;
    const uint32_t cx = t.key - row;
    const int n = static_cast<int>(threadIdx.x & 31u);
    // Targets far from the first (particles outside the grid share its boundary
    // cells) wait for a subgroup of their own, so that the filter's half
    // precision holds every member.  The first is always taken.
    const float ex = t.x.x - xf, ey = t.x.y - s.oy, ez = t.x.z - s.oz;
    const float e2 = ex * ex + ey * ey + ez * ez;
    s.member = t.active && ((rem >> n) & 1u) && cx < static_cast<uint32_t>(g.dx) &&
               cx - c0 <= static_cast<uint32_t>(g.span) && e2 < 900.0f * g.prune_h2;
    s.member = s.member || n == first;
    const uint32_t mem = static_cast<uint32_t>(__ballot(s.member));
    rem &= ~mem;
    const int last = 31 - __builtin_clz(mem);
    const float fx = grid_offset(t.x.x, g.ox, g.spacing, g.dx);
    s.x0 = lane_f32(fx, first);
    s.x1 = lane_f32(fx, last);
    s.ox = 0.5f * (xf + lane_f32(t.x.x, last));
    // A target within `edge` of its cell's y or z face may see, through the
    // rounding of cell coordinates, a particle one row beyond the reach.
    const float fy = grid_offset(t.x.y, g.oy, g.spacing, g.dy) - static_cast<float>(s.cy) * g.spacing;
    const float fz = grid_offset(t.x.z, g.oz, g.spacing, g.dz) - static_cast<float>(s.cz) * g.spacing;
    const float hi = g.spacing - g.edge;
    const int ry = g.reach + (__ballot(s.member && (fy < g.edge || fy > hi)) != 0ull ? 1 : 0);
    const int rz = g.reach + (__ballot(s.member && (fz < g.edge || fz > hi)) != 0ull ? 1 : 0);
    s.y0 = max(s.cy - ry, 0);
    s.z0 = max(s.cz - rz, 0);
    s.ny = min(s.cy + ry, g.dy - 1) - s.y0 + 1;
    s.nz = min(s.cz + rz, g.dz - 1) - s.z0 + 1;
    return s;
}

// Candidate run [b, e) of grid row (ry, rz) for a subgroup (empty: b = e = 0);
// the row is inside the grid.
__device__ __forceinline__ void subgroup_row(const GridView& g, const Subgroup& s,
                                             const uint32_t* __restrict__ cs,
                                             const uint32_t* __restrict__ ce,
                                             const uint4* __restrict__ bins, uint32_t n, int ry,
                                             int rz, uint32_t& b, uint32_t& e) {
    b = 0u;
    e = 0u;
    // Distance from the subgroup's cells to the row, less the rounding of cell
    // coordinates.
    const float gy = fmaxf(0.0f, static_cast<float>(abs(ry - s.cy) - 1) * g.spacing - 2.0f * g.edge);
    const float gz = fmaxf(0.0f, static_cast<float>(abs(rz - s.cz) - 1) * g.spacing - 2.0f * g.edge);
    const float d2 = gy * gy + gz * gz;
    if (d2 >= g.prune_h2) return;
    const float w = __builtin_amdgcn_sqrtf(g.prune_h2 - d2);
    const float xl = (s.x0 - w) * g.inv_spacing, xh = (s.x1 + w) * g.inv_spacing;
    const int lo = max(0, static_cast<int>(floorf(xl)));
    const int hi = min(g.dx - 1, static_cast<int>(floorf(xh)));
    if (lo > hi) return;
    const uint32_t row = g.cell_offset + static_cast<uint32_t>(g.dx) * (ry + g.dy * rz);
    // Particles of cell lo below the window and of cell hi up to its end, from
    // the cells' cumulative x-bin counts; loaded beside the cell ranges and
    // ignored for an empty cell (whose counts are an earlier step's).
    const uint8_t* const count = reinterpret_cast<const uint8_t*>(bins);
    const int k_lo = xbin_of(xl - static_cast<float>(lo)), k_hi = xbin_of(xh - static_cast<float>(hi));
    const uint32_t below = count[static_cast<size_t>(row + lo) * kXBins + max(k_lo - 1, 0)];
    const uint32_t upto = count[static_cast<size_t>(row + hi) * kXBins + k_hi];
    // The run starts at the first non-empty cell and ends at the last one: an
    // empty cell holds SPH_EMPTY_CELL as start and end, the largest start and,
    // as a signed value, the smallest end.
    uint32_t first = kEmptyCell, s_lo = kEmptyCell, s_hi = kEmptyCell;
    int last = -1;
    for (int cx = lo; cx <= hi; cx += 8) {
        uint32_t a[8];
        int z[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            const uint32_t c = row + min(cx + u, hi);
            a[u] = cs[c];
            z[u] = static_cast<int>(ce[c]);
        }
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            first = min(first, a[u]);
            last = max(last, z[u]);
        }
        if (cx == lo) s_lo = a[0];
        s_hi = a[7];  // the last iteration's is cell hi's
    }
    if (last < 0) return;
    uint32_t end = static_cast<uint32_t>(last);
    end = min(end, n);
    if (s_lo != kEmptyCell && k_lo > 0 && below != kXBinUnbinned) first = s_lo + below;
    if (s_hi != kEmptyCell && upto != kXBinUnbinned) end = min(end, s_hi + upto);
    if (first < end) {
        b = first;
        e = end;
    }
}

// The margin of the matrix filter, in units of h^2, for a target at squared
// distance q = u^2 from the origin.  A candidate in range is at most u + 1 from
// it; its coordinates are off by 2^-10 of their size (rounded towards zero),
// the target's by 2^-11, its |x|^2 by 2^-10: together at most
// 2^-10 (3 u (u + 1) + (u + 1)^2) <= 2^-10 (7 q + 4).
__device__ __forceinline__ float group_margin(float q) { return (7.0f * q + 5.0f) * 0x1p-10f; }

// Waits for the wave's loads into LDS.
__device__ __forceinline__ void wait_vmem() { __builtin_amdgcn_s_waitcnt(0x0f70); }

// Waits for the wave's LDS reads.
__device__ __forceinline__ void wait_lds() { __builtin_amdgcn_s_waitcnt(0xc07f); }

// Active lanes each copy 16 bytes from `src` to LDS at `to` + 16 lane (`to`
// wave-uniform), without passing through registers.
__device__ __forceinline__ void lds_copy16(const float4* src, uint32_t to) {
    __builtin_amdgcn_global_load_lds(
        reinterpret_cast<const __attribute__((address_space(1))) void*>(
            reinterpret_cast<uintptr_t>(src)),
        reinterpret_cast<__attribute__((address_space(3))) void*>(to), 16, 0, 0);
}

// A wave's tile: the hit masks of the ring's words (64 lanes each; the first
// once more past the last, so that the word after any is 256 bytes on), the
// list's rows, and the words' candidates, kArrays float4 each: (x, .), (v, .) and
// one more.  A word's slots from 60 on are beyond any target's range for good: a
// lane that has nothing to take points there.
constexpr uint32_t kRing = 4, kWordSlots = 60;
template <uint32_t kArrays>
struct PairTile {
    static constexpr uint32_t kRows = 256u * (kRing + 1u);
    static constexpr uint32_t kSlots = 2048u;           // kRows + 8 * 65 rounded up
    static constexpr uint32_t kArray = 1024u * kRing;   // from one array to the next
    static constexpr uint32_t kBytes = kSlots + kArrays * kArray;
    static_assert(kRows + 8u * 65u <= kSlots, "64 rows and the end");
};
constexpr uint32_t kTileAlign = 256u * kRing;  // of a tile's LDS address

// Row r of a subgroup's ny x nz rows.
__device__ __forceinline__ void row_of(const Subgroup& s, uint32_t r, int& y, int& z) {
    uint32_t q;
    if (s.ny <= 3 && s.ny * s.nz <= 64)  // wave-uniform; the usual reach
        q = (r * (s.ny == 3 ? 43u : s.ny == 2 ? 64u : 128u)) >> 7;  // r < 64
    else
        q = r / static_cast<uint32_t>(s.ny);
    z = s.z0 + static_cast<int>(q);
    y = s.y0 + static_cast<int>(r - q * static_cast<uint32_t>(s.ny));
}

// A candidate whose position is not finite is replaced by a far one, so it meets
// no one (targets that far, or not finite, are not walked here: walk_targets).
constexpr float kFar = 1e15f, kFar2 = 3e30f;

// Walks the candidates of a group in the internal x-order: their arrays a0 (x, .),
// a1 and a2 (kArrays of them).  pair(q0, ..) evaluates this lane's target with one
// candidate; every8() is called after at most nine of them, and at the end.
// tile: LDS address of the wave's PairTile.  Returns the targets left out, those of
// subgroups that the filter does not hold.
template <uint32_t kArrays, class F, class G>
__device__ __forceinline__ uint32_t walk_group(const GridView& g, const GroupTargets& t, float inv_h,
                                           const uint32_t* __restrict__ cs,
                                           const uint32_t* __restrict__ ce,
                                           const uint4* __restrict__ bins, uint32_t n,
                                           const float4* __restrict__ a0,
                                           const float4* __restrict__ a1,
                                           const float4* __restrict__ a2, uint32_t tile, F&& pair,
                                           G&& every8) {
    typedef PairTile<kArrays> T;
    const uint32_t lane = threadIdx.x & 63u;
    // The slots nobody is near.
    if (lane < 4u * kRing) {
        const uint32_t at = tile + T::kSlots + 1024u * (lane >> 2) + 16u * (kWordSlots + (lane & 3u));
        lds_write<v4f>(at, v4f{kFar, kFar, kFar, 0.0f});
#pragma unroll
        for (uint32_t k = 1; k < kArrays; ++k)
            lds_write<v4f>(at + k * T::kArray, v4f{0.0f, 0.0f, 0.0f, 0.0f});
    }
    uint32_t turn = 0u;
    uint32_t rem = static_cast<uint32_t>(__ballot(t.active)), left = 0u;
    while (rem) {
        const uint32_t before = rem;
        const Subgroup s = next_subgroup(g, t, rem);
        if (s.far) {
            left |= before & ~rem;
            continue;
        }
        // Fills the words: out of the members' range, yet finite in FP16 (an
        // infinity would make the products NaN, and its sign a hit).
        const v4f far = {s.ox + 100.0f * __builtin_amdgcn_rcpf(inv_h), s.oy, s.oz, 0.0f};
        const uint64_t members = __ballot(s.member);
        const uint32_t rows = static_cast<uint32_t>(s.ny) * static_cast<uint32_t>(s.nz);
        for (uint32_t row0 = 0; row0 < rows; row0 += 64u) {
            uint32_t rb = 0u, re = 0u;
            if (row0 + lane < rows) {
                int y, z;
                row_of(s, row0 + lane, y, z);
                subgroup_row(g, s, cs, ce, bins, n, y, z, rb, re);
            }
            // The list: the rows that are not empty, as (its end in the list,
            // first particle less its start), and an end that is never reached.
            const uint32_t len = re - rb;
            const uint32_t end = wave_scan_add(len);
            const uint32_t total = lane_u32(end, 63);
            if (total == 0u) continue;
            uint64_t live = __ballot(len != 0u);
            const uint32_t place = __builtin_amdgcn_mbcnt_hi(
                static_cast<uint32_t>(live >> 32),
                __builtin_amdgcn_mbcnt_lo(static_cast<uint32_t>(live), 0u));
            if (len != 0u) lds_write<v2u>(tile + T::kRows + 8u * place, v2u{end, rb + len - end});
            if (lane == 0u)
                lds_write<v2u>(tile + T::kRows + 8u * static_cast<uint32_t>(__builtin_popcountll(live)),
                               v2u{0xFFFFFFFFu, 0u});
            // From here on, not held through the look-up of the rows: with them the
            // density pass spilled four registers a group (24 scenes of 4096..98304:
            // force 90 us, now 88.5; a million at rest 113, now 109).
            uint32_t place_in_wave = lane;
            asm volatile("" : "+v"(place_in_wave));
            const uint32_t half = place_in_wave >> 5;
            // A lane half converts 32 of 64 candidates; the first product takes the lower
            // half's (the upper half's target operand is 0), the second the upper's.
            // Row m of a product reads slot 2 r + q of its 32, where (q, r) are the lane
            // half and accumulator that receive row m: a lane's 32 mask bits are the even
            // (half 0) or odd slots of 64, so a target's hits, which lie together along a
            // row, fall evenly on its two lanes.  The rows of slots 60 to 63 read others;
            // their bits are dropped.
            const uint32_t m = place_in_wave & 31u;
            const uint32_t slot_of_row = 2u * (4u * (m >> 3) + (m & 3u)) + ((m >> 2) & 1u) + 32u * half;
            const uint32_t row_slot =
                tile + T::kSlots + 16u * (slot_of_row < kWordSlots ? slot_of_row : slot_of_row - 4u);
            const uint32_t mask0 = tile + 4u * place_in_wave;
            // Target operands of the filter, in units of h: columns
            // (-2 x, -2 y, -2 z, 1, c, c') against rows (x, y, z, |x|^2, 1, 1), with
            // c + c' = |x|^2 - 1 - margin.
            const float sx = -s.ox * inv_h, sy = -s.oy * inv_h, sz = -s.oz * inv_h;
            const float ix = __builtin_fmaf(t.x.x, inv_h, sx), iy = __builtin_fmaf(t.x.y, inv_h, sy),
                        iz = __builtin_fmaf(t.x.z, inv_h, sz);
            const float qi = ix * ix + iy * iy + iz * iz;
            float ci = s.member && qi < 1e4f ? qi - 1.0f - group_margin(qi) : 6e4f;
            asm volatile("" : "+v"(ci));  // here, not before the rows: registers
            const _Float16 c_hi = static_cast<_Float16>(ci);
            const v8h none = {0, 0, 0, 0, 0, 0, 0, 0},
                      col = {static_cast<_Float16>(-2.0f * ix), static_cast<_Float16>(-2.0f * iy),
                             static_cast<_Float16>(-2.0f * iz), 1, c_hi,
                             static_cast<_Float16>(ci - static_cast<float>(c_hi)), 0, 0},
                      cols[2] = {half ? none : col, half ? col : none};
            // Word w holds, of every 4 words candidates, four from 4 w on.  This
            // lane copies its slot's ones, one word after the other: `at` in the
            // list, in a row that ends at entry.x, whose table entry is at row.
            const uint32_t words = (total + kWordSlots - 1u) / kWordSlots;
            uint32_t at = 4u * words * (lane >> 2) + (lane & 3u), row = tile + T::kRows;
            for (; live; live &= live - 1u)
                row += at >= lane_u32(end, static_cast<int>(__builtin_ctzll(live))) ? 8u : 0u;
            wave_sync();
            v2u entry = lds_read<v2u>(row);
            auto stage = [&](uint32_t w) {
                const uint32_t to = tile + T::kSlots + 1024u * (w % kRing);
                while (__ballot(at >= entry.x) != 0ull) {  // rows of less than four
                    row += at >= entry.x ? 8u : 0u;
                    entry = lds_read<v2u>(row);
                }
                if (lane < kWordSlots) {
                    if (at < total) {
                        const uint32_t j = at + entry.y;
                        lds_copy16(a0 + j, to);
                        if (kArrays > 1) lds_copy16(a1 + j, to + T::kArray);
                        if (kArrays > 2) lds_copy16(a2 + j, to + 2u * T::kArray);
                    } else {
                        lds_write<v4f>(to + 16u * lane, far);
#pragma unroll
                        for (uint32_t k = 1; k < kArrays; ++k)
                            lds_write<v4f>(to + k * T::kArray + 16u * lane,
                                           v4f{0.0f, 0.0f, 0.0f, 0.0f});
                    }
                }
                at += 4u;
                row += at >= entry.x ? 8u : 0u;
                entry = lds_read<v2u>(row);
            };
            auto set_mask = [&](uint32_t w, uint32_t bits) {
                lds_write<uint32_t>(mask0 + 256u * (w % kRing), bits);
                if (w % kRing == 0u) lds_write<uint32_t>(mask0 + 256u * kRing, bits);
            };
            // Each member's lane takes the set bits of its words in order.  The
            // word after the last one filtered has the mask 1, a bit that stays
            // set: a lane there, or one that is no member, takes a slot that
            // nobody is near.  word: where the lane's current word is, whose
            // first slot is at 4 word + to_slots; one candidate is on its way
            // while another is evaluated.
            const uint32_t to_slots = tile + T::kSlots + 16u * half - 4u * mask0;
            uint32_t word = mask0, cur = 1u, nxt = 1u, wrap = 256u * kRing - 1u;
            asm("" : "+v"(wrap));  // one and-or, which takes one scalar operand
            auto next_word = [&](uint32_t w) { return ((w + 256u) & wrap) | tile; };
            auto filter = [&](uint32_t w) {
                const uint32_t from = row_slot + 1024u * (w % kRing);
                const v4f x = lds_read<v4f>(from);
                keep4(x);
                float dx = __builtin_fmaf(x.x, inv_h, sx), dy = __builtin_fmaf(x.y, inv_h, sy),
                      dz = __builtin_fmaf(x.z, inv_h, sz);
                float q = dx * dx + dy * dy + dz * dz;
                if (__ballot(!(q < kFar2)) != 0ull && !(q < kFar2)) {
                    lds_write<v4f>(from, far);
                    dx = 100.0f;
                    dy = dz = 0.0f;
                    q = 1e4f;
                }
                const v2h xy = __builtin_amdgcn_cvt_pkrtz(dx, dy),
                          zq = __builtin_amdgcn_cvt_pkrtz(dz, q);
                const v8h rows8 = {static_cast<_Float16>(xy.x), static_cast<_Float16>(xy.y),
                                   static_cast<_Float16>(zq.x), static_cast<_Float16>(zq.y),
                                   1, 1, 0, 0};
                uint32_t bits = 0u;
#pragma unroll
                for (int k = 0; k < 2; ++k) {
                    const v16f d =
                        __builtin_amdgcn_mfma_f32_32x32x16_f16(rows8, cols[k], v16f{}, 0, 0, 0);
#pragma unroll
                    for (int r = 0; r < 16 - 2 * k; ++r)
                        bits = __builtin_amdgcn_alignbit(bits, __float_as_uint(d[r]), 31);
                    __builtin_amdgcn_sched_barrier(0);  // one product's registers at a time
                }
                // No word is empty: slot 60 or 61 stands in for none.
                bits = max(bits << 2, 2u);
                set_mask(w, bits);
                set_mask(w + 1u, 1u);
                wave_sync();
                // Lanes that waited for this word or read ahead to it.
                cur = s.member && word == mask0 + 256u * (w % kRing) ? bits : cur;
                nxt = lds_read<uint32_t>(word + 256u);
            };
            auto take = [&](v4f* q) {
                const uint32_t z = __builtin_clz(cur);
                uint32_t first = 4u * word + to_slots;
                asm("" : "+v"(first));  // two shift-and-adds, not three instructions
                const uint32_t p = 32u * z + first;
#pragma unroll
                for (uint32_t k = 0; k < kArrays; ++k) q[k] = lds_read<v4f>(p + k * T::kArray);
                cur &= ~(0x80000000u >> z) | 1u;
                const bool over = cur == 0u;
                cur = over ? nxt : cur;
                word = over ? next_word(word) : word;
                nxt = lds_read<uint32_t>(word + 256u);
            };
            auto eval = [&](const v4f* q) {
#pragma unroll
                for (uint32_t k = 0; k < kArrays; ++k) keep4(q[k]);
                if constexpr (kArrays == 1)
                    pair(q[0]);
                else if constexpr (kArrays == 2)
                    pair(q[0], q[1]);
                else
                    pair(q[0], q[1], q[2]);
            };
            uint32_t staged = 0u, filtered = 0u, oldest = 0u, oldest_word = mask0;
            do stage(staged);
            while (++staged < min(words, kRing));
            wait_vmem();
            wave_sync();
            do filter(filtered);
            while (++filtered < min(words, kRing - 1u));
            v4f qa[kArrays], qb[kArrays];
            take(qa);
            for (;;) {
                take(qb);
                eval(qa);
                take(qa);
                eval(qb);
                if ((++turn & 3u) == 0u) {
                    asm volatile("");  // a branch, not selects on every turn
                    every8();
                }
                // Someone is still in the oldest word.
                if ((__ballot(word == oldest_word) & members) != 0ull) continue;
                if (++oldest == words) break;
                oldest_word = next_word(oldest_word);
                if (filtered < words) {
                    wait_vmem();
                    filter(filtered++);
                    if (staged < words) {
                        wait_lds();  // of the word that goes
                        stage(staged++);
                    }
                }
            }
            eval(qa);
            every8();
            wait_lds();
            wave_sync();
        }
    }
    return left;
}

// What a direct scan reads.
struct DirectScan {
    GridView g;
    const uint32_t *cs, *ce;
    uint32_t n;
    const float4 *a0, *a1, *a2;
};

// A kernel's first arguments again, from memory: values that only the direct scan
// needs are then not held in registers through the group walk (force of one million
// settled 192 us held, 187 read again).
template <class Args>
__device__ __forceinline__ Args first_arguments() {
    static_assert(sizeof(Args) % 4 == 0, "copied by words");
    typedef const __attribute__((address_space(4))) uint32_t* Words;
    Words p = reinterpret_cast<Words>(
        reinterpret_cast<uintptr_t>(__builtin_amdgcn_kernarg_segment_ptr()));
    asm volatile("" : "+s"(p));
    Args a;
    uint32_t w[sizeof(Args) / 4];
#pragma unroll
    for (uint32_t k = 0; k < sizeof(Args) / 4; ++k) w[k] = p[k];
    __builtin_memcpy(&a, w, sizeof(Args));
    return a;
}

// Candidate runs [b, e) of kRows rows (ry, rz) of a target's stencil (empty rows
// and rows outside it: b >= e), the cells as in probe_row_run.  The loads of all
// rows go out together.
template <int kRows>
__device__ __forceinline__ void direct_rows(const GridView& g, const Probe& pr, const uint32_t* cs,
                                            const uint32_t* ce, uint32_t n, const int* ry, const int* rz, uint32_t* b, uint32_t* e) {
    uint32_t first[kRows], more[kRows], start[kRows][3];
    int end[kRows][3];
#pragma unroll
    for (int u = 0; u < kRows; ++u) {
        const float gy = slab_gap(pr.fy, ry[u], g.spacing), gz = slab_gap(pr.fz, rz[u], g.spacing);
        const float w2 = g.prune_h2 - (gy * gy + gz * gz);
        const float w = __builtin_amdgcn_sqrtf(fmaxf(w2, 0.0f));
        const int lo = max(pr.sx, static_cast<int>(floorf((pr.fx - w) * g.inv_spacing)));
        const int hi = min(pr.ex, static_cast<int>(floorf((pr.fx + w) * g.inv_spacing)));
        const bool some = w2 > 0.0f && ry[u] <= pr.ey && rz[u] <= pr.ez && lo <= hi;
        first[u] = some ? g.cell_offset + static_cast<uint32_t>(g.dx) * (ry[u] + g.dy * rz[u]) + lo
                        : g.cell_offset;  // any
        more[u] = some ? static_cast<uint32_t>(hi - lo) : 0u;
        b[u] = some ? 0u : 0x80000000u;  // no start is larger: a row of none stays empty
#pragma unroll
        for (uint32_t k = 0; k < 3; ++k) {
            const uint32_t c = first[u] + min(k, more[u]);
            start[u][k] = cs[c];
            end[u][k] = static_cast<int>(ce[c]);
        }
    }
#pragma unroll
    for (int u = 0; u < kRows; ++u) {
        // An empty cell's start is the largest, its end (as signed) the smallest.
        b[u] = max(b[u], min(start[u][0], min(start[u][1], start[u][2])));
        int last = max(end[u][0], max(end[u][1], end[u][2]));
        for (uint32_t k = 3; k <= more[u]; ++k) {  // cells of less than h
            b[u] = min(b[u], cs[first[u] + k]);
            last = max(last, static_cast<int>(ce[first[u] + k]));
        }
        e[u] = min(static_cast<uint32_t>(max(last, 0)), n);
    }
}

// This lane's half of its target's rows, three at a time: the next row to look up
// and the candidate runs [b, e) of the last three.
struct DirectRows {
    Probe pr;
    int y, z;
    uint32_t b[3], e[3];
};
__device__ __forceinline__ void next_rows(const DirectScan& d, DirectRows& r) {
    int ry[3], rz[3];
#pragma unroll
    for (int u = 0; u < 3; ++u, r.y += 2) {
        for (; r.y > r.pr.ey; r.y -= r.pr.ey - r.pr.sy + 1) ++r.z;
        ry[u] = r.y;
        rz[u] = r.z;
    }
    direct_rows<3>(d.g, r.pr, d.cs, d.ce, d.n, ry, rz, r.b, r.e);
}
__device__ __forceinline__ DirectRows first_rows(const DirectScan& d, const GroupTargets& t) {
    DirectRows r;
    r.pr = make_probe(d.g, t.x.x, t.x.y, t.x.z);
    r.y = r.pr.sy + ((threadIdx.x & 32u) != 0u ? 1 : 0);
    r.z = r.pr.sz;
    next_rows(d, r);
    return r;
}

// The candidates of the targets in `todo` (a mask of 32) by a direct scan: each
// lane walks every other row of its target's own stencil (r: the first three) and
// evaluates the candidates in range alone, r = 0 only with kSelf.  Bound by latency:
// three rows are looked up together and four candidates read together (a step of one
// million particles at 1 a cell, one row and candidate after the other: 386 us, now
// 335).
template <uint32_t kArrays, bool kSelf, class F, class G>
__device__ __forceinline__ void walk_direct(const DirectScan& d, DirectRows r, const GroupTargets& t,
                                            uint32_t todo, F&& pair, G&& every8) {
    if (((todo >> (threadIdx.x & 31u)) & 1u) == 0u) return;
    constexpr uint32_t kAhead = 4;
    const float h2 = d.g.h * d.g.h;
    uint32_t turn = 0u;
    auto run = [&](uint32_t b, uint32_t e) {
        for (uint32_t j = b; j < e; j += kAhead) {
            v4f q0[kAhead], q1[kAhead], q2[kAhead];
#pragma unroll
            for (uint32_t k = 0; k < kAhead; ++k) {
                const uint32_t at = min(j + k, e - 1u);
                q0[k] = *reinterpret_cast<const v4f*>(d.a0 + at);
                if constexpr (kArrays > 1) q1[k] = *reinterpret_cast<const v4f*>(d.a1 + at);
                if constexpr (kArrays > 2) q2[k] = *reinterpret_cast<const v4f*>(d.a2 + at);
            }
#pragma unroll
            for (uint32_t k = 0; k < kAhead; ++k) {
                const float dx = t.x.x - q0[k].x, dy = t.x.y - q0[k].y, dz = t.x.z - q0[k].z;
                const float r2 = dx * dx + dy * dy + dz * dz;
                if (j + k >= e || !(r2 < h2) || !(kSelf || r2 > 0.0f)) continue;  // a NaN too
                if constexpr (kArrays == 1)
                    pair(q0[k]);
                else if constexpr (kArrays == 2)
                    pair(q0[k], q1[k]);
                else
                    pair(q0[k], q1[k], q2[k]);
            }
            if ((++turn & 1u) == 0u) every8();
        }
    };
    for (;;) {
#pragma unroll
        for (int u = 0; u < 3; ++u) run(r.b[u], r.e[u]);
        if (r.z > r.pr.ez) break;
        next_rows(d, r);
    }
    every8();
}

// Whether the group's targets lie in few places: at most three runs of the same
// 2^g.run_bits cells, which are about the subgroups that walk_group would take one
// after the other, each with a look-up of rows, a wait and two lanes per member.
// A step of spray (us; direct scans from 3 runs on / 4 / 5 / 7 / never): one million
// at 0.2 a cell 327 / 327 / 337 / 342 / 945, at 1 a cell 342 / 345 / 393 / 473 / 470, at 4 a
// cell 341 / 320 / 320 / 324 / 315; a film of 200,000 one cell thick across the rows, 16
// a cell, 165 / 154 / 163 / 165 / 160.  (From 5 runs on with fewer loads together.)
constexpr uint32_t kMaxRuns = 3;
__device__ __forceinline__ bool few_runs(const GridView& g, const GroupTargets& t) {
    const uint32_t active = static_cast<uint32_t>(__ballot(t.active));
    const uint32_t from = lane_u32(t.key, 0) >> g.run_bits;
    const uint32_t to = lane_u32(t.key, 31 - __builtin_clz(active)) >> g.run_bits;
    if (to - from < kMaxRuns) return true;  // nearly all groups of a dense state
    const uint32_t run = t.key >> g.run_bits;
    const uint32_t before = static_cast<uint32_t>(__builtin_amdgcn_update_dpp(
        0, static_cast<int>(run), 0x138, 0xf, 0xf, false));  // wave_shr:1
    const uint32_t heads = static_cast<uint32_t>(__ballot(t.active && run != before)) | 1u;
    return static_cast<uint32_t>(__builtin_popcount(heads)) <= kMaxRuns;
}

// Whether some lane has more candidates in its first three rows than a direct scan is
// the faster for: spread groups at the surface of a dense state are walked together.
// A step (us, limit 28 / 40 / 56 / 72 / 100): 32,000 with a fifth above a pool 102 / 102 /
// 87 / 85 / 73, a film across the rows, 200,000, at 4 a cell 145 / 129 / 129 / 130 / 130,
// at 16 a cell 166 / 167 / 161 / 153 / 154; 24 scenes of 4096 to 98304, 24 steps, 5421 /
// 5417 / 5414 / 5429 / 5439.  Without a limit a step of one settled million took 9 us
// more.
constexpr uint32_t kMostCandidates = 72;
__device__ __forceinline__ bool many_candidates(const DirectRows& r, const GroupTargets& t) {
    uint32_t count = 0u;
#pragma unroll
    for (int u = 0; u < 3; ++u) count += r.e[u] > r.b[u] ? r.e[u] - r.b[u] : 0u;
    return __ballot(t.active && count > kMostCandidates) != 0ull;
}

// The sums of a group's targets: walk_group, which multiplies what a candidate
// out of range carries (v, A, B, ..) by 0.  That is no 0 if it is infinite or a
// NaN, so a target whose sums are not finite is taken again by a direct scan,
// which leaves such candidates out: then they are those of its neighbours.
// Targets that the filter does not hold are scanned directly too, and so are groups
// that are spread over many places.
// finite(): whether this lane's sums are; reset(): makes them 0; scan(): the
// DirectScan.
template <uint32_t kArrays, bool kSelf, class F, class G, class Ok, class Reset, class Scan>
__device__ __forceinline__ void walk_targets(const GridView& g, const GroupTargets& t, float inv_h,
                                             const uint32_t* __restrict__ cs,
                                             const uint32_t* __restrict__ ce,
                                             const uint4* __restrict__ bins, uint32_t n,
                                             const float4* __restrict__ a0,
                                             const float4* __restrict__ a1,
                                             const float4* __restrict__ a2, uint32_t tile,
                                             F&& pair, G&& every8, Ok&& finite, Reset&& reset,
                                             Scan&& scan) {
    uint32_t todo = static_cast<uint32_t>(__ballot(t.active));
    bool together = few_runs(g, t);
    DirectScan d;
    DirectRows rows;
    if (!together) {
        d = scan();
        rows = first_rows(d, t);
        together = many_candidates(rows, t);
    }
    if (together) {
        todo = walk_group<kArrays>(g, t, inv_h, cs, ce, bins, n, a0, a1, a2, tile, pair, every8);
        const uint64_t bad = __ballot(t.active && !finite());
        todo |= static_cast<uint32_t>(bad) | static_cast<uint32_t>(bad >> 32);
        if (todo == 0u) return;
        d = scan();
        rows = first_rows(d, t);
    }
    if ((todo >> (threadIdx.x & 31u)) & 1u) reset();
    walk_direct<kArrays, kSelf>(d, rows, t, todo, pair, every8);
}

}  // namespace sph
