// pairtile.hpp -- one wave walks the neighbours of 32 consecutive targets,
// with the matrix cores as the range filter.
//
// A wave owns a group of 32 targets, two lanes each (lane l and l + 32 share
// target l & 31 and take its even and its odd candidates).  The
// group's candidates -- the particles of every grid row that the group's
// x-window reaches -- are staged once, back to back, in the wave's own LDS
// tile, so there are no block barriers and no per-row phases.  For each 64
// staged candidates two V_MFMA_F32_32X32X8_F16 products form
//   |x_j - o|^2 - 2 (x_i - o).(x_j - o) + |x_i - o|^2 - h^2 - margin
// (o: a point among the targets) for all 32 targets in FP16, whose sign bits are
// the lanes' hit masks: one VALU instruction per 64 pairs instead of the seven
// of a distance test.  The margin covers the rounding of that form (its bound is
// at group_margin), so the masks hold every pair in range; a lane then takes
// its set bits in order and evaluates each pair from the staged global
// coordinates with the exact test, so the pairs summed and their values are
// those of a direct scan.
//
// The index of a candidate in the group's list decides the lane that takes it
// and its place in the order, so a target's sums depend on its group alone: not
// on the block size or the grid.
#pragma once

#include <type_traits>

#include "neighbors.hpp"

namespace sph {

constexpr uint32_t kGroupTargets = 32;
typedef float v2f __attribute__((ext_vector_type(2)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef float v16f __attribute__((ext_vector_type(16)));
typedef __fp16 v2h __attribute__((ext_vector_type(2)));
typedef _Float16 v4h __attribute__((ext_vector_type(4)));

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

__device__ __forceinline__ uint32_t uniform_u32(uint32_t v) {
    return static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(v)));
}
__device__ __forceinline__ uint32_t lane_u32(uint32_t v, int lane) {
    return static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(v), lane));
}
__device__ __forceinline__ float lane_f32(float v, int lane) {
    return __uint_as_float(lane_u32(__float_as_uint(v), lane));
}

// Inclusive prefix sum over the wave's 64 lanes (every lane active).
__device__ __forceinline__ uint32_t wave_scan_add(uint32_t v) {
    auto step = [&](auto ctrl, auto rows) {
        v += static_cast<uint32_t>(__builtin_amdgcn_update_dpp(
            0, static_cast<int>(v), decltype(ctrl)::value, decltype(rows)::value, 0xf, false));
    };
    step(std::integral_constant<int, 0x111>{}, std::integral_constant<int, 0xf>{});  // row_shr:1
    step(std::integral_constant<int, 0x112>{}, std::integral_constant<int, 0xf>{});  // row_shr:2
    step(std::integral_constant<int, 0x114>{}, std::integral_constant<int, 0xf>{});  // row_shr:4
    step(std::integral_constant<int, 0x118>{}, std::integral_constant<int, 0xf>{});  // row_shr:8
    step(std::integral_constant<int, 0x142>{}, std::integral_constant<int, 0xa>{});  // row_bcast:15
    step(std::integral_constant<int, 0x143>{}, std::integral_constant<int, 0xc>{});  // row_bcast:31
    return v;
}

// Targets of one group: lane l holds target l & 31 (both halves the same).
struct GroupTargets {
    float4 x;        // position (any w)
    uint32_t key;    // cell of the grid's own cell array (cell_offset taken off)
    bool active;
};

// A subgroup: the targets of a group that share a grid row and span at most
// g.span cells along it.
struct Subgroup {
    bool member;          // this lane's target
    int cy, cz;           // the row
    float x0, x1;         // first and last x offset from the grid origin (clamped into it)
    float ox, oy, oz;     // origin of the filter's coordinates: near the targets
    int y0, z0, ny, nz;   // rows reached: ny x nz from (y0, z0), inside the grid
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

// Lanes below `lanes` each copy 16 bytes from src[step * lane] to LDS at
// `to` + 16 lane (`to` wave-uniform), without passing through registers.
__device__ __forceinline__ void lds_copy16(const float4* src, uint32_t step, uint32_t to,
                                           uint32_t lanes) {
    const uint32_t lane = threadIdx.x & 63u;
    if (lane < lanes)
        __builtin_amdgcn_global_load_lds(
            reinterpret_cast<const __attribute__((address_space(1))) void*>(
                reinterpret_cast<uintptr_t>(src + step * lane)),
            reinterpret_cast<__attribute__((address_space(3))) void*>(to), 16, 0, 0);
}

// t / d for a quotient below 2^20 (d > 0; inv_d ~ 1 / d).
__device__ __forceinline__ uint32_t small_quotient(uint32_t t, uint32_t d, float inv_d) {
    uint32_t q = static_cast<uint32_t>(static_cast<float>(t) * inv_d);
    q -= q * d > t ? 1u : 0u;
    q += t - q * d >= d ? 1u : 0u;
    return q;
}

// A wave's tile of kCap candidates (a multiple of 64): their (x, .) as float4,
// with kVelocity their (v, .) too, and the 64 lanes' mask words of every 64
// candidates.  The two slots and the mask words past the last ones in use are
// where a lane that has finished points (it reads one word ahead).
template <uint32_t kCap, bool kVelocity>
struct PairTile {
    static constexpr uint32_t kSlots = 16u * (kCap + 2u);
    static constexpr uint32_t kMask = kVelocity ? 2u * kSlots : kSlots;
    static constexpr uint32_t kBytes = kMask + 4u * (kCap + 128u);
};

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

// A candidate whose position is not finite is replaced by a far one, and a
// target whose position is not finite is evaluated from -kFar, so neither meets
// anyone (it keeps its own NaN, and no pair adds one to a sum).
constexpr float kFar = 1e15f, kFar2 = 3e30f;

__device__ __forceinline__ float4 target_position(const GroupTargets& t) {
    const float q = t.x.x * t.x.x + t.x.y * t.x.y + t.x.z * t.x.z;
    return q < kFar2 ? t.x : make_float4(-kFar, -kFar, -kFar, t.x.w);
}

// Walks the candidates of a group: their (x, .) in `xs` and, with kVelocity,
// (v, .) in `vs`, in the internal x-order.  pair(xv...) evaluates this lane's
// target with one candidate: pair(x) or pair(x, v); every8() is called after at
// most nine of them, and at the end.
// tile: LDS address of the wave's PairTile; a longer list is taken kCap
// candidates at a time.
template <uint32_t kCap, bool kVelocity, class F, class G>
__device__ __forceinline__ void walk_group(const GridView& g, const GroupTargets& t, float inv_h,
                                           const uint32_t* __restrict__ cs,
                                           const uint32_t* __restrict__ ce,
                                           const uint4* __restrict__ bins, uint32_t n,
                                           const float4* __restrict__ xs,
                                           const float4* __restrict__ vs, uint32_t tile, F&& pair,
                                           G&& every8) {
    typedef PairTile<kCap, kVelocity> T;
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t half = lane >> 5;
    // A lane half converts 32 of 64 candidates; the first product takes the lower
    // half's (the upper half's target operand is 0), the second the upper's.
    // Row m of a product reads slot 2 r + q of its 32, where (q, r) are the lane
    // half and accumulator that receive row m: a lane's 32 mask bits
    // are the even (half 0) or odd slots of 64, so a target's hits, which lie
    // together along a row, fall evenly on its two lanes.
    const uint32_t m = lane & 31u;
    const uint32_t slot_of_row = 2u * (4u * (m >> 3) + (m & 3u)) + ((m >> 2) & 1u);
    uint32_t rem = static_cast<uint32_t>(__ballot(t.active));
    while (rem) {
        const Subgroup s = next_subgroup(g, t, rem);
        // Fills a tile to whole words: out of the members' range, yet finite in
        // FP16 (an infinity would make the products NaN, and its sign a hit).
        const v4f far = {s.ox + 100.0f * __builtin_amdgcn_rcpf(inv_h), s.oy, s.oz, 0.0f};
        // Target operands of the filter, in units of h: columns (-2 x, -2 y, -2 z, 1)
        // against rows (x, y, z, |x|^2), added to the column's |x|^2 - 1 - margin.
        const float sx = -s.ox * inv_h, sy = -s.oy * inv_h, sz = -s.oz * inv_h;
        const float ix = __builtin_fmaf(t.x.x, inv_h, sx), iy = __builtin_fmaf(t.x.y, inv_h, sy),
                    iz = __builtin_fmaf(t.x.z, inv_h, sz);
        const float qi = ix * ix + iy * iy + iz * iz;
        const float ci = s.member && qi < 1e4f ? qi - 1.0f - group_margin(qi) : 1e30f;
        const v4h none = {0, 0, 0, 0},
                  col = {static_cast<_Float16>(-2.0f * ix), static_cast<_Float16>(-2.0f * iy),
                         static_cast<_Float16>(-2.0f * iz), 1},
                  cols[2] = {half ? none : col, half ? col : none};
        v16f base;
#pragma unroll
        for (int r = 0; r < 16; ++r) base[r] = ci;
        const uint32_t rows = static_cast<uint32_t>(s.ny) * static_cast<uint32_t>(s.nz);
        for (uint32_t row0 = 0; row0 < rows; row0 += 64u) {
            uint32_t rb = 0u, re = 0u;
            if (row0 + lane < rows) {
                int y, z;
                row_of(s, row0 + lane, y, z);
                subgroup_row(g, s, cs, ce, bins, n, y, z, rb, re);
            }
            const uint32_t len = re - rb;
            const uint32_t end = wave_scan_add(len);
            const uint32_t total = lane_u32(end, 63);
            const int live_rows = static_cast<int>(min(64u, rows - row0));
            // A list longer than the tile is taken in `parts`, part p holding
            // every parts-th candidate from p on: each part then has its share
            // of every target's neighbours, and the lanes stay even.  (Modelled
            // takes per lane at 24 particles per h^3, 50 of them neighbours, with
            // 256 candidates at a time: 106 one stretch after the other, 77 so.)
            const uint32_t parts = (total + kCap - 1u) / kCap;
            const float inv_parts = __builtin_amdgcn_rcpf(static_cast<float>(parts));
            for (uint32_t part = 0; part < parts; ++part) {
                const uint32_t cnt = (total - part + parts - 1u) / parts;
                // Slots [first, past) of this lane's row.
                const uint32_t past = small_quotient(end - part + parts - 1u, parts, inv_parts);
                const uint32_t first = small_quotient(end - len - part + parts - 1u, parts, inv_parts);
                for (int r = 0; r < live_rows; ++r) {
                    const uint32_t s0 = lane_u32(first, r), s1 = lane_u32(past, r);
                    // Particle of slot k: its row's first one plus its place.
                    const uint32_t from = lane_u32(rb + len - end, r) + part;
                    for (uint32_t k = s0; k < s1; k += 64u) {
                        lds_copy16(xs + (from + parts * k), parts, tile + 16u * k, s1 - k);
                        if (kVelocity)
                            lds_copy16(vs + (from + parts * k), parts, tile + T::kSlots + 16u * k,
                                       s1 - k);
                    }
                }
                const uint32_t words = (cnt + 63u) >> 6;
                // Far candidates up to the end of the last 64, and two beyond
                // for the finished lanes: those are any target's, so out of
                // everyone's range wherever it is.
                for (uint32_t k = cnt + lane; k < 64u * words + 2u; k += 64u) {
                    lds_write<v4f>(tile + 16u * k,
                                   k < 64u * words ? far : v4f{kFar, kFar, kFar, 0.0f});
                    if (kVelocity)
                        lds_write<v4f>(tile + T::kSlots + 16u * k, v4f{0.0f, 0.0f, 0.0f, 0.0f});
                }
                const uint32_t mask0 = tile + T::kMask + 4u * lane;
                const uint32_t end_mask = mask0 + 256u * words;
                lds_write<uint32_t>(end_mask, 0x80000000u);
                lds_write<uint32_t>(end_mask + 256u, 0x80000000u);
                wait_vmem();
                wave_sync();
                for (uint32_t w = 0; w < words; ++w) {
                    const uint32_t at = tile + 16u * (64u * w + 32u * half + slot_of_row);
                    const v4f x = lds_read<v4f>(at);
                    keep4(x);
                    float dx = __builtin_fmaf(x.x, inv_h, sx), dy = __builtin_fmaf(x.y, inv_h, sy),
                          dz = __builtin_fmaf(x.z, inv_h, sz);
                    float q = dx * dx + dy * dy + dz * dz;
                    if (__ballot(!(q < kFar2)) != 0ull && !(q < kFar2)) {
                        lds_write<v4f>(at, far);
                        dx = 100.0f;
                        dy = dz = 0.0f;
                        q = 1e4f;
                    }
                    const v2h xy = __builtin_amdgcn_cvt_pkrtz(dx, dy),
                              zq = __builtin_amdgcn_cvt_pkrtz(dz, q);
                    const v4h rows8 = {static_cast<_Float16>(xy.x), static_cast<_Float16>(xy.y),
                                       static_cast<_Float16>(zq.x), static_cast<_Float16>(zq.y)};
                    uint32_t bits = 0u;
#pragma unroll
                    for (int k = 0; k < 2; ++k) {
                        const v16f d =
                            __builtin_amdgcn_mfma_f32_32x32x8f16(rows8, cols[k], base, 0, 0, 0);
#pragma unroll
                        for (int r = 0; r < 16; ++r)
                            bits = __builtin_amdgcn_alignbit(bits, __float_as_uint(d[r]), 31);
                    }
                    // No word is empty: the last slot stands in for none, and
                    // the exact test of pair() turns it down.
                    lds_write<uint32_t>(mask0 + 256u * w, max(bits, 1u));
                }
                wave_sync();
                // Each member's lane takes the set bits of its words in order;
                // a lane that has finished (or is no member) keeps taking the
                // far candidate past the end.  word: where the lane's current
                // word is, whose first slot is at 4 word + to_slots.  One
                // candidate is on its way while another is evaluated.
                const uint32_t to_slots = tile + 16u * half - 4u * mask0;
                uint32_t word = s.member ? mask0 : end_mask;
                uint32_t cur = lds_read<uint32_t>(word), nxt = lds_read<uint32_t>(word + 256u);
                auto take = [&](v4f& x, v4f& v) {
                    const uint32_t z = __builtin_clz(cur);
                    uint32_t first = 4u * word + to_slots;
                    asm("" : "+v"(first));  // two shift-and-adds, not three instructions
                    const uint32_t p = 32u * z + first;
                    x = lds_read<v4f>(p);
                    if (kVelocity) v = lds_read<v4f>(p + T::kSlots);
                    cur &= ~(0x80000000u >> z);
                    const bool over = cur == 0u;
                    cur = over ? nxt : cur;
                    word = over ? min(word + 256u, end_mask) : word;
                    nxt = lds_read<uint32_t>(word + 256u);
                };
                auto eval = [&](const v4f& x, const v4f& v) {
                    keep4(x);
                    if constexpr (kVelocity)
                        pair(x, v);
                    else
                        pair(x);
                };
                v4f xa, va, xb, vb;
                take(xa, va);
                uint32_t turn = 0u;
                do {
                    take(xb, vb);
                    eval(xa, va);
                    take(xa, va);
                    eval(xb, vb);
                    if ((++turn & 3u) == 0u) {
                        asm volatile("");  // a branch, not selects on every turn
                        every8();
                    }
                } while (__ballot(word != end_mask) != 0ull);
                eval(xa, va);
                every8();
                wave_sync();
            }
        }
    }
}

}  // namespace sph
