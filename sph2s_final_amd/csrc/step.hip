// step.hip -- the single-scale SPH step on gfx950.
//
// Pass order of Solver::Advance (SPH2S_FINAL_SINGLE_SCALE/Solver.cu:1082-1198):
//   hash+hist      cell hash per particle fused with the radix-sort digit
//                  histograms, plus the empty-cell reset of the ranges
//                  (computeHashs :401-424 and the two cudaMemsets :1118-1127)
//   radix passes   stable (hash, slot) sort          (thrust, :1110-1115)
//   k_order        cell start/end (reorderAndComputeCellStartEndD :478-534),
//                  internal x-order of each cell (reads the state through the
//                  sort's permutation) and its x-bin table, and the state in
//                  sorted slots when a pass needs it
//   k_density      Poly6 density                    (:536-599, :198-229)
//   k_force        spiky pressure + viscosity Laplacian (+ tension) fused with
//                  symplectic Euler and the wall clamp (:601-711, :713-755)
//
// State layout: float4 pos = (x, y, z, persistent id bits), float4 vel =
// (vx, vy, vz, 0), one 16-byte load per particle.  Within one row (cy, cz)
// of the grid the cells cx are consecutive hashes, so a stencil row of up to
// three cells is one contiguous run of sorted particles.
#include <vector>

#include "neighbors.hpp"
#include "diagnostics.hpp"
#include "pairtile.hpp"
#include "pairwalk.hpp"
#include "walls.hpp"

namespace sph {
namespace {

constexpr int kBlock = 256;

// Internal x-order: slot s of the sorted order (cell c, run [b, e)) moves to
// b + rank, its rank by (x, sorted slot) among the cell's particles, so each
// cell's particles are sorted by x (deterministically: ties keep the sorted
// order).  Cells are short (tens to a few hundred particles), so the rank is
// a direct count over the cell.  The block stages
// the x of every particle in its cells' runs in LDS (lanes of one cell then
// read the same LDS word each step); runs beyond the staged range are read
// from global memory.  The state of sorted slot j is pos[perm[j]], vel[perm[j]]
// of the previous order; with kCopy it is also written to tpos[j], tvel[j].
//
// A run's bounds are where neighbouring sorted keys differ: inside the block
// from ballots, beyond it from the 64 keys on either side, and only for a cell
// of more particles by a search of the sorted keys.  The first and last slot of
// a run write the cell's range.  Bound by latency (two rounds of loads) and, at
// one million, by its 76 MB (15 us at the card's copy rate).  Before, the ranges
// were a kernel of their own and the ranks compared floats and slots apart: us
// at 4096 particles / one million 4.6 + 5.8 / 4.8 + 23, now 4.5 / 19.
constexpr int kXorderTile = 2048;

// Bits that order as unsigned like the floats do (-0 as 0; NaNs of either sign
// beyond the infinities), and back.
__device__ __forceinline__ uint32_t ordered_bits(float x) {
    const uint32_t u = x == x ? __float_as_uint(x + 0.0f) : 0x7FC00000u;
    return u ^ (static_cast<uint32_t>(static_cast<int32_t>(u) >> 31) | 0x80000000u);
}
__device__ __forceinline__ float from_ordered(uint32_t u) {
    return __uint_as_float(u ^ ((u >> 31) ? 0x80000000u : 0xFFFFFFFFu));
}

// The first index in [lo, hi) of the sorted keys that holds `key` or more
// (kAfter: more than `key`), or hi.  All lanes of a wave call it; 64 probes a
// round.
template <bool kAfter>
__device__ __forceinline__ uint32_t search_keys(const uint32_t* __restrict__ skeys, uint32_t lo,
                                                uint32_t hi, uint32_t key, uint32_t num_cells) {
    const uint32_t lane = threadIdx.x & 63u;
    while (lo < hi) {
        const uint32_t step = (hi - lo + 63u) / 64u;
        const uint32_t at = lo + lane * step;
        const uint32_t k = at < hi ? min(skeys[at], num_cells - 1) : 0xFFFFFFFFu;
        const uint64_t found = __ballot(kAfter ? k > key : k >= key);  // lanes past hi among them
        const uint32_t f = found ? static_cast<uint32_t>(__builtin_ctzll(found)) : 64u;
        if (f > 0u) lo += (f - 1u) * step + 1u;
        if (f > 0u && f < 64u) hi = min(hi, lo + step - 1u);
        if (f == 0u) hi = lo;
    }
    return lo;
}

template <bool kBatched, bool kCopy>
__global__ __launch_bounds__(kBlock) void k_order(const uint32_t* __restrict__ skeys,
                                                  const uint32_t* __restrict__ perm,
                                                  const float4* __restrict__ pos,
                                                  const float4* __restrict__ vel,
                                                  float4* __restrict__ tpos,
                                                  float4* __restrict__ tvel,
                                                  uint32_t* __restrict__ cell_start,
                                                  uint32_t* __restrict__ cell_end,
                                                  const uint32_t* __restrict__ n_dev, StepParams p,
                                                  const SceneParams* __restrict__ scenes,
                                                  float4* __restrict__ ipos,
                                                  float4* __restrict__ ivel,
                                                  uint32_t* __restrict__ i2r,
                                                  uint4* __restrict__ bins) {
    __shared__ uint32_t xs_tile[kXorderTile];
    __shared__ uint64_t heads[kBlock / 64];
    __shared__ uint32_t edge[2];  // where the block's first run starts, its last run ends
    const uint32_t n = *n_dev;
    const uint32_t block0 = blockIdx.x * kBlock;
    if (block0 >= n) return;  // block-uniform
    const uint32_t wave = uniform_u32(threadIdx.x >> 6), lane = threadIdx.x & 63u;
    const uint32_t s = block0 + threadIdx.x, end = min(block0 + kBlock, n);
    const bool active = s < n;
    // Keys are clamped cell hashes (< num_cells) and perm is a permutation of
    // [0, n); the min() guards keep every access in bounds regardless.
    auto key_at = [&](uint32_t j) { return min(skeys[j], p.num_cells - 1); };
    auto source = [&](uint32_t j) { return min(perm[j], n - 1); };
    // Two rounds of loads: the keys and the sources of the block's slots and of
    // 64 slots on either side (waves 0 and 1 look at the keys there, 2 and 3
    // take the x), then the states.
    const uint32_t own = active ? s : end - 1u;
    const uint32_t src = source(own);
    const uint32_t key = key_at(own);
    const uint32_t before = key_at(max(own, 1u) - 1u);
    const bool low = (wave & 1u) == 0u;  // the slots below the block, nearest first, or above it
    const bool in = low ? lane < block0 : end + lane < n;
    const uint32_t at = in ? (low ? block0 - 1u - lane : end + lane) : own;
    const uint32_t key_last = key_at(end - 1u);
    const uint32_t* const list = wave < 2u ? skeys : perm;
    const uint32_t beside = min(list[at], (wave < 2u ? p.num_cells : n) - 1u);
    // As vectors: a struct copy of which the x is used here goes through an array
    // in LDS, whose index reads the dispatch packet in host memory (10 us).
    const v4f xs = *reinterpret_cast<const v4f*>(pos + src);
    const v4f vs = *reinterpret_cast<const v4f*>(vel + src);
    if (wave >= 2u && in) xs_tile[low ? 63u - lane : 64u + (end - block0) + lane] = ordered_bits(pos[beside].x);
    if (active) xs_tile[64u + threadIdx.x] = ordered_bits(xs.x);
    const bool head = active && (s == 0u || before != key);
    const uint64_t wave_heads = __ballot(head);
    if (lane == 0u) heads[wave] = wave_heads;
    if (wave == 0u) {
        const uint32_t k0 = uniform_u32(key);  // block0's
        const uint64_t other = ~__ballot(in && beside == k0);
        uint32_t b = block0;
        if ((wave_heads & 1u) == 0u)
            b = other ? block0 - static_cast<uint32_t>(__builtin_ctzll(other))
                      : search_keys<false>(skeys, 0u, block0 - 64u, k0, p.num_cells);
        if (lane == 0u) edge[0] = b;
    } else if (wave == 1u) {
        const uint32_t k1 = uniform_u32(key_last);
        const uint64_t other = ~__ballot(in && beside == k1);
        const uint32_t e = other ? end + static_cast<uint32_t>(__builtin_ctzll(other))
                                 : search_keys<true>(skeys, min(end + 64u, n), n, k1, p.num_cells);
        if (lane == 0u) edge[1] = e;
    }
    __syncthreads();
    // This slot's run [b, e): heads of its own wave, or of the nearest wave that
    // has one (wave-uniform), or the block's edge.
    uint32_t b = edge[0], e = edge[1];
    for (uint32_t w = 0; w < wave; ++w)
        if (const uint64_t m = heads[w])
            b = block0 + 64u * w + 63u - static_cast<uint32_t>(__builtin_clzll(m));
    for (uint32_t w = kBlock / 64; --w > wave;)
        if (const uint64_t m = heads[w]) e = block0 + 64u * w + static_cast<uint32_t>(__builtin_ctzll(m));
    const uint64_t upto_lane = ~0ull >> (63u - lane);
    if (const uint64_t m = wave_heads & upto_lane)
        b = block0 + 64u * wave + 63u - static_cast<uint32_t>(__builtin_clzll(m));
    if (const uint64_t m = wave_heads & ~upto_lane)
        e = block0 + 64u * wave + static_cast<uint32_t>(__builtin_ctzll(m));
    // The x of slots [from, upto) are staged, from `tile` on.
    uint32_t from = block0 - min(block0, 64u), upto = min(end + 64u, n);
    const uint32_t* tile = xs_tile + 64u - (block0 - from);
    if (edge[0] < from || edge[1] > upto) {  // block-uniform: a run that reaches further
        from = edge[0];
        upto = min(edge[1], from + kXorderTile);
        tile = xs_tile;
        __syncthreads();
        for (uint32_t k = threadIdx.x; k < upto - from; k += kBlock)
            xs_tile[k] = ordered_bits(pos[source(from + k)].x);
        __syncthreads();
    }
    if (!active) return;
    if (head) cell_start[key] = s;
    if (e == s + 1u) cell_end[key] = e;
    if (kCopy) {
        *reinterpret_cast<v4f*>(tpos + s) = xs;
        *reinterpret_cast<v4f*>(tvel + s) = vs;
    }
    const bool staged = b >= from && e <= upto;
    // rank: particles before s in (x, sorted slot) order; xg: the smallest x
    // after it, which is the x of the next particle in the cell's x-order.  One
    // 64-bit compare a candidate, which counts s itself too.
    uint32_t upto_s = 0, next = 0xFFFFFFFFu;
    const uint64_t mine = static_cast<uint64_t>(ordered_bits(xs.x)) << 32 | s;
    auto count = [&](uint32_t j, uint32_t u) {
        const bool after = (static_cast<uint64_t>(u) << 32 | j) > mine;
        upto_s += after ? 0u : 1u;
        next = after ? min(next, u) : next;
    };
    if (staged) {
        const uint32_t* const xr = tile + (b - from);
        const uint32_t m = e - b;
        uint32_t k = 0;
        for (; k + 4u <= m; k += 4u) {
            const uint32_t u0 = xr[k], u1 = xr[k + 1], u2 = xr[k + 2], u3 = xr[k + 3];
            count(b + k, u0);
            count(b + k + 1, u1);
            count(b + k + 2, u2);
            count(b + k + 3, u3);
        }
        for (; k < m; ++k) count(b + k, xr[k]);
    } else {
        for (uint32_t j = b; j < e; ++j) count(j, ordered_bits(pos[source(j)].x));
    }
    const uint32_t rank = upto_s - 1u;
    const float xg = from_ordered(next);
    const uint32_t q = b + rank;
    *reinterpret_cast<v4f*>(ipos + q) = xs;
    *reinterpret_cast<v4f*>(ivel + q) = vs;
    i2r[q] = s;

    // The cell's x-bin table: cumulative counts of its kXBins x-bins (one
    // byte each).  Bins are non-decreasing along the x-order, so the particle
    // of rank r holds the count r + 1 for every bin from its own up to (not
    // including) the next particle's bin, or up to the last bin if it is the
    // cell's last particle; the first particle also writes 0 for the bins
    // below its own.  Every entry is written by exactly one particle.  Cells
    // of more than kXBinMax particles get the all-ones marker (no trimming).
    uint8_t* t = reinterpret_cast<uint8_t*>(bins + static_cast<size_t>(key) * kXBinQuads);
    const uint32_t cnt = e - b;
    if (cnt > kXBinMax) {
        if (rank == 0)
            for (int k = 0; k < kXBins; ++k) t[k] = static_cast<uint8_t>(kXBinUnbinned);
        return;
    }
    float ox = p.ox, spacing = p.spacing, inv = 1.0f / p.spacing;
    int dx = p.dx;
    if (kBatched) {
        const GridView& g = scenes[__float_as_uint(vs.w)].g;
        ox = g.ox;
        spacing = g.spacing;
        inv = g.inv_spacing;
        dx = g.dx;
    }
    // A NaN x, last in its cell (which is the row's first), is in the last bin.
    const float cx = static_cast<float>(cell_coord(xs.x, ox, spacing, dx));
    auto bin = [&](float x) {
        const float f = (x - ox) * inv - cx;
        return f < 1.0f ? xbin_of(f) : kXBins - 1;
    };
    const int kq = bin(xs.x);
    const int kn = (rank + 1 < cnt) ? max(kq, bin(xg)) : kXBins;
    if (rank == 0)
        for (int k = 0; k < kq; ++k) t[k] = 0u;
    const uint8_t c = static_cast<uint8_t>(rank + 1);
    for (int k = kq; k < kn; ++k) t[k] = c;
}


// Launch shapes of the neighbour passes, selected at run time by the tune word
// (StepParams::tune; 0 = the defaults).  Every shape computes bit-identical
// results: a target's sums depend on its group of 32 alone (pairtile.hpp), and
// the shape only decides which wave handles which group.  Walled scenes' passes in
// row order have one shape.
//   bits 0-3   density, bits 4-7 force: waves per block (kTileWaves)
//   bits 8-11  density grid:       one block per its waves' groups, or a
//   bits 12-15 force grid:         persistent grid of 1, 2, 4, 8 blocks per CU
//                                  looping over those blocks
//   bits 16-17 density block size, bits 18-19 force block size: 256 (0), 128
//              (1), 512 (2) threads, as far as the block's LDS goes; a non-zero
//              field needs waves-per-block field 0
//   bits 20-21 density, bits 22-23 force: groups taken by a wave one after the
//              other, 1 (0) or 2 (1), with the default block (single scenes)
//
typedef PairTile<1> DensityTile;
typedef PairTile<2> ForceTile;
// Waves share nothing but the launch, so the number is a matter of tails and is left
// to the tuner.  Density / force of 15 steps in ms with 4 waves, 1, 2, 3 and 5: 4.1 million
// in 64 scenes 5.26 / 7.45, 4.91 / 6.72, 5.02 / 7.06, 5.17 / 7.61, 7.22 / 11.1; one million
// 1.54 / 2.12, 1.47 / 2.01 with 1; 32,768 0.343 / 0.387 with either.  Values 6 to 9 were
// variants of their own once and stay valid words.
constexpr uint32_t kTileWaves[] = {4, 1, 2, 3, 5, 6, 4, 4, 4, 4};
constexpr uint32_t kMaxBlockLds = 64u << 10;
// Groups in a row that one XCD takes (32, 128 and 512: within 2%).
constexpr uint32_t kXcdChunkGroups = 128;
constexpr uint32_t kPersistPerCu[] = {0, 1, 2, 4, 8};
constexpr int kWavesPerBlock = kBlock / 64;
const SceneParams* const kNoScenes = nullptr;

// Internal x-order of a neighbour pass: the pass reads the internal-order
// state, trims rows with the cells' x-bins and writes results at i2r[slot].
struct XOrder {
    const uint32_t* i2r;
    const uint4* bins;
    const float4* bacc;  // force: boundary acceleration per sorted slot (or NULL)
    // force: device error word; the integration ORs kDevErrNonFinite into it
    // when it writes a NaN or infinite position or velocity (or NULL).
    uint32_t* err = nullptr;
};
constexpr uint32_t kNumCus = 256;

struct LaunchShape {
    dim3 grid, block;
    uint32_t nvb;     // blocks of `block` waves to cover
    uint32_t per;     // groups per wave
    uint32_t lds;     // bytes of LDS per block
    uint32_t chunk;   // consecutive blocks that one XCD takes
};

inline LaunchShape launch_shape(uint32_t groups, uint32_t tile_bytes, uint32_t waves_idx,
                                uint32_t persist_idx, uint32_t block_idx, uint32_t per) {
    LaunchShape s;
    uint32_t waves = block_idx == 1 ? 2u : block_idx == 2 ? 8u : kTileWaves[std::min(waves_idx, 9u)];
    waves = std::min(waves, kMaxBlockLds / tile_bytes);
    s.lds = waves * tile_bytes;
    s.per = per;
    s.chunk = std::max(1u, kXcdChunkGroups / (waves * per));
    s.nvb = std::max(1u, (groups + waves * per - 1) / (waves * per));
    s.block = dim3(64u * waves);
    uint32_t g = s.nvb;
    if (persist_idx > 0 && persist_idx < 5) {
        g = std::min(s.nvb, kPersistPerCu[persist_idx] * kNumCus);
        // A multiple of the XCD count keeps each virtual block on the XCD the
        // chunked mapping assigns it to.
        if (g > kNumXcds) g -= g % kNumXcds;
    }
    s.grid = dim3(g);
    return s;
}

// The pair arithmetic below is written with explicit fused multiply-adds and
// contraction off, so every kernel that evaluates a pair rounds it the same
// way whatever the surrounding code: the launch variants of a pass, which
// inline it into different code, give identical sums.
__device__ __forceinline__ float dist2(float dx, float dy, float dz) {
#pragma clang fp contract(off)
    return __builtin_fmaf(dz, dz, __builtin_fmaf(dy, dy, dx * dx));
}

// Poly6 weight in units of h^2: a = 1 - r^2 / h^2 clamped to [0, 1] (one
// fused multiply-add with the clamp modifier), so (h^2 - r^2)^3 = h^6 a^3 for
// r < h and the term is 0 otherwise; a = 1 for r = 0.
__device__ __forceinline__ float poly6_unit(const float4& xi, const v4f& xj, float inv_h2) {
#pragma clang fp contract(off)
    const float dx = xi.x - xj.x, dy = xi.y - xj.y, dz = xi.z - xj.z;
    const float r2 = dist2(dx, dy, dz);
    return __builtin_amdgcn_fmed3f(__builtin_fmaf(-r2, inv_h2, 1.0f), 0.0f, 1.0f);
}

// The first arguments of k_density and k_force, in their order (arrays: of the
// candidates), and their direct scan's view of them.
struct WalkArguments {
    GridView g;
    const uint32_t *cs, *ce, *n_dev;
    const float4 *a0, *a1;
    const SceneParams* scenes;
};
static_assert(offsetof(WalkArguments, cs) == (sizeof(GridView) + 7) / 8 * 8, "as kernel arguments lie");
template <bool kBatched>
__device__ __forceinline__ DirectScan scan_again(uint32_t scene) {
    const WalkArguments w = first_arguments<WalkArguments>();
    return DirectScan{kBatched ? w.scenes[scene].g : w.g, w.cs, w.ce, *w.n_dev, w.a0, w.a1, nullptr};
}

// computeDensitiesPressuresD + computeDensityCell (Solver.cu:198-229,536-599):
// rho_i = m c6 sum_{r_ij < h} (h^2 - r_ij^2)^3, self included, evaluated as
// (m c6 h^6) sum a^3 with a = 1 - r_ij^2 / h^2 (poly6_unit).  Terms are added in
// FP32, with kKahan at most nine in a row, whose sums are added in FP64.
// Also emits the per-particle factors the force pass needs for every
// neighbour j: A_j = k (rho_j - rho0) / rho_j^2 and B_j = 1 / rho_j, packed
// with the state as (x, A) and (v, B), which the force pass copies to LDS as
// they lie.  Bound by VALU issue (92% of its time over a dam break of one million, by
// counters, with 89% of the lanes active).
// Against one lane per target with a block-staged tile per grid row (us, before
// -> now): 4096 particles 29 -> 18, 24 scenes of 4096..98304 72 -> 63, one
// million 138 -> 134, one million at rest 95 -> 80.  At one million 23 of them go
// to finding the rows, 22 to the filter products and their masks, and most of the
// rest is takes and staging.  Five waves per SIMD (96 VGPRs): with four 63 and
// 143, with six (spills) 67 and 144 us.
// Batched scenes (kBatched): a group's constants come from scenes[id]; runs
// never leave a scene because each scene's cells occupy their own range of the
// global cell array.
template <bool kKahan, bool kFinalize, bool kBatched>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(5))) void k_density(
    GridView g_in, const uint32_t* __restrict__ cs, const uint32_t* __restrict__ ce,
    const uint32_t* __restrict__ n_dev, const float4* __restrict__ ipos,
    const float4* __restrict__ ivel, const SceneParams* __restrict__ scenes,
    const uint32_t* __restrict__ skeys, StepParams p_in, float* __restrict__ rho,
    float2* __restrict__ aux, float4* __restrict__ ixa, float4* __restrict__ ivb,
    const uint4* __restrict__ groups, uint32_t n_groups, XOrder xo, LaunchShape sh) {
    extern __shared__ __align__(kTileAlign) unsigned char lds[];
    const uint32_t wave = uniform_u32(threadIdx.x >> 6), waves = blockDim.x >> 6;
    const uint32_t tile = lds_address(lds) + wave * DensityTile::kBytes;
    const uint32_t n = *n_dev;
    for (uint32_t vb = blockIdx.x; vb < sh.nvb; vb += gridDim.x) {
        const uint32_t first = (xcd_local_block(vb, sh.nvb, sh.chunk) * waves + wave) * sh.per;
        for (uint32_t group = first; group < first + sh.per; ++group) {
            const GroupRange gr = group_range<kBatched>(group, n, groups, n_groups);
            if (gr.start >= gr.end) continue;
            const StepParams& p = kBatched ? scenes[gr.scene].p : p_in;
            const GridView& g = kBatched ? scenes[gr.scene].g : g_in;
            uint32_t s;
            const GroupTargets t = load_targets(g, gr, ipos, skeys, s);
            const float4 xi = t.x;
            const float inv_h2 = p.inv_h2;
            double sum64 = 0.0;
            float sum32 = 0.0f;
            walk_targets<1, true>(
                g, t, p.inv_h, cs, ce, xo.bins, n, ipos, nullptr, nullptr, tile, [&](const v4f& x) {
#pragma clang fp contract(off)
                    const float a = poly6_unit(xi, x, inv_h2);
                    sum32 = __builtin_fmaf(a * a, a, sum32);
                },
                [&] {
                    if (kKahan) {
                        sum64 += static_cast<double>(sum32);
                        sum32 = 0.0f;
                    }
                },
                [] { return true; },
                [&] {
                    sum64 = 0.0;
                    sum32 = 0.0f;
                },
                [&] { return scan_again<kBatched>(gr.scene); });
            const float r = p.c6m_h6 * (kKahan ? static_cast<float>(both_halves(sum64))
                                               : both_halves(sum32));
            if (t.active && (threadIdx.x & 32u) == 0u) {
                const uint32_t o = xo.i2r[s];
                rho[o] = r;
                if (kFinalize) {
                    const float4 v = ivel[s];
                    const float inv = __builtin_amdgcn_rcpf(r);
                    const float A = p.stiffness * (r - p.rest_density) * inv * inv;
                    ixa[s] = make_float4(t.x.x, t.x.y, t.x.z, A);
                    ivb[s] = make_float4(v.x, v.y, v.z, inv);
                    if (aux) aux[o] = make_float2(A, inv);
                }
            }
        }
    }
}

// Pair sums of the force pass for one target i (position xi, velocity vi,
// A_i): pressure P, viscosity V and tension T.
template <bool kTension>
struct PairSums {
    float Px = 0.f, Py = 0.f, Pz = 0.f;
    float Vx = 0.f, Vy = 0.f, Vz = 0.f;
    float Tx = 0.f, Ty = 0.f, Tz = 0.f;

    // xa = (x_j, A_j), vb = (v_j, B_j), x_j finite.  Branch-free: out of range
    // (h - r) clamps to 0, and at r = 0 it is 0 too (0 * inf is a NaN, which
    // the clamp takes to 0), with 1 / r held finite, so such a pair adds 0 if
    // v, A and B are finite (walk_targets sees to the others).
    __device__ __forceinline__ void add(const float4& xi, const float4& vi, float ai, float h,
                                        float h2, const v4f& xa, const v4f& vb) {
#pragma clang fp contract(off)
        const float dx = xi.x - xa.x, dy = xi.y - xa.y, dz = xi.z - xa.z;
        const float r2 = dist2(dx, dy, dz);
        const float rs = __builtin_amdgcn_rsqf(r2);
        const float hr = __builtin_amdgcn_fmed3f(__builtin_fmaf(-r2, rs, h), 0.0f, h);
        const float inv_r = __builtin_amdgcn_fmed3f(rs, 0.0f, 2e19f);
        const float tpr = (ai + xa.w) * hr * hr * inv_r;
        Px = __builtin_fmaf(tpr, dx, Px);
        Py = __builtin_fmaf(tpr, dy, Py);
        Pz = __builtin_fmaf(tpr, dz, Pz);
        const float tvs = hr * vb.w;
        Vx = __builtin_fmaf(tvs, vb.x - vi.x, Vx);
        Vy = __builtin_fmaf(tvs, vb.y - vi.y, Vy);
        Vz = __builtin_fmaf(tvs, vb.z - vi.z, Vz);
        if (kTension) {
            const float a = __builtin_amdgcn_fmed3f(h2 - r2, 0.0f, h2);
            const float w = a * a * a;
            Tx = __builtin_fmaf(w, dx, Tx);
            Ty = __builtin_fmaf(w, dy, Ty);
            Tz = __builtin_fmaf(w, dz, Tz);
        }
    }

    __device__ __forceinline__ bool finite() const {
        return __builtin_isfinite(((Px + Py) + (Pz + Vx)) + ((Vy + Vz) + ((Tx + Ty) + Tz)));
    }
};

// The force pass's result for target i at sorted slot o: the acceleration
// (plus the boundary acceleration bacc[o] when bacc is non-NULL), then, with
// kIntegrate, integrateD (Solver.cu:713-755): v += dt a; x += dt v; and the
// wall clamp.  Without kIntegrate only the acceleration is written.
template <bool kTension, bool kIntegrate>
__device__ __forceinline__ void force_finish(const PairSums<kTension>& S, const StepParams& p,
                                             const float4& xi, const float4& vi,
                                             const float2& ai, uint32_t o,
                                             const float4* __restrict__ bacc, float dt,
                                             float4* __restrict__ pos, float4* __restrict__ vel,
                                             float4* __restrict__ accel,
                                             uint32_t* __restrict__ err) {
#pragma clang fp contract(off)
    const float vc = p.visc * ai.y;
    float ax = __builtin_fmaf(vc, S.Vx, p.c45m * S.Px) + p.gx;
    float ay = __builtin_fmaf(vc, S.Vy, p.c45m * S.Py) + p.gy;
    float az = __builtin_fmaf(vc, S.Vz, p.c45m * S.Pz) + p.gz;
    if (kTension) {
        const float tc = p.tens * ai.y;
        ax = __builtin_fmaf(-tc, S.Tx, ax);
        ay = __builtin_fmaf(-tc, S.Ty, ay);
        az = __builtin_fmaf(-tc, S.Tz, az);
    }
    if (bacc) {  // a_i = f_i / rho_i + b_i + g (Solver.cu:708-710)
        const float4 b = bacc[o];
        ax += b.x;
        ay += b.y;
        az += b.z;
    }
    if (!kIntegrate) {
        accel[o] = make_float4(ax, ay, az, 0.0f);
        return;
    }
    float vx = __builtin_fmaf(dt, ax, vi.x), vy = __builtin_fmaf(dt, ay, vi.y),
          vz = __builtin_fmaf(dt, az, vi.z);
    float x = __builtin_fmaf(dt, vx, xi.x), y = __builtin_fmaf(dt, vy, xi.y),
          z = __builtin_fmaf(dt, vz, xi.z);
    if (p.flags & SPH_FLAG_WALL_CLAMP) {
        const float e = p.restitution;
        if (x < p.lox) { x = p.lox; vx = -e * vx; }
        if (x > p.hix) { x = p.hix; vx = -e * vx; }
        if (y < p.loy) { y = p.loy; vy = -e * vy; }
        if (y > p.hiy) { y = p.hiy; vy = -e * vy; }
        if (z < p.loz) { z = p.loz; vz = -e * vz; }
        if (z > p.hiz) { z = p.hiz; vz = -e * vz; }
    }
    pos[o] = make_float4(x, y, z, xi.w);
    vel[o] = make_float4(vx, vy, vz, vi.w);
    if (accel) accel[o] = make_float4(ax, ay, az, 0.0f);
    // A NaN or infinity in any component makes the sum non-finite.
    if (err && !__builtin_isfinite(((x + y) + (z + vx)) + (vy + vz))) atomicOr(err, kDevErrNonFinite);
}

// a_i = m c45 sum_j (A_i + A_j)(h-r)^2/r x_ij            (pressure)
//     + (mu m c45 / rho_i) sum_j B_j (h-r)(v_j - v_i)     (viscosity)
//     - (sigma m c6 / rho_i) sum_j (h^2-r^2)^3 x_ij       (tension)
//     + g,                     0 < r_ij < h
// which is f_i / rho_i of Solver.cu:231-309,601-711 with rho_i factored out,
// fused with integrateD (Solver.cu:713-755) and the wall clamp.
//
// With kIntegrate = false (two-scale own-set pass, XSPH) the kernel only writes
// the acceleration, gravity included, to accel.
//
// Bound by VALU issue (95% of its time over a dam break of one million, by counters,
// with 92% of the lanes active).  A queue of hits per lane, filled by distance tests on a
// block-staged tile, spent most of its time on lanes waiting for the slowest
// and on block barriers; two lanes per target with the matrix filter's masks
// take (us, before -> now): 4096 particles 50 -> 20, 24 scenes of 4096..98304
// 116 -> 90, one million 320 -> 200, one million at rest 150 -> 110.
template <bool kTension, bool kIntegrate, bool kBatched>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(4))) void k_force(
    GridView g_in, const uint32_t* __restrict__ cs, const uint32_t* __restrict__ ce,
    const uint32_t* __restrict__ n_dev, const float4* __restrict__ ixa,
    const float4* __restrict__ ivb, const SceneParams* __restrict__ scenes,
    const float4* __restrict__ ipos, const float4* __restrict__ ivel,
    const uint32_t* __restrict__ skeys, StepParams p_in, float dt, float4* __restrict__ pos,
    float4* __restrict__ vel, float4* __restrict__ accel, const uint4* __restrict__ groups,
    uint32_t n_groups, XOrder xo, LaunchShape sh) {
    extern __shared__ __align__(kTileAlign) unsigned char lds[];
    const uint32_t wave = uniform_u32(threadIdx.x >> 6), waves = blockDim.x >> 6;
    const uint32_t tile = lds_address(lds) + wave * ForceTile::kBytes;
    const uint32_t n = *n_dev;
    for (uint32_t vb = blockIdx.x; vb < sh.nvb; vb += gridDim.x) {
        const uint32_t first = (xcd_local_block(vb, sh.nvb, sh.chunk) * waves + wave) * sh.per;
        for (uint32_t group = first; group < first + sh.per; ++group) {
            const GroupRange gr = group_range<kBatched>(group, n, groups, n_groups);
            if (gr.start >= gr.end) continue;
            const StepParams& p = kBatched ? scenes[gr.scene].p : p_in;
            const GridView& g = kBatched ? scenes[gr.scene].g : g_in;
            uint32_t s;
            const GroupTargets t = load_targets(g, gr, ixa, skeys, s);
            const float4 xi = t.x;
            const float4 vi = ivb[t.active ? s : gr.start];
            PairSums<kTension> S;
            walk_targets<2, false>(
                g, t, p.inv_h, cs, ce, xo.bins, n, ixa, ivb, nullptr, tile,
                [&](const v4f& x, const v4f& v) { S.add(xi, vi, t.x.w, p.h, p.h2, x, v); }, [] {},
                [&] { return S.finite(); }, [&] { S = PairSums<kTension>{}; },
                [&] { return scan_again<kBatched>(gr.scene); });
            S.Px = both_halves(S.Px);
            S.Py = both_halves(S.Py);
            S.Pz = both_halves(S.Pz);
            S.Vx = both_halves(S.Vx);
            S.Vy = both_halves(S.Vy);
            S.Vz = both_halves(S.Vz);
            if (kTension) {
                S.Tx = both_halves(S.Tx);
                S.Ty = both_halves(S.Ty);
                S.Tz = both_halves(S.Tz);
            }
            if (t.active && (threadIdx.x & 32u) == 0u) {
                float4 x = t.x, v = vi;
                if (kIntegrate) {  // the id and tag words come with the unpacked state
                    x.w = ipos[s].w;
                    v.w = ivel[s].w;
                }
                force_finish<kTension, kIntegrate>(S, p, x, v, make_float2(t.x.w, vi.w), xo.i2r[s],
                                                   xo.bacc, dt, pos, vel, accel, xo.err);
            }
        }
    }
}

// ---- walled scenes ---------------------------------------------------------
// One lane per target and the sums in row order: density in plain FP32 per grid
// row with the rows' sums combined by Kahan compensation, force in one chain.
// A boundary particle's push rises so steeply that the last bits of a velocity
// grow by 10^4 within four steps (200,000 particles in the reference's tank:
// largest velocity difference, over the RMS velocity, of the same sums in the
// group walk's order 3e-4 to 1.6e-3, by the initial jitter), so scenes with
// walls keep this order of additions and with it their trajectories.  The group
// walk would take the four steps from 826 to 739 us.  The XSPH and two-scale forms,
// which integrate in a later kernel, take the group walk with walls too.  Neither
// order is the nearer one to 64 bits: four XSPH steps of that tank were off by at
// most 1.16e-3, 7.7e-4 and 8.1e-4 of the RMS velocity (three initial jitters) with
// sums by rows and by 1.11e-3, 7.6e-4 and 8.0e-4 with the walk's, the RMS by 1.92e-5 with
// both; the orders differ by 2e-4 to 6e-4, inputs moved by one unit in the last place
// by 2.6e-3 to 5.3e-3 (two scales: 3e-4 to 4.5e-3 against 7e-3 to 2.4e-2 in the low set,
// 1e-2 to 0.2 against 0.27 to 1.0 in the high one).
constexpr int kRowDensityTile = 1280, kRowForceTile = 640, kRowList = 16, kRowScan = 8;

__device__ __forceinline__ v4f as_v4f(const float4& q) { return v4f{q.x, q.y, q.z, q.w}; }

template <bool kKahan>
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(6))) void k_density_rows(
    const float4* __restrict__ ipos, const float4* __restrict__ ivel,
    const uint32_t* __restrict__ cs, const uint32_t* __restrict__ ce, StepParams p, GridView g,
    const uint32_t* __restrict__ n_dev, float* __restrict__ rho, float4* __restrict__ ixa,
    float4* __restrict__ ivb, XOrder xo) {
    __shared__ float4 tile[kRowDensityTile];
    __shared__ uint32_t red[2 * kWavesPerBlock];
    const uint32_t n = *n_dev;
    const uint32_t s = xcd_local_block(blockIdx.x, gridDim.x) * kBlock + threadIdx.x;
    const bool active = s < n;
    const float4 xi = active ? ipos[s] : make_float4(0.f, 0.f, 0.f, 0.f);
    const Probe pr = make_probe(g, xi.x, xi.y, xi.z);
    const float inv_h2 = p.inv_h2;
    float sum = 0.0f, comp = 0.0f;
    auto row = [&](uint32_t m, auto&& load) {
#pragma clang fp contract(off)
        float rs = 0.0f;
        auto add = [&](const float4& q) {
            const float a = poly6_unit(xi, as_v4f(q), inv_h2);
            rs = __builtin_fmaf(a * a, a, rs);
        };
        uint32_t k = 0;
        for (; k + 8 <= m; k += 8) {
            float4 q[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) q[u] = load(k + u);
#pragma unroll
            for (int u = 0; u < 8; ++u) add(q[u]);
        }
        for (; k < m; ++k) add(load(k));
        if (kKahan) {
            const float y = rs - comp;
            const float t = sum + y;
            comp = (t - sum) - y;
            sum = t;
        } else {
            sum += rs;
        }
    };
    walk_stencil_staged<kBlock, kRowDensityTile, true>(
        g, pr, cs, ce, n, active, red, [&](uint32_t k, uint32_t j) { tile[k] = ipos[j]; },
        [&](uint32_t t0, uint32_t t1, uint32_t) {
            row(t1 - t0, [&](uint32_t k) {
                const float4 q = tile[t0 + k];
                keep_lds_quad(q);
                return q;
            });
        },
        [&](uint32_t b, uint32_t e) { row(e - b, [&](uint32_t k) { return ipos[b + k]; }); },
        xo.bins);
    if (!active) return;
    const float r = p.c6m_h6 * sum;
    const float inv = __builtin_amdgcn_rcpf(r);
    const float4 v = ivel[s];
    rho[xo.i2r[s]] = r;
    ixa[s] = make_float4(xi.x, xi.y, xi.z, p.stiffness * (r - p.rest_density) * inv * inv);
    ivb[s] = make_float4(v.x, v.y, v.z, inv);
}

// In-range candidates are appended to the lane's column of an LDS list, and
// their pair terms evaluated, in order, when some lane's column is full and at
// the end of every row.
template <bool kTension>
__global__ __launch_bounds__(kBlock) void k_force_rows(
    const float4* __restrict__ ipos, const float4* __restrict__ ivel,
    const float4* __restrict__ ixa, const float4* __restrict__ ivb,
    const uint32_t* __restrict__ cs, const uint32_t* __restrict__ ce, StepParams p, GridView g,
    const uint32_t* __restrict__ n_dev, float dt, float4* __restrict__ pos,
    float4* __restrict__ vel, float4* __restrict__ accel, XOrder xo) {
    __shared__ float4 tp[kRowForceTile + kRowScan];
    __shared__ float4 tv[kRowForceTile + kRowScan];
    __shared__ uint16_t list[kRowList][kBlock];
    __shared__ uint32_t red[2 * kWavesPerBlock];
    const uint32_t n = *n_dev;
    const uint32_t s = xcd_local_block(blockIdx.x, gridDim.x) * kBlock + threadIdx.x;
    const bool active = s < n;
    const float4 zero = make_float4(0.f, 0.f, 0.f, 0.f);
    const float4 xi = active ? ixa[s] : zero, vi = active ? ivb[s] : zero;
    const Probe pr = make_probe(g, xi.x, xi.y, xi.z);
    PairSums<kTension> S;
    uint32_t cnt = 0;
    auto pair = [&](const float4& x, const float4& v) {
        S.add(xi, vi, xi.w, p.h, p.h2, as_v4f(x), as_v4f(v));
    };
    // 0 < r2 < h2 as one unsigned compare: r2 >= +0 is a sum of squares, and
    // for non-negative floats the bit patterns order like the values.
    const uint32_t h2_bits_m1 = __float_as_uint(p.h2) - 1u;
    auto in_range = [&](const float4& q) {
        return __float_as_uint(dist2(xi.x - q.x, xi.y - q.y, xi.z - q.z)) - 1u < h2_bits_m1;
    };
    // Two list entries are fetched per step so their tile reads overlap.
    auto flush = [&]() {
        uint32_t k = 0;
        for (; k + 2 <= cnt; k += 2) {
            const uint32_t t0 = list[k][threadIdx.x], t1 = list[k + 1][threadIdx.x];
            const float4 a0 = tp[t0], b0 = tv[t0], a1 = tp[t1], b1 = tv[t1];
            pair(a0, b0);
            pair(a1, b1);
        }
        if (k < cnt) {
            const uint32_t t0 = list[k][threadIdx.x];
            pair(tp[t0], tv[t0]);
        }
        cnt = 0;
    };
    walk_stencil_staged<kBlock, kRowForceTile, true, kRowScan>(
        g, pr, cs, ce, n, active, red,
        [&](uint32_t k, uint32_t j) {
            tp[k] = ixa[j];
            tv[k] = ivb[j];
        },
        [&](uint32_t t0, uint32_t t1, uint32_t) {
            // Whole groups of candidates are loaded before any test (the tile is
            // padded); every candidate's index is written at the queue tail and
            // the tail advances only for in-range ones.
            for (uint32_t t = t0; t < t1; t += kRowScan) {
                float4 c[kRowScan];
#pragma unroll
                for (int u = 0; u < kRowScan; ++u) c[u] = tp[t + u];
#pragma unroll
                for (int u = 0; u < kRowScan; ++u) {
                    keep_lds_quad(c[u]);
                    const bool hit = (t + u < t1) & in_range(c[u]);  // no short circuit
                    list[cnt][threadIdx.x] = static_cast<uint16_t>(t + u);
                    cnt += hit ? 1u : 0u;
                }
                if (__ballot(cnt > kRowList - kRowScan) != 0ull) flush();
            }
            flush();
        },
        [&](uint32_t b, uint32_t e) {
            for (uint32_t j = b; j < e; ++j) {
                const float4 x = ixa[j];
                if (in_range(x)) pair(x, ivb[j]);
            }
        },
        xo.bins);
    if (!active) return;
    float4 x = xi, v = vi;
    x.w = ipos[s].w;
    v.w = ivel[s].w;
    force_finish<kTension, true>(S, p, x, v, make_float2(xi.w, vi.w), xo.i2r[s], xo.bacc, dt, pos,
                                 vel, accel, xo.err);
}

// XSPH integrator (integrateXSPHD, SINGLE_SCALE/Solver.cu:346-395, 757-853,
// with each axis taking its own correction component): in sorted order, after
// the force pass has written every particle's acceleration,
//   v'_i = v_i + dt a_i,  v''_i = v'_i + eps m c6 sum_{r < h} B_j (h^2 - r^2)^3 (v'_j - v'_i),
//   x'_i = x_i + dt v''_i, then the wall clamp.
// The block-staged stencil walk holds (x_j, B_j) and v'_j per candidate.
constexpr int kXsphTile = 512;

__global__ __launch_bounds__(kBlock) void k_xsph_integrate(
    const float4* __restrict__ tpos, const float4* __restrict__ tvel,
    const float2* __restrict__ aux, const float4* __restrict__ accel,
    const uint32_t* __restrict__ cs, const uint32_t* __restrict__ ce, StepParams p, GridView g,
    const uint32_t* __restrict__ n_dev, float dt, float4* __restrict__ pos,
    float4* __restrict__ vel) {
    __shared__ float4 tx[kXsphTile];
    __shared__ float4 tv[kXsphTile];
    __shared__ uint32_t red[2 * kWavesPerBlock];
    const uint32_t n = *n_dev;
    const uint32_t s = xcd_local_block(blockIdx.x, gridDim.x) * kBlock + threadIdx.x;
    const bool active = s < n;
    const float4 xi = active ? tpos[s] : make_float4(0.f, 0.f, 0.f, 0.f);
    float4 vi = active ? tvel[s] : make_float4(0.f, 0.f, 0.f, 0.f);
    if (active) {
        const float4 a = accel[s];
        vi.x += dt * a.x;
        vi.y += dt * a.y;
        vi.z += dt * a.z;
    }
    const Probe pr = make_probe(g, xi.x, xi.y, xi.z);
    float Sx = 0.f, Sy = 0.f, Sz = 0.f;
    auto pair = [&](const float4& xb, const float4& v) {
        const float dx = xi.x - xb.x, dy = xi.y - xb.y, dz = xi.z - xb.z;
        const float r2 = dist2(dx, dy, dz);
        if (r2 < p.h2) {
            const float a = p.h2 - r2;
            const float w = a * a * a * xb.w;
            Sx += w * (v.x - vi.x);
            Sy += w * (v.y - vi.y);
            Sz += w * (v.z - vi.z);
        }
    };
    auto vprime = [&](uint32_t j) {
        const float4 v = tvel[j], a = accel[j];
        return make_float4(v.x + dt * a.x, v.y + dt * a.y, v.z + dt * a.z, 0.0f);
    };
    walk_stencil_staged<kBlock, kXsphTile>(
        g, pr, cs, ce, n, active, red,
        [&](uint32_t k, uint32_t j) {
            const float4 x = tpos[j];
            tx[k] = make_float4(x.x, x.y, x.z, aux[j].y);
            tv[k] = vprime(j);
        },
        [&](uint32_t t0, uint32_t t1, uint32_t) {
            for (uint32_t t = t0; t < t1; ++t) {
                const float4 q = tx[t], v = tv[t];
                keep_lds_quad(q);
                keep_lds_quad(v);
                pair(q, v);
            }
        },
        [&](uint32_t b, uint32_t e) {
            for (uint32_t j = b; j < e; ++j) {
                const float4 x = tpos[j];
                pair(make_float4(x.x, x.y, x.z, aux[j].y), vprime(j));
            }
        });
    if (!active) return;
    float vx = vi.x + p.xsph * Sx, vy = vi.y + p.xsph * Sy, vz = vi.z + p.xsph * Sz;
    float x = xi.x + dt * vx, y = xi.y + dt * vy, z = xi.z + dt * vz;
    if (p.flags & SPH_FLAG_WALL_CLAMP) {
        const float e = p.restitution;
        if (x < p.lox) { x = p.lox; vx = -e * vx; }
        if (x > p.hix) { x = p.hix; vx = -e * vx; }
        if (y < p.loy) { y = p.loy; vy = -e * vy; }
        if (y > p.hiy) { y = p.hiy; vy = -e * vy; }
        if (z < p.loz) { z = p.loz; vz = -e * vz; }
        if (z > p.hiz) { z = p.hiz; vz = -e * vz; }
    }
    pos[s] = make_float4(x, y, z, xi.w);
    vel[s] = make_float4(vx, vy, vz, vi.w);
}

// Launches.  All density and force passes run in the internal x-order.  The
// group passes take the tune word (the tension forms run the default shape);
// walled scenes have one shape.
inline uint32_t group_count(uint32_t cap_n, uint32_t n_groups) {
    return n_groups ? n_groups : (cap_n + kGroupTargets - 1) / kGroupTargets;
}

template <bool kKahan, bool kFinalize, bool kBatched>
void launch_density(uint32_t tune, uint32_t cap_n, hipStream_t st, const StepBuffers& b,
                    const StepParams& p, const GridView& g, float2* aux, const SceneParams* scenes,
                    const XOrder& xo) {
    const uint32_t n_groups = group_count(cap_n, kBatched ? b.n_groups : 0u);
    const LaunchShape sh =
        launch_shape(n_groups, DensityTile::kBytes, tune & 0xFu, (tune >> 8) & 0xFu,
                     (tune >> 16) & 0x3u, kBatched ? 1u : 1u + ((tune >> 20) & 1u));
    hipLaunchKernelGGL((k_density<kKahan, kFinalize, kBatched>), sh.grid, sh.block, sh.lds, st,
                       g, b.cell_start, b.cell_end, b.n_dev, b.ipos, b.ivel, scenes, b.skeys, p, b.rho,
                       aux, b.ixa, b.ivb, b.groups, n_groups, xo, sh);
}

template <bool kTension, bool kIntegrate, bool kBatched>
void launch_force(uint32_t tune, uint32_t cap_n, hipStream_t st, const StepBuffers& b,
                  const StepParams& p, const GridView& g, float dt, float4* pos, float4* vel,
                  float4* accel, const SceneParams* scenes, const XOrder& xo) {
    if (kTension) tune = 0u;
    const uint32_t n_groups = group_count(cap_n, kBatched ? b.n_groups : 0u);
    const LaunchShape sh =
        launch_shape(n_groups, ForceTile::kBytes, (tune >> 4) & 0xFu, (tune >> 12) & 0xFu,
                     (tune >> 18) & 0x3u, kBatched ? 1u : 1u + ((tune >> 22) & 1u));
    hipLaunchKernelGGL((k_force<kTension, kIntegrate, kBatched>), sh.grid, sh.block, sh.lds, st,
                       g, b.cell_start, b.cell_end, b.n_dev, b.ixa, b.ivb, scenes, b.ipos, b.ivel,
                       b.skeys, p, dt, pos, vel, accel, b.groups, n_groups, xo, sh);
}

__global__ void k_pack_state(const float* __restrict__ pxyz, const float* __restrict__ vxyz,
                             uint32_t n, float4* __restrict__ pos, float4* __restrict__ vel) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    pos[i] = make_float4(pxyz[3 * i], pxyz[3 * i + 1], pxyz[3 * i + 2], __uint_as_float(i));
    if (vxyz)
        vel[i] = make_float4(vxyz[3 * i], vxyz[3 * i + 1], vxyz[3 * i + 2], 0.0f);
    else
        vel[i] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
}

__global__ void k_export_aos(const float4* __restrict__ src, uint32_t n, float* __restrict__ dst) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float4 v = src[i];
    dst[3 * i] = v.x;
    dst[3 * i + 1] = v.y;
    dst[3 * i + 2] = v.z;
}

inline dim3 blocks_for(uint32_t n) { return dim3((n + kBlock - 1) / kBlock); }

// Whether a step's sums are taken in row order (k_density_rows).
inline bool row_order(const StepParams& p, const StepBuffers& b) {
    return b.walls && b.bacc && !(p.flags & SPH_FLAG_XSPH);
}

}  // namespace

int launch_pass(int pass, const StepParams& p, const StepBuffers& b, float dt,
                uint32_t key_bits, bool write_accel, hipStream_t stream) {
    if (p.n == 0) return SPH_OK;
    const GridView g = make_grid_view(p.ox, p.oy, p.oz, p.spacing, p.dx, p.dy, p.dz, p.h);
    switch (pass) {
        case kPassHash: {
            if (block_sort_fits(p.n)) break;  // with the sort
            const int rc = hash_hist_cells(p, b.n_dev, b.pos, b.keys, key_bits, b.sort_temp,
                                           b.sort_temp_bytes, b.cell_start, b.cell_end, stream);
            if (rc != SPH_OK) return rc;
            break;
        }
        case kPassSort: {
            const int rc =
                block_sort_fits(p.n)
                    ? sort_cells_block(p, b.n_dev, b.pos, b.skeys, b.perm, key_bits, b.cell_start,
                                       b.cell_end, stream)
                    : sort_cells(p, b.keys, b.skeys, b.perm, key_bits, b.sort_temp, stream);
            if (rc != SPH_OK) return rc;
            break;
        }
        case kPassReorder: {
            if (!b.ipos) return set_error(SPH_ERR_INVALID_ARGUMENT, "step buffers lack the x-order");
            // The sorted copies tpos / tvel are read by the colour, wall and
            // XSPH passes and by the two-scale step.
            const bool copy = b.color || (b.walls && b.bacc) || (p.flags & SPH_FLAG_XSPH) ||
                              b.keep_sorted;
            hipLaunchKernelGGL((copy ? k_order<false, true> : k_order<false, false>),
                               blocks_for(p.n), dim3(kBlock), 0, stream, b.skeys, b.perm, b.pos,
                               b.vel, b.tpos, b.tvel, b.cell_start, b.cell_end, b.n_dev, p,
                               kNoScenes, b.ipos, b.ivel, b.i2r, b.xbins);
            break;
        }
        case kPassDensity:
            if (!b.ipos) return set_error(SPH_ERR_INVALID_ARGUMENT, "step buffers lack the x-order");
            if (row_order(p, b)) {
                hipLaunchKernelGGL((p.flags & SPH_FLAG_KAHAN) ? k_density_rows<true>
                                                              : k_density_rows<false>,
                                   blocks_for(p.n), dim3(kBlock), 0, stream, b.ipos, b.ivel,
                                   b.cell_start, b.cell_end, p, g, b.n_dev, b.rho, b.ixa, b.ivb,
                                   XOrder{b.i2r, b.xbins});
                break;
            }
            // Only the XSPH pass reads A, B in the sorted order.
            if (float2* const aux = (p.flags & SPH_FLAG_XSPH) ? b.aux : nullptr;
                p.flags & SPH_FLAG_KAHAN)
                launch_density<true, true, false>(p.tune, p.n, stream, b, p, g, aux, kNoScenes,
                                                 XOrder{b.i2r, b.xbins});
            else
                launch_density<false, true, false>(p.tune, p.n, stream, b, p, g, aux, kNoScenes,
                                                 XOrder{b.i2r, b.xbins});
            break;
        case kPassForce: {
            float4* acc = write_accel ? b.accel : nullptr;
            if (!b.ipos) return set_error(SPH_ERR_INVALID_ARGUMENT, "step buffers lack the x-order");
            if (b.color) {  // colour values from the force pass's inputs
                const int rc = launch_energy_color(b.tpos, b.tvel, b.cell_start, b.cell_end,
                                                   b.n_dev, p.n, g, p.mass, b.color, stream);
                if (rc != SPH_OK) return rc;
            }
            const bool walls = b.walls && b.bacc;
            if (walls) {
                const int rc = launch_wall_accel(*b.walls, b.tpos, b.n_dev, p.n, b.bacc, stream);
                if (rc != SPH_OK) return rc;
            }
            if (p.flags & SPH_FLAG_XSPH) {
                // Accelerations of every particle first (sorted order), then
                // the XSPH integration, which reads its neighbours' ones.
                const XOrder xa{b.i2r, b.xbins, walls ? b.bacc : nullptr};
                float4* const no_state = nullptr;
                if (p.tens != 0.0f)
                    launch_force<true, false, false>(p.tune, p.n, stream, b, p, g, 0.0f, no_state,
                                                    no_state, b.accel, kNoScenes, xa);
                else
                    launch_force<false, false, false>(p.tune, p.n, stream, b, p, g, 0.0f, no_state,
                                                    no_state, b.accel, kNoScenes, xa);
                hipLaunchKernelGGL(k_xsph_integrate, blocks_for(p.n), dim3(kBlock), 0, stream,
                                   b.tpos, b.tvel, b.aux, b.accel, b.cell_start, b.cell_end, p, g,
                                   b.n_dev, dt, b.pos, b.vel);
                break;
            }
            const XOrder xo{b.i2r, b.xbins, walls ? b.bacc : nullptr,
                            radix_sort_error_word(b.sort_temp)};
            if (row_order(p, b))
                hipLaunchKernelGGL((p.tens != 0.0f) ? k_force_rows<true> : k_force_rows<false>,
                                   blocks_for(p.n), dim3(kBlock), 0, stream, b.ipos, b.ivel, b.ixa,
                                   b.ivb, b.cell_start, b.cell_end, p, g, b.n_dev, dt, b.pos, b.vel,
                                   acc, xo);
            else if (p.tens != 0.0f)
                launch_force<true, true, false>(p.tune, p.n, stream, b, p, g, dt, b.pos, b.vel, acc,
                                               kNoScenes, xo);
            else
                launch_force<false, true, false>(p.tune, p.n, stream, b, p, g, dt, b.pos, b.vel, acc,
                                               kNoScenes, xo);
            break;
        }
        default:
            return set_error(SPH_ERR_INVALID_ARGUMENT, "unknown pass");
    }
    SPH_HIP(hipGetLastError());
    return SPH_OK;
}

int launch_step(const StepParams& p, const StepBuffers& b, float dt, uint32_t key_bits,
                bool write_accel, hipStream_t stream) {
    for (int pass = 0; pass < kNumPasses; ++pass) {
        const int rc = launch_pass(pass, p, b, dt, key_bits, write_accel, stream);
        if (rc != SPH_OK) return rc;
    }
    return SPH_OK;
}

// The two-scale own-set passes in the internal x-order: density without the
// A/B finalisation (the complementary sums complete it), the internal-order
// copy of the finalised A/B, then the force without integration.  Results
// land at the sorted slots, as in the sorted-order passes above.
int launch_density_own_x(const StepParams& p, const StepBuffers& b, hipStream_t stream) {
    if (p.n == 0) return SPH_OK;
    if (!b.ipos) return set_error(SPH_ERR_INVALID_ARGUMENT, "step buffers lack the x-order");
    const GridView g = make_grid_view(p.ox, p.oy, p.oz, p.spacing, p.dx, p.dy, p.dz, p.h);
    const XOrder xo{b.i2r, b.xbins};
    if (p.flags & SPH_FLAG_KAHAN)
        launch_density<true, false, false>(p.tune, p.n, stream, b, p, g, nullptr, kNoScenes, xo);
    else
        launch_density<false, false, false>(p.tune, p.n, stream, b, p, g, nullptr, kNoScenes, xo);
    SPH_HIP(hipGetLastError());
    return SPH_OK;
}

// The packed internal state of the force pass from the final A, B: (x, A) and
// (v, B).
__global__ __launch_bounds__(kBlock) void k_gather_aux(const float2* __restrict__ aux,
                                                       const uint32_t* __restrict__ i2r,
                                                       const uint32_t* __restrict__ n_dev,
                                                       const float4* __restrict__ ipos,
                                                       const float4* __restrict__ ivel,
                                                       float4* __restrict__ ixa,
                                                       float4* __restrict__ ivb) {
    const uint32_t s = blockIdx.x * kBlock + threadIdx.x;
    if (s >= *n_dev) return;
    const float4 x = ipos[s], v = ivel[s];
    const float2 a = aux[i2r[s]];
    ixa[s] = make_float4(x.x, x.y, x.z, a.x);
    ivb[s] = make_float4(v.x, v.y, v.z, a.y);
}

int launch_gather_aux(const StepParams& p, const StepBuffers& b, hipStream_t stream) {
    if (p.n == 0) return SPH_OK;
    hipLaunchKernelGGL(k_gather_aux, blocks_for(p.n), dim3(kBlock), 0, stream, b.aux, b.i2r,
                       b.n_dev, b.ipos, b.ivel, b.ixa, b.ivb);
    SPH_HIP(hipGetLastError());
    return SPH_OK;
}

int launch_force_own_x(const StepParams& p, const GridView& g, const StepBuffers& b,
                       float4* accel_own, hipStream_t stream) {
    if (p.n == 0) return SPH_OK;
    if (!b.ipos) return set_error(SPH_ERR_INVALID_ARGUMENT, "step buffers lack the x-order");
    float4* const no_state = nullptr;
    const XOrder xo{b.i2r, b.xbins};
    if (p.tens != 0.0f)
        launch_force<true, false, false>(p.tune, p.n, stream, b, p, g, 0.0f, no_state, no_state,
                                        accel_own, kNoScenes, xo);
    else
        launch_force<false, false, false>(p.tune, p.n, stream, b, p, g, 0.0f, no_state, no_state,
                                        accel_own, kNoScenes, xo);
    SPH_HIP(hipGetLastError());
    return SPH_OK;
}

// Pair work of the most recent step, over its internal x-order: the candidates in
// every particle's own stencil rows (the nine rows and any rows beyond; a group's
// list holds those of 32 particles) and the pairs with 0 < r < h among them.  Wave sums, then one 64-bit atomic
// per wave per counter.
__global__ __launch_bounds__(kBlock) void k_count_pairs(const float4* __restrict__ ipos,
                                                        const uint32_t* __restrict__ cs,
                                                        const uint32_t* __restrict__ ce,
                                                        const uint4* __restrict__ bins,
                                                        const uint32_t* __restrict__ n_dev,
                                                        GridView g, float h2,
                                                        unsigned long long* __restrict__ out) {
    const uint32_t n = *n_dev;
    const uint32_t s = blockIdx.x * kBlock + threadIdx.x;
    uint32_t cand = 0, nbr = 0;
    if (s < n) {
        const float4 xi = ipos[s];
        const Probe pr = make_probe(g, xi.x, xi.y, xi.z);
        const uint32_t h2_bits_m1 = __float_as_uint(h2) - 1u;
        auto run = [&](uint32_t b, uint32_t e) {
            if (b >= e) return;
            cand += e - b;
            for (uint32_t j = b; j < e; ++j) {
                const float4 xj = ipos[j];
                const float r2 = dist2(xi.x - xj.x, xi.y - xj.y, xi.z - xj.z);
                nbr += (__float_as_uint(r2) - 1u < h2_bits_m1) ? 1u : 0u;
            }
        };
        for (int rz = pr.sz; rz <= pr.ez; ++rz)
            for (int ry = pr.sy; ry <= pr.ey; ++ry) {
                uint32_t b, e;
                probe_row<true>(g, pr, cs, ce, bins, n, ry, rz, b, e);
                run(b, e);
            }
    }
    cand = __ockl_wfred_add_u32(cand);
    nbr = __ockl_wfred_add_u32(nbr);
    if ((threadIdx.x & 63) == 0) {
        atomicAdd(&out[0], static_cast<unsigned long long>(cand));
        atomicAdd(&out[1], static_cast<unsigned long long>(nbr));
    }
}

int launch_count_pairs(const StepParams& p, const StepBuffers& b, unsigned long long* out,
                       hipStream_t stream) {
    if (p.n == 0 || !b.ipos) return SPH_OK;
    const GridView g = make_grid_view(p.ox, p.oy, p.oz, p.spacing, p.dx, p.dy, p.dz, p.h);
    hipLaunchKernelGGL(k_count_pairs, blocks_for(p.n), dim3(kBlock), 0, stream, b.ipos,
                       b.cell_start, b.cell_end, b.xbins, b.n_dev, g, p.h2, out);
    SPH_HIP(hipGetLastError());
    return SPH_OK;
}

int launch_pack_state(const float* pxyz, const float* vxyz, uint32_t n, float4* pos,
                      float4* vel, hipStream_t stream) {
    if (n == 0) return SPH_OK;
    hipLaunchKernelGGL(k_pack_state, blocks_for(n), dim3(kBlock), 0, stream, pxyz, vxyz, n, pos,
                       vel);
    SPH_HIP(hipGetLastError());
    return SPH_OK;
}

int launch_export_aos(const float4* src, uint32_t n, float* dst, hipStream_t stream) {
    if (n == 0) return SPH_OK;
    hipLaunchKernelGGL(k_export_aos, blocks_for(n), dim3(kBlock), 0, stream, src, n, dst);
    SPH_HIP(hipGetLastError());
    return SPH_OK;
}

int launch_batch_pass(int pass, const StepParams& cap, const StepBuffers& b,
                      const SceneParams* scenes, bool kahan, bool tension, float dt,
                      uint32_t key_bits, bool write_accel, hipStream_t stream) {
    if (cap.n == 0) return SPH_OK;
    const GridView g0 = make_grid_view(cap.ox, cap.oy, cap.oz, cap.spacing, cap.dx, cap.dy, cap.dz,
                                       cap.h);
    switch (pass) {
        case kPassHash: {
            if (block_sort_fits(b.segments.largest)) break;  // with the sort
            const int rc = hash_hist_cells_batched(cap, b.n_dev, b.pos, b.vel, scenes, b.keys,
                                                   key_bits, b.sort_temp, b.sort_temp_bytes,
                                                   b.cell_start, b.cell_end, stream);
            if (rc != SPH_OK) return rc;
            break;
        }
        case kPassSort: {
            const int rc =
                block_sort_fits(b.segments.largest)
                    ? sort_cells_block_batched(cap, b.segments, b.pos, scenes, b.skeys, b.perm,
                                               b.cell_start, b.cell_end, stream)
                    : sort_cells(cap, b.keys, b.skeys, b.perm, key_bits, b.sort_temp, stream);
            if (rc != SPH_OK) return rc;
            break;
        }
        case kPassReorder: {
            // No pass of a batched step reads the sorted copies.
            if (!b.ipos) return set_error(SPH_ERR_INVALID_ARGUMENT, "step buffers lack the x-order");
            hipLaunchKernelGGL((k_order<true, false>), blocks_for(cap.n), dim3(kBlock), 0, stream,
                               b.skeys, b.perm, b.pos, b.vel, nullptr, nullptr, b.cell_start,
                               b.cell_end, b.n_dev, cap, scenes, b.ipos, b.ivel, b.i2r, b.xbins);
            break;
        }
        case kPassDensity:
            if (!b.ipos) return set_error(SPH_ERR_INVALID_ARGUMENT, "step buffers lack the x-order");
            if (kahan)
                launch_density<true, true, true>(cap.tune, cap.n, stream, b, cap, g0, nullptr, scenes,
                                                XOrder{b.i2r, b.xbins});
            else
                launch_density<false, true, true>(cap.tune, cap.n, stream, b, cap, g0, nullptr, scenes,
                                                XOrder{b.i2r, b.xbins});
            break;
        case kPassForce: {
            if (!b.ipos) return set_error(SPH_ERR_INVALID_ARGUMENT, "step buffers lack the x-order");
            float4* acc = write_accel ? b.accel : nullptr;
            const XOrder xo{b.i2r, b.xbins, nullptr, radix_sort_error_word(b.sort_temp)};
            if (tension)
                launch_force<true, true, true>(cap.tune, cap.n, stream, b, cap, g0, dt, b.pos, b.vel, acc,
                                              scenes, xo);
            else
                launch_force<false, true, true>(cap.tune, cap.n, stream, b, cap, g0, dt, b.pos, b.vel, acc,
                                              scenes, xo);
            break;
        }
        default:
            return set_error(SPH_ERR_INVALID_ARGUMENT, "unknown pass");
    }
    SPH_HIP(hipGetLastError());
    return SPH_OK;
}

}  // namespace sph

namespace sph {

bool tune_word_valid(uint32_t tune, bool batched) {
    const uint32_t dtile = tune & 0xFu, fvar = (tune >> 4) & 0xFu;
    const uint32_t dblock = (tune >> 16) & 0x3u, fblock = (tune >> 18) & 0x3u;
    const uint32_t dppl = (tune >> 20) & 0x3u, fppl = (tune >> 22) & 0x3u;
    return (tune >> 24) == 0u && dtile <= 5u && fvar <= 9u && ((tune >> 8) & 0xFu) <= 4u &&
           ((tune >> 12) & 0xFu) <= 4u && dblock <= 2u && fblock <= 2u && dppl <= 1u &&
           fppl <= 1u && (dblock == 0u || dtile == 0u) && (fblock == 0u || fvar == 0u) &&
           (dppl == 0u || (dtile == 0u && dblock == 0u)) &&
           (fppl == 0u || (fvar == 0u && fblock == 0u)) && (!batched || (dppl | fppl) == 0u);
}

int tune_pass(bool force, bool one_shape, uint32_t groups, bool batched,
              const std::function<int(uint32_t, float&)>& time, TunedPass& out) {
    const uint32_t tile = force ? ForceTile::kBytes : DensityTile::kBytes;
    const int waves = force ? 4 : 0, grid = force ? 12 : 8, block = force ? 18 : 16,
              pairs = force ? 22 : 20;
    out = TunedPass{};
    int rc = time(0u, out.default_ms);
    out.best_ms = out.default_ms;
    std::vector<LaunchShape> seen;
    auto is_new = [&](uint32_t w) {
        const LaunchShape s = launch_shape(groups, tile, (w >> waves) & 0xFu, (w >> grid) & 0xFu,
                                           (w >> block) & 0x3u, 1u + ((w >> pairs) & 1u));
        for (const LaunchShape& o : seen)
            if (o.grid.x == s.grid.x && o.block.x == s.block.x && o.per == s.per) return false;
        seen.push_back(s);
        return true;
    };
    auto consider = [&](uint32_t w) {
        float ms = 0.0f;
        if (rc != SPH_OK || one_shape || !is_new(w)) return;
        rc = time(w, ms);
        if (rc == SPH_OK && ms < out.best_ms) {
            out.best_ms = ms;
            out.word = w;
        }
    };
    (void)is_new(0u);
    for (uint32_t v = 1; v <= (force ? 9u : 5u); ++v) consider(v << waves);
    for (uint32_t v = 1; v <= 2; ++v) consider(v << block);
    if (!batched) consider(1u << pairs);
    const uint32_t shape = out.word;
    for (uint32_t v = 1; v <= 4; ++v) consider(shape | (v << grid));
    return rc;
}

int tune_neighbour_passes(StepParams p, const StepBuffers& b, const SceneParams* scenes,
                          bool kahan, bool tension, float dt, uint32_t key_bits, uint32_t reps,
                          hipStream_t stream, uint32_t* tune_out, float* ms_out) {
    if (p.n == 0) return set_error(SPH_ERR_INVALID_ARGUMENT, "autotune: no particles");
    reps = std::max(reps, 1u);
    auto run = [&](int pass, uint32_t tune) {
        p.tune = tune;
        return scenes ? launch_batch_pass(pass, p, b, scenes, kahan, tension, dt, key_bits, false,
                                          stream)
                      : launch_pass(pass, p, b, dt, key_bits, false, stream);
    };
    // The force pass integrates into pos/vel: keep the state to restore it.
    void* saved = nullptr;
    const size_t bytes = 16 * static_cast<size_t>(p.n);
    SPH_HIP(hipMalloc(&saved, 2 * bytes));
    hipEvent_t e0 = nullptr, e1 = nullptr;
    int rc = SPH_OK;
    auto fail = [&](int code) {
        if (e0) (void)hipEventDestroy(e0);
        if (e1) (void)hipEventDestroy(e1);
        (void)hipStreamSynchronize(stream);
        (void)hipFree(saved);
        return code;
    };
    hipError_t e = hipMemcpyAsync(saved, b.pos, bytes, hipMemcpyDeviceToDevice, stream);
    if (e == hipSuccess)
        e = hipMemcpyAsync(static_cast<char*>(saved) + bytes, b.vel, bytes,
                           hipMemcpyDeviceToDevice, stream);
    if (e == hipSuccess) e = hipEventCreate(&e0);
    if (e == hipSuccess) e = hipEventCreate(&e1);
    if (e != hipSuccess) return fail(hip_error(e, "autotune setup", __FILE__, __LINE__));
    for (int pass = kPassHash; pass <= kPassReorder && rc == SPH_OK; ++pass) rc = run(pass, 0u);
    if (rc != SPH_OK) return fail(rc);
    // Mean milliseconds of one launch of `pass` with tune word t (after one
    // untimed launch).
    auto time_pass = [&](int pass, uint32_t t, float& ms) -> int {
        int r = run(pass, t);
        if (r != SPH_OK) return r;
        SPH_HIP(hipEventRecord(e0, stream));
        for (uint32_t i = 0; i < reps && r == SPH_OK; ++i) r = run(pass, t);
        if (r != SPH_OK) return r;
        SPH_HIP(hipEventRecord(e1, stream));
        SPH_HIP(hipEventSynchronize(e1));
        SPH_HIP(hipEventElapsedTime(&ms, e0, e1));
        ms /= static_cast<float>(reps);
        return SPH_OK;
    };
    // Walled scenes and the force with tension have one shape.
    const bool rows = !scenes && row_order(p, b);
    const uint32_t groups = group_count(p.n, scenes ? b.n_groups : 0u);
    TunedPass density, force;
    rc = tune_pass(false, rows, groups, scenes != nullptr,
                   [&](uint32_t w, float& ms) { return time_pass(kPassDensity, w, ms); }, density);
    if (rc == SPH_OK) rc = run(kPassDensity, density.word);  // the force pass's input
    if (rc == SPH_OK)
        rc = tune_pass(true, rows || tension, groups, scenes != nullptr,
                       [&](uint32_t w, float& ms) { return time_pass(kPassForce, w, ms); }, force);
    if (rc != SPH_OK) return fail(rc);
    e = hipMemcpyAsync(b.pos, saved, bytes, hipMemcpyDeviceToDevice, stream);
    if (e == hipSuccess)
        e = hipMemcpyAsync(b.vel, static_cast<char*>(saved) + bytes, bytes,
                           hipMemcpyDeviceToDevice, stream);
    if (e != hipSuccess) return fail(hip_error(e, "autotune restore", __FILE__, __LINE__));
    *tune_out = density.word | force.word;
    if (ms_out) {
        ms_out[0] = density.default_ms;
        ms_out[1] = density.best_ms;
        ms_out[2] = force.default_ms;
        ms_out[3] = force.best_ms;
    }
    return fail(SPH_OK);
}

}  // namespace sph
