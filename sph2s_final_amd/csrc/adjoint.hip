// adjoint.hip -- differentiable batched rollout: T steps of the batched
// single-scale step and the reverse-mode adjoint of a loss on the final
// positions with respect to the initial positions and velocities and every
// scene's stiffness and viscosity.  The reference has no differentiation; the
// forward step it differentiates is Solver::Advance
// (SPH2S_FINAL_SINGLE_SCALE/Solver.cu:1082-1198) with the wall clamp.
//
// Forward form per step (sorted slot order, scene constants per particle):
//   rho_i = c6m sum_j (h^2 - r^2)^3                       (r < h, self included)
//   A_i = k (rho_i - rho0) / rho_i^2,  B_i = 1 / rho_i
//   a_i = C45 sum_j (A_i + A_j) F_ij x_ij + Vc B_i sum_j (h - r) B_j (v_j - v_i) + g
//         F = (h - r)^2 / r, C45 = m 45/(pi h^6), Vc = mu C45    (0 < r < h)
//   v' = v + dt a,  x' = x + dt v',  then the wall clamp.
// Adjoint per step, topology frozen (the pair sets of the forward step):
//   k_adj_integrate  clamp and symplectic Euler: abar = dL/da, direct dL/dx, dL/dv
//   k_adj_force      dL/dA_i = C45 sum_j F x_ij.(abar_i - abar_j)
//                    dL/dB_i = Vc sum_j (h - r) B_j (v_j - v_i).(abar_i - abar_j)
//                    dL/drho_i = dL/dA_i k (2 rho0 - rho_i) B_i^3 - dL/dB_i B_i^2
//                    dL/dx_i += C45 sum_j (A_i + A_j) [F dA + F'/r (x_ij.dA) x_ij]
//                               - Vc B_i sum_j B_j (v_j - v_i).dA x_ij / r
//                    dL/dv_i += Vc B_i sum_j (h - r) B_j (abar_j - abar_i)
//                    dL/dk += dL/dA_i (rho_i - rho0) B_i^2,
//                    dL/dmu += C45 B_i sum_j (h - r) B_j (v_j - v_i).abar_i
//                    (dA = abar_i - abar_j, F'/r = -(h - r)(h + r)/r^3)
//   k_adj_density    dL/dx_i += -6 c6m sum_j (h^2 - r^2)^2 (dL/drho_i + dL/drho_j) x_ij,
//                    written at the step's input slot perm[i].
// The pair sums use that j is a neighbour of i iff i is one of j's.
//
// The adjoint passes run in the forward step's internal x-order (cells sorted
// by x inside, stencil rows trimmed with the cells' x-bins), like the forward
// neighbour passes; the adjoint of the step's outputs is gathered from the
// sorted slots and the result scattered to the step's input slots
// perm[i2r[q]].
//
// Memory: the state is checkpointed every K steps; the backward sweep
// recomputes each K-step segment from its checkpoint, keeping every step's
// x-ordered state packed with the A/B factors, accelerations, densities,
// permutations, cell ranges and x-bin tables (60 B per particle + 40 B per cell
// per step), then runs the adjoint passes over the segment in reverse.  The
// forward writes the last segment's records itself, so that segment is never
// recomputed.  Parameter gradients accumulate in FP64 per group of 32 slots
// (a group always belongs to the same scene) and are reduced per scene in a
// fixed order, so the result is deterministic.
#include <algorithm>
#include <cmath>
#include <new>
#include <vector>

#include "batch.hpp"
#include "pairtile.hpp"

using namespace sph;

namespace {

constexpr int kBlock = 256;
inline dim3 blocks_for(uint32_t n) { return dim3((n + kBlock - 1) / kBlock); }

__device__ __forceinline__ uint32_t scene_of(const uint32_t* __restrict__ off, uint32_t n_scenes,
                                             uint32_t i) {
    uint32_t lo = 0, hi = n_scenes;  // off[lo] <= i < off[hi]
    while (hi - lo > 1) {
        const uint32_t mid = (lo + hi) >> 1;
        if (off[mid] <= i)
            lo = mid;
        else
            hi = mid;
    }
    return lo;
}

// State from AoS device arrays in global id order: pos.w = id, vel.w = scene.
__global__ void k_pack_batch(const float* __restrict__ p3, const float* __restrict__ v3,
                             const uint32_t* __restrict__ off, uint32_t n_scenes, uint32_t n,
                             float4* __restrict__ pos, float4* __restrict__ vel) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const uint32_t sc = scene_of(off, n_scenes, i);
    pos[i] = make_float4(p3[3 * i], p3[3 * i + 1], p3[3 * i + 2], __uint_as_float(i));
    vel[i] = v3 ? make_float4(v3[3 * i], v3[3 * i + 1], v3[3 * i + 2], __uint_as_float(sc))
                : make_float4(0.f, 0.f, 0.f, __uint_as_float(sc));
}

// out[id] = pos[s].xyz (ids are a permutation of [0, n)).
__global__ void k_export_by_id(const float4* __restrict__ pos, uint32_t n, float* __restrict__ out) {
    const uint32_t s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= n) return;
    const float4 x = pos[s];
    const uint32_t id = min(__float_as_uint(x.w), n - 1);
    out[3 * id] = x.x;
    out[3 * id + 1] = x.y;
    out[3 * id + 2] = x.z;
}

// Adjoint seed in the final state's slot order: gx[s] = g[id(s)], gv = 0.
__global__ void k_seed(const float4* __restrict__ pos, const float* __restrict__ g, uint32_t n,
                       float4* __restrict__ gx, float4* __restrict__ gv) {
    const uint32_t s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= n) return;
    const uint32_t id = min(__float_as_uint(pos[s].w), n - 1);
    gx[s] = make_float4(g[3 * id], g[3 * id + 1], g[3 * id + 2], 0.f);
    gv[s] = make_float4(0.f, 0.f, 0.f, 0.f);
}

__global__ void k_unpack3(const float4* __restrict__ src, uint32_t n, float* __restrict__ dst) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float4 v = src[i];
    dst[3 * i] = v.x;
    dst[3 * i + 1] = v.y;
    dst[3 * i + 2] = v.z;
}

// Clamp and symplectic Euler.  The pre-clamp position is recomputed with the
// forward kernel's expressions from the stored sorted state and acceleration.
// Half a wave per group of the batch's table, which holds the scene.
__global__ __launch_bounds__(kBlock) void k_adj_integrate(
    const float4* __restrict__ ixa, const float4* __restrict__ ivb,
    const float4* __restrict__ accel, const uint32_t* __restrict__ i2r,
    const float4* __restrict__ gx, const float4* __restrict__ gv,
    const SceneParams* __restrict__ scenes, const uint4* __restrict__ groups, uint32_t n_groups,
    const uint32_t* __restrict__ n_dev, float dt, float4* __restrict__ abar,
    float4* __restrict__ gxd, float4* __restrict__ gvd) {
    const uint32_t n = *n_dev;
    const uint32_t group = (xcd_local_block(blockIdx.x, gridDim.x) * kBlock + threadIdx.x) / kGroupTargets;
    if (group >= n_groups) return;
    const uint4 gr = groups[group];
    const uint32_t s = gr.x + threadIdx.x % kGroupTargets;
    if (s >= min(gr.y, n)) return;
    // s: internal slot; the step's outputs (and their adjoints) sit at its
    // sorted slot i2r[s].
    const uint32_t o = min(i2r[s], n - 1);
    const float4 xi = ixa[s], vi = ivb[s], ai = accel[o], gxi = gx[o], gvi = gv[o];
    const StepParams& p = scenes[gr.z].p;
    const bool clamp = (p.flags & SPH_FLAG_WALL_CLAMP) != 0u;
    const float e = p.restitution;
    auto axis = [&](float x, float v, float a, float gxo, float gvo, float lo, float hi, float& ga,
                    float& gxr, float& gvr) {
        const float vp = v + dt * a;
        const float xp = x + dt * vp;
        float gxp = gxo, gvp = gvo;
        if (clamp && (xp < lo || xp > hi)) {
            gxp = 0.0f;
            gvp = -e * gvo;
        }
        gvp += dt * gxp;
        gxr = gxp;
        gvr = gvp;
        ga = dt * gvp;
    };
    float4 A, X, V;
    axis(xi.x, vi.x, ai.x, gxi.x, gvi.x, p.lox, p.hix, A.x, X.x, V.x);
    axis(xi.y, vi.y, ai.y, gxi.y, gvi.y, p.loy, p.hiy, A.y, X.y, V.y);
    axis(xi.z, vi.z, ai.z, gxi.z, gvi.z, p.loz, p.hiz, A.z, X.z, V.z);
    A.w = X.w = V.w = 0.0f;
    abar[s] = A;
    gxd[s] = X;
    gvd[s] = V;
}

typedef PairTile<3> AdjForceTile;
typedef PairTile<1> AdjDensityTile;
// One wave per block: the force adjoint's tile, 14 KB, then has 11 waves on a
// CU, where blocks of four leave room for 8 (197 against 235 us at one million).
constexpr uint32_t kAdjForceWaves = 1, kAdjDensityWaves = 4;
constexpr uint32_t kAdjChunkGroups = 128;  // groups in a row that one XCD takes

// The wave's group and its targets; the cells come from the positions, as the
// step's sort took them.
template <uint32_t kWavesPerBlock>
__device__ __forceinline__ GroupRange adjoint_group(uint32_t n, const uint4* __restrict__ groups,
                                                    uint32_t n_groups) {
    const uint32_t block = xcd_local_block(blockIdx.x, gridDim.x, kAdjChunkGroups / kWavesPerBlock);
    return group_range<true>(block * kWavesPerBlock + uniform_u32(threadIdx.x >> 6), n, groups,
                             n_groups);
}

__device__ __forceinline__ GroupTargets adjoint_targets(const GridView& g, const GroupRange& r,
                                                        const float4* __restrict__ xs, uint32_t& s) {
    GroupTargets t;
    s = r.start + (threadIdx.x & 31u);
    t.active = s < r.end;
    t.x = xs[t.active ? s : r.start];
    t.key = cell_hash(t.x.x, t.x.y, t.x.z, g.ox, g.oy, g.oz, g.spacing, g.dx, g.dy, g.dz);
    return t;
}

// Force-pair adjoint; see the file comment for the terms.  The group walk
// (pairtile.hpp) with (x, A), (v, B) and abar per candidate; a pair out of range
// or coincident adds 0 (walk_targets sees to what is not finite).  Writes (x, dL/drho) packed for the density adjoint, and
// adds each group's parameter terms, in FP64, to the group's own accumulators.
// Bound by VALU issue.  Against a queue of hits per lane on a block-staged tile
// (us, one million in 16 scenes): 233 -> 197.
__global__ __launch_bounds__(64 * kAdjForceWaves) __attribute__((amdgpu_waves_per_eu(3)))
void k_adj_force(
    const float4* __restrict__ ixa, const float4* __restrict__ ivb, const float* __restrict__ rho,
    const uint32_t* __restrict__ i2r, const float4* __restrict__ abar,
    const uint32_t* __restrict__ cs, const uint32_t* __restrict__ ce,
    const uint4* __restrict__ bins, const SceneParams* __restrict__ scenes,
    const uint4* __restrict__ groups, uint32_t n_groups, const uint32_t* __restrict__ n_dev,
    float4* __restrict__ xg, float4* __restrict__ gxd, float4* __restrict__ gvd,
    double* __restrict__ kacc, double* __restrict__ macc) {
    __shared__ __align__(kTileAlign) unsigned char lds[kAdjForceWaves * AdjForceTile::kBytes];
    const uint32_t wave = uniform_u32(threadIdx.x >> 6);
    const uint32_t n = *n_dev;
    const GroupRange gr = adjoint_group<kAdjForceWaves>(n, groups, n_groups);
    if (gr.start >= gr.end) return;
    const StepParams& p = scenes[gr.scene].p;
    const GridView& g = scenes[gr.scene].g;
    uint32_t s;
    const GroupTargets t = adjoint_targets(g, gr, ixa, s);
    const float4 xi = t.x;
    const uint32_t own = t.active ? s : gr.start;
    const float4 vi = ivb[own], bi = abar[own];
    const float h = p.h;
    // 0 < r2 < h2 as one unsigned compare (r2 >= +0; non-negative floats order
    // like their bit patterns).
    const uint32_t h2_bits_m1 = __float_as_uint(p.h2) - 1u;
    float sumA = 0.f, S1 = 0.f, Sd = 0.f;  // Sd: sum (h - r) B_j dv.dA
    float gPx = 0.f, gPy = 0.f, gPz = 0.f;   // sum (A_i + A_j)[F dA + F'/r (x.dA) x]
    float gVx = 0.f, gVy = 0.f, gVz = 0.f;   // sum B_j (dv.dA) x / r
    float gWx = 0.f, gWy = 0.f, gWz = 0.f;   // sum (h - r) B_j dA
    walk_targets<3, false>(
        g, t, p.inv_h, cs, ce, bins, n, ixa, ivb, abar,
        lds_address(lds) + wave * AdjForceTile::kBytes,
        [&](const v4f& xa, const v4f& vb, const v4f& bj) {
            const float dx = xi.x - xa.x, dy = xi.y - xa.y, dz = xi.z - xa.z;
            const float r2 = dx * dx + dy * dy + dz * dz;
            const float rs = __builtin_amdgcn_rsqf(r2);
            const float hr = __builtin_amdgcn_fmed3f(h - r2 * rs, 0.0f, h);
            const float inv_r = __float_as_uint(r2) - 1u < h2_bits_m1 ? rs : 0.0f;
            const float hi = hr * inv_r, F = hr * hi;
            const float Fr = -hi * (h + r2 * inv_r) * inv_r * inv_r;
            const float ax = bi.x - bj.x, ay = bi.y - bj.y, az = bi.z - bj.z;
            const float ux = vb.x - vi.x, uy = vb.y - vi.y, uz = vb.z - vi.z;
            const float xdA = dx * ax + dy * ay + dz * az;
            const float udA = ux * ax + uy * ay + uz * az;
            sumA += F * xdA;
            const float wB = hr * vb.w;
            S1 += wB * (ux * bi.x + uy * bi.y + uz * bi.z);
            Sd += wB * udA;
            const float pa = t.x.w + xa.w;
            const float cP = pa * Fr * xdA, pF = pa * F;
            gPx += pF * ax + cP * dx;
            gPy += pF * ay + cP * dy;
            gPz += pF * az + cP * dz;
            const float cV = vb.w * udA * inv_r;
            gVx += cV * dx;
            gVy += cV * dy;
            gVz += cV * dz;
            gWx += wB * ax;
            gWy += wB * ay;
            gWz += wB * az;
        },
        [] {},
        [&] {
            return __builtin_isfinite(((sumA + S1) + (Sd + gPx)) + ((gPy + gPz) + (gVx + gVy)) +
                                      ((gVz + gWx) + (gWy + gWz)));
        },
        [&] {
            sumA = S1 = Sd = 0.f;
            gPx = gPy = gPz = gVx = gVy = gVz = gWx = gWy = gWz = 0.f;
        },
        [&] { return DirectScan{g, cs, ce, n, ixa, ivb, abar}; });
    sumA = both_halves(sumA);
    S1 = both_halves(S1);
    Sd = both_halves(Sd);
    gPx = both_halves(gPx);
    gPy = both_halves(gPy);
    gPz = both_halves(gPz);
    gVx = both_halves(gVx);
    gVy = both_halves(gVy);
    gVz = both_halves(gVz);
    gWx = both_halves(gWx);
    gWy = both_halves(gWy);
    gWz = both_halves(gWz);
    const float Bi = vi.w, ri = rho[min(i2r[own], n - 1)];
    const float gA = p.c45m * sumA, gB = p.visc * Sd;
    // The lower lane half sums the group's stiffness terms, the upper one its
    // viscosity terms, in a fixed order.
    const bool upper = (threadIdx.x & 32u) != 0u;
    double acc = !t.active ? 0.0
                           : static_cast<double>(upper ? p.c45m * Bi * S1
                                                       : gA * (ri - p.rest_density) * Bi * Bi);
#pragma unroll
    for (int d = 16; d > 0; d >>= 1) acc += __shfl_xor(acc, d);
    const uint32_t group = gr.index;
    if ((threadIdx.x & 31u) == 0u) (upper ? macc : kacc)[group] += acc;
    if (!t.active || upper) return;
    xg[s] = make_float4(t.x.x, t.x.y, t.x.z,
                        gA * p.stiffness * (2.0f * p.rest_density - ri) * Bi * Bi * Bi - gB * Bi * Bi);
    const float vb = p.visc * Bi;
    float4 X = gxd[s], V = gvd[s];
    X.x += p.c45m * gPx - vb * gVx;
    X.y += p.c45m * gPy - vb * gVy;
    X.z += p.c45m * gPz - vb * gVz;
    V.x -= vb * gWx;
    V.y -= vb * gWy;
    V.z -= vb * gWz;
    gxd[s] = X;
    gvd[s] = V;
}

// Density-pair adjoint, then the scatter to the step's input order.  The group
// walk with (x, dL/drho) per candidate.
// Bound by VALU issue; one lane per target with block-staged rows took (us, one
// million in 16 scenes) 121, this 84 to 92.
__global__ __launch_bounds__(64 * kAdjDensityWaves) __attribute__((amdgpu_waves_per_eu(5)))
void k_adj_density(
    const float4* __restrict__ xg, const uint32_t* __restrict__ cs,
    const uint32_t* __restrict__ ce, const uint4* __restrict__ bins,
    const uint32_t* __restrict__ i2r, const uint32_t* __restrict__ perm,
    const SceneParams* __restrict__ scenes, const uint4* __restrict__ groups, uint32_t n_groups,
    const uint32_t* __restrict__ n_dev, const float4* __restrict__ gxd,
    const float4* __restrict__ gvd, float4* __restrict__ gx, float4* __restrict__ gv) {
    __shared__ __align__(kTileAlign) unsigned char lds[kAdjDensityWaves * AdjDensityTile::kBytes];
    const uint32_t wave = uniform_u32(threadIdx.x >> 6);
    const uint32_t n = *n_dev;
    const GroupRange gr = adjoint_group<kAdjDensityWaves>(n, groups, n_groups);
    if (gr.start >= gr.end) return;
    const StepParams& p = scenes[gr.scene].p;
    const GridView& g = scenes[gr.scene].g;
    uint32_t s;
    const GroupTargets t = adjoint_targets(g, gr, xg, s);
    const float4 xi = t.x;
    const float inv_h2 = p.inv_h2;
    // Sums of a^2 (g_i + g_j) x_ij with a = 1 - r^2 / h^2 clamped to [0, 1]
    // (one clamped fused multiply-add): the pair's (h^2 - r^2)^2 is h^4 a^2,
    // and a = 0 out of range.  A coincident pair (x_ij = 0) adds zero.
    float sx = 0.f, sy = 0.f, sz = 0.f;
    walk_targets<1, false>(
        g, t, p.inv_h, cs, ce, bins, n, xg, nullptr, nullptr,
        lds_address(lds) + wave * AdjDensityTile::kBytes,
        [&](const v4f& q) {
            const float dx = xi.x - q.x, dy = xi.y - q.y, dz = xi.z - q.z;
            const float r2 = dx * dx + dy * dy + dz * dz;
            const float a = __builtin_amdgcn_fmed3f(__builtin_fmaf(-r2, inv_h2, 1.0f), 0.0f, 1.0f);
            const float c = a * a * (t.x.w + q.w);
            sx += c * dx;
            sy += c * dy;
            sz += c * dz;
        },
        [] {}, [&] { return __builtin_isfinite(sx + sy + sz); }, [&] { sx = sy = sz = 0.f; },
        [&] { return DirectScan{g, cs, ce, n, xg, nullptr, nullptr}; });
    sx = both_halves(sx);
    sy = both_halves(sy);
    sz = both_halves(sz);
    if (!t.active) return;
    const uint32_t q = min(perm[min(i2r[s], n - 1)], n - 1);
    if ((threadIdx.x & 32u) != 0u) {
        gv[q] = gvd[s];
        return;
    }
    const float k6 = -6.0f * p.c6m * (p.h2 * p.h2);
    float4 X = gxd[s];
    X.x += k6 * sx;
    X.y += k6 * sy;
    X.z += k6 * sz;
    gx[q] = X;
}

// Per-scene sums of the groups' FP64 accumulators in a fixed order: one block
// per scene, strided partial sums, then a tree in LDS.  (One million particles
// in 16 scenes, one sum per group instead of one per particle: 71 -> 11 us.)
__global__ __launch_bounds__(kBlock) void k_scene_reduce(const double* __restrict__ kacc,
                                                         const double* __restrict__ macc,
                                                         const uint4* __restrict__ groups,
                                                         uint32_t n_groups,
                                                         double* __restrict__ out) {
    __shared__ double sk[kBlock], sm[kBlock];
    const uint32_t sc = blockIdx.x;
    auto first_of = [&](uint32_t scene) {  // the first group of a scene or a later one
        uint32_t lo = 0, hi = n_groups;
        while (lo < hi) {
            const uint32_t mid = (lo + hi) >> 1;
            if (groups[mid].z < scene)
                lo = mid + 1;
            else
                hi = mid;
        }
        return lo;
    };
    const uint32_t b = first_of(sc), e = first_of(sc + 1);
    double a = 0.0, m = 0.0;
    for (uint32_t i = b + threadIdx.x; i < e; i += kBlock) {
        a += kacc[i];
        m += macc[i];
    }
    sk[threadIdx.x] = a;
    sm[threadIdx.x] = m;
    __syncthreads();
    for (int w = kBlock / 2; w > 0; w >>= 1) {
        if (static_cast<int>(threadIdx.x) < w) {
            sk[threadIdx.x] += sk[threadIdx.x + w];
            sm[threadIdx.x] += sm[threadIdx.x + w];
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        out[2 * sc] = sk[0];
        out[2 * sc + 1] = sm[0];
    }
}

size_t al(size_t x) { return (x + 255) & ~static_cast<size_t>(255); }

}  // namespace

// One recomputed step's record inside a segment.
struct RolloutSlot {
    float4 *ixa, *ivb;  // (x, A), (v, B), internal order
    float4* accel;      // sorted slots
    float* rho;         // sorted slots
    uint32_t *perm, *i2r, *cell_start, *cell_end;
    uint4* xbins;
    hipGraphExec_t graph = nullptr;
};

struct sph_rollout {
    sph_batch* b = nullptr;
    float dt = 0.0f;
    uint32_t n_steps = 0, every = 1, n_ckpt = 0;
    void* arena = nullptr;
    size_t arena_bytes = 0;
    float4 *ckpt_pos = nullptr, *ckpt_vel = nullptr;
    std::vector<RolloutSlot> slot;
    float4 *gx, *gv, *abar, *gxd, *gvd;
    float4* xg;  // (x, dL/drho), internal order
    double *kacc, *macc, *red;
    hipEvent_t ev_in = nullptr, ev_out = nullptr;
    // With more than one segment the backward keeps two sets of K records:
    // the recomputation of one segment (on stream rs) overlaps the adjoint of
    // the next later one (on the batch's stream).
    uint32_t n_sets = 1;
    hipStream_t rs = nullptr;
    hipEvent_t ev_rec[2] = {nullptr, nullptr}, ev_adj[2] = {nullptr, nullptr}, ev_seed = nullptr;
    bool have_forward = false;
};

namespace {

// The rollout runs on the batch's own stream, ordered after the caller's
// stream (NULL: the null stream) on entry and before it on exit.
int enter(sph_rollout* r, void* stream) {
    SPH_HIP(hipEventRecord(r->ev_in, static_cast<hipStream_t>(stream)));
    SPH_HIP(hipStreamWaitEvent(r->b->stream, r->ev_in, 0));
    return SPH_OK;
}

int leave(sph_rollout* r, void* stream) {
    SPH_HIP(hipEventRecord(r->ev_out, r->b->stream));
    SPH_HIP(hipStreamWaitEvent(static_cast<hipStream_t>(stream), r->ev_out, 0));
    return SPH_OK;
}

StepBuffers slot_buffers(const sph_rollout* r, const RolloutSlot& s) {
    StepBuffers sb = r->b->buf;
    sb.ixa = s.ixa;
    sb.ivb = s.ivb;
    sb.i2r = s.i2r;
    sb.xbins = s.xbins;
    sb.accel = s.accel;
    sb.rho = s.rho;
    sb.perm = s.perm;
    sb.cell_start = s.cell_start;
    sb.cell_end = s.cell_end;
    return sb;
}

int slot_graph(sph_rollout* r, RolloutSlot& s) {
    if (s.graph) return SPH_OK;
    hipStream_t st = r->b->stream;
    hipGraph_t g = nullptr;
    SPH_HIP(hipStreamBeginCapture(st, hipStreamCaptureModeThreadLocal));
    const int rc = batch_step(r->b, slot_buffers(r, s), r->dt, true, st);
    const hipError_t e = hipStreamEndCapture(st, &g);
    if (rc != SPH_OK) {
        if (g) (void)hipGraphDestroy(g);
        return rc;
    }
    if (e != hipSuccess) return hip_error(e, "hipStreamEndCapture", __FILE__, __LINE__);
    const hipError_t ei = hipGraphInstantiate(&s.graph, g, nullptr, nullptr, 0);
    (void)hipGraphDestroy(g);
    if (ei != hipSuccess) {
        s.graph = nullptr;
        return hip_error(ei, "hipGraphInstantiate", __FILE__, __LINE__);
    }
    return SPH_OK;
}

int adjoint_step(sph_rollout* r, const RolloutSlot& s) {
    sph_batch* b = r->b;
    hipStream_t st = b->stream;
    const uint4* const groups = b->buf.groups;
    const uint32_t ng = b->buf.n_groups;
    hipLaunchKernelGGL(k_adj_integrate, blocks_for(ng * kGroupTargets), dim3(kBlock), 0, st, s.ixa,
                       s.ivb, s.accel, s.i2r, r->gx, r->gv, b->scenes, groups, ng, b->buf.n_dev,
                       r->dt, r->abar, r->gxd, r->gvd);
    hipLaunchKernelGGL(k_adj_force, dim3((ng + kAdjForceWaves - 1) / kAdjForceWaves),
                       dim3(64 * kAdjForceWaves), 0, st, s.ixa, s.ivb, s.rho, s.i2r, r->abar,
                       s.cell_start, s.cell_end, s.xbins, b->scenes, groups, ng, b->buf.n_dev,
                       r->xg, r->gxd, r->gvd, r->kacc, r->macc);
    hipLaunchKernelGGL(k_adj_density, dim3((ng + kAdjDensityWaves - 1) / kAdjDensityWaves),
                       dim3(64 * kAdjDensityWaves), 0, st, r->xg, s.cell_start, s.cell_end, s.xbins,
                       s.i2r, s.perm, b->scenes, groups, ng, b->buf.n_dev, r->gxd, r->gvd, r->gx,
                       r->gv);
    SPH_HIP(hipGetLastError());
    return SPH_OK;
}

}  // namespace

extern "C" {

int sph_rollout_destroy(sph_rollout* r) {
    if (!r) return SPH_OK;
    if (r->b && r->b->stream) (void)hipStreamSynchronize(r->b->stream);
    if (r->rs) (void)hipStreamSynchronize(r->rs);
    for (auto& s : r->slot)
        if (s.graph) (void)hipGraphExecDestroy(s.graph);
    if (r->arena) (void)hipFree(r->arena);
    if (r->ev_in) (void)hipEventDestroy(r->ev_in);
    if (r->ev_out) (void)hipEventDestroy(r->ev_out);
    for (int k = 0; k < 2; ++k) {
        if (r->ev_rec[k]) (void)hipEventDestroy(r->ev_rec[k]);
        if (r->ev_adj[k]) (void)hipEventDestroy(r->ev_adj[k]);
    }
    if (r->ev_seed) (void)hipEventDestroy(r->ev_seed);
    if (r->rs) (void)hipStreamDestroy(r->rs);
    if (r->b) sph_batch_destroy(r->b);
    delete r;
    return SPH_OK;
}

int sph_rollout_create(const sph_config* cfgs, uint32_t n_scenes, const uint32_t* counts,
                       float dt, uint32_t n_steps, uint32_t checkpoint_every, sph_rollout** out) {
    if (!out) return set_error(SPH_ERR_INVALID_ARGUMENT, "out is null");
    *out = nullptr;
    if (!(dt > 0.0f) || !std::isfinite(dt)) return set_error(SPH_ERR_INVALID_ARGUMENT, "dt must be > 0");
    if (checkpoint_every == 0) return set_error(SPH_ERR_INVALID_ARGUMENT, "checkpoint_every must be >= 1");
    for (uint32_t s = 0; cfgs && s < n_scenes; ++s)
        if (cfgs[s].tension != 0.0f)
            return set_error(SPH_ERR_UNSUPPORTED, "rollout: tension is not differentiated");
    auto* r = new (std::nothrow) sph_rollout;
    if (!r) return set_error(SPH_ERR_INVALID_ARGUMENT, "out of host memory");
    int rc = batch_alloc(cfgs, n_scenes, counts, &r->b);
    if (rc != SPH_OK) {
        delete r;
        return rc;
    }
    r->dt = dt;
    r->n_steps = n_steps;
    r->every = std::min(checkpoint_every, std::max(n_steps, 1u));
    r->n_ckpt = (n_steps + r->every - 1) / r->every;
    const size_t N = r->b->n, C = r->b->total_cells, S = r->b->n_scenes,
                 G = r->b->buf.n_groups;
    const uint32_t K = n_steps ? r->every : 0u;
    const size_t n_stored = r->n_ckpt ? r->n_ckpt - 1 : 0;  // the last segment keeps records
    r->n_sets = (r->n_ckpt > 1) ? 2u : 1u;
    std::vector<size_t> sizes = {al(16 * N * n_stored), al(16 * N * n_stored)};
    for (uint32_t k = 0; k < K * r->n_sets; ++k)
        for (size_t v : {16 * N, 4 * N, 16 * N, 16 * N, 4 * N, 4 * N, 4 * C, 4 * C, kXBinBytes * C})
            sizes.push_back(al(v));
    for (size_t v : {16 * N, 16 * N, 16 * N, 16 * N, 16 * N, 16 * N, 8 * G, 8 * G, 16 * S})
        sizes.push_back(al(v));
    size_t total = 0;
    for (size_t v : sizes) total += v;
    hipError_t e = hipMalloc(&r->arena, total);
    if (e == hipSuccess) e = hipEventCreateWithFlags(&r->ev_in, hipEventDisableTiming);
    if (e == hipSuccess) e = hipEventCreateWithFlags(&r->ev_out, hipEventDisableTiming);
    if (r->n_sets > 1) {
        if (e == hipSuccess) e = hipStreamCreateWithFlags(&r->rs, hipStreamNonBlocking);
        for (int k = 0; k < 2; ++k) {
            if (e == hipSuccess) e = hipEventCreateWithFlags(&r->ev_rec[k], hipEventDisableTiming);
            if (e == hipSuccess) e = hipEventCreateWithFlags(&r->ev_adj[k], hipEventDisableTiming);
        }
        if (e == hipSuccess) e = hipEventCreateWithFlags(&r->ev_seed, hipEventDisableTiming);
    }
    if (e != hipSuccess) {
        sph_rollout_destroy(r);
        return hip_error(e, "rollout allocation", __FILE__, __LINE__);
    }
    r->arena_bytes = total;
    char* a = static_cast<char*>(r->arena);
    size_t i = 0;
    auto take = [&]() {
        void* p = a;
        a += sizes[i++];
        return p;
    };
    r->ckpt_pos = static_cast<float4*>(take());
    r->ckpt_vel = static_cast<float4*>(take());
    r->slot.resize(static_cast<size_t>(K) * r->n_sets);
    for (auto& s : r->slot) {
        s.accel = static_cast<float4*>(take());
        s.rho = static_cast<float*>(take());
        s.ixa = static_cast<float4*>(take());
        s.ivb = static_cast<float4*>(take());
        s.perm = static_cast<uint32_t*>(take());
        s.i2r = static_cast<uint32_t*>(take());
        s.cell_start = static_cast<uint32_t*>(take());
        s.cell_end = static_cast<uint32_t*>(take());
        s.xbins = static_cast<uint4*>(take());
    }
    r->gx = static_cast<float4*>(take());
    r->gv = static_cast<float4*>(take());
    r->abar = static_cast<float4*>(take());
    r->gxd = static_cast<float4*>(take());
    r->gvd = static_cast<float4*>(take());
    r->xg = static_cast<float4*>(take());
    r->kacc = static_cast<double*>(take());
    r->macc = static_cast<double*>(take());
    r->red = static_cast<double*>(take());
    *out = r;
    return SPH_OK;
}

int sph_rollout_info(const sph_rollout* r, uint32_t* n_particles, uint32_t* n_scenes,
                     size_t* device_bytes) {
    if (!r) return set_error(SPH_ERR_INVALID_ARGUMENT, "rollout is null");
    if (n_particles) *n_particles = r->b->n;
    if (n_scenes) *n_scenes = r->b->n_scenes;
    if (device_bytes) *device_bytes = r->arena_bytes;
    return SPH_OK;
}

int sph_rollout_forward(sph_rollout* r, const float* pos0, const float* vel0,
                        const float* stiffness, const float* viscosity, float* final_pos,
                        void* stream) {
    if (!r || !pos0) return set_error(SPH_ERR_INVALID_ARGUMENT, "null argument");
    sph_batch* b = r->b;
    const uint32_t n = b->n;
    int rc = enter(r, stream);
    if (rc != SPH_OK) return rc;
    rc = batch_set_parameters(b, stiffness, viscosity);
    if (rc != SPH_OK) return rc;
    hipLaunchKernelGGL(k_pack_batch, blocks_for(n), dim3(kBlock), 0, b->stream, pos0, vel0,
                       b->part_offset_dev, b->n_scenes, n, b->buf.pos, b->buf.vel);
    SPH_HIP(hipGetLastError());
    // The last segment runs through the segment-record graphs, so the backward
    // sweep starts from records the forward already wrote.
    const uint32_t last0 = r->n_ckpt ? (r->n_ckpt - 1) * r->every : 0u;
    for (uint32_t t = 0; t < r->n_steps; ++t) {
        if (t % r->every == 0 && t < last0) {
            const size_t o = static_cast<size_t>(t / r->every) * n;
            SPH_HIP(hipMemcpyAsync(r->ckpt_pos + o, b->buf.pos, 16 * size_t(n),
                                   hipMemcpyDeviceToDevice, b->stream));
            SPH_HIP(hipMemcpyAsync(r->ckpt_vel + o, b->buf.vel, 16 * size_t(n),
                                   hipMemcpyDeviceToDevice, b->stream));
        }
        if (t >= last0) {
            RolloutSlot& sl = r->slot[t - last0];
            rc = slot_graph(r, sl);
            if (rc != SPH_OK) return rc;
            SPH_HIP(hipGraphLaunch(sl.graph, b->stream));
        } else {
            rc = sph_batch_advance(b, r->dt, 1);
            if (rc != SPH_OK) return rc;
        }
    }
    if (final_pos) {
        hipLaunchKernelGGL(k_export_by_id, blocks_for(n), dim3(kBlock), 0, b->stream, b->buf.pos,
                           n, final_pos);
        SPH_HIP(hipGetLastError());
    }
    r->have_forward = true;
    return leave(r, stream);
}

int sph_rollout_backward(sph_rollout* r, const float* grad_final, float* grad_pos0,
                         float* grad_vel0, double* grad_stiffness, double* grad_viscosity,
                         void* stream) {
    if (!r || !grad_final) return set_error(SPH_ERR_INVALID_ARGUMENT, "null argument");
    if (!r->have_forward)
        return set_error(SPH_ERR_INVALID_ARGUMENT, "rollout: backward needs a forward first");
    sph_batch* b = r->b;
    const uint32_t n = b->n;
    int rc = enter(r, stream);
    if (rc != SPH_OK) return rc;
    hipLaunchKernelGGL(k_seed, blocks_for(n), dim3(kBlock), 0, b->stream, b->buf.pos, grad_final,
                       n, r->gx, r->gv);
    SPH_HIP(hipGetLastError());
    SPH_HIP(hipMemsetAsync(r->kacc, 0, 8 * size_t(b->buf.n_groups), b->stream));
    SPH_HIP(hipMemsetAsync(r->macc, 0, 8 * size_t(b->buf.n_groups), b->stream));
    // Segment c's records live in set (last - c) % 2 (the forward wrote the
    // last segment's into set 0).  Segment c - 1 is recomputed on rs while
    // the batch's stream runs the adjoint of segment c; a set is refilled only
    // after the adjoint that read it, and read only after its recomputation.
    const uint32_t last = r->n_ckpt ? r->n_ckpt - 1 : 0u;
    const uint32_t K = r->every;
    auto set_of = [&](uint32_t c) { return (last - c) & 1u; };
    auto slot_of = [&](uint32_t c, uint32_t t) -> RolloutSlot& {
        return r->slot[static_cast<size_t>(set_of(c)) * K + (t - c * K)];
    };
    // Every graph exists before any of them is queued (captures run on the
    // batch's stream).
    for (auto& sl : r->slot) {
        rc = slot_graph(r, sl);
        if (rc != SPH_OK) return rc;
    }
    hipStream_t rs = r->n_sets > 1 ? r->rs : b->stream;
    if (r->n_sets > 1) {  // the seed reads the final state the recomputation overwrites
        SPH_HIP(hipEventRecord(r->ev_seed, b->stream));
        SPH_HIP(hipStreamWaitEvent(rs, r->ev_seed, 0));
    }
    bool adj_done[2] = {false, false};
    for (uint32_t c = r->n_ckpt; c-- > 0;) {
        const uint32_t t0 = c * r->every, t1 = std::min(r->n_steps, t0 + r->every);
        if (c >= 1) {  // recompute segment c - 1 on rs, overlapping the adjoint of c
            const uint32_t p = c - 1, ps = set_of(p);
            if (r->n_sets > 1 && adj_done[ps]) SPH_HIP(hipStreamWaitEvent(rs, r->ev_adj[ps], 0));
            const size_t o = static_cast<size_t>(p) * n;
            SPH_HIP(hipMemcpyAsync(b->buf.pos, r->ckpt_pos + o, 16 * size_t(n),
                                   hipMemcpyDeviceToDevice, rs));
            SPH_HIP(hipMemcpyAsync(b->buf.vel, r->ckpt_vel + o, 16 * size_t(n),
                                   hipMemcpyDeviceToDevice, rs));
            const uint32_t p1 = std::min(r->n_steps, p * K + K);
            for (uint32_t t = p * K; t < p1; ++t) SPH_HIP(hipGraphLaunch(slot_of(p, t).graph, rs));
            if (r->n_sets > 1) SPH_HIP(hipEventRecord(r->ev_rec[ps], rs));
        }
        if (c < last && r->n_sets > 1) SPH_HIP(hipStreamWaitEvent(b->stream, r->ev_rec[set_of(c)], 0));
        for (uint32_t t = t1; t-- > t0;) {
            rc = adjoint_step(r, slot_of(c, t));
            if (rc != SPH_OK) return rc;
        }
        if (r->n_sets > 1) {
            SPH_HIP(hipEventRecord(r->ev_adj[set_of(c)], b->stream));
            adj_done[set_of(c)] = true;
        }
    }
    // The state now holds a recomputed segment's end (or, with one segment,
    // the forward's final state, whose records the adjoint has consumed).
    r->have_forward = false;
    if (grad_pos0)
        hipLaunchKernelGGL(k_unpack3, blocks_for(n), dim3(kBlock), 0, b->stream, r->gx, n,
                           grad_pos0);
    if (grad_vel0)
        hipLaunchKernelGGL(k_unpack3, blocks_for(n), dim3(kBlock), 0, b->stream, r->gv, n,
                           grad_vel0);
    hipLaunchKernelGGL(k_scene_reduce, dim3(b->n_scenes), dim3(kBlock), 0, b->stream, r->kacc,
                       r->macc, b->buf.groups, b->buf.n_groups, r->red);
    SPH_HIP(hipGetLastError());
    if (grad_stiffness || grad_viscosity) {
        std::vector<double> h(2 * size_t(b->n_scenes));
        SPH_HIP(hipMemcpyAsync(h.data(), r->red, 16 * size_t(b->n_scenes), hipMemcpyDeviceToHost,
                               b->stream));
        SPH_HIP(hipStreamSynchronize(b->stream));
        for (uint32_t s = 0; s < b->n_scenes; ++s) {
            if (grad_stiffness) grad_stiffness[s] = h[2 * s];
            if (grad_viscosity) grad_viscosity[s] = h[2 * s + 1];
        }
    }
    return leave(r, stream);
}

int sph_rollout_synchronize(sph_rollout* r) {
    if (!r) return set_error(SPH_ERR_INVALID_ARGUMENT, "rollout is null");
    SPH_HIP(hipStreamSynchronize(r->b->stream));
    return SPH_OK;
}

int sph_rollout_device_errors(sph_rollout* r, uint32_t* bits) {
    if (!r) return set_error(SPH_ERR_INVALID_ARGUMENT, "rollout is null");
    return sph_batch_device_errors(r->b, bits);
}

}  // extern "C"
