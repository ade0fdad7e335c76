// pyramid.hip — min-depth (Hi-Z) pyramid for gfx950, and the device depth rasteriser for synthetic requests.
//
// Replaces DepthPyramidGeneration.comp.glsl:13-19 dispatched once per mip with a barrier in between
// (vulkanDraw.cpp:554-622). Each level texel is the MIN over the non-zero-weight texels of the bilinear
// footprint of its centre in the level above (level 0 samples the depth buffer), the rule in cull_math.h.
//
// Single pass for power-of-two bases: each workgroup owns a tile of level 0 (32 x 32 texels), writes it,
// and reduces it in registers down to 1 x 1 (levels 1..5, exact 2:1 with edge clamp). The last workgroup
// (the highest-numbered one, waiting on flagged words) reduces the remaining levels from the
// 1-texel-per-tile image. Other bases go by regions, also in one launch (pyramid_region_kernel), and those too large for
// either take one launch per level with the general footprint rule.
#include "bz_internal.h"
#include "synth_rng.h"

namespace bz {

namespace {

constexpr uint32_t kPyrBlock = 512;
constexpr uint32_t kTile = kPyrTile;  // level-0 tile edge of a workgroup: eight waves of 32 x 4 texels
constexpr unsigned long long kTailFlag = 1ull << 63;
constexpr uint32_t kLdsJobs = 1024;  // batched: job start table staged in LDS up to this many jobs

__device__ __forceinline__ float min4(float a, float b, float c, float d)
{
    return glsl_min(glsl_min(a, b), glsl_min(c, d));
}

typedef float float4_unaligned __attribute__((ext_vector_type(4), aligned(4)));  // one 16-byte load at any dword
typedef float float2_unaligned __attribute__((ext_vector_type(2), aligned(4)));  // one 8-byte load at any dword

// A quad_perm of the four lanes of each quad.
template <int A, int B, int C, int D>
__device__ __forceinline__ float quad_perm(float v)
{
    return __int_as_float(
        __builtin_amdgcn_update_dpp(0, __float_as_int(v), A | B << 2 | C << 4 | D << 6, 0xf, 0xf, true));
}
// min of the value in the lane whose bit `off` is clear and the one whose bit is set, in that order, for both lanes.
__device__ __forceinline__ float min_across(float v, uint32_t lane, uint32_t off)
{
    const float o = __shfl_xor(v, (int)off, 64);
    return (lane & off) ? glsl_min(o, v) : glsl_min(v, o);
}

// Orders a wave's LDS writes before its later LDS reads.
__device__ __forceinline__ void wave_lds_sync()
{
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0)
    __builtin_amdgcn_wave_barrier();
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
}

// One flagged word of the tail: waits until it is there (bounded; giving up sets *err) and clears it, so the next build
// starts from zero.
__device__ __forceinline__ float tail_finish(const PyrBuildJob& J, uint32_t idx, unsigned long long w, uint32_t* err)
{
    uint32_t spins = 0;
    while (!(w & kTailFlag)) {
        if (++spins > J.spin_limit) {
            atomicExch(err, 1u);
            break;
        }
        __builtin_amdgcn_s_sleep(1);
        w = __hip_atomic_load(&J.tail[idx], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    __hip_atomic_store(&J.tail[idx], 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return __uint_as_float((uint32_t)w);
}

struct PyrSmem {
    float l2[64];                                              // level 2 of the tile: a row of 8 per wave
    float a[kPyrTailTexels * 4u], b[kPyrTailTexels];          // the tile image, then the tail's levels in turn
};

// One workgroup's tile of a single-pass (power-of-two) pyramid, levels 0 to 5: a lane owns two level-0 texels side by side
// and a wave 32 x 4 (16 lanes across, so every store of level 0 covers whole 128-byte lines), so that levels 1 and 2 come
// from exchanges between its lanes; levels 3 to 5 from exchanges within the first wave, which reads the eight waves'
// rows from LDS behind the only barrier. Texels outside the base are +infinity, which no minimum takes over a texel, so
// every power-of-two extent down to 1 x 1 goes the same way.
// What bounded a build before was the levels as much as the depth image: a barrier and an LDS round trip per level held
// each workgroup's slots for half as long again as its loads (2560 x 1440 depth onto 2048 x 1024: level 0 alone 7.2 us,
// with its levels 10.8, the whole build 14.5; now 12.4. 1920 x 1080 onto 1024 x 1024: 8.9 -> 8.2; 64 pyramids of the batch
// with exact 2:1: 85 -> 78 us). Lanes in Morton order, which need no LDS up to level 4, store level 0 in 64-byte pieces:
// level 0 alone 10.5 us. Four texels a lane and 256 threads: 11.5, but 8.2 instead of 6.6 us for 1024 x 512.
__device__ __forceinline__ void pyramid_tile(const PyrBuildJob& J, uint32_t tile, PyrSmem& sm, uint32_t* err)
{
    const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t tx = tile % J.tiles_x, ty = tile / J.tiles_x, bw = J.base_w, bh = J.base_h;
    const uint32_t x1 = tx * (kTile / 2u) + (lane & 15u);                // the lane's level-1 column
    const uint32_t x0 = 2u * x1, y0 = ty * kTile + wave * 4u + (lane >> 4);  // and its first level-0 texel
    const float inf = __builtin_inff();
    float ta = inf, tb = inf;  // level-0 texels
    // ---- level 0 from the depth image; every load of a lane is issued before the first minimum
    if (J.w == 2u * bw && J.h == 2u * bh && bw >= 2u && ((uintptr_t)J.depth & 15u) == 0) {
        // exactly 2:1: the footprint of texel (x, y) is depth {2x, 2x+1} x {2y, 2y+1} (frac(tx) = 0.5 on both axes)
        if (x0 < bw && y0 < bh) {
            const float4* p = reinterpret_cast<const float4*>(J.depth + (size_t)(2u * y0) * J.w) + x1;
            const float4 r0 = p[0], r1 = p[J.w / 4u];
            ta = min4(r0.x, r0.y, r1.x, r1.y);
            tb = min4(r0.z, r0.w, r1.z, r1.w);
        }
    } else {
        // general ratio: the footprint rule; the base extent is a power of two, so (x + 0.5) / W equals
        // (x + 0.5) * (1 / W) exactly
        const float rbw = 1.0f / (float)bw, rbh = 1.0f / (float)bh;
        const uint32_t xa = x0 < bw ? x0 : bw - 1u, xb = x0 + 1u < bw ? x0 + 1u : bw - 1u, y = y0 < bh ? y0 : bh - 1u;
        const Footprint f = footprint(((float)xa + 0.5f) * rbw, ((float)y + 0.5f) * rbh, J.w, J.h);
        const Footprint e = footprint(((float)xb + 0.5f) * rbw, ((float)y + 0.5f) * rbh, J.w, J.h);
        const float *r0 = J.depth + (size_t)f.y0 * J.w, *r1 = J.depth + (size_t)f.y1 * J.w;
        float a0, a1, a2, a3, b0, b1, b2, b3;
        if (J.w <= 2u * bw && J.w >= 4u) {
            // At most two depth texels per base texel: the two footprints lie within four texels of a row (their
            // positions differ by at most 2, so floor of the second is at most 2 further, and one more for its right
            // neighbour), read as one 16-byte load that starts early enough to end inside the row. Eight 4-byte
            // loads touched each line four times (1366 x 768 onto 1024 x 512: 7.2 us).
            const uint32_t xs = f.x0 < J.w - 4u ? f.x0 : J.w - 4u;
            const float4_unaligned p = *reinterpret_cast<const float4_unaligned*>(r0 + xs);
            const float4_unaligned q = *reinterpret_cast<const float4_unaligned*>(r1 + xs);
            auto pick = [](float4_unaligned r, uint32_t i) {
                const float lo = i & 1u ? r.y : r.x, hi = i & 1u ? r.w : r.z;
                return i & 2u ? hi : lo;
            };
            a0 = pick(p, f.x0 - xs);
            a1 = pick(p, f.x1 - xs);
            a2 = pick(q, f.x0 - xs);
            a3 = pick(q, f.x1 - xs);
            b0 = pick(p, e.x0 - xs);
            b1 = pick(p, e.x1 - xs);
            b2 = pick(q, e.x0 - xs);
            b3 = pick(q, e.x1 - xs);
        } else if (J.w >= 2u) {
            // More depth texels per base texel: each footprint's two texels of a row as one 8-byte load, which starts a
            // texel early where the footprint is the row's last one. With eight 4-byte loads a 4096 x 4096 depth onto
            // 1024 x 1024 took 13.2 us, and 10.4 for one level only; now 9.2 and 5.8.
            const uint32_t xa = f.x0 < J.w - 2u ? f.x0 : J.w - 2u, xe = e.x0 < J.w - 2u ? e.x0 : J.w - 2u;
            const float2_unaligned p = *reinterpret_cast<const float2_unaligned*>(r0 + xa);
            const float2_unaligned q = *reinterpret_cast<const float2_unaligned*>(r1 + xa);
            const float2_unaligned u = *reinterpret_cast<const float2_unaligned*>(r0 + xe);
            const float2_unaligned v = *reinterpret_cast<const float2_unaligned*>(r1 + xe);
            a0 = f.x0 > xa ? p.y : p.x;
            a1 = f.x1 > xa ? p.y : p.x;
            a2 = f.x0 > xa ? q.y : q.x;
            a3 = f.x1 > xa ? q.y : q.x;
            b0 = e.x0 > xe ? u.y : u.x;
            b1 = e.x1 > xe ? u.y : u.x;
            b2 = e.x0 > xe ? v.y : v.x;
            b3 = e.x1 > xe ? v.y : v.x;
        } else {  // a depth image one texel wide
            a0 = a1 = b0 = b1 = r0[0];
            a2 = a3 = b2 = b3 = r1[0];
        }
        if (x0 < bw && y0 < bh) ta = min4(a0, a1, a2, a3);
        if (x0 + 1u < bw && y0 < bh) tb = min4(b0, b1, b2, b3);
    }
    if (y0 < bh) {  // (8-byte aligned: even pitch, and the levels start at the allocation's start)
        if (x0 + 1u < bw) *reinterpret_cast<float2*>(J.texels + (size_t)y0 * bw + x0) = make_float2(ta, tb);
        else if (x0 < bw) J.texels[(size_t)y0 * bw + x0] = ta;  // a base one texel wide
    }
    if (J.mips == 1u) return;
    // ---- levels 1 and 2: (x1, y0 / 2) >> (L - 1) is the lane's texel of level L, stored by the first lane of its group
    const uint32_t levels = J.tile_levels;
    auto store = [&](uint32_t L, uint32_t x, uint32_t y, float t) {
        const uint32_t w = level_dim(bw, L);
        if (L < levels && x < w && y < level_dim(bh, L)) J.texels[J.level_offset[L] + (size_t)y * w + x] = t;
    };
    float v = min_across(glsl_min(ta, tb), lane, 16u);
    if ((lane & 16u) == 0u) store(1u, x1, y0 >> 1, v);
    v = min_across(glsl_min(quad_perm<0, 0, 2, 2>(v), quad_perm<1, 1, 3, 3>(v)), lane, 32u);
    if ((lane & 49u) == 0u) {
        store(2u, x1 >> 1, y0 >> 2, v);
        sm.l2[wave * 8u + (lane >> 1)] = v;
    }
    __syncthreads();
    // ---- levels 3 to 5: lane = level-2 texel (lane & 7, lane >> 3) of the tile
    const uint32_t n_tiles = J.tiles_x * J.tiles_y;
    const bool tail = levels < J.mips && tile + 1u == n_tiles;
    if (wave && !tail) return;
    {
        const uint32_t lx = lane & 7u, ly = lane >> 3;
        v = sm.l2[lane];
        v = min_across(glsl_min(quad_perm<0, 0, 2, 2>(v), quad_perm<1, 1, 3, 3>(v)), lane, 8u);
        if (wave == 0u && ((lx | ly) & 1u) == 0u) store(3u, tx * 4u + (lx >> 1), ty * 4u + (ly >> 1), v);
        v = min_across(glsl_min(quad_perm<0, 0, 0, 0>(v), quad_perm<2, 2, 2, 2>(v)), lane, 16u);
        if (wave == 0u && ((lx | ly) & 3u) == 0u) store(4u, tx * 2u + (lx >> 2), ty * 2u + (ly >> 2), v);
        v = min_across(min_across(v, lane, 4u), lane, 32u);
        if (tid == 0u) store(5u, tx, ty, v);
    }
    if (levels >= J.mips) return;
    // ---- hand each tile's 1x1 value to the highest-numbered workgroup, which reduces the tail levels. The value
    // travels in a 64-bit agent-scope atomic word with a presence flag; the receiving workgroup clears each word
    // after reading it, so every build starts with all words zero. Neither a release fence (an L2 write-back per
    // workgroup) nor a shared completion counter (a serialised atomic per workgroup) is needed.
    if (!tail) {
        if (tid == 0)
            __hip_atomic_store(&J.tail[tile], kTailFlag | __float_as_uint(v), __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_AGENT);
        return;
    }
    // the tile image (one texel per tile, level 5): the words of a thread are loaded together, before the first wait
    constexpr uint32_t KW = kPyrTailTexels * 4u / kPyrBlock;
    unsigned long long w[KW];
#pragma unroll
    for (uint32_t k = 0; k < KW; ++k) {
        const uint32_t i = tid + k * kPyrBlock;
        w[k] = i < n_tiles ? __hip_atomic_load(&J.tail[i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : 0ull;
    }
#pragma unroll
    for (uint32_t k = 0; k < KW; ++k) {
        const uint32_t i = tid + k * kPyrBlock;
        if (i < n_tiles) sm.a[i] = i == tile ? v : tail_finish(J, i, w[k], err);
    }
    uint32_t nw = J.tiles_x, nh = J.tiles_y, cw, ch;
    float* g;
    float* src = sm.a;
    float* dst = sm.b;
    bool one_wave = false;
    // the remaining levels in LDS; from the first of at most 64 texels on, by one wave
    for (uint32_t L = levels; L < J.mips; ++L) {
        if (one_wave) wave_lds_sync();
        else __syncthreads();
        cw = nw;
        ch = nh;
        nw = cw > 1u ? cw >> 1 : 1u;
        nh = ch > 1u ? ch >> 1 : 1u;
        if (!one_wave && nw * nh <= 64u) {
            if (wave) return;
            one_wave = true;
        }
        const uint32_t nshift = (uint32_t)__builtin_ctz(nw), dx = cw > 1u ? 1u : 0u, dy = ch > 1u ? cw : 0u;
        g = J.texels + J.level_offset[L];
        for (uint32_t t = tid; t < nw * nh; t += kPyrBlock) {
            const float* p = src + (t >> nshift) * (dy ? 2u * cw : cw) + (t & (nw - 1u)) * (1u + dx);
            const float m = min4(p[0], p[dx], p[dy], p[dx + dy]);
            dst[t] = m;
            g[t] = m;
        }
        float* tmp = src;
        src = dst;
        dst = tmp;
    }
}

__global__ __launch_bounds__(kPyrBlock) void pyramid_kernel(PyrBuildJob J, uint32_t* err)
{
    __shared__ PyrSmem sm;
    pyramid_tile(J, blockIdx.x, sm, err);
}

// Last entry of the ascending table `starts` that is <= x (searched in LDS when staged there).
__device__ __forceinline__ uint32_t last_le(const uint32_t* starts, uint32_t n, uint32_t x)
{
    uint32_t lo = 0, hi = n - 1u;
    while (lo < hi) {
        const uint32_t mid = (lo + hi + 1u) >> 1;
        if (starts[mid] <= x) lo = mid;
        else hi = mid - 1u;
    }
    return lo;
}

// Many pyramids in one launch: workgroup (x, y) builds level-0 tile x of job y; workgroups past the job's tiles return
// at once. The job index is the workgroup's y, so no table of first workgroups is searched (the search's load cost
// each workgroup a round trip: the 256-view batch 336.6 us against 314.6 us), and the descriptor is read in place with
// scalar loads. Within a job, workgroups are dispatched in tile order, so the job's last tile (which waits on the others'
// hand-off words) starts after every tile it waits for.
__global__ __launch_bounds__(kPyrBlock) void pyramid_batch_kernel(const PyrBuildJob* __restrict__ jobs, uint32_t* err)
{
    __shared__ PyrSmem sm;
    const PyrBuildJob& J = jobs[blockIdx.y];
    if (blockIdx.x >= J.tiles_x * J.tiles_y) return;
    pyramid_tile(J, blockIdx.x, sm, err);
}

// The same for a few jobs, which come in the kernel arguments.
__global__ __launch_bounds__(kPyrBlock) void pyramid_few_kernel(PyrArgs jobs, uint32_t* err)
{
    __shared__ PyrSmem sm;
    const PyrBuildJob& J = jobs.j[blockIdx.y];
    if (blockIdx.x >= J.tiles_x * J.tiles_y) return;
    pyramid_tile(J, blockIdx.x, sm, err);
}

// The coordinates of a footprint along one axis: texels i0 and i1 (equal when the second has no weight) of `src` texels
// below texel x of `dst` (footprint() of cull_math.h, axis by axis).
__device__ __forceinline__ void footprint_axis(uint32_t x, uint32_t dst, uint32_t src, uint32_t& i0, uint32_t& i1)
{
    const float u = ((float)x + 0.5f) / (float)dst;
    const float t = u * (float)src - 0.5f, f = floorf(t);
    i0 = clamp_texel(f, src);
    i1 = (t - f) > 0.0f ? clamp_texel(f + 1.0f, src) : i0;
}

// Extents that are not powers of two, in one launch. A workgroup owns kRegionTile x kRegionTile texels of level K (the
// last of `tile_levels`) and, of every level below, the texels from the first one under its own first texel to the first
// one under the next tile's; it computes those and the few of its neighbours' that its own footprints reach into (the
// plan's `need`), level by level in LDS, and stores what it owns. Level K then goes to the highest-numbered workgroup as
// flagged words, like the tile image of the power-of-two build, which reduces the levels that remain. One launch per
// level, as larger bases still take, costs a launch and a round trip per level for ever fewer texels (800 x 450 with 10
// mips: 10.2 us against 21.5 us of kernels, 30 us a build where the host is the bound). Two texels of level 4 and axis per
// workgroup: 350 workgroups for 800 x 450, each computing at most 47 x 47 texels of level 0 for 32 x 32 of its own.
constexpr uint32_t kRegionBlock = 512;
struct RegionSmem {
    uint32_t c0[2][kRegionLevels][kRegionMax], c1[2][kRegionLevels][kRegionMax];  // per axis and level: footprint
    float a[kRegionTail];                       // level 0, 2, 4 of the region; then the tail's image ...
    float b[kRegionTail / 2u];                  // levels 1, 3; then its levels in turn (half: an image one texel wide)
};
static_assert(kRegionMax * kRegionMax <= kRegionTail, "the region's level 0 fits the tail's image");

__global__ __launch_bounds__(kRegionBlock) void pyramid_region_kernel(PyrBuildJob J, uint32_t* err)
{
    __shared__ RegionSmem sm;
    const uint32_t tid = threadIdx.x, lx = tid & 31u, ly = tid >> 5;
    const uint32_t K = J.tile_levels - 1u;
    const PyrRegion* px = J.plan + (size_t)(blockIdx.x % J.tiles_x) * kRegionLevels;
    const PyrRegion* py = J.plan + (size_t)(J.tiles_x + blockIdx.x / J.tiles_x) * kRegionLevels;
    for (uint32_t q = tid; q < 2u * kRegionLevels * kRegionMax; q += kRegionBlock) {
        const uint32_t axis = q / (kRegionLevels * kRegionMax), L = q / kRegionMax % kRegionLevels, i = q % kRegionMax;
        const PyrRegion* p = axis ? py : px;
        if (L <= K && p[L].begin + i < p[L].need) {
            const uint32_t base = axis ? J.base_h : J.base_w;
            const uint32_t src = L ? level_dim(base, L - 1u) : (axis ? J.h : J.w), off = L ? p[L - 1u].begin : 0u;
            uint32_t i0, i1;
            footprint_axis(p[L].begin + i, level_dim(base, L), src, i0, i1);
            sm.c0[axis][L][i] = i0 - off;
            sm.c1[axis][L][i] = i1 - off;
        }
    }
    __syncthreads();
    // ---- level 0 from the depth image: the loads of three texels of a thread before the first minimum
    {
        const PyrRegion rx = px[0], ry = py[0];
        const uint32_t nw = rx.need - rx.begin, nh = ry.need - ry.begin;
        for (uint32_t x = lx; x < nw; x += 32u) {
            const uint32_t x0 = sm.c0[0][0][x], x1 = sm.c1[0][0][x];
            for (uint32_t yb = ly; yb < nh; yb += 48u) {
                float d[3][4];
#pragma unroll
                for (uint32_t k = 0; k < 3u; ++k) {
                    const uint32_t y = yb + 16u * k < nh ? yb + 16u * k : yb;
                    const float* r0 = J.depth + (size_t)sm.c0[1][0][y] * J.w;
                    const float* r1 = J.depth + (size_t)sm.c1[1][0][y] * J.w;
                    d[k][0] = r0[x0];
                    d[k][1] = r0[x1];
                    d[k][2] = r1[x0];
                    d[k][3] = r1[x1];
                }
#pragma unroll
                for (uint32_t k = 0; k < 3u; ++k) {
                    const uint32_t y = yb + 16u * k;
                    if (y >= nh) continue;
                    const float m = min4(d[k][0], d[k][1], d[k][2], d[k][3]);
                    sm.a[y * kRegionMax + x] = m;
                    if (rx.begin + x < rx.end && ry.begin + y < ry.end)
                        J.texels[(size_t)(ry.begin + y) * J.base_w + rx.begin + x] = m;
                }
            }
        }
    }
    const bool handoff = J.tile_levels < J.mips;
    for (uint32_t L = 1; L <= K; ++L) {
        __syncthreads();
        const float* src = (L & 1u) ? sm.a : sm.b;
        float* dst = (L & 1u) ? sm.b : sm.a;
        const uint32_t ps = (L & 1u) ? kRegionMax : kRegionMax / 2u, pd = (L & 1u) ? kRegionMax / 2u : kRegionMax;
        const PyrRegion rx = px[L], ry = py[L];
        const uint32_t nw = rx.need - rx.begin, nh = ry.need - ry.begin, W = level_dim(J.base_w, L);
        float* g = J.texels + J.level_offset[L];
        for (uint32_t y = ly; y < nh; y += 16u) {
            const float* r0 = src + sm.c0[1][L][y] * ps;
            const float* r1 = src + sm.c1[1][L][y] * ps;
            for (uint32_t x = lx; x < nw; x += 32u) {
                const uint32_t x0 = sm.c0[0][L][x], x1 = sm.c1[0][L][x];
                const float m = min4(r0[x0], r0[x1], r1[x0], r1[x1]);
                dst[y * pd + x] = m;
                if (rx.begin + x < rx.end && ry.begin + y < ry.end) {
                    const size_t at = (size_t)(ry.begin + y) * W + rx.begin + x;
                    g[at] = m;
                    if (L == K && handoff)
                        __hip_atomic_store(&J.tail[at], kTailFlag | __float_as_uint(m), __ATOMIC_RELAXED,
                                           __HIP_MEMORY_SCOPE_AGENT);
                }
            }
        }
    }
    if (!handoff || blockIdx.x + 1u < gridDim.x) return;
    // ---- the tail: level K from all workgroups (this one's too), then the levels that remain, in LDS
    __syncthreads();
    uint32_t nw = level_dim(J.base_w, K), nh = level_dim(J.base_h, K);
    constexpr uint32_t KW = 8;  // words of a thread in flight
    for (uint32_t i0 = 0; i0 < nw * nh; i0 += KW * kRegionBlock) {
        unsigned long long w[KW];
#pragma unroll
        for (uint32_t k = 0; k < KW; ++k) {
            const uint32_t i = i0 + k * kRegionBlock + tid;
            w[k] = i < nw * nh ? __hip_atomic_load(&J.tail[i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : 0ull;
        }
#pragma unroll
        for (uint32_t k = 0; k < KW; ++k) {
            const uint32_t i = i0 + k * kRegionBlock + tid;
            if (i < nw * nh) sm.a[i] = tail_finish(J, i, w[k], err);
        }
    }
    const float* src = sm.a;
    float* dst = sm.b;
    for (uint32_t L = J.tile_levels; L < J.mips; ++L) {
        __syncthreads();
        const uint32_t cw = nw, ch = nh;
        nw = level_dim(J.base_w, L);
        nh = level_dim(J.base_h, L);
        float* g = J.texels + J.level_offset[L];
        for (uint32_t y = ly; y < nh; y += 16u) {
            uint32_t y0, y1;
            footprint_axis(y, nh, ch, y0, y1);
            for (uint32_t x = lx; x < nw; x += 32u) {
                uint32_t x0, x1;
                footprint_axis(x, nw, cw, x0, x1);
                const float m = min4(src[y0 * cw + x0], src[y0 * cw + x1], src[y1 * cw + x0], src[y1 * cw + x1]);
                dst[y * nw + x] = m;
                g[y * nw + x] = m;
            }
        }
        const float* done = dst;
        dst = dst == sm.b ? sm.a : sm.b;
        src = done;
    }
}

// General per-level footprint reduction (any sizes).
__global__ void pyramid_level_kernel(const float* __restrict__ src, uint32_t sw, uint32_t sh, float* __restrict__ dst,
                                     uint32_t dw, uint32_t dh)
{
    const uint32_t x = blockIdx.x * 16u + (threadIdx.x & 15u);
    const uint32_t y = blockIdx.y * 16u + (threadIdx.x >> 4);
    if (x >= dw || y >= dh) return;
    const float u = ((float)x + 0.5f) / (float)dw;
    const float v = ((float)y + 0.5f) / (float)dh;
    const Footprint f = footprint(u, v, sw, sh);
    dst[(size_t)y * dw + x] = footprint_min(src, sw, f);
}

// Synthetic depth: one workgroup per 64 x 64 pixel tile. The workgroup regenerates the rectangles from the seed in
// chunks, keeps those overlapping its tile in LDS, and each pixel (16 per thread, in registers) takes the max
// (nearest, reverse-z) of the ground plane and its covering rectangles. max is exact, so the order of the LDS list
// does not matter.
constexpr uint32_t kRasterTile = kSynthTile;
constexpr uint32_t kMaxRects = kSynthMaxRects;
constexpr uint32_t kRectChunk = 512;
constexpr uint32_t kRasterPix = kRasterTile * kRasterTile / 256;

__device__ __forceinline__ void synth_depth_tile(uint64_t seed, uint32_t W, uint32_t H, uint32_t n_rects, float p11, float znear,
                                 float* __restrict__ depth, uint32_t bx, uint32_t by, int4* s_rect, float* s_depth,
                                 uint32_t* s_n)
{
    const int32_t tx0 = (int32_t)(bx * kRasterTile), ty0 = (int32_t)(by * kRasterTile);
    const int32_t tx1 = tx0 + (int32_t)kRasterTile, ty1 = ty0 + (int32_t)kRasterTile;
    float d[kRasterPix];
#pragma unroll
    for (uint32_t k = 0; k < kRasterPix; ++k) {
        const uint32_t t = threadIdx.x + k * 256u;
        const int32_t y = ty0 + (int32_t)(t / kRasterTile);
        d[k] = synth_plane_depth((uint32_t)(y < (int32_t)H ? y : 0), H, p11, znear);
    }
    for (uint32_t r0 = 0; r0 < n_rects; r0 += kRectChunk) {
        if (threadIdx.x == 0) *s_n = 0;
        __syncthreads();
        const uint32_t r1 = r0 + kRectChunk < n_rects ? r0 + kRectChunk : n_rects;
        for (uint32_t r = r0 + threadIdx.x; r < r1; r += 256) {
            const SynthRect sr = synth_rect(seed, W, H, r);
            if (sr.x0 < tx1 && sr.x1 > tx0 && sr.y0 < ty1 && sr.y1 > ty0) {
                const uint32_t slot = atomicAdd(s_n, 1u);
                s_rect[slot] = make_int4(sr.x0, sr.y0, sr.x1, sr.y1);
                s_depth[slot] = sr.depth;
            }
        }
        __syncthreads();
        const uint32_t n = *s_n;
        for (uint32_t j = 0; j < n; ++j) {
            const int4 rc = s_rect[j];
            const float rd = s_depth[j];
#pragma unroll
            for (uint32_t k = 0; k < kRasterPix; ++k) {
                const uint32_t t = threadIdx.x + k * 256u;
                const int32_t x = tx0 + (int32_t)(t % kRasterTile), y = ty0 + (int32_t)(t / kRasterTile);
                if (x >= rc.x && x < rc.z && y >= rc.y && y < rc.w) d[k] = glsl_max(d[k], rd);
            }
        }
        __syncthreads();  // the list is rewritten by the next chunk
    }
#pragma unroll
    for (uint32_t k = 0; k < kRasterPix; ++k) {
        const uint32_t t = threadIdx.x + k * 256u;
        const int32_t x = tx0 + (int32_t)(t % kRasterTile), y = ty0 + (int32_t)(t / kRasterTile);
        if (x < (int32_t)W && y < (int32_t)H) depth[(size_t)y * W + x] = d[k];
    }
}

__global__ __launch_bounds__(256) void synth_depth_kernel(uint64_t seed, uint32_t W, uint32_t H, uint32_t n_rects,
                                                          float p11, float znear, float* __restrict__ depth)
{
    __shared__ int4 s_rect[kRectChunk];
    __shared__ float s_depth[kRectChunk];
    __shared__ uint32_t s_n;
    synth_depth_tile(seed, W, H, n_rects, p11, znear, depth, blockIdx.x, blockIdx.y, s_rect, s_depth, &s_n);
}

// Many depth buffers in one launch (workgroup b rasterises tile b - wg_start of the job whose range holds b).
__global__ __launch_bounds__(256) void synth_depth_batch_kernel(const SynthJob* __restrict__ jobs,
                                                                const uint32_t* __restrict__ starts, uint32_t n_jobs)
{
    __shared__ int4 s_rect[kRectChunk];
    __shared__ float s_depth[kRectChunk];
    __shared__ uint32_t s_n;
    __shared__ uint32_t s_start[kLdsJobs];
    uint32_t j;
    if (n_jobs <= kLdsJobs) {
        for (uint32_t k = threadIdx.x; k < n_jobs; k += 256) s_start[k] = starts[k];
        __syncthreads();
        j = last_le(s_start, n_jobs, blockIdx.x);
    } else {
        j = last_le(starts, n_jobs, blockIdx.x);
    }
    const SynthJob J = jobs[j];
    const uint32_t local = blockIdx.x - J.wg_start;
    if (local == 0 && J.tail_zero)
        for (uint32_t k = threadIdx.x; k < J.n_tail; k += 256) J.tail_zero[k] = 0ull;
    synth_depth_tile(J.seed, J.w, J.h, J.occluders, J.p11, J.znear, J.depth, local % J.tiles_x, local / J.tiles_x,
                     s_rect, s_depth, &s_n);
}

}  // namespace

hipError_t launch_pyramid(const PyrBuildJob& job, uint32_t* err, hipStream_t st)
{
    hipLaunchKernelGGL(pyramid_kernel, dim3(job.tiles_x * job.tiles_y), dim3(kPyrBlock), 0, st, job, err);
    return hipGetLastError();
}

hipError_t launch_pyramid_batch(const PyrBuildJob* jobs_host, const PyrBuildJob* jobs_dev, uint32_t n_jobs,
                                uint32_t* err, hipStream_t st)
{
    if (n_jobs == 0) return hipSuccess;
    uint32_t max_tiles = 1;
    for (uint32_t k = 0; k < n_jobs; ++k) {
        const uint32_t t = jobs_host[k].tiles_x * jobs_host[k].tiles_y;
        max_tiles = t > max_tiles ? t : max_tiles;
    }
    if (n_jobs <= kArgPyrJobs) {
        PyrArgs a;
        for (uint32_t k = 0; k < kArgPyrJobs; ++k) a.j[k] = jobs_host[k < n_jobs ? k : 0u];
        hipLaunchKernelGGL(pyramid_few_kernel, dim3(max_tiles, n_jobs), dim3(kPyrBlock), 0, st, a, err);
        return hipGetLastError();
    }
    constexpr uint32_t kMaxGridY = 65535;  // jobs per launch (the grid's y extent); more go in further launches
    for (uint32_t j0 = 0; j0 < n_jobs; j0 += kMaxGridY) {
        const uint32_t n = n_jobs - j0 < kMaxGridY ? n_jobs - j0 : kMaxGridY;
        hipLaunchKernelGGL(pyramid_batch_kernel, dim3(max_tiles, n), dim3(kPyrBlock), 0, st, jobs_dev + j0, err);
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    return hipGetLastError();
}

// The regions of one axis (kRegionLevels per tile): the same float arithmetic as the kernel's footprints.
bool plan_region_axis(uint32_t base, uint32_t K, PyrRegion* out)
{
    const uint32_t n = level_dim(base, K), tiles = (n + kRegionTile - 1u) / kRegionTile;
    auto at = [&](uint32_t L, uint32_t x, uint32_t& i0, uint32_t& i1) {  // footprint of level L's texel x in level L - 1
        const uint32_t src = level_dim(base, L - 1u);
        const Footprint f = footprint(((float)x + 0.5f) / (float)level_dim(base, L), 0.0f, src, 1u);
        i0 = f.x0;
        i1 = f.x1;
    };
    for (uint32_t t = 0; t < tiles; ++t) {
        PyrRegion* r = out + (size_t)t * kRegionLevels;
        for (uint32_t L = 0; L < kRegionLevels; ++L) r[L] = PyrRegion{ 0u, 0u, 0u };
        r[K].begin = t * kRegionTile;
        r[K].end = t + 1u < tiles ? (t + 1u) * kRegionTile : n;
        r[K].need = r[K].end;
        for (uint32_t L = K; L >= 1u; --L) {
            uint32_t i0, i1;
            at(L, r[L].begin, i0, i1);
            r[L - 1u].begin = t ? i0 : 0u;
            if (t + 1u < tiles) at(L, r[L].end, r[L - 1u].end, i1);
            else r[L - 1u].end = level_dim(base, L - 1u);
            at(L, r[L].need - 1u, i0, i1);
            r[L - 1u].need = i1 + 1u > r[L - 1u].end ? i1 + 1u : r[L - 1u].end;
            const uint32_t room = ((L - 1u) & 1u) ? kRegionMax / 2u : kRegionMax;
            if (r[L - 1u].need - r[L - 1u].begin > room) return false;
        }
    }
    return true;
}

hipError_t launch_pyramid_region(const PyrBuildJob& job, uint32_t* err, hipStream_t st)
{
    hipLaunchKernelGGL(pyramid_region_kernel, dim3(job.tiles_x * job.tiles_y), dim3(kRegionBlock), 0, st, job, err);
    return hipGetLastError();
}

hipError_t launch_pyramid_level(const float* src, uint32_t sw, uint32_t sh, float* dst, uint32_t dw, uint32_t dh,
                                hipStream_t st)
{
    hipLaunchKernelGGL(pyramid_level_kernel, dim3((dw + 15) / 16, (dh + 15) / 16), dim3(256), 0, st, src, sw, sh, dst,
                       dw, dh);
    return hipGetLastError();
}

hipError_t launch_synth_depth_batch(const SynthJob* jobs_dev, const uint32_t* starts_dev, uint32_t n_jobs,
                                    uint32_t total_wgs, hipStream_t st)
{
    if (n_jobs == 0 || total_wgs == 0) return hipSuccess;
    hipLaunchKernelGGL(synth_depth_batch_kernel, dim3(total_wgs), dim3(256), 0, st, jobs_dev, starts_dev, n_jobs);
    return hipGetLastError();
}

hipError_t launch_synth_depth(uint64_t seed, uint32_t w, uint32_t h, uint32_t occluders, float p11, float znear,
                              float* depth, hipStream_t st)
{
    if (occluders > kMaxRects) return hipErrorInvalidValue;
    hipLaunchKernelGGL(synth_depth_kernel, dim3((w + kRasterTile - 1) / kRasterTile, (h + kRasterTile - 1) / kRasterTile),
                       dim3(256), 0, st, seed, w, h, occluders, p11, znear, depth);
    return hipGetLastError();
}

}  // namespace bz
