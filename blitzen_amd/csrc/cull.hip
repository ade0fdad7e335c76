// cull.hip — gfx950 draw-cull kernels (early / late / plain / temporal / onpc passes).
//
// Replaces InitialDrawCull.comp.glsl:12-58, LateDrawCull.comp.glsl:13-71, TransparentDrawCull.comp.glsl:13-65,
// OnpcDrawCull.comp.glsl:11-52 and drawOccTemporal.hlsl:13-64. The per-object arithmetic is in cull_math.h.
//
// Two kernels per pass, both HBM-streaming, with no wait between workgroups:
//   decide: tiles of BLOCK x ITEMS objects, each wave a run of 64 x ITEMS neighbouring ones. Every object stream
//           of the tile is loaded at once (coalesced SoA float4 / uint32 loads); sphere -> view space and frustum
//           test for every object; the frustum survivors of each wave are compacted into LDS so the Hi-Z test
//           (two square roots, five divisions, a 2x2 gather) runs on dense lanes, and likewise the emitting objects
//           for LOD selection. Emitting objects are ranked with wave64 ballots and the waves' totals in (wave, item)
//           order, i.e. ascending object order, and written as (objectId, LOD) to the tile's staging slot; the
//           tile's count goes to counts[tile]. The LATE pass also writes visibility here.
//   emit:   each workgroup takes a run of tiles, adds the counts of the job's earlier tiles (a block reduction) to
//           get its output base, and writes DrawIndexedIndirect commands in order, plus the draw count.
// The output order is ascending objectId, independent of scheduling (the reference appends in atomicAdd order).
// A pass over few objects is one kernel (fused_kernel, late_tile_kernel): each tile adds up the counts that the tiles
// before it publish. For many tiles, and as a decoupled look-back, that was measured slower: cross-XCD status visibility
// costs ~1 us per round trip and the first generation of workgroups waits for the slowest of them.
#include "bz_internal.h"
#include "fuse.h"

namespace bz {

namespace {

__device__ __forceinline__ uint32_t wave_incl_scan(uint32_t v, uint32_t lane)
{
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        uint32_t t = __shfl_up(v, off, 64);
        if (lane >= (uint32_t)off) v += t;
    }
    return v;
}

// Small tables staged in LDS per workgroup when they fit: surface radii and LOD ranges (512 surfaces, 6 KiB),
// LOD errors (2048 LODs, 8 KiB) and the pyramid's level offsets. Larger tables are gathered from global memory.
constexpr uint32_t kLdsSurfaces = 512;
constexpr uint32_t kLdsLods = 2048;

template <int BLOCK, int ITEMS, bool LDS_TAB>
struct TileSmem {
    float surf_rad[LDS_TAB ? kLdsSurfaces : 1];
    uint2 surf_lod[LDS_TAB ? kLdsSurfaces : 1];
    float lod_err[LDS_TAB ? kLdsLods : 1];
    float4 cand[BLOCK];               // per-wave compaction area: one chunk of 64 entries per wave
    uint2 cand2[BLOCK];
    uint32_t lvl[kMaxMips];
    uint32_t wtot[2][BLOCK / 64];     // per-wave totals of the emitting objects, by the tile's parity
    uint32_t ctot[2][BLOCK / 64];     // frame cache: per-wave totals of the survivors
    uint32_t csum[BLOCK / 64];        // cluster mode: per-wave sums of the emitting objects' cluster counts
    uint32_t last;                    // one-launch passes: the number of the launch before
    uint32_t red[2 * (BLOCK / 64)];   // and the reduction of the earlier tiles' counts
};

// Pass families compiled separately so the visibility stream is loaded unconditionally where it is used.
enum : int { MODE_EARLY = 0, MODE_LATE = 1, MODE_OTHER = 2 };  // OTHER: PLAIN, TEMPORAL, ONPC (runtime-uniform)

// Orders a wave's LDS writes before its later LDS reads (the compaction areas are private to a wave): a compiler
// barrier, then a wait on LDS operations only (lgkmcnt(0); vmcnt and expcnt left at their maxima), so global loads in
// flight, such as the next tile's prefetch, are not waited on.
__device__ __forceinline__ void wave_lds_sync()
{
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    __builtin_amdgcn_s_waitcnt(0xC07F);
    __builtin_amdgcn_wave_barrier();
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
}

// Per-wave compaction of a lane predicate over ITEMS items: slot[k] = this lane's position among the wave's set
// entries in (item, lane) order; returns the wave's total.
template <int ITEMS>
__device__ __forceinline__ uint32_t wave_compact(const bool (&pred)[ITEMS], uint32_t (&slot)[ITEMS], uint32_t lane)
{
    uint32_t total = 0;
#pragma unroll
    for (int k = 0; k < ITEMS; ++k) {
        const unsigned long long m = __ballot(pred[k]);
        slot[k] = total + (uint32_t)__popcll(m & ((1ull << lane) - 1ull));
        total += (uint32_t)__popcll(m);
    }
    return total;
}

// Object streams of one tile held in registers. Indices are clamped into the job so every load is issued without
// waiting on another; out-of-range lanes are discarded afterwards. Item k of a thread is object tile_object + 64 k of
// the job: a wave's objects are consecutive, so that their order within the tile is (wave, item, lane) and a wave ranks
// its own without its neighbours. The indices are recomputed from the tile's number where they are needed, not kept: two
// tiles' streams are live at once, and 64 registers a thread is what a fourth workgroup per CU fits in.
template <int ITEMS>
struct Streams {
    uint32_t vis[ITEMS], surf[ITEMS];
    float4 w[ITEMS];  // world-space centre, scale
};

template <int BLOCK, int ITEMS>
__device__ __forceinline__ uint32_t tile_object(uint32_t tile_in_job)
{
    return tile_in_job * (uint32_t)(BLOCK * ITEMS) + (threadIdx.x >> 6) * (64u * ITEMS) + (threadIdx.x & 63u);
}
// Item k's object, clamped into the job (jobs always hold at least one object).
__device__ __forceinline__ uint32_t clamped_object(const CullJob& J, uint32_t i)
{
    return J.begin + (i < J.n ? i : J.n - 1u);
}

// Loads of the per-object streams. NT: marked non-temporal (streaming, evicted first), for the passes that read each
// stream once and gather no Hi-Z texels: an EARLY pass recording a frame cache (its LATE pass reads the records, not
// these streams again: 4% faster per frame), PLAIN and ONPC (4%). Without the cache the LATE pass re-reads the same
// streams and finds part of them still in the last-level cache, which the hint would give up (2.5% slower per frame),
// and passes with a Hi-Z test keep their texels cached better without it, so those keep the default policy.
typedef float nt_float4 __attribute__((ext_vector_type(4)));
template <bool NT>
__device__ __forceinline__ float4 stream_load(const float4* p)
{
    if constexpr (NT) {
        const nt_float4 v = __builtin_nontemporal_load(reinterpret_cast<const nt_float4*>(p));
        return make_float4(v.x, v.y, v.z, v.w);
    } else {
        return *p;
    }
}
template <bool NT, class T>
__device__ __forceinline__ T stream_load(const T* p)
{
    if constexpr (NT) return __builtin_nontemporal_load(p);
    else return *p;
}

// The visibility stream (EARLY, LATE).
template <int BLOCK, int ITEMS, int MODE, bool NT = false>
__device__ __forceinline__ void issue_vis(const CullJob& J, uint32_t tile_in_job, Streams<ITEMS>& s)
{
    const uint32_t i0 = tile_object<BLOCK, ITEMS>(tile_in_job);
#pragma unroll
    for (int k = 0; k < ITEMS; ++k) {
        s.vis[k] = 0u;
        if (MODE == MODE_EARLY || MODE == MODE_LATE)
            s.vis[k] = stream_load<NT>(J.vis_in + clamped_object(J, i0 + 64u * k));
    }
}

// The surface-id and world-space sphere streams: for every object, or in EARLY only for last-frame-visible ones (which
// waits for the visibility stream first).
// ALL (EARLY recording a frame cache): every object's streams are loaded, not only the last-frame-visible ones.
template <int BLOCK, int ITEMS, int MODE, bool ALL = false, bool NT = false>
__device__ __forceinline__ void issue_objects(const CullJob& J, uint32_t tile_in_job, Streams<ITEMS>& s)
{
    const SceneDev& S = J.scene;
    const uint32_t i0 = tile_object<BLOCK, ITEMS>(tile_in_job);
#pragma unroll
    for (int k = 0; k < ITEMS; ++k) {
        const uint32_t g = clamped_object(J, i0 + 64u * k);
        s.surf[k] = 0u;
        s.w[k] = make_float4(0.f, 0.f, 0.f, 0.f);
        if (MODE != MODE_EARLY || ALL || (i0 + 64u * k < J.n && s.vis[k] != 0u)) {
            s.surf[k] = S.obj_surf16 ? (uint32_t)stream_load<NT>(S.obj_surf16 + g) : stream_load<NT>(S.obj_surf + g);
            s.w[k] = stream_load<NT>(S.world + g);
        }
    }
}

template <int BLOCK, int ITEMS, int MODE, bool ALL = false, bool NT = false>
__device__ __forceinline__ void issue_tile(const CullJob& J, uint32_t tile_in_job, Streams<ITEMS>& s)
{
    issue_vis<BLOCK, ITEMS, MODE, NT>(J, tile_in_job, s);
    issue_objects<BLOCK, ITEMS, MODE, ALL, NT>(J, tile_in_job, s);
}

// Small tables into LDS (surface radii and LOD ranges, LOD errors) plus the pyramid's level offsets. All loads of a
// thread are issued before its first LDS write. The caller places the barrier.
template <int BLOCK, int ITEMS, bool LDS_TAB>
__device__ __forceinline__ void stage_tables(const CullJob& J, TileSmem<BLOCK, ITEMS, LDS_TAB>& sm)
{
    const uint32_t tid = threadIdx.x;
    const SceneDev& S = J.scene;
    if constexpr (LDS_TAB) {
        constexpr int SPT = (kLdsSurfaces + BLOCK - 1) / BLOCK, LPT = (kLdsLods + BLOCK - 1) / BLOCK;
        float t_rad[SPT];
        uint2 t_lod[SPT];
        float t_err[LPT];
#pragma unroll
        for (int j = 0; j < SPT; ++j) {
            const uint32_t t = tid + (uint32_t)j * BLOCK;
            const uint32_t tt = t < S.n_surfaces ? t : 0u;
            t_rad[j] = S.surf_sphere[tt].w;
            t_lod[j] = S.surf_lod[tt];
        }
#pragma unroll
        for (int j = 0; j < LPT; ++j) {
            const uint32_t t = tid + (uint32_t)j * BLOCK;
            t_err[j] = S.lod_error[t < S.n_lods ? t : 0u];
        }
#pragma unroll
        for (int j = 0; j < SPT; ++j) {
            const uint32_t t = tid + (uint32_t)j * BLOCK;
            if (t < S.n_surfaces) {
                sm.surf_rad[t] = t_rad[j];
                sm.surf_lod[t] = t_lod[j];
            }
        }
#pragma unroll
        for (int j = 0; j < LPT; ++j) {
            const uint32_t t = tid + (uint32_t)j * BLOCK;
            if (t < S.n_lods) sm.lod_err[t] = t_err[j];
        }
    }
    if (tid < (uint32_t)kMaxMips) {  // level offsets from the extent (no load): sum of the smaller levels' areas
        uint32_t off = 0;
        for (uint32_t L = 0; L < tid; ++L) off += level_dim(J.pyr.base_w, L) * level_dim(J.pyr.base_h, L);
        sm.lvl[tid] = off;
    }
}

struct NoPrefetch {
    __device__ __forceinline__ void operator()() const {}
};

// By the last tile of a one-launch pass: the commands of the tiles that left theirs, as (objectId, LOD) entries.
__device__ __forceinline__ void settle_staged(const CullJob& J, uint32_t tile_size, const uint2* staging, const FuseDev& fuse,
                                              uint32_t launch, uint32_t left)
{
    fuse_settle(fuse, launch, left, J.n_tiles, [&](uint32_t t, uint32_t first, uint32_t n) {
        for (uint32_t e = threadIdx.x; e < n; e += 64u) {
            const uint2 en = staging[(size_t)t * tile_size + e];
            if (first + e < J.capacity) write_command(J.cmds, first + e, en.x, J.scene.lod_draw[en.y]);
        }
    });
}

// Decides one tile whose streams are in `s` (the decide kernel's body). Called by all threads of the workgroup.
// `prefetch` is invoked once, after the tile's last global gather (the Hi-Z texels), so loads it issues stay in
// flight through the rest of the tile (vmcnt retires in issue order: nothing later waits on them).
// CL (cluster object pass): ccounts[gtile] also receives the sum of the emitting objects' LOD cluster counts.
// CACHE (EARLY with all streams loaded): every frustum survivor of the tile is recorded in the frame cache `fc`.
// INST (LOD-instanced output): each emitting object also adds 1 to its LOD's bin of the workgroup's LDS histogram.
// FUSED (one tile per workgroup): the tile's commands are written here and not staged for an emit launch (staged only
// where the tile leaves them to the last one).
template <int BLOCK, int ITEMS, int MODE, bool HIZ, bool LDS_TAB, bool CL = false, bool CACHE = false, bool INST = false,
          bool FUSED = false, class Prefetch>
__device__ __forceinline__ void process_tile(const CullJob& J, uint32_t tile_in_job, uint32_t gtile, uint32_t parity,
                                             const Streams<ITEMS>& s, uint32_t* counts, uint2* staging,
                                             uint32_t* ccounts,
                                             TileSmem<BLOCK, ITEMS, LDS_TAB>& sm, Prefetch&& prefetch,
                                             FrameCacheDev fc = FrameCacheDev{}, uint32_t* lds_hist = nullptr,
                                             FuseDev fuse = FuseDev{}, uint32_t launch = 0u)
{
    constexpr bool lds_tab = LDS_TAB;
    constexpr int NW = BLOCK / 64;
    constexpr uint32_t TILE = BLOCK * ITEMS;
    constexpr bool late = MODE == MODE_LATE;
    const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t pass = J.pass;
    const uint32_t i0 = tile_object<BLOCK, ITEMS>(tile_in_job);  // item k: object i0 + 64 k of the job
    const SceneDev& S = J.scene;

    float cx[ITEMS], cy[ITEMS], cz[ITEMS], rad[ITEMS];
    if (lds_tab) {
#pragma unroll
        for (int k = 0; k < ITEMS; ++k) rad[k] = sm.surf_rad[s.surf[k]];
    } else {
#pragma unroll
        for (int k = 0; k < ITEMS; ++k) rad[k] = S.surf_sphere[s.surf[k]].w;
    }

    // ---- sphere -> view space + frustum for every object
    bool vis_new[ITEMS], emit[ITEMS], frus[ITEMS];
#pragma unroll
    for (int k = 0; k < ITEMS; ++k) {
        world_to_view(J.view, s.w[k].x, s.w[k].y, s.w[k].z, cx[k], cy[k], cz[k]);
        rad[k] = rad[k] * s.w[k].w;
        frus[k] = i0 + 64u * k < J.n && frustum_visible(J.view, cx[k], cy[k], cz[k], rad[k]);
        vis_new[k] = frus[k] && (MODE != MODE_EARLY || s.vis[k] != 0u);
    }
    float4* cand = sm.cand + wave * 64u;
    uint2* cand2 = sm.cand2 + wave * 64u;

    // ---- Hi-Z on the wave's frustum survivors, compacted onto dense lanes in chunks of 64. The texel gathers are
    // issued by every lane (idle lanes read a clamped, in-bounds texel) and the prefetch is issued right after the
    // first chunk's gathers: vmcnt retires in issue order, so waiting for the gathers does not wait for the prefetch.
    if constexpr (HIZ) {
        uint32_t slot[ITEMS];
        const uint32_t n = wave_compact<ITEMS>(vis_new, slot, lane);
        bool res[ITEMS];
#pragma unroll
        for (int k = 0; k < ITEMS; ++k) res[k] = vis_new[k];
        auto chunk = [&](uint32_t c0, auto&& between) {
#pragma unroll
            for (int k = 0; k < ITEMS; ++k)
                if (vis_new[k] && slot[k] - c0 < 64u) cand[slot[k] - c0] = make_float4(cx[k], cy[k], cz[k], rad[k]);
            wave_lds_sync();
            const bool act = c0 + lane < n;
            const float4 c = cand[lane];
            float a0 = 0.f, a1 = 0.f, a2 = 0.f, a3 = 0.f;
            const bool test =
                act && project_sphere(c.x, c.y, c.z, c.w, J.view.znear, J.view.p00, J.view.p11, a0, a1, a2, a3);
            const float width = (a2 - a0) * J.view.pyrW;
            const float height = (a3 - a1) * J.view.pyrH;
            const uint32_t L = hiz_level(glsl_max(width, height), J.pyr.mips);
            const uint32_t W = level_dim(J.pyr.base_w, L), H = level_dim(J.pyr.base_h, L);
            const Footprint f = footprint((a0 + a2) * 0.5f, (a1 + a3) * 0.5f, W, H);
            float d00, d01, d10, d11;
            footprint_texels(J.pyr.texels + sm.lvl[L], W, f, d00, d01, d10, d11);
            __builtin_amdgcn_sched_barrier(0);  // keep the gathers ahead of the prefetch in issue order
            between();
            __builtin_amdgcn_sched_barrier(0);
            if (act) {
                const float d = glsl_min(glsl_min(d00, d01), glsl_min(d10, d11));
                // a sphere crossing the near plane is not tested and stays visible
                cand2[lane].x = (test ? (J.view.znear / (c.z - c.w) > d) : true) ? 1u : 0u;
            }
            wave_lds_sync();
#pragma unroll
            for (int k = 0; k < ITEMS; ++k)
                if (vis_new[k] && slot[k] - c0 < 64u) res[k] = cand2[slot[k] - c0].x != 0u;
            wave_lds_sync();
        };
        chunk(0u, prefetch);  // always runs (all lanes idle when n == 0): the prefetch is issued unconditionally
        for (uint32_t c0 = 64u; c0 < n; c0 += 64u) chunk(c0, NoPrefetch{});
#pragma unroll
        for (int k = 0; k < ITEMS; ++k) vis_new[k] = res[k];
    } else {
        prefetch();
    }

    // ---- LOD selection on the wave's emitting objects (with a frame cache: on every frustum survivor, a superset),
    // compacted onto dense lanes in chunks of 64
#pragma unroll
    for (int k = 0; k < ITEMS; ++k) emit[k] = late ? (vis_new[k] && s.vis[k] == 0u) : vis_new[k];
    bool lsel[ITEMS];
#pragma unroll
    for (int k = 0; k < ITEMS; ++k) lsel[k] = CACHE ? frus[k] : emit[k];
    uint32_t eslot[ITEMS], lod_abs[ITEMS];
    const uint32_t ne = wave_compact<ITEMS>(lsel, eslot, lane);
#pragma unroll
    for (int k = 0; k < ITEMS; ++k) lod_abs[k] = 0u;
    for (uint32_t c0 = 0; c0 < ne; c0 += 64u) {
#pragma unroll
        for (int k = 0; k < ITEMS; ++k)
            if (lsel[k] && eslot[k] - c0 < 64u) {
                cand[eslot[k] - c0] = make_float4(cx[k], cy[k], cz[k], rad[k]);
                cand2[eslot[k] - c0] = make_uint2(__float_as_uint(s.w[k].w), s.surf[k]);
            }
        wave_lds_sync();
        if (c0 + lane < ne) {
            const float4 c = cand[lane];
            const uint2 e = cand2[lane];
            const float scale = __uint_as_float(e.x);
            const uint2 lo = lds_tab ? sm.surf_lod[e.y] : S.surf_lod[e.y];
            const float len = sqrtf((c.x * c.x + c.y * c.y) + c.z * c.z);
            const float distance = glsl_max(len - c.w, 0.0f);
            const float threshold = (distance * J.view.lodTarget) / scale;
            uint32_t idx = 0;  // the last LOD whose error is below the threshold: four errors read at a time
            for (uint32_t l0 = 1; l0 < lo.y; l0 += 4u) {
                uint32_t l[4];
                float err[4];
#pragma unroll
                for (uint32_t j = 0; j < 4u; ++j) {
                    l[j] = l0 + j < lo.y ? l0 + j : lo.y - 1u;
                    err[j] = lds_tab ? sm.lod_err[lo.x + l[j]] : S.lod_error[lo.x + l[j]];
                }
#pragma unroll
                for (uint32_t j = 0; j < 4u; ++j)
                    if (err[j] < threshold) idx = l[j];
            }
            cand2[lane].x = (pass == PASS_ONPC) ? idx : idx + lo.x;
        }
        wave_lds_sync();
#pragma unroll
        for (int k = 0; k < ITEMS; ++k)
            if (lsel[k] && eslot[k] - c0 < 64u) lod_abs[k] = cand2[eslot[k] - c0].x;
        wave_lds_sync();
    }

    if constexpr (INST) {  // the LOD histogram of the workgroup's tiles (LDS)
#pragma unroll
        for (int k = 0; k < ITEMS; ++k)
            if (emit[k]) atomicAdd(&lds_hist[lod_abs[k]], 1u);
    }

    if constexpr (CL) {  // the tile's cluster total, for the expansion's record offsets
        uint32_t cc = 0;
#pragma unroll
        for (int k = 0; k < ITEMS; ++k)
            if (emit[k]) cc += S.lod_cluster[lod_abs[k]].y;
#pragma unroll
        for (int off = 32; off >= 1; off >>= 1) cc += __shfl_xor(cc, off, 64);
        if (lane == 0) sm.csum[wave] = cc;
    }

    // ---- visibility; ranks in (wave, item, lane) order -> staging
    if (late) {
#pragma unroll
        for (int k = 0; k < ITEMS; ++k)
            if (i0 + 64u * k < J.n) J.vis_out[J.begin + i0 + 64u * k] = vis_new[k] ? 1u : 0u;
    }
    // A wave's ranks come from its own ballots (without a frame cache those of the LOD compaction); the waves' totals
    // go through LDS, and each wave adds up the totals before its own. One barrier per tile: the totals alternate between
    // two sets by the tile's parity, so a wave that is a tile ahead does not overwrite what a slower one still reads.
    uint32_t erank[ITEMS], etot = ne;
    if constexpr (CACHE) etot = wave_compact<ITEMS>(emit, erank, lane);
    if (lane == 0) {
        sm.wtot[parity][wave] = etot;
        if constexpr (CACHE) sm.ctot[parity][wave] = ne;
    }
    __syncthreads();
    uint32_t before = 0, total = 0, cbefore = 0, ctotal = 0;
#pragma unroll
    for (uint32_t w = 0; w < (uint32_t)NW; ++w) {
        const uint32_t x = sm.wtot[parity][w];
        before += w < wave ? x : 0u;
        total += x;
        if constexpr (CACHE) {
            const uint32_t y = sm.ctot[parity][w];
            cbefore += w < wave ? y : 0u;
            ctotal += y;
        }
    }
    if (tid == 0) {
        if constexpr (FUSED) fuse_publish(fuse, launch, gtile, total);
        else counts[gtile] = total;
        if constexpr (CACHE) fc.counts[gtile] = ctotal;
        if constexpr (CL) {
            uint32_t tot = 0;
#pragma unroll
            for (int w = 0; w < NW; ++w) tot += sm.csum[w];
            ccounts[gtile] = tot;
        }
    }
    if constexpr (!FUSED) {
        uint2* stage = staging + (size_t)gtile * TILE + before;
#pragma unroll
        for (int k = 0; k < ITEMS; ++k)
            if (emit[k]) stage[CACHE ? erank[k] : eslot[k]] = make_uint2(J.begin + i0 + 64u * k, lod_abs[k]);
    }
    if constexpr (CACHE) {
        const size_t cb = (size_t)gtile * TILE + cbefore;
#pragma unroll
        for (int k = 0; k < ITEMS; ++k)
            if (frus[k]) {
                fc.sph[cb + eslot[k]] = make_float4(cx[k], cy[k], cz[k], rad[k]);
                fc.meta[cb + eslot[k]] = make_uint2(J.begin + i0 + 64u * k, lod_abs[k]);
            }
    }
    if constexpr (FUSED) {
        // the draw data is gathered while the earlier tiles' words arrive
        uint2 d[ITEMS];
#pragma unroll
        for (int k = 0; k < ITEMS; ++k) d[k] = emit[k] ? S.lod_draw[lod_abs[k]] : make_uint2(0u, 0u);
        const bool last_tile = gtile + 1u == J.n_tiles;
        uint32_t prefix, left = 0;
        const bool mine = fuse_prefix<BLOCK>(fuse, launch, gtile, last_tile, sm.red, prefix, left, [&] {
            uint2* stage = staging + (size_t)gtile * TILE + before;
#pragma unroll
            for (int k = 0; k < ITEMS; ++k)
                if (emit[k]) stage[CACHE ? erank[k] : eslot[k]] = make_uint2(J.begin + i0 + 64u * k, lod_abs[k]);
        });
        if (!mine) return;
        if (tid == 0 && last_tile) *J.count = prefix + total;
#pragma unroll
        for (int k = 0; k < ITEMS; ++k) {
            const uint32_t pos = prefix + before + (CACHE ? erank[k] : eslot[k]);
            if (emit[k] && pos < J.capacity) write_command(J.cmds, pos, J.begin + i0 + 64u * k, d[k]);
        }
        if (last_tile) settle_staged(J, TILE, staging, fuse, launch, left);
    }
}

// One tile, loads and decision (non-persistent form, used by the batched kernel and the cluster object pass).
template <int BLOCK, int ITEMS, int MODE, bool HIZ, bool LDS_TAB, bool CL = false>
__device__ __forceinline__ void decide_tile(const CullJob& J, uint32_t tile_in_job, uint32_t gtile, uint32_t* counts,
                                            uint2* staging, TileSmem<BLOCK, ITEMS, LDS_TAB>& sm,
                                            uint32_t* ccounts = nullptr)
{
    constexpr bool NT = MODE == MODE_OTHER && !HIZ;  // PLAIN / ONPC: streamed once, no Hi-Z
    Streams<ITEMS> s;
    issue_vis<BLOCK, ITEMS, MODE, NT>(J, tile_in_job, s);
    if (MODE != MODE_EARLY) issue_objects<BLOCK, ITEMS, MODE, false, NT>(J, tile_in_job, s);
    stage_tables<BLOCK, ITEMS>(J, sm);
    if (MODE == MODE_EARLY) issue_objects<BLOCK, ITEMS, MODE, false, NT>(J, tile_in_job, s);
    __syncthreads();  // staged tables visible
    process_tile<BLOCK, ITEMS, MODE, HIZ, LDS_TAB, CL>(J, tile_in_job, gtile, 0u, s, counts, staging, ccounts, sm,
                                                        NoPrefetch{});
}

// Persistent decide for one view: workgroup b takes tiles b, b + G, b + 2G, ... (no workgroup waits on another, so
// any residency is safe). Tables are staged once; the next tile's streams are issued while the current one is
// decided (two register sets, alternating, so no register copy waits on a load in flight).
// INST: workgroup b takes the contiguous tiles of chunk b instead (chunk_range), counts
// its emitting objects per LOD in LDS and writes the counts to row b of ih.hist.
template <int BLOCK, int ITEMS, int MODE, bool HIZ, bool LDS_TAB, bool CACHE = false, bool INST = false>
__global__ __launch_bounds__(BLOCK) void decide_kernel(CullJob J, uint32_t* counts, uint2* staging, FrameCacheDev fc,
                                                       InstHistDev ih)
{
    __shared__ TileSmem<BLOCK, ITEMS, LDS_TAB> sm;
    __shared__ uint32_t s_hist[INST ? kInstLdsBins : 1];
    constexpr bool NT = (MODE == MODE_EARLY && CACHE) || (MODE == MODE_OTHER && !HIZ);
    uint32_t t, t_end, step;
    if constexpr (INST) {
        chunk_range(blockIdx.x, ih.tiles_per_chunk, ih.n_long, J.n_tiles, t, t_end);
        step = 1;
        for (uint32_t i = threadIdx.x; i < ih.n_lods; i += BLOCK) s_hist[i] = 0u;  // (ordered by the barrier below)
    } else {
        t = blockIdx.x;
        t_end = J.n_tiles;
        step = gridDim.x;
    }
    Streams<ITEMS> A, B;
    issue_tile<BLOCK, ITEMS, MODE, CACHE, NT>(J, t, A);
    stage_tables<BLOCK, ITEMS>(J, sm);
    __syncthreads();
    while (true) {
        {
            const uint32_t tn = t + step;
            // past the last tile, tile n_tiles is issued: every lane is out of range and clamped to the job's last
            // object, so each stream costs one cache line (discarded). A branch around the loads instead was 2.7 us
            // slower per pass, re-issuing the current tile 2.2 us slower (with non-temporal loads its lines are
            // fetched again).
            process_tile<BLOCK, ITEMS, MODE, HIZ, LDS_TAB, false, CACHE, INST>(J, t, t, 0u, A, counts, staging, nullptr,
                                                                                sm, [&]() {
                issue_tile<BLOCK, ITEMS, MODE, CACHE, NT>(J, tn < t_end ? tn : J.n_tiles, B);
            }, fc, s_hist);
            t = tn;
            if (t >= t_end) break;
        }
        {
            const uint32_t tn = t + step;
            process_tile<BLOCK, ITEMS, MODE, HIZ, LDS_TAB, false, CACHE, INST>(J, t, t, 1u, B, counts, staging, nullptr,
                                                                                sm, [&]() {
                issue_tile<BLOCK, ITEMS, MODE, CACHE, NT>(J, tn < t_end ? tn : J.n_tiles, A);
            }, fc, s_hist);
            t = tn;
            if (t >= t_end) break;
        }
    }
    if constexpr (INST) {
        __syncthreads();
        uint32_t* row = ih.hist + (size_t)blockIdx.x * ih.n_lods;
        for (uint32_t i = threadIdx.x; i < ih.n_lods; i += BLOCK) row[i] = s_hist[i];
    }
}

// A pass over few objects in one launch: one tile per workgroup, which also writes the tile's commands. A workgroup's first
// command follows from the counts that the workgroups before it publish. Every object's streams are loaded at once, in
// EARLY too (the visibility's round trip costs more than the other objects' bytes here); the tables are read from global
// memory, as for the batches.
template <int BLOCK, int ITEMS, int MODE, bool HIZ, bool CACHE>
__global__ __launch_bounds__(BLOCK) void fused_kernel(CullJob J, FrameCacheDev fc, uint2* left, FuseDev fuse)
{
    __shared__ TileSmem<BLOCK, ITEMS, false> sm;
    const uint32_t last = fuse_last(fuse);  // (no branch: its wait comes behind the streams' loads)
    Streams<ITEMS> s;
    issue_tile<BLOCK, ITEMS, MODE, true, false>(J, blockIdx.x, s);
    stage_tables<BLOCK, ITEMS>(J, sm);
    if (threadIdx.x == 0) sm.last = last;
    __syncthreads();
    const uint32_t launch = fuse_launch(sm.last);
    process_tile<BLOCK, ITEMS, MODE, HIZ, false, false, CACHE, false, true>(
        J, blockIdx.x, blockIdx.x, 0u, s, nullptr, left, nullptr, sm, NoPrefetch{}, fc, nullptr, fuse, launch);
}

// Last entry of the ascending table `starts` that is <= t.
__device__ __forceinline__ uint32_t find_job(const uint32_t* starts, uint32_t n_jobs, uint32_t t)
{
    uint32_t lo = 0, hi = n_jobs - 1;
    while (lo < hi) {
        const uint32_t mid = (lo + hi + 1) >> 1;
        if (starts[mid] <= t) lo = mid;
        else hi = mid - 1;
    }
    return lo;
}

constexpr uint32_t kLdsJobs = 1024;  // batched: job start table staged in LDS up to this many jobs

// One tile of a batch: t of all, the job's own tile t - tile_start. Which job a tile belongs to goes to tile_job for the
// emit.
template <int BLOCK, int ITEMS>
__device__ __forceinline__ void decide_batch_tile(const CullJob& J, uint32_t jb, uint32_t t, uint32_t* counts,
                                                  uint2* staging, uint32_t* tile_job,
                                                  TileSmem<BLOCK, ITEMS, false>& sm)
{
    const uint32_t tt = t - J.tile_start;
    if (threadIdx.x == 0) tile_job[t] = jb;
    if (J.pass == PASS_LATE) decide_tile<BLOCK, ITEMS, MODE_LATE, true, false>(J, tt, t, counts, staging, sm);
    else if (J.hiz) decide_tile<BLOCK, ITEMS, MODE_OTHER, true, false>(J, tt, t, counts, staging, sm);
    else decide_tile<BLOCK, ITEMS, MODE_OTHER, false, false>(J, tt, t, counts, staging, sm);
}

// Batched decide: one launch over the (job, tile) work list of many views; workgroup b takes global tile b. The job
// lookup searches the jobs' first tiles: up to kArgJobs jobs they come in the kernel argument `sa` (scalar loads
// from the kernarg segment, no barrier; the 256-view batch decides in 402.8 us against 414.3 us with the LDS copy),
// up to kLdsJobs they are staged in LDS (one coalesced read), beyond that the compact global table is searched. The
// job itself is read in place with scalar loads (its index is wave-uniform), with no LDS copy and barrier: the
// 256-view graph 0.732 ms against 0.742 ms with the copy. The surface and LOD tables are read from global memory
// (they stay in the L2), not staged in LDS: each workgroup decides a single tile, and staging the whole tables for it
// cost more (the 256-view graph 0.78 ms against 0.76 ms).
template <int BLOCK, int ITEMS>
__global__ __launch_bounds__(BLOCK) void decide_batch_kernel(const CullJob* __restrict__ jobs,
                                                             const uint32_t* __restrict__ starts, uint32_t n_jobs,
                                                             uint32_t* counts, uint2* staging, uint32_t* tile_job,
                                                             JobStartsArg sa)
{
    __shared__ TileSmem<BLOCK, ITEMS, false> sm;
    __shared__ uint32_t s_start[kLdsJobs];
    const uint32_t t = blockIdx.x;
    uint32_t jb;
    if (n_jobs <= kArgJobs) {
        jb = find_job(sa.v, n_jobs, t);
    } else if (n_jobs <= kLdsJobs) {
        for (uint32_t k = threadIdx.x; k < n_jobs; k += BLOCK) s_start[k] = starts[k];
        __syncthreads();
        jb = find_job(s_start, n_jobs, t);
    } else {
        jb = find_job(starts, n_jobs, t);
    }
    jb = __builtin_amdgcn_readfirstlane(jb);
    decide_batch_tile<BLOCK, ITEMS>(jobs[jb], jb, t, counts, staging, tile_job, sm);
}

// The same for a few jobs, which come whole in the kernel arguments (unused entries start past every tile).
__device__ __forceinline__ uint32_t few_job(const JobArgs& a, uint32_t t)
{
    uint32_t jb = 0;
#pragma unroll
    for (uint32_t k = 1; k < kArgFullJobs; ++k) jb += a.j[k].tile_start <= t ? 1u : 0u;
    return __builtin_amdgcn_readfirstlane(jb);
}

template <int BLOCK, int ITEMS>
__global__ __launch_bounds__(BLOCK) void decide_few_kernel(JobArgs jobs, uint32_t* counts, uint2* staging,
                                                           uint32_t* tile_job)
{
    __shared__ TileSmem<BLOCK, ITEMS, false> sm;
    const uint32_t jb = few_job(jobs, blockIdx.x);
    decide_batch_tile<BLOCK, ITEMS>(jobs.j[jb], jb, blockIdx.x, counts, staging, tile_job, sm);
}

// Cluster object pass (PreClusterDrawCull.comp.glsl:13-47): the PLAIN (or, with a pyramid, TEMPORAL) decision of
// every object, its LOD, and per tile the number of emitting objects (counts), their (objectId, LOD) list (staging)
// and the sum of their LOD cluster counts (ccounts). One workgroup per tile. The register cap keeps two
// items per thread at four 512-thread workgroups a CU (68 registers without it: 1 M objects took a second round, 11.8
// against 10.1 us).
template <int BLOCK, int ITEMS, bool HIZ, bool LDS_TAB>
__global__ __launch_bounds__(BLOCK) __attribute__((amdgpu_waves_per_eu(ITEMS == 2 ? 8 : 4)))
void decide_cluster_kernel(CullJob J, uint32_t* counts, uint2* staging, uint32_t* ccounts)
{
    __shared__ TileSmem<BLOCK, ITEMS, LDS_TAB> sm;
    decide_tile<BLOCK, ITEMS, MODE_OTHER, HIZ, LDS_TAB, true>(J, blockIdx.x, blockIdx.x, counts, staging, sm, ccounts);
}

template <int BLOCK, int ITEMS>
hipError_t launch_cluster_objects_t(const CullJob& job, const CompactScratch& s, uint32_t* ccounts, hipStream_t st)
{
    const bool lds = job.scene.n_surfaces <= kLdsSurfaces && job.scene.n_lods <= kLdsLods;
    const dim3 g(job.n_tiles), b(BLOCK);
#define BZ_CL_LAUNCH(HZ, LT) \
    hipLaunchKernelGGL((decide_cluster_kernel<BLOCK, ITEMS, HZ, LT>), g, b, 0, st, job, s.counts, s.staging, ccounts)
    if (job.hiz) {
        if (lds) BZ_CL_LAUNCH(true, true);
        else BZ_CL_LAUNCH(true, false);
    } else {
        if (lds) BZ_CL_LAUNCH(false, true);
        else BZ_CL_LAUNCH(false, false);
    }
#undef BZ_CL_LAUNCH
    return hipGetLastError();
}

// ------------------------------------------------------------------------------------------------ emit
constexpr uint32_t kEmitBlock = 256;
constexpr uint32_t kEmitTiles = kEmitBlock / 64;  // one tile per wave
constexpr uint32_t kEmitWideBlock = 1024;         // jobs of more than kScanTiles tiles: 16 tiles per workgroup
constexpr uint32_t kEmitSumTiles = 32768;         // up to these the workgroup adds up the earlier tiles' counts
constexpr uint32_t kEmitUnroll = 2;               // entries per lane in flight (a tile emits ~70 on average)

template <uint32_t BLOCK, bool WIDE>
struct EmitSmem {
    uint32_t red[BLOCK / 64];
    uint32_t cnt[BLOCK / 64 + 1];                            // exclusive prefix of the workgroup's tile counts
    alignas(16) uint2 buf[WIDE ? BLOCK / 64 : 1][64u * 3u];  // the waves' commands
};

// A workgroup barrier for LDS only: waits for this wave's LDS operations (lgkmcnt(0)) but not for its global loads in
// flight (vmcnt and expcnt left at their maxima), then s_barrier.
__device__ __forceinline__ void block_lds_sync()
{
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    __builtin_amdgcn_s_waitcnt(0xC07F);
    __builtin_amdgcn_s_barrier();
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
}

// The commands of up to 64 staged entries (lane l holds entry l; the first cnt count), at cmds[pos0 ...), put together in
// the wave's LDS and stored as 16-byte words (a command is 24 bytes: the words are 8-byte aligned, the last may be half a
// one). For the large jobs, whose emit is bound by its stores: three 8-byte words per lane, 24 bytes apart, touch every
// line of the output three times (16 777 216 objects, 1.6 M commands: 82.9 -> 81.7 us). A small job waits longer for the
// LDS than it saves (4 194 304-object frame 57.7 -> 57.9 us) and keeps the plain stores.
__device__ __forceinline__ void write_wave_commands(uint2* buf, uint32_t* cmds, uint32_t pos0, uint32_t cnt,
                                                    uint32_t object, uint2 draw)
{
    typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
    typedef uint32_t u32x4_at8 __attribute__((ext_vector_type(4), aligned(8)));
    const uint32_t lane = threadIdx.x & 63u;
    write_command(reinterpret_cast<uint32_t*>(buf), lane, object, draw);
    wave_lds_sync();
    uint32_t* out = cmds + (size_t)pos0 * 6u;
    const uint32_t words = cnt * 6u;
#pragma unroll
    for (uint32_t k = 0; k < 2u; ++k) {
        const uint32_t i = (k * 64u + lane) * 4u;
        if (i >= words) break;
        const u32x4 v = *reinterpret_cast<const u32x4*>(reinterpret_cast<const uint32_t*>(buf) + i);
        if (i + 4u <= words) *reinterpret_cast<u32x4_at8*>(out + i) = v;
        else *reinterpret_cast<uint2*>(out + i) = make_uint2(v.x, v.y);
    }
    wave_lds_sync();
}

// Writes the commands of tiles [t0, t1) of one job (t1 - t0 <= BLOCK / 64; tile_size >= 64 * kEmitUnroll). One round
// of loads gets the counts of the job's earlier tiles (reduced to the output base; 16 per thread and round), or
// with `scanned` (the exclusive prefix of all counts) two entries of it, the workgroup's own counts and,
// before any count is known, the first 64 * kEmitUnroll staging entries of each wave's tile (in bounds: every tile
// owns tile_size slots); each wave gathers its entries' LOD draw data while the block scan of the counts runs, then
// writes tile t0 + w's commands in order. Longer tiles continue in rounds of kEmitUnroll entries per lane.
template <uint32_t BLOCK, bool WIDE>
__device__ __forceinline__ void emit_tiles(const CullJob& J, uint32_t t0, uint32_t t1, uint32_t tile_size,
                                           const uint32_t* counts, const uint2* staging, const uint32_t* scanned,
                                           EmitSmem<BLOCK, WIDE>& sm)
{
    constexpr uint32_t NW = BLOCK / 64u;
    const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6;
    const uint32_t nt = t1 - t0;
    const uint32_t tw = t0 + (wave < nt ? wave : 0u);  // this wave's tile (clamped for waves without one)
    const uint2* stage = staging + (size_t)tw * tile_size;
    const uint2* lod_draw = J.scene.lod_draw;
    uint2 ent[kEmitUnroll], d[kEmitUnroll];
#pragma unroll
    for (uint32_t u = 0; u < kEmitUnroll; ++u) ent[u] = stage[u * 64u + lane];  // speculative: checked against c below
    const uint32_t c = wave < nt ? counts[tw] : 0u;
    // the job's earlier tiles: every load of a thread issued before the first add (16 per pass)
    uint32_t part = 0;
    const uint32_t own = tid < nt ? counts[t0 + tid] : 0u;
    if (scanned) {  // one lane takes the difference of the scanned prefixes; the reduction below adds it
        if (tid == 0) part = scanned[t0] - scanned[J.tile_start];
    } else for (uint32_t u0 = J.tile_start; u0 < t0; u0 += 16u * BLOCK) {
        uint32_t v[16];
#pragma unroll
        for (int j = 0; j < 16; ++j) {
            const uint32_t u = u0 + (uint32_t)j * BLOCK + tid;
            v[j] = u < t0 ? counts[u] : 0u;
        }
#pragma unroll
        for (int j = 0; j < 16; ++j) part += v[j];
    }
#pragma unroll
    for (uint32_t u = 0; u < kEmitUnroll; ++u)
        d[u] = u * 64u + lane < c ? lod_draw[ent[u].y] : make_uint2(0u, 0u);  // in flight through the scan
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) part += __shfl_xor(part, off, 64);
    if (lane == 0) sm.red[wave] = part;
    if (wave == 0) {
        uint32_t v = own;
#pragma unroll
        for (int off = 1; off < (int)NW; off <<= 1) {
            const uint32_t t = __shfl_up(v, off, 64);
            if (lane >= (uint32_t)off) v += t;
        }
        if (lane < NW) sm.cnt[lane + 1] = v;
        if (lane == 0) sm.cnt[0] = 0;
    }
    block_lds_sync();
    uint32_t prefix = 0;
#pragma unroll
    for (uint32_t w = 0; w < NW; ++w) prefix += sm.red[w];
    if (tid == 0 && t1 == J.tile_start + J.n_tiles) *J.count = prefix + sm.cnt[nt];
    if (wave >= nt) return;
    const uint32_t base = prefix + sm.cnt[wave];
    for (uint32_t e0 = 0; e0 < c; e0 += 64u * kEmitUnroll) {
        if (e0) {
#pragma unroll
            for (uint32_t u = 0; u < kEmitUnroll; ++u) {
                const uint32_t e = e0 + u * 64u + lane;
                ent[u] = stage[e < c ? e : 0u];  // objectId, absolute LOD (entry 0 exists whenever c > 0)
            }
#pragma unroll
            for (uint32_t u = 0; u < kEmitUnroll; ++u) d[u] = lod_draw[ent[u].y];
        }
#pragma unroll
        for (uint32_t u = 0; u < kEmitUnroll; ++u) {
            if constexpr (WIDE) {
                const uint32_t e = e0 + u * 64u, pos = base + e;
                if (e < c && pos < J.capacity) {  // uniform
                    const uint32_t room = J.capacity - pos, left = c - e < 64u ? c - e : 64u;
                    write_wave_commands(sm.buf[wave], J.cmds, pos, left < room ? left : room, ent[u].x, d[u]);
                }
            } else {
                const uint32_t e = e0 + u * 64u + lane;
                const uint32_t pos = base + e;
                if (e < c && pos < J.capacity) write_command(J.cmds, pos, ent[u].x, d[u]);
            }
        }
    }
}

template <uint32_t BLOCK, bool WIDE>
__global__ __launch_bounds__(BLOCK) void emit_kernel(CullJob J, uint32_t tile_size, const uint32_t* counts,
                                                     const uint2* staging, const uint32_t* prefix)
{
    __shared__ EmitSmem<BLOCK, WIDE> sm;
    const uint32_t t0 = blockIdx.x * (BLOCK / 64u);
    const uint32_t t1 = t0 + BLOCK / 64u < J.n_tiles ? t0 + BLOCK / 64u : J.n_tiles;
    emit_tiles<BLOCK, WIDE>(J, t0, t1, tile_size, counts, staging, prefix, sm);
}

// Batched emit of one tile by one wave: its count, its first 64 * kEmitUnroll entries and its job's number are loaded
// together; then the counts of the job's earlier tiles (or two words of the scanned prefix) together with the entries'
// draw data; then it writes its commands. The waves of a workgroup share nothing: tiles of different jobs meet in one
// workgroup, and splitting it at the job boundaries, with a search for each job and two barriers, cost a round trip per
// boundary (64 views: 10.0 us, now 7.4).
__device__ __forceinline__ void emit_batch_tile(const CullJob& J, uint32_t t, uint32_t c, uint2 (&ent)[kEmitUnroll],
                                                const uint2* stage, const uint32_t* counts, const uint32_t* scanned)
{
    const uint32_t lane = threadIdx.x & 63u;
    const uint2* lod_draw = J.scene.lod_draw;
    uint2 d[kEmitUnroll];
#pragma unroll
    for (uint32_t u = 0; u < kEmitUnroll; ++u)
        d[u] = u * 64u + lane < c ? lod_draw[ent[u].y] : make_uint2(0u, 0u);
    uint32_t base;
    if (scanned) {
        base = scanned[t] - scanned[J.tile_start];
    } else {
        uint32_t part = 0;
        for (uint32_t u0 = J.tile_start; u0 < t; u0 += 16u * 64u) {
            uint32_t v[16];
#pragma unroll
            for (uint32_t k = 0; k < 16u; ++k) {
                const uint32_t u = u0 + k * 64u + lane;
                v[k] = u < t ? counts[u] : 0u;
            }
#pragma unroll
            for (uint32_t k = 0; k < 16u; ++k) part += v[k];
        }
#pragma unroll
        for (int off = 32; off >= 1; off >>= 1) part += __shfl_xor(part, off, 64);
        base = part;
    }
    if (lane == 0 && t + 1u == J.tile_start + J.n_tiles) *J.count = base + c;
    for (uint32_t e0 = 0; e0 < c; e0 += 64u * kEmitUnroll) {
        if (e0) {
#pragma unroll
            for (uint32_t u = 0; u < kEmitUnroll; ++u) {
                const uint32_t e = e0 + u * 64u + lane;
                ent[u] = stage[e < c ? e : 0u];
            }
#pragma unroll
            for (uint32_t u = 0; u < kEmitUnroll; ++u) d[u] = lod_draw[ent[u].y];
        }
#pragma unroll
        for (uint32_t u = 0; u < kEmitUnroll; ++u) {
            const uint32_t e = e0 + u * 64u + lane;
            if (e < c && base + e < J.capacity) write_command(J.cmds, base + e, ent[u].x, d[u]);
        }
    }
}

__global__ __launch_bounds__(kEmitBlock) void emit_batch_kernel(const CullJob* __restrict__ jobs, uint32_t total_tiles,
                                                                uint32_t tile_size, const uint32_t* counts,
                                                                const uint2* staging, const uint32_t* tile_job,
                                                                const uint32_t* prefix)
{
    const uint32_t t = blockIdx.x * kEmitTiles + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if (t >= total_tiles) return;
    const uint2* stage = staging + (size_t)t * tile_size;
    uint2 ent[kEmitUnroll];
#pragma unroll
    for (uint32_t u = 0; u < kEmitUnroll; ++u) ent[u] = stage[u * 64u + (threadIdx.x & 63u)];  // checked against c
    emit_batch_tile(jobs[__builtin_amdgcn_readfirstlane(tile_job[t])], t, counts[t], ent, stage, counts, prefix);
}

__global__ __launch_bounds__(kEmitBlock) void emit_few_kernel(JobArgs jobs, uint32_t total_tiles, uint32_t tile_size,
                                                              const uint32_t* counts, const uint2* staging,
                                                              const uint32_t* prefix)
{
    const uint32_t t = blockIdx.x * kEmitTiles + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if (t >= total_tiles) return;
    const uint2* stage = staging + (size_t)t * tile_size;
    uint2 ent[kEmitUnroll];
#pragma unroll
    for (uint32_t u = 0; u < kEmitUnroll; ++u) ent[u] = stage[u * 64u + (threadIdx.x & 63u)];
    emit_batch_tile(jobs.j[few_job(jobs, t)], t, counts[t], ent, stage, counts, prefix);
}

// The emit launch of one job whose decide launch wrote s.counts / s.staging. Up to kScanTiles tiles, 4 per workgroup. Above,
// 16 per workgroup of 1024 threads: each workgroup still adds up all the counts before its own, one round of loads per
// 16 384 tiles, but there are a quarter as many workgroups to do so, and that costs less than a scan launch between the
// two kernels, which one workgroup runs while the others wait (with the scan / without: 4199 tiles 29.3 / 26.5 us, 11 719
// tiles 62.8 / 57.8, 16 384 tiles 82.9 / 78.1, 23 438 tiles 114.1 / 108.5; 512 threads at 16 384 tiles 78.3). The sums
// grow with the square of the tiles: from three rounds on (46 875 tiles: 137.1 / 139.2 us) the scan is the better one.
hipError_t launch_emit(const CullJob& job, uint32_t tile_size, const CompactScratch& s, hipStream_t st)
{
    const uint32_t* prefix = nullptr;
    if (job.n_tiles > kEmitSumTiles) {
        const hipError_t e = launch_scan_counts(s.counts, job.n_tiles, s.prefix, st);
        if (e != hipSuccess) return e;
        prefix = s.prefix;
    }
#define BZ_EMIT(B, W) \
    hipLaunchKernelGGL((emit_kernel<B, W>), dim3((job.n_tiles + B / 64u - 1u) / (B / 64u)), dim3(B), 0, st, job, \
                       tile_size, (const uint32_t*)s.counts, (const uint2*)s.staging, prefix)
    if (job.n_tiles <= kScanTiles) BZ_EMIT(kEmitBlock, false);
    else if (!prefix) BZ_EMIT(kEmitWideBlock, true);
    else BZ_EMIT(kEmitBlock, true);
#undef BZ_EMIT
    return hipGetLastError();
}

// LATE pass from a frame cache: the EARLY pass of the same view, transforms and range recorded each tile's frustum
// survivors (view-space sphere, objectId, LOD index) in ascending objectId order. A workgroup reads its survivors
// only: objects outside the frustum are invisible (visibility 0, no command), survivors take the Hi-Z test, and the
// visible ones read their current visibility (as LateDrawCull.comp.glsl:51 does, so any write to it since the EARLY
// pass is seen) and, when newly visible, are emitted with their recorded LOD -- the same arithmetic on the same values
// as the full LATE pass, so the commands, count and visibility are identical.
//
// One 256-thread workgroup per recorded tile: its survivors in rounds of 256, the first loaded together with the tile's
// count, each with the Hi-Z test; then the current visibility of the survivors that pass it (gathered after the test: a
// survivor occluded now is not emitted whatever it was, and a tenth of them pass); then the visibility of the whole tile
// (coalesced 16-byte stores; 0 outside the frustum) and the newly visible survivors' commands in survivor order. No
// transform, surface or LOD table is read. Workgroups of 512 threads per 4096 objects, which this replaced, were all
// resident at once, so that their loads, tests and stores ran in step across the GPU, and a region that is all in view
// (neighbouring ids, neighbouring objects) was one workgroup's, in four rounds of 1024 (4 194 304 objects at random: frame
// 58.0 -> 56.9 us; 1 048 576 in region order: 50.2 -> 43.3; 131 072 in region order, one launch: 35.7 -> 24.4).
constexpr uint32_t kLtBlock = 256;
template <int TILE, bool FUSED>
__global__ __launch_bounds__(kLtBlock) void late_tile_kernel(CullJob J, FrameCacheDev fc, uint32_t* counts,
                                                             uint2* staging, FuseDev fuse)
{
    constexpr uint32_t NW = kLtBlock / 64, ROUNDS = TILE / kLtBlock;
    __shared__ uint32_t s_new[TILE / 32], s_lvl[kMaxMips], s_tot[ROUNDS][NW], s_red[2 * NW], s_last;
    const uint32_t t = blockIdx.x, tid = threadIdx.x, lane = tid & 63u, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t base = t * TILE, nt = J.n - base < TILE ? J.n - base : TILE, obj0 = J.begin + base;
    const uint32_t last = FUSED ? fuse_last(fuse) : 0u;
    const size_t slot0 = (size_t)t * TILE + tid;
    float4 sp = fc.sph[slot0];
    uint2 mt = fc.meta[slot0];
    const uint32_t n = __builtin_amdgcn_readfirstlane(fc.counts[t]);
    if (tid < (uint32_t)kMaxMips) {
        uint32_t off = 0;
        for (uint32_t L = 0; L < tid; ++L) off += level_dim(J.pyr.base_w, L) * level_dim(J.pyr.base_h, L);
        s_lvl[tid] = off;
    }
    if (tid < TILE / 32) s_new[tid] = 0u;
    if (FUSED && tid == 0) s_last = last;
    __syncthreads();
    const uint32_t launch = FUSED ? fuse_launch(s_last) : 0u;
    uint32_t before = 0;      // the tile's commands of the rounds so far
    bool emit[ROUNDS];        // FUSED: a round's commands wait for the tile's first slot
    uint32_t rank[ROUNDS], obj[ROUNDS], lod[ROUNDS];
#pragma unroll
    for (uint32_t r = 0; r < ROUNDS; ++r) {
        emit[r] = false;
        rank[r] = obj[r] = lod[r] = 0u;
        if (r * kLtBlock < n) {  // uniform
            const uint32_t e = r * kLtBlock + tid;
            if (r) {
                sp = fc.sph[slot0 + r * kLtBlock];
                mt = fc.meta[slot0 + r * kLtBlock];
            }
            const uint32_t local = mt.x - obj0;
            if (e < n && local < nt) {  // (an entry outside the tile can only come from a mismatched cache)
                float a0 = 0.f, a1 = 0.f, a2 = 0.f, a3 = 0.f;
                const bool test =
                    project_sphere(sp.x, sp.y, sp.z, sp.w, J.view.znear, J.view.p00, J.view.p11, a0, a1, a2, a3);
                // a sphere crossing the near plane is not tested and stays visible
                const bool vis = test ? occlusion_visible(J.view, J.pyr, s_lvl, a0, a1, a2, a3, sp.z, sp.w) : true;
                if (vis) atomicOr(&s_new[local >> 5], 1u << (local & 31u));
                emit[r] = vis && J.vis_in[mt.x] == 0u;  // the current visibility (LateDrawCull:51), where it decides
            }
            const unsigned long long m = __ballot(emit[r]);
            rank[r] = (uint32_t)__popcll(m & ((1ull << lane) - 1ull));
            obj[r] = mt.x;
            lod[r] = mt.y;
            if (lane == 0) s_tot[r][wave] = (uint32_t)__popcll(m);
            __syncthreads();
            uint32_t total = 0;
#pragma unroll
            for (uint32_t w = 0; w < NW; ++w) {
                const uint32_t x = s_tot[r][w];
                rank[r] += w < wave ? x : 0u;
                total += x;
            }
            rank[r] += before;
            before += total;
            if constexpr (!FUSED)
                if (emit[r]) staging[(size_t)t * TILE + rank[r]] = make_uint2(obj[r], lod[r]);
        }
    }
    if (n == 0) __syncthreads();  // (s_new cleared; with survivors a round's barrier has followed its last bit)
    if (tid == 0) {
        if constexpr (FUSED) fuse_publish(fuse, launch, t, before);
        else counts[t] = before;
    }
    // the visibility is next read by the following frame's EARLY pass: stored non-temporal
    typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
    if (nt == TILE && ((uintptr_t)(J.vis_out + obj0) & 15u) == 0) {
        for (uint32_t i = tid; i < TILE / 4u; i += kLtBlock) {
            const uint32_t b = s_new[i >> 3] >> ((i & 7u) * 4u);
            const u32x4 v = { b & 1u, (b >> 1) & 1u, (b >> 2) & 1u, (b >> 3) & 1u };
            __builtin_nontemporal_store(v, reinterpret_cast<u32x4*>(J.vis_out + obj0) + i);
        }
    } else {
        for (uint32_t i = tid; i < nt; i += kLtBlock)
            __builtin_nontemporal_store((s_new[i >> 5] >> (i & 31u)) & 1u, J.vis_out + obj0 + i);
    }
    if constexpr (FUSED) {
        uint2 d[ROUNDS];
#pragma unroll
        for (uint32_t r = 0; r < ROUNDS; ++r) d[r] = emit[r] ? J.scene.lod_draw[lod[r]] : make_uint2(0u, 0u);
        const bool last_tile = t + 1u == J.n_tiles;
        uint32_t prefix, left = 0;
        const bool mine = fuse_prefix<kLtBlock>(fuse, launch, t, last_tile, s_red, prefix, left, [&] {
#pragma unroll
            for (uint32_t r = 0; r < ROUNDS; ++r)
                if (emit[r]) staging[(size_t)t * TILE + rank[r]] = make_uint2(obj[r], lod[r]);
        });
        if (!mine) return;
        if (tid == 0 && last_tile) *J.count = prefix + before;
#pragma unroll
        for (uint32_t r = 0; r < ROUNDS; ++r) {
            const uint32_t pos = prefix + rank[r];
            if (emit[r] && pos < J.capacity) write_command(J.cmds, pos, obj[r], d[r]);
        }
        if (last_tile) settle_staged(J, TILE, staging, fuse, launch, left);
    }
}

// Persistent grid: `per_cu` workgroups per CU, or (per_cu == 0) as many as are resident at once per CU.
template <int BLOCK, int ITEMS, int MODE, bool HIZ, bool LDS_TAB, bool CACHE = false, bool INST = false>
void launch_decide(const CullJob& job, uint32_t n_cu, uint32_t per_cu, uint32_t* counts, uint2* staging, hipStream_t st,
                   const FrameCacheDev& fc = FrameCacheDev{}, const InstHistDev& ih = InstHistDev{})
{
    static int resident = 0;
    if (resident == 0) {
        int r = 0;
        if (hipOccupancyMaxActiveBlocksPerMultiprocessor(
                &r, decide_kernel<BLOCK, ITEMS, MODE, HIZ, LDS_TAB, CACHE, INST>, BLOCK, 0) != hipSuccess ||
            r < 1)
            r = 1;
        resident = r;
    }
    uint64_t grid = (uint64_t)n_cu * (per_cu ? per_cu : (uint32_t)resident);
    if (grid > job.n_tiles) grid = job.n_tiles;
    if (grid == 0) grid = 1;
    if (INST) grid = job.n_tiles ? (job.n_tiles - ih.n_long) / ih.tiles_per_chunk : 1;  // one chunk per workgroup
    hipLaunchKernelGGL((decide_kernel<BLOCK, ITEMS, MODE, HIZ, LDS_TAB, CACHE, INST>), dim3((uint32_t)grid),
                       dim3(BLOCK), 0, st, job, counts, staging, fc, ih);
}

// Workgroups per CU of the instanced decide (as launch_decide counts them for the persistent grid).
template <int BLOCK, int ITEMS>
uint32_t inst_resident()
{
    static int resident = 0;
    if (resident == 0) {
        int r = 0;
        if (hipOccupancyMaxActiveBlocksPerMultiprocessor(
                &r, decide_kernel<BLOCK, ITEMS, MODE_OTHER, false, true, false, true>, BLOCK, 0) != hipSuccess ||
            r < 1)
            r = 1;
        resident = r;
    }
    return (uint32_t)resident;
}

// The decide of the LOD-instanced output: PLAIN decisions plus the chunks' LOD histograms.
template <int BLOCK, int ITEMS>
hipError_t launch_decide_inst_t(const CullJob& job, const CompactScratch& s, uint32_t n_cu, uint32_t per_cu,
                                const InstHistDev& ih, hipStream_t st)
{
    const bool lds = job.scene.n_surfaces <= kLdsSurfaces && job.scene.n_lods <= kLdsLods;
    const FrameCacheDev none{};
    if (lds) launch_decide<BLOCK, ITEMS, MODE_OTHER, false, true, false, true>(job, n_cu, per_cu, s.counts, s.staging,
                                                                               st, none, ih);
    else launch_decide<BLOCK, ITEMS, MODE_OTHER, false, false, false, true>(job, n_cu, per_cu, s.counts, s.staging, st,
                                                                            none, ih);
    return hipGetLastError();
}

template <int BLOCK, int ITEMS, int MODE, bool HIZ, bool CACHE = false>
void launch_mode(const CullJob& job, uint32_t n_cu, uint32_t per_cu, uint32_t* counts, uint2* staging, hipStream_t st,
                 const FrameCacheDev& fc = FrameCacheDev{})
{
    const bool lds = job.scene.n_surfaces <= kLdsSurfaces && job.scene.n_lods <= kLdsLods;
    if (lds) launch_decide<BLOCK, ITEMS, MODE, HIZ, true, CACHE>(job, n_cu, per_cu, counts, staging, st, fc);
    else launch_decide<BLOCK, ITEMS, MODE, HIZ, false, CACHE>(job, n_cu, per_cu, counts, staging, st, fc);
}

template <int BLOCK, int ITEMS>
hipError_t launch_cull_t(const CullJob& job, const CompactScratch& s, uint32_t n_cu, uint32_t per_cu, hipStream_t st,
                         const FrameCacheDev* fc, bool with_emit = true)
{
    const bool h = job.hiz != 0;
    if (job.pass == PASS_EARLY && fc) {
        if (h) launch_mode<BLOCK, ITEMS, MODE_EARLY, true, true>(job, n_cu, per_cu, s.counts, s.staging, st, *fc);
        else launch_mode<BLOCK, ITEMS, MODE_EARLY, false, true>(job, n_cu, per_cu, s.counts, s.staging, st, *fc);
    } else if (job.pass == PASS_EARLY) {
        if (h) launch_mode<BLOCK, ITEMS, MODE_EARLY, true>(job, n_cu, per_cu, s.counts, s.staging, st);
        else launch_mode<BLOCK, ITEMS, MODE_EARLY, false>(job, n_cu, per_cu, s.counts, s.staging, st);
    } else if (job.pass == PASS_LATE) {
        launch_mode<BLOCK, ITEMS, MODE_LATE, true>(job, n_cu, per_cu, s.counts, s.staging, st);
    } else {
        if (h) launch_mode<BLOCK, ITEMS, MODE_OTHER, true>(job, n_cu, per_cu, s.counts, s.staging, st);
        else launch_mode<BLOCK, ITEMS, MODE_OTHER, false>(job, n_cu, per_cu, s.counts, s.staging, st);
    }
    hipError_t e = hipGetLastError();
    if (e != hipSuccess || !with_emit) return e;
    return launch_emit(job, (uint32_t)(BLOCK * ITEMS), s, st);
}

FuseDev fuse_dev(const FuseScratch& s, uint32_t wait_limit)
{
    return FuseDev{ s.words, s.err, wait_limit < kFusePatience ? wait_limit : kFusePatience };
}

hipError_t launch_fused_t(const CullJob& job, const FrameCacheDev& fc, bool record, uint2* left, const FuseDev& f,
                          hipStream_t st)
{
    const dim3 g(job.n_tiles), b(kFuseBlock);
#define BZ_FUSED(M, HZ, CA) \
    hipLaunchKernelGGL((fused_kernel<kFuseBlock, kFuseItems, M, HZ, CA>), g, b, 0, st, job, fc, left, f)
    const bool h = job.hiz != 0;
    if (job.pass == PASS_EARLY && record) {
        if (h) BZ_FUSED(MODE_EARLY, true, true);
        else BZ_FUSED(MODE_EARLY, false, true);
    } else if (job.pass == PASS_EARLY) {
        if (h) BZ_FUSED(MODE_EARLY, true, false);
        else BZ_FUSED(MODE_EARLY, false, false);
    } else if (job.pass == PASS_LATE) {
        BZ_FUSED(MODE_LATE, true, false);
    } else if (h) {
        BZ_FUSED(MODE_OTHER, true, false);
    } else {
        BZ_FUSED(MODE_OTHER, false, false);
    }
#undef BZ_FUSED
    return hipGetLastError();
}

template <int BLOCK, int ITEMS>
hipError_t launch_cull_batch_t(const CullJob* jobs_host, const CullJob* jobs, const uint32_t* starts, uint32_t n_jobs,
                               uint32_t total_tiles, uint32_t max_job_tiles, const CompactScratch& s, hipStream_t st)
{
    const bool few = n_jobs <= kArgFullJobs;
    JobArgs ja;
    if (few) {
        for (uint32_t k = 0; k < kArgFullJobs; ++k) {
            ja.j[k] = jobs_host[k < n_jobs ? k : 0u];
            if (k >= n_jobs) ja.j[k].tile_start = 0xffffffffu;
        }
        hipLaunchKernelGGL((decide_few_kernel<BLOCK, ITEMS>), dim3(total_tiles), dim3(BLOCK), 0, st, ja, s.counts,
                           s.staging, s.tile_job);
    } else {
        // entries past n_jobs are never searched; they are filled so the argument is fully defined
        JobStartsArg sa;
        for (uint32_t k = 0; k < kArgJobs; ++k) sa.v[k] = k < n_jobs ? jobs_host[k].tile_start : 0xffffffffu;
        hipLaunchKernelGGL((decide_batch_kernel<BLOCK, ITEMS>), dim3(total_tiles), dim3(BLOCK), 0, st, jobs, starts,
                           n_jobs, s.counts, s.staging, s.tile_job, sa);
    }
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    const uint32_t* prefix = nullptr;
    if (max_job_tiles > kScanTiles) {  // the batch's global prefix; each job takes differences of it
        e = launch_scan_counts(s.counts, total_tiles, s.prefix, st);
        if (e != hipSuccess) return e;
        prefix = s.prefix;
    }
    const dim3 g((total_tiles + kEmitTiles - 1) / kEmitTiles), b(kEmitBlock);
    if (few)
        hipLaunchKernelGGL(emit_few_kernel, g, b, 0, st, ja, total_tiles, (uint32_t)(BLOCK * ITEMS),
                           (const uint32_t*)s.counts, (const uint2*)s.staging, prefix);
    else
        hipLaunchKernelGGL(emit_batch_kernel, g, b, 0, st, jobs, total_tiles, (uint32_t)(BLOCK * ITEMS),
                           (const uint32_t*)s.counts, (const uint2*)s.staging, (const uint32_t*)s.tile_job, prefix);
    return hipGetLastError();
}

}  // namespace

#define BZ_TUNING_TABLE(X) \
    X(256, 2) X(256, 4) X(512, 2) X(512, 4)

hipError_t launch_cull(const CullJob& job, const CompactScratch& s, uint32_t block, uint32_t items, uint32_t n_cu,
                       uint32_t per_cu, hipStream_t st, const FrameCacheDev* cache)
{
#define X(B, I) \
    if (block == B && items == I) return launch_cull_t<B, I>(job, s, n_cu, per_cu, st, cache);
    BZ_TUNING_TABLE(X)
#undef X
    return hipErrorInvalidValue;
}

hipError_t launch_fused(const CullJob& job, const FuseScratch& s, uint32_t wait_limit, hipStream_t st,
                        const FrameCacheDev* cache)
{
    const FrameCacheDev fc = cache ? *cache : FrameCacheDev{};
    return launch_fused_t(job, fc, cache != nullptr, s.left, fuse_dev(s, wait_limit), st);
}

hipError_t launch_decide_only(const CullJob& job, const CompactScratch& s, uint32_t block, uint32_t items,
                              uint32_t n_cu, uint32_t per_cu, hipStream_t st, const InstHistDev* ih)
{
#define X(B, I)                                                                                                      \
    if (block == B && items == I)                                                                                     \
        return ih ? launch_decide_inst_t<B, I>(job, s, n_cu, per_cu, *ih, st)                                         \
                  : launch_cull_t<B, I>(job, s, n_cu, per_cu, st, nullptr, false);
    BZ_TUNING_TABLE(X)
#undef X
    return hipErrorInvalidValue;
}

void decide_inst_chunks(const CullJob& job, uint32_t block, uint32_t items, uint32_t n_cu, uint32_t per_cu,
                        uint32_t* tiles_per_chunk, uint32_t* n_long, uint32_t* n_chunks)
{
    uint32_t resident = 1;
#define X(B, I) \
    if (block == B && items == I) resident = inst_resident<B, I>();
    BZ_TUNING_TABLE(X)
#undef X
    // one chunk fewer than the workgroups that fit at once (one round, each workgroup a contiguous run of tiles, the
    // lengths differing by at most one tile): the scatter launch has a workgroup per chunk plus one for the commands,
    // and with as many chunks as slots it holds one workgroup more than three per CU (C1 size: scatter 15.6 us
    // against 12.8 us)
    uint64_t slots = (uint64_t)n_cu * (per_cu ? per_cu : resident);
    if (slots > 1) slots -= 1;
    if (slots > job.n_tiles) slots = job.n_tiles;
    if (slots == 0) slots = 1;
    *n_chunks = (uint32_t)slots;
    *tiles_per_chunk = (uint32_t)(job.n_tiles / slots);
    *n_long = (uint32_t)(job.n_tiles % slots);
    if (*tiles_per_chunk == 0) {  // (an empty job: one chunk of no tiles)
        *tiles_per_chunk = 1;
        *n_long = 0;
    }
}

hipError_t launch_late_fused(const CullJob& job, const FrameCacheDev& cache, const FuseScratch& s, uint32_t wait_limit,
                             hipStream_t st)
{
    hipLaunchKernelGGL((late_tile_kernel<kFuseBlock * kFuseItems, true>), dim3(job.n_tiles), dim3(kLtBlock), 0, st, job,
                       cache, (uint32_t*)nullptr, s.left, fuse_dev(s, wait_limit));
    return hipGetLastError();
}

hipError_t launch_late_cached(const CullJob& job, const CompactScratch& s, const FrameCacheDev& cache, uint32_t rec,
                              hipStream_t st)
{
    const dim3 g(job.n_tiles), b(kLtBlock);
#define BZ_LATE(T) \
    hipLaunchKernelGGL((late_tile_kernel<T, false>), g, b, 0, st, job, cache, s.counts, s.staging, FuseDev{})
    switch (rec) {
    case 512: BZ_LATE(512); break;
    case 1024: BZ_LATE(1024); break;
    case 2048: BZ_LATE(2048); break;
    default: return hipErrorInvalidValue;
    }
#undef BZ_LATE
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? launch_emit(job, rec, s, st) : e;
}

hipError_t launch_cluster_objects(const CullJob& job, const CompactScratch& s, uint32_t* ccounts, uint32_t block,
                                  uint32_t items, hipStream_t st)
{
#define X(B, I) \
    if (block == B && items == I) return launch_cluster_objects_t<B, I>(job, s, ccounts, st);
    BZ_TUNING_TABLE(X)
#undef X
    return hipErrorInvalidValue;
}

hipError_t launch_cull_batch(const CullJob* jobs_host, const CullJob* jobs_dev, const uint32_t* starts_dev,
                             uint32_t n_jobs, uint32_t total_tiles, uint32_t max_job_tiles, const CompactScratch& s,
                             uint32_t block, uint32_t items, hipStream_t st)
{
    if (n_jobs == 0 || total_tiles == 0) return hipSuccess;
#define X(B, I)                                                                                                      \
    if (block == B && items == I)                                                                                     \
        return launch_cull_batch_t<B, I>(jobs_host, jobs_dev, starts_dev, n_jobs, total_tiles, max_job_tiles, s, st);
    BZ_TUNING_TABLE(X)
#undef X
    return hipErrorInvalidValue;
}

// ------------------------------------------------------------------------------------------------
// exclusive prefix of tile counts (jobs of more than kScanTiles tiles)
// ------------------------------------------------------------------------------------------------
constexpr uint32_t kScanBlock = 1024;
constexpr uint32_t kScanPer = 8;  // consecutive counts per thread and round

// One workgroup walks the counts in rounds of kScanBlock * kScanPer. Each round is loaded and stored coalesced
// (thread t takes words t, t + kScanBlock, ...) through an LDS tile, in which thread t then owns kScanPer consecutive
// counts: an exclusive scan of its 8 counts, a wave scan of the thread totals and a block scan of the wave totals give
// each count its prefix (plus the rounds before); the last word is the total. The LDS tile has one spare word per 32,
// so the 8-word strided accesses spread over the banks.
__device__ __forceinline__ uint32_t scan_lds_index(uint32_t i) { return i + (i >> 5); }

__global__ __launch_bounds__(kScanBlock) void scan_counts_kernel(const uint32_t* __restrict__ counts, uint32_t n,
                                                                 uint32_t* __restrict__ prefix)
{
    constexpr uint32_t NW = kScanBlock / 64, R = kScanBlock * kScanPer;
    __shared__ uint32_t wsum[NW];
    __shared__ uint32_t tile[R + R / 32];
    const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6;
    uint32_t carry = 0;
    for (uint32_t r0 = 0; r0 < n; r0 += R) {
        uint32_t c[kScanPer];
#pragma unroll
        for (uint32_t k = 0; k < kScanPer; ++k) {
            const uint32_t i = r0 + k * kScanBlock + tid;
            c[k] = i < n ? counts[i] : 0u;
        }
#pragma unroll
        for (uint32_t k = 0; k < kScanPer; ++k) tile[scan_lds_index(k * kScanBlock + tid)] = c[k];
        __syncthreads();
        uint32_t v[kScanPer], own = 0;
#pragma unroll
        for (uint32_t k = 0; k < kScanPer; ++k) {
            const uint32_t x = tile[scan_lds_index(tid * kScanPer + k)];
            v[k] = own;
            own += x;
        }
        const uint32_t incl = wave_incl_scan(own, lane);
        if (lane == 63) wsum[wave] = incl;
        __syncthreads();
        uint32_t before = 0, total = 0;
#pragma unroll
        for (uint32_t w = 0; w < NW; ++w) {
            before += w < wave ? wsum[w] : 0u;
            total += wsum[w];
        }
        const uint32_t base = carry + before + (incl - own);
#pragma unroll
        for (uint32_t k = 0; k < kScanPer; ++k) tile[scan_lds_index(tid * kScanPer + k)] = base + v[k];
        __syncthreads();
#pragma unroll
        for (uint32_t k = 0; k < kScanPer; ++k) {
            const uint32_t i = r0 + k * kScanBlock + tid;
            if (i < n) prefix[i] = tile[scan_lds_index(k * kScanBlock + tid)];
        }
        carry += total;
        __syncthreads();  // wsum and the tile are rewritten by the next round
    }
    if (threadIdx.x == 0) prefix[n] = carry;
}

hipError_t launch_scan_counts(const uint32_t* counts, uint32_t n, uint32_t* prefix, hipStream_t st)
{
    hipLaunchKernelGGL(scan_counts_kernel, dim3(1), dim3(kScanBlock), 0, st, counts, n, prefix);
    return hipGetLastError();
}

// ------------------------------------------------------------------------------------------------
// small helpers
// ------------------------------------------------------------------------------------------------
__global__ void fill_u32_kernel(uint32_t* p, uint32_t value, uint64_t n)
{
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (uint64_t)gridDim.x * blockDim.x)
        p[i] = value;
}

hipError_t launch_fill_u32(uint32_t* p, uint32_t value, uint64_t n, hipStream_t st)
{
    if (n == 0) return hipSuccess;
    uint64_t blocks = (n + 255) / 256;
    if (blocks > 65536) blocks = 65536;
    hipLaunchKernelGGL(fill_u32_kernel, dim3((uint32_t)blocks), dim3(256), 0, st, p, value, n);
    return hipGetLastError();
}

// Transform updates, in two launches so that an id named more than once in one commit takes its last occurrence
// (UpdateObjectTransform copies updates into the staging buffer in call order, vulkanDraw.cpp:816-820):
//   mark:    copies ids from the pinned slot into device memory; update i raises winner[id] to i + 1;
//   scatter: update i reads its 32-byte record over the host link and writes it into the position/scale and quaternion
//            streams, and its object's world-space sphere, only if it is the winner, which then clears winner[id] (the
//            array is all zero between commits; a non-winner compares its own i + 1 and never matches, whether it reads
//            before or after that clear).
// Ids >= n_xf are skipped and set err[2].
// The host link bounds both. One thread reads a whole record, and everything else that it needs before (id, winner,
// surface): 41 943 updates 38.0 us, 200 000 152 us; with the records' loads issued first 38.5 and 161, with a thread per
// 16-byte half 44.3 and 175. Writing the spheres costs 0.8 us of the 38.0.
__global__ __launch_bounds__(256) void mark_staged_transforms_kernel(const uint32_t* __restrict__ ids, uint32_t n,
                                                                     uint32_t n_xf, uint32_t* __restrict__ dev_ids,
                                                                     uint32_t* winner, uint32_t* err)
{
    const uint32_t i = blockIdx.x * 256u + threadIdx.x;
    if (i >= n) return;
    const uint32_t id = ids[i];
    dev_ids[i] = id;
    if (id >= n_xf) {
        atomicOr(&err[2], 1u);
        return;
    }
    atomicMax(&winner[id], i + 1u);
}

// World-space bounding sphere of an object, and its transform's scale.
__device__ __forceinline__ float4 world_sphere(const float4& sph, const float4& ps, const float4& q)
{
    float4 w;
    sphere_to_world(sph.x, sph.y, sph.z, ps.x, ps.y, ps.z, ps.w, q.x, q.y, q.z, q.w, w.x, w.y, w.z);
    w.w = ps.w;
    return w;
}

__device__ __forceinline__ float4 object_surface(const SceneDev& S, uint32_t obj)
{
    return S.surf_sphere[S.obj_surf16 ? (uint32_t)S.obj_surf16[obj] : S.obj_surf[obj]];
}

// The spheres of the objects that use the workgroup's updated transforms (scenes with obj_xf): thread i's transform is used
// by `len` objects, listed from objs[first]. The lists, end to end, are dealt to the threads, so that one of many objects does
// not hold a thread up; four objects of a thread in flight. An update then costs what it moves: a launch that looked at the
// stamp of every object's transform instead took, for 41 943 of 4 194 304 transforms in random order, 31 us besides.
struct SpreadSmem {
    float4 ps[256], q[256];
    uint32_t end[256], off[256];  // of each list: its end in the sequence, and what takes a place in it to its index in objs
    uint32_t wsum[4];
};
__device__ __forceinline__ void spread_spheres(const XfTarget& to, uint32_t first, uint32_t len, const float4& ps,
                                               const float4& q, SpreadSmem& sm)
{
    constexpr uint32_t U = 4;
    const uint32_t tid = threadIdx.x, wave = tid >> 6;
    uint32_t end = wave_incl_scan(len, tid & 63u);
    if ((tid & 63u) == 63u) sm.wsum[wave] = end;
    sm.ps[tid] = ps;
    sm.q[tid] = q;
    __syncthreads();
    for (uint32_t w = 0; w < wave; ++w) end += sm.wsum[w];
    sm.end[tid] = end;
    sm.off[tid] = first - (end - len);
    __syncthreads();
    const uint32_t total = sm.end[255];
    for (uint32_t r0 = 0; r0 < total; r0 += U * 256u) {
        uint32_t j[U], obj[U];
        float4 sph[U];
#pragma unroll
        for (uint32_t u = 0; u < U; ++u) {
            const uint32_t r = r0 + u * 256u + tid;
            j[u] = 0;  // the first list that ends behind r
#pragma unroll
            for (uint32_t step = 128; step; step >>= 1)
                if (sm.end[j[u] + step - 1u] <= r) j[u] += step;
            obj[u] = r < total ? to.objs[sm.off[j[u]] + r] : 0u;
        }
#pragma unroll
        for (uint32_t u = 0; u < U; ++u) sph[u] = object_surface(to.scene, obj[u]);
#pragma unroll
        for (uint32_t u = 0; u < U; ++u)
            if (r0 + u * 256u + tid < total) to.world[obj[u]] = world_sphere(sph[u], sm.ps[j[u]], sm.q[j[u]]);
    }
}
// The list of an updated transform; a long one is left to the next launch.
__device__ __forceinline__ void spread_list(const XfTarget& to, uint32_t id, bool updated, uint32_t& first, uint32_t& len)
{
    first = updated ? to.first[id] : 0u;
    len = updated ? to.first[id + 1u] - first : 0u;
    if (len > xf_inline(to.per_block)) {
        to.stamp[id] = to.version;
        len = 0u;
    }
}

template <bool SHARED>
__global__ __launch_bounds__(256) void scatter_staged_transforms_kernel(const uint32_t* __restrict__ dev_ids,
                                                                        const float4* __restrict__ records, uint32_t n,
                                                                        XfTarget to)
{
    if constexpr (SHARED) {
        __shared__ SpreadSmem sm;
        const uint32_t i = blockIdx.x * to.per_block + threadIdx.x;
        const uint32_t id = threadIdx.x < to.per_block && i < n ? dev_ids[i] : 0xffffffffu;
        const bool wins = id < to.scene.n_transforms && to.winner[id] == i + 1u;
        float4 ps = make_float4(0.f, 0.f, 0.f, 0.f), q = ps;
        if (wins) {
            ps = records[2u * i];
            q = records[2u * i + 1u];
        }
        uint32_t first, len;
        spread_list(to, id, wins, first, len);  // (its loads behind the records')
        if (wins) {
            to.xf_ps[id] = ps;
            to.xf_q[id] = q;
            to.winner[id] = 0u;
        }
        spread_spheres(to, first, len, ps, q, sm);
    } else {
        const uint32_t i = blockIdx.x * 256u + threadIdx.x;
        if (i >= n) return;
        const uint32_t id = dev_ids[i];
        if (id >= to.scene.n_transforms || to.winner[id] != i + 1u) return;
        const bool sphere = id < to.scene.n_objects;
        const float4 sph = sphere ? object_surface(to.scene, id) : make_float4(0.f, 0.f, 0.f, 0.f);
        const float4 ps = records[2u * i], q = records[2u * i + 1u];
        to.xf_ps[id] = ps;
        to.xf_q[id] = q;
        to.winner[id] = 0u;
        if (sphere) to.world[id] = world_sphere(sph, ps, q);
    }
}

// Updates that name every id once (and in range), up to kDistinctUpdates of them: straight from the pinned slot to the
// streams in one launch. Calls with 4096 updates 11.5 us against 14.3 in two launches, 10 485 16.2 against 18.6, 16 384 21.1
// against 22.8, 24 576 27.7 against 28.7, but 41 943 51.5 against 39.1: ids and records read over the link at once slow each
// other down when there are many.
template <bool SHARED>
__global__ __launch_bounds__(256) void scatter_distinct_transforms_kernel(const uint32_t* __restrict__ ids,
                                                                          const float4* __restrict__ records,
                                                                          uint32_t n, XfTarget to)
{
    if constexpr (SHARED) {
        __shared__ SpreadSmem sm;
        const uint32_t i = blockIdx.x * to.per_block + threadIdx.x;
        const bool mine = threadIdx.x < to.per_block && i < n;
        const uint32_t id = mine ? ids[i] : 0xffffffffu;
        float4 ps = make_float4(0.f, 0.f, 0.f, 0.f), q = ps;
        if (mine) {
            ps = records[2u * i];
            q = records[2u * i + 1u];
        }
        uint32_t first, len;
        const bool valid = id < to.scene.n_transforms;
        spread_list(to, id, valid, first, len);
        if (valid) {
            to.xf_ps[id] = ps;
            to.xf_q[id] = q;
        }
        spread_spheres(to, first, len, ps, q, sm);
    } else {
        const uint32_t i = blockIdx.x * 256u + threadIdx.x;
        if (i >= n) return;
        const uint32_t id = ids[i];
        const float4 ps = records[2u * i], q = records[2u * i + 1u];
        if (id >= to.scene.n_transforms) return;  // (the caller has looked: only a caller's race on its ids gets here)
        to.xf_ps[id] = ps;
        to.xf_q[id] = q;
        if (id < to.scene.n_objects) to.world[id] = world_sphere(object_surface(to.scene, id), ps, q);
    }
}

// World-space spheres of all the scene's objects.
__global__ __launch_bounds__(256) void world_spheres_kernel(SceneDev S, float4* __restrict__ world)
{
    const uint32_t i = blockIdx.x * 256u + threadIdx.x;
    if (i >= S.n_objects) return;
    const uint32_t x = S.obj_xf ? S.obj_xf[i] : i;
    world[i] = world_sphere(object_surface(S, i), S.xf_ps[x], S.xf_q[x]);
}

// The spheres of the objects of a transform that many use, a wave per piece of at most kXfChunk of them: those whose
// transform carries the stamp of the update just scattered.
__global__ __launch_bounds__(256) void chunk_spheres_kernel(XfTarget to)
{
    const uint32_t c = blockIdx.x * 4u + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63u;
    if (c >= to.n_chunks) return;
    const XfChunk ck = to.chunks[c];
    if (to.stamp[ck.xf] != to.version) return;
    const float4 ps = to.xf_ps[ck.xf], q = to.xf_q[ck.xf];
    constexpr uint32_t U = kXfChunk / 64u;
    uint32_t obj[U];
    float4 sph[U];
#pragma unroll
    for (uint32_t u = 0; u < U; ++u) {
        const uint32_t k = ck.begin + u * 64u + lane;
        obj[u] = to.objs[k < ck.end ? k : ck.begin];
    }
#pragma unroll
    for (uint32_t u = 0; u < U; ++u) sph[u] = object_surface(to.scene, obj[u]);
#pragma unroll
    for (uint32_t u = 0; u < U; ++u)
        if (ck.begin + u * 64u + lane < ck.end) to.world[obj[u]] = world_sphere(sph[u], ps, q);
}

// Adds 1 to counter[x] for every active lane and gives each lane the count before it. The lanes of the first two transforms
// met are added together: where one transform is many objects', they would otherwise queue up at its counter.
__device__ __forceinline__ uint32_t count_up(uint32_t* counter, uint32_t x, bool active)
{
    const uint32_t lane = threadIdx.x & 63u;
    uint32_t place = 0;
    for (uint32_t round = 0; round < 2u; ++round) {
        const unsigned long long todo = __ballot(active);
        if (!todo) return place;
        const uint32_t x0 = __shfl(x, __ffsll(todo) - 1, 64);
        const unsigned long long same = __ballot(active && x == x0);
        uint32_t base = 0;
        if (lane == (uint32_t)__ffsll(same) - 1u) base = atomicAdd(&counter[x0], (uint32_t)__popcll(same));
        base = __shfl(base, __ffsll(same) - 1, 64);
        if (active && x == x0) {
            place = base + (uint32_t)__popcll(same & ((1ull << lane) - 1ull));
            active = false;
        }
    }
    return active ? atomicAdd(&counter[x], 1u) : place;
}

__global__ __launch_bounds__(256) void list_count_kernel(const uint32_t* __restrict__ obj_xf, uint32_t n, uint32_t* counts)
{
    const uint32_t i = blockIdx.x * 256u + threadIdx.x;
    count_up(counts, i < n ? obj_xf[i] : 0u, i < n);
}

__global__ __launch_bounds__(256) void list_fill_kernel(const uint32_t* __restrict__ obj_xf, uint32_t n, uint32_t* next,
                                                        uint32_t* __restrict__ objs)
{
    const uint32_t i = blockIdx.x * 256u + threadIdx.x;
    const uint32_t place = count_up(next, i < n ? obj_xf[i] : 0u, i < n);
    if (i < n) objs[place] = i;
}

// next[t] = first[t], the number of lists that are not empty
__global__ __launch_bounds__(256) void list_start_kernel(const uint32_t* __restrict__ first, uint32_t n_xf, uint32_t* next,
                                                         uint32_t* used)
{
    const uint32_t t = blockIdx.x * 256u + threadIdx.x;
    if (t < n_xf) next[t] = first[t];
    const unsigned long long m = __ballot(t < n_xf && first[t + 1u] != first[t]);
    if ((threadIdx.x & 63u) == 0 && m) atomicAdd(used, (uint32_t)__popcll(m));
}

__global__ __launch_bounds__(256) void list_chunks_kernel(const uint32_t* __restrict__ first, uint32_t n_xf, uint32_t most,
                                                          XfChunk* __restrict__ chunks, uint32_t* n_chunks)
{
    const uint32_t t = blockIdx.x * 256u + threadIdx.x;
    if (t >= n_xf) return;
    const uint32_t b = first[t], e = first[t + 1u];
    if (e - b <= most) return;
    const uint32_t n = (e - b + kXfChunk - 1u) / kXfChunk, slot = atomicAdd(n_chunks, n);
    for (uint32_t k = 0; k < n; ++k) {
        const uint32_t k0 = b + k * kXfChunk;
        chunks[slot + k] = XfChunk{ t, k0, e - k0 < kXfChunk ? e : k0 + kXfChunk };
    }
}

hipError_t launch_list_objects(const uint32_t* obj_xf, uint32_t n, uint32_t n_xf, uint32_t* work, uint32_t* first,
                               uint32_t* objs, hipStream_t st)
{
    const dim3 go((n + 255u) / 256u), gt((n_xf + 255u) / 256u), b(256);
    hipError_t e = launch_fill_u32(work, 0u, (uint64_t)n_xf + 1u, st);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(list_count_kernel, go, b, 0, st, obj_xf, n, work);
    e = launch_scan_counts(work, n_xf, first, st);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(list_start_kernel, gt, b, 0, st, (const uint32_t*)first, n_xf, work, work + n_xf);
    hipLaunchKernelGGL(list_fill_kernel, go, b, 0, st, obj_xf, n, work, objs);
    return hipGetLastError();
}

hipError_t launch_list_chunks(const uint32_t* first, uint32_t n_xf, uint32_t most, XfChunk* chunks, uint32_t* n_chunks,
                              hipStream_t st)
{
    const hipError_t e = launch_fill_u32(n_chunks, 0u, 1u, st);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(list_chunks_kernel, dim3((n_xf + 255u) / 256u), dim3(256), 0, st, first, n_xf, most, chunks,
                       n_chunks);
    return hipGetLastError();
}

hipError_t launch_world_spheres(const SceneDev& scene, float4* world, hipStream_t st)
{
    if (scene.n_objects == 0) return hipSuccess;
    hipLaunchKernelGGL(world_spheres_kernel, dim3((scene.n_objects + 255u) / 256u), dim3(256), 0, st, scene, world);
    return hipGetLastError();
}

hipError_t launch_scatter_staged_transforms(const uint32_t* ids, const float4* records, uint32_t n, bool distinct,
                                            const XfTarget& to, uint32_t* dev_ids, uint32_t* err, hipStream_t st)
{
    if (n == 0) return hipSuccess;
    const bool shared = to.scene.obj_xf != nullptr && to.scene.n_objects != 0;
    const uint32_t per = shared ? to.per_block : 256u;
    const dim3 g((uint32_t)(((uint64_t)n + per - 1u) / per)), g256((n + 255u) / 256u), b(256);
    if (distinct && n <= kDistinctUpdates) {
        if (shared) hipLaunchKernelGGL(scatter_distinct_transforms_kernel<true>, g, b, 0, st, ids, records, n, to);
        else hipLaunchKernelGGL(scatter_distinct_transforms_kernel<false>, g, b, 0, st, ids, records, n, to);
    } else {
        hipLaunchKernelGGL(mark_staged_transforms_kernel, g256, b, 0, st, ids, n, to.scene.n_transforms, dev_ids, to.winner,
                           err);
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
        const uint32_t* di = dev_ids;
        if (shared) hipLaunchKernelGGL(scatter_staged_transforms_kernel<true>, g, b, 0, st, di, records, n, to);
        else hipLaunchKernelGGL(scatter_staged_transforms_kernel<false>, g, b, 0, st, di, records, n, to);
    }
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess || to.n_chunks == 0) return e;
    hipLaunchKernelGGL(chunk_spheres_kernel, dim3((to.n_chunks + 3u) / 4u), b, 0, st, to);
    return hipGetLastError();
}

}  // namespace bz
