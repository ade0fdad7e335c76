// fuse.h — device helpers of the passes that decide and write their commands in one launch: the draw command record, and
// the counts that workgroups publish for the ones after them.
#pragma once
#include "bz_internal.h"
#include "fuse_words.h"

namespace bz {

__device__ __forceinline__ void write_command(uint32_t* cmds, uint32_t pos, uint32_t object, uint2 draw)
{
    uint2* cmd = reinterpret_cast<uint2*>(cmds + (size_t)pos * 6u);
    cmd[0] = make_uint2(object, draw.x);  // objectId, indexCount
    cmd[1] = make_uint2(1u, draw.y);       // instanceCount, firstIndex
    cmd[2] = make_uint2(0u, 0u);           // vertexOffset, firstInstance
}

// The words that a launch's workgroups hand each other, each with the launch's number above its value: a word of another
// launch is not taken, so nothing is cleared between launches (fuse_words.h).
struct FuseDev {
    unsigned long long* words;  // [0] number of the last launch, [1] of the last one in which a tile left its commands
                                // (32 bits each), [kFuseFirst + tile] the tiles' command counts, [kFuseFirst + kFuseTiles +
                                // tile] of a tile that left its commands: 1 left, 2 taken by the one that writes them
    uint32_t* err;              // set when the last tile gives its wait up
    uint32_t patience;          // looks at words not there yet before a tile leaves its commands
};
enum : uint32_t { kFuseLeft = 1, kFuseTaken = 2 };
__device__ __forceinline__ unsigned long long fuse_load(const FuseDev& fuse, uint32_t word)
{
    return __hip_atomic_load(&fuse.words[word], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void fuse_store(const FuseDev& fuse, uint32_t word, uint32_t launch, uint32_t value)
{
    __hip_atomic_store(&fuse.words[word], (unsigned long long)launch << 32 | value, __ATOMIC_RELAXED,
                       __HIP_MEMORY_SCOPE_AGENT);
}

// Takes the commands that a tile left; one thread does.
__device__ __forceinline__ bool fuse_claim(const FuseDev& fuse, uint32_t word, uint32_t launch)
{
    unsigned long long is = (unsigned long long)launch << 32 | kFuseLeft;
    return __hip_atomic_compare_exchange_strong(&fuse.words[word], &is, (unsigned long long)launch << 32 | kFuseTaken,
                                                __ATOMIC_ACQ_REL, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Takes words [first, first + n) of this launch, a thread every BLOCK-th, its loads (KW at a time) ahead of its first wait.
// false: `limit` looks were not enough for one of this thread's words (which is then taken as it is).
template <uint32_t BLOCK, class Take>
__device__ __forceinline__ bool fuse_take(const FuseDev& fuse, uint32_t launch, uint32_t first, uint32_t n, uint32_t limit,
                                          Take&& take)
{
    constexpr uint32_t KW = 4;
    const uint32_t tid = threadIdx.x;
    uint32_t spins = 0;
    for (uint32_t u0 = 0; u0 < n; u0 += KW * BLOCK) {
        unsigned long long w[KW];
#pragma unroll
        for (uint32_t k = 0; k < KW; ++k) {
            const uint32_t u = u0 + k * BLOCK + tid;
            w[k] = u < n ? fuse_load(fuse, first + u) : (unsigned long long)launch << 32;
        }
#pragma unroll
        for (uint32_t k = 0; k < KW; ++k) {
            while ((uint32_t)(w[k] >> 32) != launch && spins <= limit && ++spins <= limit) {
                __builtin_amdgcn_s_sleep(1);
                w[k] = fuse_load(fuse, first + u0 + k * BLOCK + tid);
            }
            take((uint32_t)w[k]);
        }
    }
    return spins <= limit;
}

// Sum of the counts of the tiles before `tile`, by the whole workgroup (red: 2 * BLOCK / 64 LDS words; one barrier). false,
// for all of it: a count has not come.
template <uint32_t BLOCK>
__device__ __forceinline__ bool fuse_sum(const FuseDev& fuse, uint32_t launch, uint32_t tile, uint32_t limit, uint32_t* red,
                                         uint32_t& prefix)
{
    constexpr uint32_t NW = BLOCK / 64u;
    uint32_t part = 0;
    const bool here =
        fuse_take<BLOCK>(fuse, launch, kFuseFirst, tile, limit, [&](uint32_t count) { part += count; });
    const uint32_t missing = __all(here) ? 0u : 1u;
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) part += __shfl_xor(part, off, 64);
    if ((threadIdx.x & 63u) == 0) {
        red[threadIdx.x >> 6] = part;
        red[NW + (threadIdx.x >> 6)] = missing;
    }
    __syncthreads();
    prefix = 0;
    uint32_t any = 0;
#pragma unroll
    for (uint32_t w = 0; w < NW; ++w) {
        prefix += red[w];
        any |= red[NW + w];
    }
    return __builtin_amdgcn_readfirstlane(any) == 0u;
}

// Commands of the tiles before `tile`, by the whole workgroup. Every tile but the last waits for their counts only so long
// (fuse.patience): then it stores its commands with stage() and leaves them to the last tile, and false is returned.
//
// So every workgroup but a launch's last one ends whatever else is or is not running: nothing here rests on the order in
// which workgroups start. That matters with several streams: a launch's workgroups go to eight XCDs that fill
// independently, and the ones of other launches that wait can hold every slot that an earlier tile of this one needs (an
// expansion has four workgroups a CU, 128 slots an XCD, and 80 of its 640 tiles on each: two other streams are enough),
// while this one's hold the slots that those wait for. The last tiles alone, one workgroup per launch, cannot.
//
// The last tile does not wait for the others to end: it only looks whether one has left, after it has had every count. A
// tile that leaves says so first, waits until that is done, and then looks at the counts once more. If one is still missing,
// that one comes later than the tile's word, and the last tile, whose look starts after it has had that count, looks later
// still: it finds the word. If none is missing, the last tile may have looked before, and whichever of the two takes the
// word writes the commands. (The words are read and written past the L2s, all XCDs' at one place, and a load that has come
// back, or a store waited for, is done there. So the last tile needs its loads in that order, and no fence: one that writes
// its L2 back cost 1 us per pass, a frame of 65 536 objects 24.2 -> 26.3 us; this look costs 0.1.)
template <uint32_t BLOCK, class Stage>
__device__ __forceinline__ bool fuse_prefix(const FuseDev& fuse, uint32_t launch, uint32_t tile, bool last_tile,
                                            uint32_t* red, uint32_t& prefix, uint32_t& left, Stage&& stage)
{
    const bool here =
        fuse_sum<BLOCK>(fuse, launch, tile, last_tile ? BZ_DEFAULT_WAIT_LIMIT : fuse.patience, red, prefix);
    uint32_t* mark = reinterpret_cast<uint32_t*>(fuse.words + 1);
    if (last_tile) {
        if (!here && threadIdx.x == 0) atomicExch(fuse.err, 1u);
        __atomic_signal_fence(__ATOMIC_SEQ_CST);
        __builtin_amdgcn_s_waitcnt(0);
        left = __hip_atomic_load(mark, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (threadIdx.x == 0) {  // each workgroup has read the launch's number: it moves on, and a word ages
            const uint32_t aged = fuse_aged(launch, kFuseTiles);
            if (aged > tile) fuse_store(fuse, kFuseFirst + aged, 0u, 0u);
            __hip_atomic_store(reinterpret_cast<uint32_t*>(fuse.words), launch, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        return true;
    }
    if (__builtin_expect(here, 1)) return true;
    const uint32_t word = kFuseFirst + kFuseTiles + tile;
    stage();
    __threadfence();
    __syncthreads();
    if (threadIdx.x == 0) {
        fuse_store(fuse, word, launch, kFuseLeft);
        __hip_atomic_store(mark, launch, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "agent");
    }
    __syncthreads();
    if (!fuse_sum<BLOCK>(fuse, launch, tile, 0u, red, prefix)) return false;
    __syncthreads();
    if (threadIdx.x == 0) red[0] = fuse_claim(fuse, word, launch) ? 1u : 0u;
    __syncthreads();
    return __builtin_amdgcn_readfirstlane(red[0]) != 0u;
}
// The number of the launch before. The value that thread 0 reads is the workgroup's: it hands it to the others through LDS,
// ahead of a barrier that the workgroup's word is published behind, so that no read of words[0] that counts is outstanding
// once the word has arrived (a wave that used a read of its own could still be waiting for it then, and get the next one).
__device__ __forceinline__ uint32_t fuse_last(const FuseDev& fuse)
{
    return __hip_atomic_load(reinterpret_cast<uint32_t*>(fuse.words), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ uint32_t fuse_launch(uint32_t last)  // this launch's number
{
    return fuse_next(__builtin_amdgcn_readfirstlane(last));
}
__device__ __forceinline__ void fuse_publish(const FuseDev& fuse, uint32_t launch, uint32_t tile, uint32_t count)
{
    fuse_store(fuse, kFuseFirst + tile, launch, count);
}
// By the last tile, which has had every count: its first wave writes the commands of the tiles that left theirs
// (write(tile, first command, commands), 64 lanes).
template <class Write>
__device__ __forceinline__ void fuse_settle(const FuseDev& fuse, uint32_t launch, uint32_t left, uint32_t n_tiles,
                                            Write&& write)
{
    if (threadIdx.x >= 64u || __builtin_expect(__builtin_amdgcn_readfirstlane(left) != launch, 1)) return;
    uint32_t first = 0;
    for (uint32_t t = 0; t + 1u < n_tiles; ++t) {
        const uint32_t count = (uint32_t)fuse_load(fuse, kFuseFirst + t);
        uint32_t mine = 0;
        if (threadIdx.x == 0) mine = fuse_claim(fuse, kFuseFirst + kFuseTiles + t, launch) ? 1u : 0u;
        if (__builtin_amdgcn_readfirstlane(mine)) {
            __threadfence();
            write(t, first, count);
        }
        first += count;
    }
}

}  // namespace bz
