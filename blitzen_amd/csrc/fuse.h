// fuse.h — device helpers of the passes that decide and write their commands in one launch: the draw command record, and
// the counts that workgroups publish for the ones after them.
#pragma once
#include "bz_internal.h"

namespace bz {

__device__ __forceinline__ void write_command(uint32_t* cmds, uint32_t pos, uint32_t object, uint2 draw)
{
    uint2* cmd = reinterpret_cast<uint2*>(cmds + (size_t)pos * 6u);
    cmd[0] = make_uint2(object, draw.x);  // objectId, indexCount
    cmd[1] = make_uint2(1u, draw.y);       // instanceCount, firstIndex
    cmd[2] = make_uint2(0u, 0u);           // vertexOffset, firstInstance
}

// The word another workgroup publishes for a tile in one launch: the tile's command count with the launch's number above
// it. A word of another launch is not taken, so nothing is cleared between launches.
struct FuseDev {
    unsigned long long* words;  // [0] number of the last launch (32 bits), [kFuseFirst + tile] the tiles' words
    uint32_t* err;              // set when a wait gives up
};

// Commands of the tiles before `tile`, by the whole workgroup (red: BLOCK / 64 LDS words; one barrier). Every word of a
// thread is loaded before its first wait; a tile only waits on workgroups dispatched before it.
template <uint32_t BLOCK>
__device__ __forceinline__ uint32_t fuse_prefix(const FuseDev& fuse, uint32_t launch, uint32_t tile, uint32_t* red)
{
    constexpr uint32_t KW = 4;
    const uint32_t tid = threadIdx.x;
    uint32_t part = 0;
    for (uint32_t u0 = 0; u0 < tile; u0 += KW * BLOCK) {
        unsigned long long w[KW];
#pragma unroll
        for (uint32_t k = 0; k < KW; ++k) {
            const uint32_t u = u0 + k * BLOCK + tid;
            w[k] = u < tile ? __hip_atomic_load(&fuse.words[kFuseFirst + u], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)
                            : (unsigned long long)launch << 32;
        }
#pragma unroll
        for (uint32_t k = 0; k < KW; ++k) {
            uint32_t spins = 0;
            while ((uint32_t)(w[k] >> 32) != launch) {
                if (++spins > BZ_DEFAULT_WAIT_LIMIT) {
                    atomicExch(fuse.err, 1u);
                    break;
                }
                __builtin_amdgcn_s_sleep(1);
                w[k] = __hip_atomic_load(&fuse.words[kFuseFirst + u0 + k * BLOCK + tid], __ATOMIC_RELAXED,
                                         __HIP_MEMORY_SCOPE_AGENT);
            }
            part += (uint32_t)w[k];
        }
    }
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) part += __shfl_xor(part, off, 64);
    if ((tid & 63u) == 0) red[tid >> 6] = part;
    __syncthreads();
    uint32_t prefix = 0;
#pragma unroll
    for (uint32_t w = 0; w < BLOCK / 64u; ++w) prefix += red[w];
    return prefix;
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
    return __builtin_amdgcn_readfirstlane(last) + 1u;
}
__device__ __forceinline__ void fuse_publish(const FuseDev& fuse, uint32_t launch, uint32_t tile, uint32_t count)
{
    __hip_atomic_store(&fuse.words[kFuseFirst + tile], (unsigned long long)launch << 32 | count, __ATOMIC_RELAXED,
                       __HIP_MEMORY_SCOPE_AGENT);
}
// By the last tile, which has had every word: each workgroup has read the launch's number, so it can move on.
__device__ __forceinline__ void fuse_finish(const FuseDev& fuse, uint32_t launch)
{
    __hip_atomic_store(reinterpret_cast<uint32_t*>(fuse.words), launch, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

}  // namespace bz
