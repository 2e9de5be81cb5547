// Ray hand-out of the persistent traversal kernels (HIP device code for
// gfx950).
#pragma once

#include "internal.hpp"

namespace rtbvh {

// Ray hand-out of the persistent kernels.  Static (schedule 0): lane k of
// the grid takes rays k, k + stride, ...  Wave ranges (schedule 1): wave w
// owns the contiguous rays [w L, (w + 1) L), L = ceil(rays / waves), and its
// idle lanes draw the next ones in lane order as they free up, so a wave's
// lanes stay busy until its range is used up (no atomics: the cursor is
// wave-uniform).
// A value known to be equal in every lane of the wave, read from the first
// active lane so that the compiler keeps it in scalar registers.
__device__ __forceinline__ uint64_t wave_uniform(uint64_t v) {
    const uint32_t lo = uint32_t(__builtin_amdgcn_readfirstlane(int(uint32_t(v))));
    const uint32_t hi = uint32_t(__builtin_amdgcn_readfirstlane(int(uint32_t(v >> 32))));
    return (uint64_t(hi) << 32) | lo;
}

struct RaySchedule {
    uint64_t rid;
    uint64_t stride;
    uint64_t cursor;  // wave ranges: next ray of the wave's range (wave-uniform)
    uint64_t end;
    bool ranges;

    __device__ void init(const TraceParams& p) {
        stride = uint64_t(gridDim.x) * blockDim.x;
        const uint64_t tid = uint64_t(blockIdx.x) * blockDim.x + threadIdx.x;
        rid = tid;
        ranges = p.wave_ranges != 0;
        const uint64_t waves = (stride + 63) >> 6;
        const uint64_t per = (p.ray_count + waves - 1) / waves;
        const uint64_t b = (tid >> 6) * per;
        // the same for every lane of the wave (blocks are whole waves): held
        // in scalar registers
        cursor = wave_uniform(b < p.ray_count ? b : p.ray_count);
        end = wave_uniform(b + per < p.ray_count ? b + per : p.ray_count);
    }

    // This lane is idle and rays may be left for it.
    __device__ bool can_take(const TraceParams& p, bool active) const {
        return !active && (ranges ? cursor < end : rid < p.ray_count);
    }

    // Called by the whole wave when it hands out rays (takers = ballot of
    // can_take); true when this lane got ray `rid`.
    __device__ bool take(bool me, uint64_t takers) {
        if (!ranges) return me;
        // takers in the lanes below this one (v_mbcnt)
        const uint32_t below = __builtin_amdgcn_mbcnt_hi(
            uint32_t(takers >> 32), __builtin_amdgcn_mbcnt_lo(uint32_t(takers), 0u));
        const uint64_t r = cursor + below;
        cursor += uint64_t(__popcll(takers));
        if (cursor > end) cursor = end;
        if (!me || r >= end) return false;
        rid = r;
        return true;
    }

    // The lane's ray is finished (or skipped).
    __device__ void next() {
        if (!ranges) rid += stride;
    }
};

}  // namespace rtbvh
