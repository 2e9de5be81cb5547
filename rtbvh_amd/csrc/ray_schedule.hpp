// Ray hand-out of the persistent traversal kernels (HIP device code for
// gfx950).
#pragma once

#include "internal.hpp"

namespace rtbvh {

// Ray hand-out of the persistent kernels.  Static (schedule 0): lane k of
// the grid takes rays k, k + stride, ...  Runs (schedule 1): the rays are
// dealt to the waves in turn in runs of 64 consecutive ones (wave w of W owns
// runs w, w + W, ...), and a wave's idle lanes draw its next rays in order as
// they free up, so its lanes stay busy until its rays are used up (no
// atomics: the cursor is wave-uniform).  Runs keep neighbouring rays in one
// wave; dealing them in turn gives every wave a share of the whole set.  One
// contiguous range per wave, the form before, left the waves of an image's
// costly rows running alone at the end: on a 1M tree (default shape, 64 rays
// a run against one range) 2^22 / 2^24 camera rays 1344 / 2704 us against
// 1600 / 4171, 2^24 bounce rays 7.86 ms against 8.42, 2^24 shadow rays in the
// order of their origins on 4M triangles 8.37 ms against 11.39.  Runs of 128
// to 512 rays: 1380 to 1558 us for the first.  Equal shares (the rays past
// the last whole round of runs dealt in pieces of under 64) lost 1 % over 260
// launches of 700k to 16M rays, 10 % on any hit of the binary traversal.
//
// A grid of many times the resident waves keeps one contiguous range per wave
// (wave_runs 2, the compressed and 4-wide traversals only): waves spread over
// the whole set share less of the caches' traffic (2^26 bounce rays of an
// 8192 x 8192 image 24.6 ms against 26.2 in runs, a batch of 256 scenes with
// 328M rays 97 against 137 ms).  Images whose costly part is small go the
// other way: of a 16:9 image 2^26 camera rays 15.1 ms against 8.5 in runs and
// its bounce rays, whose many misses start anew at random points, 31.3 against
// 28.3.
constexpr uint32_t kRunShift = 6;

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
    // runs: positions of the wave's sequence, and the first rays of its first
    // run and of the next (all wave-uniform, in scalar registers)
    uint32_t cursor, end;
    uint64_t base, jump;
    bool runs;

    __device__ void init(const TraceParams& p) {
        stride = uint64_t(gridDim.x) * blockDim.x;
        const uint64_t tid = uint64_t(blockIdx.x) * blockDim.x + threadIdx.x;
        rid = tid;
        runs = p.wave_runs != 0;
        const uint64_t waves = (stride + 63) >> 6, wave = wave_uniform(tid >> 6);
        const uint64_t total = (p.ray_count + (1u << kRunShift) - 1) >> kRunShift;
        cursor = 0;
        if (p.wave_runs == 2) {  // one range: its runs follow each other
            const uint64_t per = (p.ray_count + waves - 1) / waves;
            base = wave * per < p.ray_count ? wave * per : p.ray_count;
            jump = uint64_t(1) << kRunShift;
            end = uint32_t(p.ray_count - base < per ? p.ray_count - base : per);
        } else {
            base = wave << kRunShift;
            jump = waves << kRunShift;
            end = wave < total ? uint32_t((total - wave + waves - 1) / waves) << kRunShift : 0u;
        }
        end = uint32_t(__builtin_amdgcn_readfirstlane(int(end)));
    }

    // This lane is idle and rays may be left for it.
    __device__ bool can_take(const TraceParams& p, bool active) const {
        return !active && (runs ? cursor < end : rid < p.ray_count);
    }

    // Called by the whole wave when it hands out rays (takers = ballot of
    // can_take); true when this lane got ray `rid`.
    __device__ bool take(const TraceParams& p, bool me, uint64_t takers) {
        if (!runs) return me;
        // takers in the lanes below this one (v_mbcnt)
        const uint32_t below = __builtin_amdgcn_mbcnt_hi(
            uint32_t(takers >> 32), __builtin_amdgcn_mbcnt_lo(uint32_t(takers), 0u));
        const uint32_t q = cursor + below;
        cursor += uint32_t(__popcll(takers));
        if (cursor > end) cursor = end;
        if (!me || q >= end) return false;
        const uint64_t r =
            base + uint64_t(q >> kRunShift) * jump + (q & ((1u << kRunShift) - 1u));
        if (r >= p.ray_count) return false;  // the last run may be short
        rid = r;
        return true;
    }

    // Called by the whole wave: no lane will take another ray once those in
    // hand (`active`) are done, given that none can now.
    __device__ bool last(const TraceParams& p, bool active) const {
        return runs || __ballot(active && rid + stride < p.ray_count) == 0;
    }

    // The lane's ray is finished (or skipped).
    __device__ void next() {
        if (!runs) rid += stride;
    }
};

}  // namespace rtbvh
