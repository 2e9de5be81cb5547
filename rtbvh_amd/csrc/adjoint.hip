// Adjoint of the ray/triangle hit (no counterpart in the reference, whose
// Moller-Trumbore test, src/builders/spatial_sah.rs:132-163, is forward only).
//
// With the hit triangle fixed by the forward pass, (t, u, v) solves
//     o + t d = (1 - u - v) v0 + u v1 + v v2,   i.e.   M x = s
// with M = [-d | e1 | e2], x = (t, u, v), s = o - v0, e1 = v1 - v0,
// e2 = v2 - v0.  For an upstream gradient g = dL/dx the adjoint is
//     lambda = M^-T g,   dL/ds = lambda,   dL/dM = -lambda x^T,
// which gives
//     dL/do  = lambda                 dL/dd  = t lambda
//     dL/dv0 = -(1 - u - v) lambda    dL/dv1 = -u lambda    dL/dv2 = -v lambda.
// The rows of M^-1 are f (e1 x e2), f (d x e2), f (e1 x d) with f = 1 / a,
// a = e1 . (d x e2) = det M (the same a as the forward test), so
//     lambda = f (g_t (e1 x e2) + g_u (d x e2) + g_v (e1 x d)).
// Ray gradients are written; vertex gradients of triangles hit by several
// rays are summed in any order (the last bits depend on it).
//
// Two forms.  adjoint_kernel adds each ray's nine vertex terms by float
// atomics; the nine scattered atomics of a ray bound it (38 G atomics/s,
// 990 us for 2^22 rays on 100k triangles).  From kBucketRays rays on, the
// terms go through buckets of consecutive triangles instead: tiles of 4096
// rays count their buckets, a scan places the runs, adjoint_records_kernel
// computes each ray's lambda once and writes it with u, v and the triangle
// into the tile's run of its bucket, and adjoint_sum_kernel adds a chunk's
// records into sums in LDS and flushes them bucket by bucket.  2^22 rays on
// 1k / 100k / 1M triangles: 168 / 237 / 388 us against 1471 / 985 / 1591 us;
// of the 237 us the records take 143 (386 MB read and written, 2.7 TB/s), the
// sums 51, counts and scan 35.  The sums' error against 64 bits is no larger:
// fewer terms are added one by one.
#include <algorithm>

#include "block_scan.hpp"
#include "internal.hpp"

namespace rtbvh {

hipError_t scan_exclusive_u32(uint32_t* data, uint32_t count, uint32_t* total, void* scratch,
                              size_t scratch_bytes, hipStream_t stream);
size_t scan_scratch_bytes(uint32_t count);

namespace {

__device__ __forceinline__ void cross3(float ax, float ay, float az, float bx, float by, float bz,
                                       float& cx, float& cy, float& cz) {
    cx = ay * bz - by * az;
    cy = az * bx - bz * ax;
    cz = ax * by - bx * ay;
}

struct AdjointArgs {
    const float* verts;
    uint32_t prim_count;
    const DevRay* rays;
    const DevHit* hits;
    uint64_t ray_count;
    const float *gt, *gu, *gv;  // gradients of t, u, v (null: zero), `step` floats apart
    uint32_t step;
    float *grad_verts, *grad_origin, *grad_dir;
};

// lambda of ray i, its hit and its triangle (prim_count or above: no hit, a
// zero lambda).
struct Lambda {
    float x, y, z, t, u, v;
    uint32_t prim;
};

__device__ __forceinline__ Lambda ray_lambda(const AdjointArgs& a, uint64_t i) {
    const float4 h = reinterpret_cast<const float4*>(a.hits)[i];
    Lambda l;
    l.x = l.y = l.z = 0.f;
    l.t = h.x;
    l.u = h.y;
    l.v = h.z;
    l.prim = __float_as_uint(h.w);
    if (l.prim < a.prim_count) {
        const float4* r4 = reinterpret_cast<const float4*>(a.rays + i);
        const float4 rb = r4[1];
        const float dx = rb.x, dy = rb.y, dz = rb.z;
        const float* p = a.verts + size_t(l.prim) * 9;
        const float e1x = p[3] - p[0], e1y = p[4] - p[1], e1z = p[5] - p[2];
        const float e2x = p[6] - p[0], e2y = p[7] - p[1], e2z = p[8] - p[2];
        float hx, hy, hz, nx, ny, nz, kx, ky, kz;
        cross3(dx, dy, dz, e2x, e2y, e2z, hx, hy, hz);     // d x e2
        cross3(e1x, e1y, e1z, e2x, e2y, e2z, nx, ny, nz);  // e1 x e2
        cross3(e1x, e1y, e1z, dx, dy, dz, kx, ky, kz);     // e1 x d
        const float det = (e1x * hx + e1y * hy) + e1z * hz;
        const float f = 1.0f / det;
        const float gt = a.gt ? a.gt[i * a.step] : 0.f, gu = a.gu ? a.gu[i * a.step] : 0.f,
                    gv = a.gv ? a.gv[i * a.step] : 0.f;
        l.x = f * (gt * nx + gu * hx + gv * kx);
        l.y = f * (gt * ny + gu * hy + gv * ky);
        l.z = f * (gt * nz + gu * hz + gv * kz);
    }
    return l;
}

__device__ __forceinline__ void write_ray_gradients(const AdjointArgs& a, uint64_t i,
                                                    const Lambda& l) {
    if (a.grad_origin) {
        a.grad_origin[i * 3] = l.x;
        a.grad_origin[i * 3 + 1] = l.y;
        a.grad_origin[i * 3 + 2] = l.z;
    }
    if (a.grad_dir) {
        const bool hit = l.prim < a.prim_count;
        a.grad_dir[i * 3] = hit ? l.t * l.x : 0.f;
        a.grad_dir[i * 3 + 1] = hit ? l.t * l.y : 0.f;
        a.grad_dir[i * 3 + 2] = hit ? l.t * l.z : 0.f;
    }
}

// The nine vertex terms of a hit, added to g.
__device__ __forceinline__ void add_vertex_terms(float* g, float lx, float ly, float lz, float u,
                                                 float v) {
    const float w0 = -(1.0f - u - v), w1 = -u, w2 = -v;
    atomicAdd(g + 0, w0 * lx);
    atomicAdd(g + 1, w0 * ly);
    atomicAdd(g + 2, w0 * lz);
    atomicAdd(g + 3, w1 * lx);
    atomicAdd(g + 4, w1 * ly);
    atomicAdd(g + 5, w1 * lz);
    atomicAdd(g + 6, w2 * lx);
    atomicAdd(g + 7, w2 * ly);
    atomicAdd(g + 8, w2 * lz);
}

__global__ void adjoint_kernel(AdjointArgs a) {
    const uint64_t i = uint64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i >= a.ray_count) return;
    const Lambda l = ray_lambda(a, i);
    if (a.grad_verts && l.prim < a.prim_count)
        add_vertex_terms(a.grad_verts + size_t(l.prim) * 9, l.x, l.y, l.z, l.u, l.v);
    write_ray_gradients(a, i, l);
}

// ---- buckets ----------------------------------------------------------------
constexpr int kBlock = 256;
constexpr uint32_t kTileRays = 4096;       // rays a block counts and places
constexpr int kSumBlock = 1024;
constexpr uint32_t kMaxBuckets = 1024;
constexpr uint32_t kMaxBucketPrims = 1024;  // 36 KB of sums in LDS
// Below this many rays the atomics are the faster form: 2^18 rays on 100k /
// 1M triangles 72 / 117 us against 83 / 211 us by buckets, 2^20 rays 270 / 420
// against 100 / 198.
constexpr uint64_t kBucketRays = 1u << 19;
constexpr uint64_t kPassRays = 1u << 22;    // rays per pass: 100 MB of records, within the MALL

// lambda, u, v and the triangle's place in its bucket: 24 bytes, 8-aligned.
struct Record {
    float2 a, b, c;
};

__global__ void __launch_bounds__(kBlock)
    adjoint_count_kernel(AdjointArgs a, uint32_t shift, uint32_t buckets, uint32_t tiles,
                         uint32_t* counts) {
    __shared__ uint32_t s_cnt[kMaxBuckets];
    for (uint32_t k = threadIdx.x; k < buckets; k += kBlock) s_cnt[k] = 0;
    __syncthreads();
    const uint64_t first = uint64_t(blockIdx.x) * kTileRays;
    for (uint32_t k = threadIdx.x; k < kTileRays; k += kBlock) {
        const uint64_t i = first + k;
        if (i >= a.ray_count) break;
        const uint32_t prim = a.hits[i].prim;
        if (prim < a.prim_count) atomicAdd(&s_cnt[prim >> shift], 1u);
    }
    __syncthreads();
    for (uint32_t k = threadIdx.x; k < buckets; k += kBlock)
        counts[size_t(k) * tiles + blockIdx.x] = s_cnt[k];
}

__global__ void __launch_bounds__(kBlock)
    adjoint_records_kernel(AdjointArgs a, uint32_t shift, uint32_t buckets, uint32_t tiles,
                           const uint32_t* offsets, Record* records) {
    __shared__ uint32_t s_next[kMaxBuckets];
    for (uint32_t k = threadIdx.x; k < buckets; k += kBlock)
        s_next[k] = offsets[size_t(k) * tiles + blockIdx.x];
    __syncthreads();
    const uint64_t first = uint64_t(blockIdx.x) * kTileRays;
    for (uint32_t k = threadIdx.x; k < kTileRays; k += kBlock) {
        const uint64_t i = first + k;
        if (i >= a.ray_count) break;
        const Lambda l = ray_lambda(a, i);
        write_ray_gradients(a, i, l);
        if (l.prim >= a.prim_count) continue;
        const uint32_t at = atomicAdd(&s_next[l.prim >> shift], 1u);
        Record r;
        r.a = make_float2(l.x, l.y);
        r.b = make_float2(l.z, l.u);
        r.c = make_float2(l.v, __uint_as_float(l.prim & ((1u << shift) - 1u)));
        records[at] = r;
    }
}

// Sum over the 8 lanes of a group, in every lane.
template <int CTRL>
__device__ __forceinline__ float dpp_get(float x) {
    return __uint_as_float(uint32_t(
        __builtin_amdgcn_update_dpp(0, int(__float_as_uint(x)), CTRL, 0xF, 0xF, true)));
}
__device__ __forceinline__ float sum8(float x) {
    x += dpp_get<0xB1>(x);   // quad_perm: the lane's pair
    x += dpp_get<0x4E>(x);   // quad_perm: the other pair
    x += dpp_get<0x141>(x);  // row_half_mirror: the other quad
    return x;
}

// Records [first, first + chunk) of the bucket-ordered array, bucket by
// bucket, kSubChunk at a time: the records are placed in LDS in the order of
// their triangles (a count, a scan, a scatter), a group of 8 lanes sums each
// triangle's nine terms, and a bucket's sums, kept in LDS by their groups, are
// added to the gradients at its end.  By atomics, also where the chunk holds
// the whole bucket: calls on other streams may be adding to the same
// gradients (rtbvh_gpu_adjoint accumulates), in either form.  Adding the terms
// by LDS atomics instead (nine a record) took 195 us for 2^22 records, 51 us
// this way.
constexpr uint32_t kSubChunk = 2 * kSumBlock;

__global__ void __launch_bounds__(kSumBlock)
    adjoint_sum_kernel(AdjointArgs a, uint32_t shift, uint32_t buckets, uint32_t tiles,
                       const uint32_t* offsets, const uint32_t* total, const Record* records,
                       uint32_t chunk) {
    extern __shared__ float s_sum[];  // 9 per triangle of a bucket
    __shared__ float s_x[kSubChunk], s_y[kSubChunk], s_z[kSubChunk], s_u[kSubChunk],
        s_v[kSubChunk];
    __shared__ uint32_t s_first[kMaxBucketPrims + 1];  // counts, then first places
    __shared__ uint32_t s_scan[kSumBlock / 64];
    const uint32_t count = *total;
    const uint32_t first = blockIdx.x * chunk;
    if (first >= count) return;  // whole block
    const uint32_t end = count - first < chunk ? count : first + chunk;
    const uint32_t prims = 1u << shift;
    const uint32_t lane8 = threadIdx.x & 7u, group = threadIdx.x >> 3;
    // the bucket that holds record `first`: the last that starts at or below it
    uint32_t lo = 0, hi = buckets;
    while (hi - lo > 1) {
        const uint32_t mid = (lo + hi) >> 1;
        if (offsets[size_t(mid) * tiles] <= first)
            lo = mid;
        else
            hi = mid;
    }
    uint32_t at = first;
    for (uint32_t b = lo; b < buckets && at < end; ++b) {
        const uint32_t next = b + 1 < buckets ? offsets[size_t(b + 1) * tiles] : count;
        const uint32_t stop = next < end ? next : end;
        if (stop <= at) continue;  // an empty bucket
        for (uint32_t k = threadIdx.x; k < prims * 9; k += kSumBlock) s_sum[k] = 0.f;
        for (; at < stop; at += kSubChunk) {
            const uint32_t m = stop - at < kSubChunk ? stop - at : kSubChunk;
            if (threadIdx.x < prims) s_first[threadIdx.x] = 0;
            __syncthreads();
            Record r[2];
            uint32_t prim[2], rank[2];
#pragma unroll
            for (uint32_t q = 0; q < 2; ++q) {
                const uint32_t k = threadIdx.x + q * kSumBlock;
                if (k < m) {
                    r[q] = records[at + k];
                    prim[q] = __float_as_uint(r[q].c.y);
                    rank[q] = atomicAdd(&s_first[prim[q]], 1u);
                }
            }
            __syncthreads();
            const uint32_t mine = threadIdx.x < prims ? s_first[threadIdx.x] : 0u;
            const uint32_t excl = block_exclusive_n<kSumBlock>(mine, s_scan, nullptr);
            if (threadIdx.x < prims) s_first[threadIdx.x] = excl;
            if (threadIdx.x == 0) s_first[prims] = m;
            __syncthreads();
#pragma unroll
            for (uint32_t q = 0; q < 2; ++q)
                if (threadIdx.x + q * kSumBlock < m) {
                    const uint32_t to = s_first[prim[q]] + rank[q];
                    s_x[to] = r[q].a.x;
                    s_y[to] = r[q].a.y;
                    s_z[to] = r[q].b.x;
                    s_u[to] = r[q].b.y;
                    s_v[to] = r[q].c.x;
                }
            __syncthreads();
            for (uint32_t p = group; p < prims; p += kSumBlock / 8) {
                float g[9] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
                const uint32_t p0 = s_first[p], p1 = s_first[p + 1];
                for (uint32_t k = p0 + lane8; k < p1; k += 8) {
                    const float lx = s_x[k], ly = s_y[k], lz = s_z[k], u = s_u[k], v = s_v[k];
                    const float w0 = -(1.0f - u - v), w1 = -u, w2 = -v;
                    g[0] += w0 * lx;
                    g[1] += w0 * ly;
                    g[2] += w0 * lz;
                    g[3] += w1 * lx;
                    g[4] += w1 * ly;
                    g[5] += w1 * lz;
                    g[6] += w2 * lx;
                    g[7] += w2 * ly;
                    g[8] += w2 * lz;
                }
                if (p0 == p1) continue;  // the same for the group's lanes
#pragma unroll
                for (int c = 0; c < 9; ++c) {
                    const float t = sum8(g[c]);
                    if (lane8 == uint32_t(c & 7)) s_sum[p * 9 + c] += t;
                }
            }
            __syncthreads();
        }
        at = stop;
        float* g = a.grad_verts + size_t(b) * prims * 9;
        const uint32_t own = a.prim_count - b * prims < prims ? a.prim_count - b * prims : prims;
        for (uint32_t k = threadIdx.x; k < own * 9; k += kSumBlock) {
            const float t = s_sum[k];
            if (t != 0.f) atomicAdd(g + k, t);
        }
        __syncthreads();
    }
}

size_t align256(size_t b) { return (b + 255) & ~size_t(255); }

// The bucket form over at most kPassRays rays at a time; false when it does
// not apply and nothing was launched (few rays, more triangles than the
// buckets hold, a capturing stream, no workspace).
bool launch_buckets(const AdjointArgs& all, hipStream_t stream, hipError_t* result) {
    if (!all.grad_verts || all.ray_count < kBucketRays || all.prim_count == 0 ||
        all.prim_count > kMaxBuckets * kMaxBucketPrims)
        return false;
    // the workspace is handed on by events, which a recorded graph must not hold
    hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(stream, &cap) != hipSuccess || cap != hipStreamCaptureStatusNone) {
        (void)hipGetLastError();
        return false;
    }
    // small buckets, so that most are flushed by one block
    uint32_t shift = 6;
    while ((all.prim_count + (1u << shift) - 1) >> shift > kMaxBuckets) ++shift;
    const uint32_t buckets = (all.prim_count + (1u << shift) - 1) >> shift;
    const uint64_t pass = std::min(all.ray_count, kPassRays);
    const uint32_t tiles = uint32_t((pass + kTileRays - 1) / kTileRays);
    const size_t sz_rec = align256(size_t(pass) * sizeof(Record));
    const size_t sz_cnt = align256(size_t(buckets) * tiles * 4);
    const size_t sz_scan = align256(scan_scratch_bytes(buckets * tiles));
    Workspace ws;
    if (workspace_acquire_on(kWsAdjoint, sz_rec + sz_cnt + sz_scan + 256, stream, &ws) !=
        hipSuccess) {
        (void)hipGetLastError();
        return false;
    }
    char* base = static_cast<char*>(ws.ptr);
    Record* records = reinterpret_cast<Record*>(base);
    uint32_t* counts = reinterpret_cast<uint32_t*>(base + sz_rec);
    void* scan = base + sz_rec + sz_cnt;
    uint32_t* total = reinterpret_cast<uint32_t*>(base + sz_rec + sz_cnt + sz_scan);
    hipError_t e = hipSuccess;
    for (uint64_t at = 0; at < all.ray_count && e == hipSuccess; at += pass) {
        AdjointArgs a = all;
        a.ray_count = std::min(pass, all.ray_count - at);
        a.rays += at;
        a.hits += at;
        if (a.gt) a.gt += at * a.step;
        if (a.gu) a.gu += at * a.step;
        if (a.gv) a.gv += at * a.step;
        if (a.grad_origin) a.grad_origin += at * 3;
        if (a.grad_dir) a.grad_dir += at * 3;
        const uint32_t t = uint32_t((a.ray_count + kTileRays - 1) / kTileRays);
        hipLaunchKernelGGL(adjoint_count_kernel, dim3(t), dim3(kBlock), 0, stream, a, shift,
                           buckets, t, counts);
        e = scan_exclusive_u32(counts, buckets * t, total, scan, sz_scan, stream);
        if (e != hipSuccess) break;
        hipLaunchKernelGGL(adjoint_records_kernel, dim3(t), dim3(kBlock), 0, stream, a, shift,
                           buckets, t, counts, records);
        // 1024 to 8192 records a block, 512 blocks or more: two a CU, but one where a
        // bucket's sums take 36 KB beside the 45 KB of records (above 524,288 triangles)
        const uint32_t chunk =
            uint32_t(std::min<uint64_t>(8192, std::max<uint64_t>(1024, a.ray_count / 512)));
        hipLaunchKernelGGL(adjoint_sum_kernel, dim3(uint32_t((a.ray_count + chunk - 1) / chunk)),
                           dim3(kSumBlock), (size_t(9) << shift) * sizeof(float), stream, a, shift,
                           buckets, t, counts, total, records, chunk);
        e = hipGetLastError();
    }
    workspace_release_on(&ws, stream);  // the next user waits for this call's work
    *result = e;
    return true;
}

}  // namespace

hipError_t launch_adjoint(const float* verts, uint32_t prim_count, const DevRay* rays,
                          const DevHit* hits, uint64_t ray_count, const float* grad_t,
                          const float* grad_u, const float* grad_v, uint32_t grad_step,
                          float* grad_verts, float* grad_origin, float* grad_dir,
                          hipStream_t stream) {
    if (ray_count == 0) return hipSuccess;
    const AdjointArgs a{verts,     prim_count, rays,   hits,      ray_count,  grad_t,
                        grad_u,    grad_v,     grad_step, grad_verts, grad_origin, grad_dir};
    hipError_t e = hipSuccess;
    if (launch_buckets(a, stream, &e)) return e;
    const uint64_t blocks = (ray_count + 255) / 256;
    hipLaunchKernelGGL(adjoint_kernel, dim3(uint32_t(blocks)), dim3(256), 0, stream, a);
    return hipGetLastError();
}

}  // namespace rtbvh
