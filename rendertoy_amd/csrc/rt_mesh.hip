// rt_mesh.hip — mesh data on the device. Per-vertex normals: Mesh.compute_normals
// (rendering/_modeling.py:48-49, a stub in the reference that raises "Not implemented yet").
//
// Definition (area-weighted vertex normals):
//   n(v) = sum of cross(P1 - P0, P2 - P0) over the (triangle t, corner k) pairs with idx[t][k] == v,
//          added in the order k = 0, 1, 2 and, within k, ascending t, starting from +0;
//   N(v) = n(v) / d, d = sqrt((x*x + y*y) + z*z) raised to 1e-300 (a NaN d stays NaN).
// Everything is FP64 from the FP32 positions, rounded once to FP32, so N is a fixed function of the
// mesh: the sum order is fixed by the pairs' numbers p = k * n_tris + t, not by scheduling.
// Vertices that no triangle uses get (0, 0, 0). Out-of-range indices are clamped to n_vertices - 1,
// as the scene build does.
//
// Pipeline (one stream): a counting placement of the pairs by vertex, whose runs are in arrival
// order, each put in order where it is summed. (Before, a stable radix sort of the pairs by vertex
// fixed the order: 133 of 219 us at 1.31 M triangles, 0.66 M vertices; now 82 us: face 34,
// scan 11, place 15, vertex 16.)
//   1. k_nrm_face   per triangle: FP64 face normal (32 B record); per pair its arrival number among
//                   its vertex's pairs (an integer atomic on the vertex's count).
//   2. k_nrm_sums, k_nrm_offsets   exclusive scan of the counts: each vertex's run in `run`; vertices
//                   of more than kSmallRun pairs are listed.
//   3. k_nrm_place  run[offset of its vertex + arrival] = p for every pair.
//   4. k_nrm_big    sorts the listed runs (none in most meshes).
//   5. k_nrm_vertex per vertex: its run in ascending p (up to 8 pairs by a sorting network in
//                   registers), the FP64 sum, float3 N at out + v * out_stride.
// A non-indexed mesh (vertices 3t, 3t+1, 3t+2) has one pair per vertex: k_nrm_direct computes it
// with no sort and no workspace.
//
// Also here: MeshVertex records <-> dense float arrays (k_mesh_pack / k_mesh_unpack), the device-side
// ingest and export of the 80-byte vertex layout of rendering/_modeling.py:22-28.
#include <cmath>

#include "rt_common.h"

namespace rt {
namespace {

constexpr uint32_t kSmallRun = 64;     // longest run k_nrm_vertex puts in order by itself
constexpr uint32_t kLdsRun = 4096;     // longest run k_nrm_big sorts in LDS
constexpr uint32_t kScanChunk = 2048;  // counts per workgroup of the scan

struct NrmWorkspace {
    double4* face;    // n_tris
    uint32_t* rank;   // 3 n_tris: arrival number of pair p
    uint32_t* run;    // 3 n_tris: the pairs by vertex
    uint32_t* count;  // n_vertices, then the number of listed vertices
    uint32_t* off;    // n_vertices
    uint32_t* sums;   // per scan chunk
    uint32_t* big;    // listed vertices
    uint64_t bytes;
};

inline uint64_t align256n(uint64_t x) { return (x + 255) & ~uint64_t(255); }

NrmWorkspace carve_nrm(char* base, uint64_t n_vertices, uint64_t n_tris) {
    NrmWorkspace w{};
    const uint64_t np = 3 * n_tris;
    uint64_t off = 0;
    auto take = [&](uint64_t bytes) {
        char* p = base ? base + off : nullptr;
        off = align256n(off + (bytes ? bytes : 4));
        return p;
    };
    w.face = (double4*)take(32 * n_tris);
    w.rank = (uint32_t*)take(4 * np);
    w.run = (uint32_t*)take(4 * np);
    w.count = (uint32_t*)take(4 * (n_vertices + 1));
    w.off = (uint32_t*)take(4 * n_vertices);
    w.sums = (uint32_t*)take(4 * ((n_vertices + kScanChunk - 1) / kScanChunk));
    w.big = (uint32_t*)take(4 * (np / kSmallRun + 1));
    w.bytes = off;
    return w;
}

RT_DEV double3 load_p64(const char* vb, uint32_t i, uint32_t stride, uint32_t off) {
    const float* p = (const float*)(vb + (uint64_t)i * stride + off);
    return make_double3((double)p[0], (double)p[1], (double)p[2]);
}

RT_DEV uint32_t clamp_index(int32_t i, uint32_t nv) {
    const uint32_t u = (uint32_t)i;
    return u < nv ? u : nv - 1;
}

// cross(b - a, c - a) in FP64 (no contraction: the library is built with -ffp-contract=off)
RT_DEV double3 face_normal(const double3 a, const double3 b, const double3 c) {
    const double e1x = b.x - a.x, e1y = b.y - a.y, e1z = b.z - a.z;
    const double e2x = c.x - a.x, e2y = c.y - a.y, e2z = c.z - a.z;
    return make_double3(e1y * e2z - e1z * e2y, e1z * e2x - e1x * e2z, e1x * e2y - e1y * e2x);
}

RT_DEV void store_normal(char* out, uint32_t v, uint32_t stride, double x, double y, double z) {
    const double sq = (x * x + y * y) + z * z;
    double d = sqrt(sq);
    d = d < 1e-300 ? 1e-300 : d;  // a NaN d is kept
    float* o = (float*)(out + (uint64_t)v * stride);
    o[0] = (float)(x / d);
    o[1] = (float)(y / d);
    o[2] = (float)(z / d);
}

__global__ void __launch_bounds__(256) k_nrm_clear(uint32_t* __restrict__ count, uint64_t n) {
    const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) count[i] = 0;
}

__global__ void __launch_bounds__(256) k_nrm_face(rt_mesh_desc m, double4* __restrict__ face,
                                                   uint32_t* __restrict__ count,
                                                   uint32_t* __restrict__ rank) {
    const uint32_t t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= m.n_tris) return;
    const char* vb = (const char*)m.vertices;
    const uint32_t i0 = clamp_index(m.indices[3 * (uint64_t)t], m.n_vertices);
    const uint32_t i1 = clamp_index(m.indices[3 * (uint64_t)t + 1], m.n_vertices);
    const uint32_t i2 = clamp_index(m.indices[3 * (uint64_t)t + 2], m.n_vertices);
    const uint32_t T = m.n_tris;
    rank[t] = atomicAdd(&count[i0], 1u);
    rank[T + t] = atomicAdd(&count[i1], 1u);
    rank[2 * T + t] = atomicAdd(&count[i2], 1u);
    const double3 f = face_normal(load_p64(vb, i0, m.vertex_stride, m.pos_offset),
                                  load_p64(vb, i1, m.vertex_stride, m.pos_offset),
                                  load_p64(vb, i2, m.vertex_stride, m.pos_offset));
    face[t] = make_double4(f.x, f.y, f.z, 0.0);
}

// Sum of one value per thread over a workgroup of 256, in every thread.
RT_DEV uint32_t block_sum(uint32_t v, uint32_t* lds) {
    for (int d = 32; d > 0; d >>= 1) v += __shfl_xor(v, d);
    if ((threadIdx.x & 63u) == 0) lds[threadIdx.x >> 6] = v;
    __syncthreads();
    const uint32_t s = lds[0] + lds[1] + lds[2] + lds[3];
    __syncthreads();
    return s;
}

// sums[b] = the counts of chunk b
__global__ void __launch_bounds__(256) k_nrm_sums(const uint32_t* __restrict__ count, uint32_t n,
                                                   uint32_t* __restrict__ sums) {
    __shared__ uint32_t lds[4];
    const uint64_t base = (uint64_t)blockIdx.x * kScanChunk;
    uint32_t v = 0;
    for (uint32_t k = threadIdx.x; k < kScanChunk; k += 256u) v += base + k < n ? count[base + k] : 0u;
    v = block_sum(v, lds);
    if (threadIdx.x == 0) sums[blockIdx.x] = v;
}

// Exclusive scan of the chunk sums in place, one workgroup: for more chunks than every chunk's
// workgroup should add up again (kSumChunks; 2 M vertices).
constexpr uint32_t kSumChunks = 1024;

__global__ void __launch_bounds__(1024) k_nrm_scan_sums(uint32_t* __restrict__ sums, uint32_t chunks) {
    __shared__ uint32_t scan[1024];
    uint32_t carry = 0;
    for (uint32_t b = 0; b < chunks; b += 1024u) {
        const uint32_t i = b + threadIdx.x, v = i < chunks ? sums[i] : 0u;
        scan[threadIdx.x] = v;
        __syncthreads();
        for (uint32_t d = 1; d < 1024; d <<= 1) {
            const uint32_t x = threadIdx.x >= d ? scan[threadIdx.x - d] : 0u;
            __syncthreads();
            scan[threadIdx.x] += x;
            __syncthreads();
        }
        if (i < chunks) sums[i] = carry + scan[threadIdx.x] - v;
        carry += scan[1023];
        __syncthreads();
    }
}

// off[i] = the counts before i (the chunks before from their sums, or, `scanned`, from their scan);
// vertices of long runs are listed
__global__ void __launch_bounds__(256) k_nrm_offsets(const uint32_t* __restrict__ count, uint32_t n,
                                                      const uint32_t* __restrict__ sums, bool scanned,
                                                      uint32_t* __restrict__ off, uint32_t* __restrict__ n_big,
                                                      uint32_t* __restrict__ big) {
    constexpr uint32_t kPer = kScanChunk / 256;
    __shared__ uint32_t lds[4], scan[256];
    uint32_t before = 0;
    if (scanned) {
        before = sums[blockIdx.x];
    } else {
        for (uint32_t b = threadIdx.x; b < blockIdx.x; b += 256u) before += sums[b];
        before = block_sum(before, lds);
    }
    const uint64_t base = (uint64_t)blockIdx.x * kScanChunk + threadIdx.x * kPer;
    uint32_t c[kPer], sum = 0;
#pragma unroll
    for (uint32_t k = 0; k < kPer; ++k) {
        c[k] = base + k < n ? count[base + k] : 0u;
        sum += c[k];
    }
    scan[threadIdx.x] = sum;
    __syncthreads();
    for (uint32_t d = 1; d < 256; d <<= 1) {
        const uint32_t x = threadIdx.x >= d ? scan[threadIdx.x - d] : 0u;
        __syncthreads();
        scan[threadIdx.x] += x;
        __syncthreads();
    }
    uint32_t at = before + scan[threadIdx.x] - sum;
#pragma unroll
    for (uint32_t k = 0; k < kPer; ++k) {
        if (base + k < n) {
            off[base + k] = at;
            if (c[k] > kSmallRun) big[atomicAdd(n_big, 1u)] = (uint32_t)(base + k);
        }
        at += c[k];
    }
}

__global__ void __launch_bounds__(256) k_nrm_place(rt_mesh_desc m, const uint32_t* __restrict__ off,
                                                    const uint32_t* __restrict__ rank,
                                                    uint32_t* __restrict__ run) {
    const uint32_t t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= m.n_tris) return;
    const uint32_t T = m.n_tris;
#pragma unroll
    for (uint32_t k = 0; k < 3; ++k) {
        const uint32_t v = clamp_index(m.indices[3 * (uint64_t)t + k], m.n_vertices), p = k * T + t;
        run[off[v] + rank[p]] = p;
    }
}

// Sorts the runs of the listed vertices, one workgroup each: a bitonic sort in LDS, or, past its size,
// the vertex's pairs collected again in order from the index list.
__global__ void __launch_bounds__(1024) k_nrm_big(rt_mesh_desc m, const uint32_t* __restrict__ n_big,
                                                   const uint32_t* __restrict__ big,
                                                   const uint32_t* __restrict__ count,
                                                   const uint32_t* __restrict__ off, uint32_t* __restrict__ run) {
    __shared__ uint32_t key[kLdsRun];
    __shared__ uint32_t waves[16];
    const uint32_t n = *n_big, tid = threadIdx.x;
    for (uint32_t b = blockIdx.x; b < n; b += gridDim.x) {
        const uint32_t v = big[b], len = count[v];
        uint32_t* out = run + off[v];
        __syncthreads();  // before the last vertex's LDS is written again
        if (len <= kLdsRun) {
            uint32_t pow2 = 1;
            while (pow2 < len) pow2 <<= 1;
            for (uint32_t i = tid; i < pow2; i += 1024u) key[i] = i < len ? out[i] : 0xFFFFFFFFu;
            for (uint32_t k = 2; k <= pow2; k <<= 1) {
                for (uint32_t d = k >> 1; d > 0; d >>= 1) {
                    __syncthreads();
                    for (uint32_t i = tid; i < pow2; i += 1024u) {
                        const uint32_t x = i ^ d;
                        if (x <= i) continue;
                        const uint32_t lo = key[i], hi = key[x];
                        if ((lo > hi) == ((i & k) == 0)) {
                            key[i] = hi;
                            key[x] = lo;
                        }
                    }
                }
            }
            __syncthreads();
            for (uint32_t i = tid; i < len; i += 1024u) out[i] = key[i];
            continue;
        }
        uint32_t done = 0;  // the same in every thread
        for (uint32_t k = 0; k < 3; ++k) {
            for (uint32_t t0 = 0; t0 < m.n_tris; t0 += 1024u) {
                const uint32_t t = t0 + tid;
                const bool mine = t < m.n_tris && clamp_index(m.indices[3 * (uint64_t)t + k], m.n_vertices) == v;
                const uint64_t mask = __ballot(mine);
                if ((tid & 63u) == 0) waves[tid >> 6] = (uint32_t)__popcll(mask);
                __syncthreads();
                uint32_t at = done, all = 0;
                for (uint32_t w = 0; w < 16u; ++w) {
                    at += w < (tid >> 6) ? waves[w] : 0u;
                    all += waves[w];
                }
                at += __builtin_amdgcn_mbcnt_hi((uint32_t)(mask >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)mask, 0u));
                if (mine) out[at] = k * m.n_tris + t;
                done += all;
                __syncthreads();
            }
        }
    }
}

// Bound by the gathers of the face records (32 B a pair, from all over the list): the 8 of a small run
// are all in flight before the first sum.
__global__ void __launch_bounds__(256) k_nrm_vertex(const uint32_t* __restrict__ count,
                                                     const uint32_t* __restrict__ off,
                                                     const uint32_t* __restrict__ run, uint32_t n_tris,
                                                     const double4* __restrict__ face,
                                                     uint32_t n_vertices, char* __restrict__ out,
                                                     uint32_t out_stride) {
    const uint32_t v = blockIdx.x * blockDim.x + threadIdx.x;
    if (v >= n_vertices) return;
    const uint32_t n = count[v];
    if (n == 0) {
        float* o = (float*)(out + (uint64_t)v * out_stride);
        o[0] = 0.0f;
        o[1] = 0.0f;
        o[2] = 0.0f;
        return;
    }
    const uint32_t* r = run + off[v];
    auto tri = [&](uint32_t p) { return p >= 2 * n_tris ? p - 2 * n_tris : (p >= n_tris ? p - n_tris : p); };
    double x = 0.0, y = 0.0, z = 0.0;
    if (n <= 8) {
        uint32_t p[8];
#pragma unroll
        for (uint32_t j = 0; j < 8; ++j) p[j] = j < n ? r[j] : 0xFFFFFFFFu;
        auto order = [&](int a, int b) {
            const uint32_t lo = p[a] < p[b] ? p[a] : p[b], hi = p[a] < p[b] ? p[b] : p[a];
            p[a] = lo;
            p[b] = hi;
        };
        // Batcher's odd-even merge sort of 8
        order(0, 1); order(2, 3); order(4, 5); order(6, 7);
        order(0, 2); order(1, 3); order(4, 6); order(5, 7);
        order(1, 2); order(5, 6);
        order(0, 4); order(1, 5); order(2, 6); order(3, 7);
        order(2, 4); order(3, 5);
        order(1, 2); order(3, 4); order(5, 6);
        double4 f[8];
#pragma unroll
        for (uint32_t j = 0; j < 8; ++j)
            if (j < n) f[j] = face[tri(p[j])];
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (uint32_t j = 0; j < 8; ++j) {
            if (j < n) {
                x = x + f[j].x;
                y = y + f[j].y;
                z = z + f[j].z;
            }
        }
    } else {
        uint32_t last = 0;
        for (uint32_t j = 0; j < n; ++j) {
            uint32_t p = r[j];
            if (n <= kSmallRun) {  // the smallest pair past the last one
                p = 0xFFFFFFFFu;
                for (uint32_t i = 0; i < n; ++i) {
                    const uint32_t q = r[i];
                    p = (j == 0 || q > last) && q < p ? q : p;
                }
                last = p;
            }
            const double4 f = face[tri(p)];
            x = x + f.x;
            y = y + f.y;
            z = z + f.z;
        }
    }
    store_normal(out, v, out_stride, x, y, z);
}

// Non-indexed mesh: vertex v < 3 n_tris is corner v % 3 of triangle v / 3, its only pair.
__global__ void __launch_bounds__(256) k_nrm_direct(rt_mesh_desc m, char* __restrict__ out,
                                                     uint32_t out_stride) {
    const uint32_t v = blockIdx.x * blockDim.x + threadIdx.x;
    if (v >= m.n_vertices) return;
    if (v >= 3 * (uint64_t)m.n_tris) {
        float* o = (float*)(out + (uint64_t)v * out_stride);
        o[0] = 0.0f;
        o[1] = 0.0f;
        o[2] = 0.0f;
        return;
    }
    const uint32_t t0 = v - v % 3u;
    const char* vb = (const char*)m.vertices;
    const double3 f = face_normal(load_p64(vb, t0, m.vertex_stride, m.pos_offset),
                                  load_p64(vb, t0 + 1, m.vertex_stride, m.pos_offset),
                                  load_p64(vb, t0 + 2, m.vertex_stride, m.pos_offset));
    store_normal(out, v, out_stride, 0.0 + f.x, 0.0 + f.y, 0.0 + f.z);
}

// MeshVertex records (80 B: P@0, N@16, C@32, T@48, B@64, float3 fields padded to 16 B) from
// dense float arrays; absent attributes, T, B and the pad words are written as zero. A wave writes
// the 64 records of its vertices as 320 consecutive 16-byte chunks, lane l taking chunks l + 64j,
// so each store instruction covers 1 KiB of contiguous output; chunk c is field c % 5 of vertex
// c / 5.
__global__ void __launch_bounds__(256) k_mesh_pack(const float* __restrict__ pos,
                                                    const float* __restrict__ nrm,
                                                    const float* __restrict__ uv, uint32_t n,
                                                    float4* __restrict__ rec) {
    const uint32_t lane = threadIdx.x & 63u;
    const uint64_t v0 = (uint64_t)blockIdx.x * blockDim.x + (threadIdx.x & ~63u);  // the wave's first vertex
    if (v0 >= n) return;
    const uint32_t nw = n - v0 < 64 ? (uint32_t)(n - v0) : 64u;
#pragma unroll
    for (uint32_t j = 0; j < 5; ++j) {
        const uint32_t c = lane + 64u * j, vl = c / 5u, f = c - 5u * vl;
        if (vl >= nw) break;
        const uint64_t v = v0 + vl;
        float4 x = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        if (f == 0) {
            x = make_float4(pos[3 * v], pos[3 * v + 1], pos[3 * v + 2], 0.0f);
        } else if (f == 1) {
            if (nrm) x = make_float4(nrm[3 * v], nrm[3 * v + 1], nrm[3 * v + 2], 0.0f);
        } else if (f == 2) {
            if (uv) x = make_float4(uv[2 * v], uv[2 * v + 1], 0.0f, 0.0f);
        }
        rec[5 * v0 + c] = x;
    }
}

// Dense P / N / C arrays out of MeshVertex records (any output may be NULL).
__global__ void __launch_bounds__(256) k_mesh_unpack(const float4* __restrict__ rec, uint32_t n,
                                                      float* __restrict__ pos,
                                                      float* __restrict__ nrm,
                                                      float* __restrict__ uv) {
    const uint32_t v = blockIdx.x * blockDim.x + threadIdx.x;
    if (v >= n) return;
    const uint64_t i3 = 3 * (uint64_t)v, i2 = 2 * (uint64_t)v;
    const float4* r = rec + 5 * (uint64_t)v;
    if (pos) {
        const float4 a = r[0];
        pos[i3] = a.x;
        pos[i3 + 1] = a.y;
        pos[i3 + 2] = a.z;
    }
    if (nrm) {
        const float4 b = r[1];
        nrm[i3] = b.x;
        nrm[i3 + 1] = b.y;
        nrm[i3 + 2] = b.z;
    }
    if (uv) {
        const float4 c = r[2];
        uv[i2] = c.x;
        uv[i2 + 1] = c.y;
    }
}

inline uint32_t nblocks(uint64_t n, uint32_t per) { return (uint32_t)((n + per - 1) / per); }

}  // namespace
}  // namespace rt

using namespace rt;

extern "C" uint64_t rt_mesh_normals_workspace_bytes(uint32_t n_vertices, uint32_t n_tris) {
    return carve_nrm(nullptr, n_vertices, n_tris).bytes;
}

extern "C" int rt_mesh_compute_normals(const rt_mesh_desc* mesh, float* normals_out,
                                       uint32_t out_stride, void* workspace, uint64_t ws_bytes,
                                       void* stream) {
    if (!mesh) return set_error(RT_EINVAL, "rt_mesh_compute_normals: mesh is NULL");
    const rt_mesh_desc& m = *mesh;
    if (m.n_vertices == 0) {
        if (m.n_tris) return set_error(RT_EINVAL, "rt_mesh_compute_normals: mesh has no vertices");
        return RT_OK;
    }
    if (!m.vertices) return set_error(RT_EINVAL, "rt_mesh_compute_normals: mesh vertices NULL");
    if (m.vertex_stride < 12 || (m.vertex_stride & 3) || (m.pos_offset & 3) ||
        m.pos_offset + 12 > m.vertex_stride)
        return set_error(RT_EINVAL, "rt_mesh_compute_normals: bad vertex stride/position offset");
    if (!m.indices && (uint64_t)m.n_tris * 3 > m.n_vertices)
        return set_error(RT_EINVAL, "rt_mesh_compute_normals: non-indexed mesh needs 3 vertices per triangle");
    if ((uint64_t)m.n_tris * 3 > 0xFFFFFFFFull)
        return set_error(RT_ECAPACITY, "rt_mesh_compute_normals: too many triangles");
    if (!normals_out) return set_error(RT_EINVAL, "rt_mesh_compute_normals: normals_out is NULL");
    if (out_stride < 12 || (out_stride & 3) || ((uintptr_t)normals_out & 3))
        return set_error(RT_EINVAL, "rt_mesh_compute_normals: output must be 4-byte aligned with stride >= 12");
    hipStream_t s = (hipStream_t)stream;
    char* out = (char*)normals_out;
    if (!m.indices) {
        hipLaunchKernelGGL(k_nrm_direct, dim3(nblocks(m.n_vertices, 256)), dim3(256), 0, s, m, out,
                           out_stride);
        return check_launch("rt_mesh_compute_normals");
    }
    const NrmWorkspace need = carve_nrm(nullptr, m.n_vertices, m.n_tris);
    if (!workspace || ws_bytes < need.bytes)
        return set_error(RT_EINVAL, "rt_mesh_compute_normals: workspace too small (need " +
                                        std::to_string(need.bytes) + " bytes)");
    if ((uintptr_t)workspace & 255)
        return set_error(RT_EINVAL, "rt_mesh_compute_normals: workspace must be 256-byte aligned");
    NrmWorkspace w = carve_nrm((char*)workspace, m.n_vertices, m.n_tris);
    const uint32_t chunks = nblocks(m.n_vertices, kScanChunk);
    uint32_t* n_big = w.count + m.n_vertices;
    hipLaunchKernelGGL(k_nrm_clear, dim3(nblocks((uint64_t)m.n_vertices + 1, 256)), dim3(256), 0, s, w.count,
                       (uint64_t)m.n_vertices + 1);
    if (m.n_tris)
        hipLaunchKernelGGL(k_nrm_face, dim3(nblocks(m.n_tris, 256)), dim3(256), 0, s, m, w.face, w.count, w.rank);
    hipLaunchKernelGGL(k_nrm_sums, dim3(chunks), dim3(256), 0, s, w.count, m.n_vertices, w.sums);
    const bool scanned = chunks > kSumChunks;
    if (scanned) hipLaunchKernelGGL(k_nrm_scan_sums, dim3(1), dim3(1024), 0, s, w.sums, chunks);
    hipLaunchKernelGGL(k_nrm_offsets, dim3(chunks), dim3(256), 0, s, w.count, m.n_vertices, w.sums, scanned, w.off,
                       n_big, w.big);
    if (m.n_tris) {
        hipLaunchKernelGGL(k_nrm_place, dim3(nblocks(m.n_tris, 256)), dim3(256), 0, s, m, w.off, w.rank, w.run);
        if (3 * (uint64_t)m.n_tris > kSmallRun)
            hipLaunchKernelGGL(k_nrm_big, dim3(64), dim3(1024), 0, s, m, n_big, w.big, w.count, w.off, w.run);
    }
    hipLaunchKernelGGL(k_nrm_vertex, dim3(nblocks(m.n_vertices, 256)), dim3(256), 0, s, w.count, w.off, w.run,
                       m.n_tris, w.face, m.n_vertices, out, out_stride);
    return check_launch("rt_mesh_compute_normals");
}

extern "C" int rt_mesh_pack(const float* pos, const float* nrm, const float* uv, uint32_t n_vertices,
                            void* records, void* stream) {
    if (n_vertices == 0) return RT_OK;
    if (!pos || !records) return set_error(RT_EINVAL, "rt_mesh_pack: positions and records are required");
    if (((uintptr_t)pos | (uintptr_t)nrm | (uintptr_t)uv) & 3)
        return set_error(RT_EINVAL, "rt_mesh_pack: arrays must be 4-byte aligned");
    if ((uintptr_t)records & 15) return set_error(RT_EINVAL, "rt_mesh_pack: records must be 16-byte aligned");
    hipLaunchKernelGGL(k_mesh_pack, dim3(nblocks(n_vertices, 256)), dim3(256), 0, (hipStream_t)stream,
                       pos, nrm, uv, n_vertices, (float4*)records);
    return check_launch("rt_mesh_pack");
}

extern "C" int rt_mesh_unpack(const void* records, uint32_t n_vertices, float* pos, float* nrm, float* uv,
                              void* stream) {
    if (n_vertices == 0) return RT_OK;
    if (!records) return set_error(RT_EINVAL, "rt_mesh_unpack: records is NULL");
    if ((uintptr_t)records & 15) return set_error(RT_EINVAL, "rt_mesh_unpack: records must be 16-byte aligned");
    if (((uintptr_t)pos | (uintptr_t)nrm | (uintptr_t)uv) & 3)
        return set_error(RT_EINVAL, "rt_mesh_unpack: arrays must be 4-byte aligned");
    hipLaunchKernelGGL(k_mesh_unpack, dim3(nblocks(n_vertices, 256)), dim3(256), 0, (hipStream_t)stream,
                       (const float4*)records, n_vertices, pos, nrm, uv);
    return check_launch("rt_mesh_unpack");
}
