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
// order, each put in order where it is summed or before. (A stable radix sort of the pairs by vertex
// fixed the order before: 133 of 219 us at 1.31 M triangles, 0.66 M vertices; now 83 us: face 34,
// scan 11, place 15, vertex 16.)
//   1. k_nrm_face   per triangle: FP64 face normal (32 B record); per pair its arrival number among
//                   its vertex's pairs (an integer atomic on the vertex's count).
//   2. k_nrm_sums, k_nrm_offsets   exclusive scan of the counts: each vertex's run in `run`; vertices
//                   of more than kNetRun pairs are listed.
//   3. k_nrm_place  run[offset of its vertex + arrival] = p for every pair.
//   4. k_nrm_order  puts the listed runs in order (none in a mesh of 5 or 6 triangles a vertex).
//   5. k_nrm_vertex per vertex: its run in ascending p (up to 8 pairs by a sorting network in
//                   registers), the FP64 sum, float3 N at out + v * out_stride.
// Triangles gathered on few vertices, us for 600,000 of random vertices of 6 : 12 : 48 : 80 : 200 : 1,000
// triangles each, and 300 hubs of 4,500: 194 : 210 : 205 : 222 : 325 : 826, 1,380. With the radix sort
// 208 : 205 : 181 : 215 : 338 : 1,158, 2,047. The pairs of one vertex are same-address atomics in k_nrm_face
// (about 14 ns each) and one lane's sum in k_nrm_vertex (140 ns each, the larger part of a hub's time).
// A non-indexed mesh (vertices 3t, 3t+1, 3t+2) has one pair per vertex: k_nrm_direct computes it
// with no sort and no workspace.
//
// Also here: MeshVertex records <-> dense float arrays (k_mesh_pack / k_mesh_unpack), the device-side
// ingest and export of the 80-byte vertex layout of rendering/_modeling.py:22-28.
#include <algorithm>
#include <cmath>

#include "rt_common.h"

namespace rt {
namespace {

constexpr uint32_t kNetRun = 8;        // longest run k_nrm_vertex puts in order in registers
constexpr uint32_t kWaveRun = 256;     // longest run a wave of k_nrm_order ranks
constexpr uint32_t kLdsRun = 4096;     // longest run, or piece of one, k_nrm_order sorts in LDS
constexpr uint32_t kScanChunk = 2048;  // counts per workgroup of the scan

struct NrmWorkspace {
    double4* face;    // n_tris
    uint32_t* rank;   // 3 n_tris: arrival number of pair p, then k_nrm_order's merges
    uint32_t* run;    // 3 n_tris: the pairs by vertex
    uint32_t* count;  // n_vertices, then the numbers of listed vertices (mid, big)
    uint32_t* off;    // n_vertices
    uint32_t* sums;   // per scan chunk
    uint32_t* mid;    // vertices of kNetRun + 1 .. kWaveRun pairs
    uint32_t* big;    // vertices of more
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
    w.count = (uint32_t*)take(4 * (n_vertices + 2));
    w.off = (uint32_t*)take(4 * n_vertices);
    w.sums = (uint32_t*)take(4 * ((n_vertices + kScanChunk - 1) / kScanChunk));
    w.mid = (uint32_t*)take(4 * (np / (kNetRun + 1) + 1));
    w.big = (uint32_t*)take(4 * (np / (kWaveRun + 1) + 1));
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
// vertices of runs that k_nrm_order puts in order are listed, listed[0] of them in `mid` and listed[1] in
// `big`, with one atomic per workgroup and list: one per vertex took 0.3 ms for 20,000 of them.
__global__ void __launch_bounds__(256) k_nrm_offsets(const uint32_t* __restrict__ count, uint32_t n,
                                                      const uint32_t* __restrict__ sums, bool scanned,
                                                      uint32_t* __restrict__ off, uint32_t* __restrict__ listed,
                                                      uint32_t* __restrict__ mid, uint32_t* __restrict__ big) {
    constexpr uint32_t kPer = kScanChunk / 256;
    __shared__ uint32_t lds[4], scan[256], s_count[2], s_base[2];
    if (threadIdx.x < 2) s_count[threadIdx.x] = 0;
    uint32_t before = 0;
    if (scanned) {
        before = sums[blockIdx.x];
    } else {
        for (uint32_t b = threadIdx.x; b < blockIdx.x; b += 256u) before += sums[b];
        before = block_sum(before, lds);
    }
    const uint64_t base = (uint64_t)blockIdx.x * kScanChunk + threadIdx.x * kPer;
    uint32_t c[kPer], sum = 0, n_mid = 0, n_big = 0;
#pragma unroll
    for (uint32_t k = 0; k < kPer; ++k) {
        c[k] = base + k < n ? count[base + k] : 0u;
        sum += c[k];
        n_mid += c[k] > kNetRun && c[k] <= kWaveRun;
        n_big += c[k] > kWaveRun;
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
    uint32_t at_mid = n_mid ? atomicAdd(&s_count[0], n_mid) : 0u, at_big = n_big ? atomicAdd(&s_count[1], n_big) : 0u;
    __syncthreads();
    if (threadIdx.x < 2 && s_count[threadIdx.x])
        s_base[threadIdx.x] = atomicAdd(&listed[threadIdx.x], s_count[threadIdx.x]);
    __syncthreads();
#pragma unroll
    for (uint32_t k = 0; k < kPer; ++k) {
        if (base + k < n) {
            off[base + k] = at;
            if (c[k] > kWaveRun)
                big[s_base[1] + at_big++] = (uint32_t)(base + k);
            else if (c[k] > kNetRun)
                mid[s_base[0] + at_mid++] = (uint32_t)(base + k);
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

// One pass of a merge sort by a workgroup of 256: src[0, n), sorted in pieces of w (a multiple of 16), to dst
// in pieces of 2 w. A thread finds where its 16 outputs begin in their two pieces and merges them.
RT_DEV void merge_pieces(const uint32_t* src, uint32_t* dst, uint64_t n, uint64_t w) {
    for (uint64_t o = 16ull * threadIdx.x; o < n; o += 16ull * 256) {
        const uint64_t a0 = o / (2 * w) * (2 * w), a1 = a0 + w < n ? a0 + w : n, b1 = a1 + w < n ? a1 + w : n;
        const uint64_t d = o - a0;  // outputs of the two pieces before these
        uint64_t lo = d > b1 - a1 ? d - (b1 - a1) : 0, hi = d < a1 - a0 ? d : a1 - a0;
        while (lo < hi) {
            const uint64_t m = (lo + hi) / 2;
            if (src[a0 + m] < src[a1 + d - 1 - m])
                lo = m + 1;
            else
                hi = m;
        }
        uint64_t i = a0 + lo, j = a1 + (d - lo);
        for (int k = 0; k < 16 && o + k < n; ++k) {
            const bool left = j >= b1 || (i < a1 && src[i] < src[j]);
            dst[o + k] = left ? src[i] : src[j];
            i += left;
            j += !left;
        }
    }
}

// Sorts run[0, n) by a workgroup of 256: pieces of kLdsRun by a bitonic sort in LDS, then merges, through
// tmp[0, n). The work grows with the run's own length; called with the same arguments by all threads.
RT_DEV void sort_run(uint32_t* run, uint32_t* tmp, uint32_t n, uint32_t* key) {
    const uint32_t tid = threadIdx.x;
    for (uint64_t base = 0; base < n; base += kLdsRun) {
        const uint32_t len = (uint32_t)(n - base < kLdsRun ? n - base : kLdsRun);
        uint32_t pow2 = 2;
        while (pow2 < len) pow2 <<= 1;
        __syncthreads();  // before the last piece's LDS is written again
        for (uint32_t i = tid; i < pow2; i += 256u) key[i] = i < len ? run[base + i] : 0xFFFFFFFFu;
        for (uint32_t k = 2; k <= pow2; k <<= 1) {
            for (uint32_t d = k >> 1; d > 0; d >>= 1) {
                __syncthreads();
                for (uint32_t q = tid; q < pow2 / 2; q += 256u) {
                    const uint32_t i = ((q & ~(d - 1)) << 1) | (q & (d - 1)), x = i + d;
                    const uint32_t lo = key[i], hi = key[x];
                    if ((lo > hi) == ((i & k) == 0)) {
                        key[i] = hi;
                        key[x] = lo;
                    }
                }
            }
        }
        __syncthreads();
        for (uint32_t i = tid; i < len; i += 256u) run[base + i] = key[i];
    }
    uint32_t *src = run, *dst = tmp;
    for (uint64_t w = kLdsRun; w < n; w *= 2) {
        __syncthreads();
        merge_pieces(src, dst, n, w);
        uint32_t* t = src;
        src = dst;
        dst = t;
    }
    if (src != run) {
        __syncthreads();
        for (uint64_t i = tid; i < n; i += 256u) run[i] = src[i];
    }
}

// Puts run[0, n) in order by one wave, K pairs in each lane (n <= 64 K): a pair's place is the number of
// smaller ones.
template <int K>
RT_DEV void rank_run(uint32_t* run, uint32_t n, uint32_t lane) {
    uint32_t p[K], rank[K];
#pragma unroll
    for (int k = 0; k < K; ++k) {
        p[k] = 64u * k + lane < n ? run[64 * k + lane] : 0xFFFFFFFFu;
        rank[k] = 0;
    }
#pragma unroll
    for (int k = 0; k < K; ++k) {
        const uint32_t here = n > 64u * k ? (n - 64u * k < 64u ? n - 64u * k : 64u) : 0u;
        for (uint32_t j = 0; j < here; ++j) {
            const uint32_t q = (uint32_t)__builtin_amdgcn_readlane((int)p[k], (int)j);
#pragma unroll
            for (int i = 0; i < K; ++i) rank[i] += q < p[i];
        }
    }
#pragma unroll
    for (int k = 0; k < K; ++k)
        if (64u * k + lane < n) run[rank[k]] = p[k];
}

// Puts the listed runs in order, a workgroup each for the big ones, a wave each for the others. Bound by the
// latency of three dependent loads per run; where no run is listed it ends at once. Random vertices of 80
// triangles, 600,000 in all: 22,500 runs in 26 us by waves, 73 by workgroups. One workgroup per run of more
// than 64 over 64 workgroups took the mesh 2,473 us in all, the index list read again for each of 300 hubs
// of 4,500 14,476.
__global__ void __launch_bounds__(256) k_nrm_order(const uint32_t* __restrict__ listed,
                                                    const uint32_t* __restrict__ mid,
                                                    const uint32_t* __restrict__ big,
                                                    const uint32_t* __restrict__ count,
                                                    const uint32_t* __restrict__ off, uint32_t* run, uint32_t* tmp) {
    __shared__ uint32_t key[kLdsRun];
    const uint32_t n_mid = listed[0], n_big = listed[1], lane = threadIdx.x & 63u;
    for (uint32_t b = blockIdx.x; b < n_big; b += gridDim.x) {
        const uint32_t v = big[b];
        sort_run(run + off[v], tmp + off[v], count[v], key);
    }
    for (uint32_t w = blockIdx.x * 4u + (threadIdx.x >> 6); w < n_mid; w += gridDim.x * 4u) {
        const uint32_t v = (uint32_t)__builtin_amdgcn_readfirstlane((int)mid[w]);
        const uint32_t n = (uint32_t)__builtin_amdgcn_readfirstlane((int)count[v]);
        uint32_t* r = run + off[v];
        if (n <= 64)
            rank_run<1>(r, n, lane);
        else if (n <= 128)
            rank_run<2>(r, n, lane);
        else
            rank_run<4>(r, n, lane);
    }
}

// Triangle of pair p.
RT_DEV uint32_t pair_tri(uint32_t p, uint32_t n_tris) {
    return p >= 2 * n_tris ? p - 2 * n_tris : (p >= n_tris ? p - n_tris : p);
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
    double x = 0.0, y = 0.0, z = 0.0;
    if (n <= kNetRun) {
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
            if (j < n) f[j] = face[pair_tri(p[j], n_tris)];
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
#pragma unroll 4
        for (uint32_t j = 0; j < n; ++j) {
            const double4 f = face[pair_tri(r[j], n_tris)];
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
    uint32_t* listed = w.count + m.n_vertices;
    hipLaunchKernelGGL(k_nrm_clear, dim3(nblocks((uint64_t)m.n_vertices + 2, 256)), dim3(256), 0, s, w.count,
                       (uint64_t)m.n_vertices + 2);
    if (m.n_tris)
        hipLaunchKernelGGL(k_nrm_face, dim3(nblocks(m.n_tris, 256)), dim3(256), 0, s, m, w.face, w.count, w.rank);
    hipLaunchKernelGGL(k_nrm_sums, dim3(chunks), dim3(256), 0, s, w.count, m.n_vertices, w.sums);
    const bool scanned = chunks > kSumChunks;
    if (scanned) hipLaunchKernelGGL(k_nrm_scan_sums, dim3(1), dim3(1024), 0, s, w.sums, chunks);
    hipLaunchKernelGGL(k_nrm_offsets, dim3(chunks), dim3(256), 0, s, w.count, m.n_vertices, w.sums, scanned, w.off,
                       listed, w.mid, w.big);
    if (m.n_tris) {
        hipLaunchKernelGGL(k_nrm_place, dim3(nblocks(m.n_tris, 256)), dim3(256), 0, s, m, w.off, w.rank, w.run);
        const uint64_t np = 3 * (uint64_t)m.n_tris;
        if (np > kNetRun)  // a wave for each of the most mid runs, up to 8 workgroups per CU
            hipLaunchKernelGGL(k_nrm_order, dim3((uint32_t)std::min<uint64_t>(np / (4 * kNetRun) + 1, 2048)), dim3(256), 0,
                               s, listed, w.mid, w.big, w.count, w.off, w.run, w.rank);
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
