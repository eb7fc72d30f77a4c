// rt_build.hip — on-device LBVH construction for rendering/_raycaster.py:26-33
// (Raycaster.__init__ -> _build_ads, a stub in the reference that only counts triangles).
//
// Pipeline (one stream; no host synchronisation):
//   1. gather      per mesh: read MeshVertex P (rendering/_modeling.py:22-28) through the optional
//                  int32 index list, write AABB centroids.
//   2. bounds      min/max of the centroids per workgroup of the gather, folded by the next kernel.
//   3. morton      30-bit Morton code of each centroid quantised to 1024^3 over those bounds.
//   4. sort        stable LSD radix sort of (code, primitive) in 4 passes of 8 bits (rt_sort.h):
//                  per-tile histogram -> per-digit row scan -> scatter, the scatter ranking keys
//                  with wave64 ballot/mbcnt multi-split so equal digits keep input order and
//                  writing each tile digit by digit from LDS.
//   5. emit        tri/shade records and padded leaf boxes in slot order, from the meshes' P/N/C.
//   6. tree        Karras 2012 binary radix tree over the extended keys (code, slot), with its boxes:
//                  bottom-up in LDS inside blocks of 1024 slots, then one wave per node that spans
//                  blocks (min/max are exact, so range unions equal the bottom-up boxes).
//   7. wide        4-wide records from the binary ones.
// PLOC (rt_tuning.builder) replaces 5-6 with locally ordered clustering over the same order.
// Every result is an integer or an exact FP32 min/max/sub, so the output is byte-identical to the
// CPU restatement under the same inputs.
#include <algorithm>
#include <cmath>
#include <utility>

#include "rt_common.h"
#include "rt_sort.h"

namespace rt {
namespace {

// LBVH tree: slots per workgroup of the local pass, and the most top boundaries of one block
constexpr int kTreeBlock = 1024;
constexpr int kTopMax = 132;
constexpr int kTopThreads = 512;

// A top boundary: its position, its diff, the code of slot p, and the ends of its node's slots
// [lo, hi1) where they lie in the boundary's block, else -1.
struct alignas(16) TopEntry {
    int32_t p, lo, hi1, diff;
    uint32_t key;
    int32_t pad[3];
};

// Global arrays of the top boundaries. By position P: pre[2 P] the box of [block start, P), suf[2 P]
// that of [P, block end), child[4 P] and child[4 P + 2] the left and right child where it is a segment.
struct TopArrays {
    TopEntry* list;    // kTopMax per block
    uint32_t* count;   // per block
    float4* pre;
    float4* suf;
    float4* child;
    float4* block;     // 2 per block: box of all its slots
};

// A mesh with triangles as the kernels after the gather read it: its first primitive and its number
// among all meshes.
struct MeshSource {
    rt_mesh_desc d;
    uint32_t base, id;
};

struct Workspace {
    float4* cent;      // n
    float4* leafbox;   // 2n: padded box of each slot (LBVH)
    MeshSource* meshes;  // of the meshes that have triangles
    uint32_t* keys0;   // n
    uint32_t* vals0;
    uint32_t* keys1;
    uint32_t* vals1;
    uint32_t* hist;    // kRadix * nblk
    uint32_t* totals;  // kRadix
    float4* partial;   // 2 per workgroup of the gather: bounds of its centroids (the space of cbox[0])
    float* cbounds;    // 8
    int32_t* parent;   // (n-1) internal then n leaves
    // PLOC builder
    int32_t* cid[2];   // n: cluster refs by position (internal id, or ~prim), ping-pong
    float4* cbox[2];   // 2n: cluster boxes by position, ping-pong
    int32_t* nn;       // n: nearest neighbour position
    int32_t* nleft;    // n-1: children and triangle count of each internal node
    int32_t* nright;
    int32_t* nsize;
    uint32_t* pos_of;  // n: Morton position of each primitive
    uint32_t* slot_of; // n: slot of each primitive
    uint32_t* fslot;   // n-1: first slot of each internal node inside a leaf
    uint32_t* scan;    // n: leaf-root sizes at their first Morton position, then their first slot
    uint32_t* part;    // per tile or chunk: counts, then the slot scan's offsets
    int32_t* state;    // 8: cluster count, nodes created and buffer per iteration parity
    uint32_t* depth;   // 1: internal ancestors of the deepest triangle of the PLOC tree
    TopArrays top;     // boundaries whose nodes span several tree blocks
    uint32_t* slot_order;  // n: primitive of each slot
    uint64_t bytes;
};

inline uint64_t align256(uint64_t x) { return (x + 255) & ~uint64_t(255); }

Workspace carve(char* base, uint64_t n) {
    Workspace w{};
    const uint64_t ni = n > 1 ? n - 1 : 1;
    uint64_t off = 0;
    auto take = [&](uint64_t bytes) {
        char* p = base ? base + off : nullptr;
        off = align256(off + bytes);
        return p;
    };
    w.cent = (float4*)take(16 * n);
    w.leafbox = (float4*)take(32 * n);
    w.meshes = (MeshSource*)take(sizeof(MeshSource) * n);
    w.keys0 = (uint32_t*)take(4 * n);
    w.vals0 = (uint32_t*)take(4 * n);
    w.keys1 = (uint32_t*)take(4 * n);
    w.vals1 = (uint32_t*)take(4 * n);
    w.hist = (uint32_t*)take(sort_hist_bytes(n));
    w.totals = (uint32_t*)take(4 * kRadix);
    w.cbounds = (float*)take(4 * 8);
    w.parent = (int32_t*)take(4 * (ni + n));
    for (int k = 0; k < 2; ++k) {
        w.cid[k] = (int32_t*)take(4 * n);
        w.cbox[k] = (float4*)take(32 * n);
    }
    w.partial = w.cbox[0];  // every workgroup of the gather has a triangle, so there are at most n
    w.nn = (int32_t*)take(4 * n);
    w.nleft = (int32_t*)take(4 * ni);
    w.nright = (int32_t*)take(4 * ni);
    w.nsize = (int32_t*)take(4 * ni);
    w.pos_of = (uint32_t*)take(4 * n);
    w.slot_of = (uint32_t*)take(4 * n);
    w.fslot = (uint32_t*)take(4 * ni);
    w.scan = (uint32_t*)take(4 * n);
    w.part = (uint32_t*)take(4 * ((n + 255) / 256));
    w.state = (int32_t*)take(4 * 8);
    w.depth = (uint32_t*)take(4);
    const uint64_t nb = (n + kTreeBlock - 1) / kTreeBlock;
    w.top.list = (TopEntry*)take(sizeof(TopEntry) * kTopMax * nb);
    w.top.count = (uint32_t*)take(4 * nb);
    w.top.pre = (float4*)take(32 * n);
    w.top.suf = (float4*)take(32 * n);
    w.top.child = (float4*)take(64 * n);
    w.top.block = (float4*)take(32 * nb);
    w.slot_order = (uint32_t*)take(4 * n);
    w.bytes = off;
    return w;
}

RT_DEV float canon(float x) { return x + 0.0f; }  // -0 -> +0

// Leaf boxes are padded by |coordinate| * 2^-14 + 2^-40 per side, wider than the world-space error
// of an FP32 Moller-Trumbore acceptance, so a box test never culls a triangle the FP32 test would
// accept: the closest hit is then independent of the traversal order (per-ray or wave-coherent).
RT_DEV float pad_of(float lo, float hi) {
    const float m = fmaxf(fabsf(lo), fabsf(hi));
    return m * 0x1p-14f + 0x1p-40f;
}

RT_DEV float3 load_f3(const char* base, uint64_t i, uint32_t stride, uint32_t off) {
    const float* p = (const float*)(base + i * stride + off);
    return make_float3(p[0], p[1], p[2]);
}

struct Box {
    float lo[3], hi[3];
};

RT_DEV Box empty_box() {
    return {{INFINITY, INFINITY, INFINITY}, {-INFINITY, -INFINITY, -INFINITY}};
}

RT_DEV Box unite(const Box& a, const Box& b) {
    Box u;
    for (int c = 0; c < 3; ++c) {
        u.lo[c] = fminf(a.lo[c], b.lo[c]);
        u.hi[c] = fmaxf(a.hi[c], b.hi[c]);
    }
    return u;
}

RT_DEV Box load_box(const float4* __restrict__ p) {
    const float4 a = p[0], b = p[1];
    return {{a.x, a.y, a.z}, {b.x, b.y, b.z}};
}

RT_DEV void store_box(float4* __restrict__ p, const Box& b) {
    p[0] = make_float4(b.lo[0], b.lo[1], b.lo[2], 0.0f);
    p[1] = make_float4(b.hi[0], b.hi[1], b.hi[2], 0.0f);
}

// Union over the wave's lanes, in every lane.
RT_DEV Box wave_unite(Box b) {
    for (int x = 1; x < 64; x <<= 1)
        for (int c = 0; c < 3; ++c) {
            b.lo[c] = fminf(b.lo[c], __shfl_xor(b.lo[c], x));
            b.hi[c] = fmaxf(b.hi[c], __shfl_xor(b.hi[c], x));
        }
    return b;
}

// Union of parts[2 i] for i < count over a workgroup of T threads, in every thread; `lds` holds two
// float4s per wave.
template <int T>
RT_DEV Box block_unite(const float4* __restrict__ parts, uint32_t count, float4* lds) {
    Box b = empty_box();
#pragma unroll 4
    for (uint32_t i = threadIdx.x; i < count; i += T) b = unite(b, load_box(parts + 2 * (uint64_t)i));
    b = wave_unite(b);
    if ((threadIdx.x & 63) == 0) store_box(lds + 2 * (threadIdx.x >> 6), b);
    __syncthreads();
    b = load_box(lds);
    for (int w = 1; w < T / 64; ++w) b = unite(b, load_box(lds + 2 * w));
    return b;
}

// Positions of triangle t of a mesh with canonical zeros, and its vertex indices; an index past the
// vertices is clamped, so a malformed list cannot read past the buffer.
RT_DEV void load_corners(const rt_mesh_desc& m, uint32_t t, uint32_t (&v)[3], float3 (&p)[3]) {
    for (int k = 0; k < 3; ++k) v[k] = 3 * t + k;
    if (m.indices) {
        const uint32_t* ix = (const uint32_t*)m.indices + 3 * (uint64_t)t;
        for (int k = 0; k < 3; ++k) v[k] = ix[k];
        for (int k = 0; k < 3; ++k) v[k] = v[k] < m.n_vertices ? v[k] : m.n_vertices - 1;
    }
    for (int k = 0; k < 3; ++k) {
        const float3 q = load_f3((const char*)m.vertices, v[k], m.vertex_stride, m.pos_offset);
        p[k] = make_float3(canon(q.x), canon(q.y), canon(q.z));
    }
}

RT_DEV Box corners_box(const float3 (&p)[3]) {
    return {{fminf(fminf(p[0].x, p[1].x), p[2].x), fminf(fminf(p[0].y, p[1].y), p[2].y),
             fminf(fminf(p[0].z, p[1].z), p[2].z)},
            {fmaxf(fmaxf(p[0].x, p[1].x), p[2].x), fmaxf(fmaxf(p[0].y, p[1].y), p[2].y),
             fmaxf(fmaxf(p[0].z, p[1].z), p[2].z)}};
}

RT_DEV Box padded(Box b) {
    for (int c = 0; c < 3; ++c) {
        const float pad = pad_of(b.lo[c], b.hi[c]);
        b.lo[c] -= pad;
        b.hi[c] += pad;
    }
    return b;
}

// The mesh of primitive p: the last one of `count` whose first primitive is not past it.
RT_DEV const MeshSource& mesh_of(const MeshSource* __restrict__ meshes, uint32_t count, uint32_t p) {
    uint32_t lo = 0, hi = count - 1;
    while (lo < hi) {
        const uint32_t mid = (lo + hi + 1) / 2;
        if (meshes[mid].base <= p)
            lo = mid;
        else
            hi = mid - 1;
    }
    return meshes[lo];
}

// One thread per triangle: the centroid of its box; the workgroup's union of centroids to `partial`, the
// mesh's description to `source` (NULL for a mesh without triangles). Everything else a triangle needs is
// read from its mesh again when its slot is known (k_emit).
__global__ void __launch_bounds__(256) k_gather(rt_mesh_desc m, uint32_t mesh_id, uint32_t n_meshes,
                                                uint32_t prim_base, float4* __restrict__ cent,
                                                int32_t* __restrict__ mesh_offsets,
                                                float4* __restrict__ partial, MeshSource* __restrict__ source) {
    __shared__ float4 wpart[4][2];
    const uint32_t t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t == 0) {
        mesh_offsets[mesh_id] = (int32_t)prim_base;
        if (mesh_id + 1 == n_meshes) mesh_offsets[n_meshes] = (int32_t)(prim_base + m.n_tris);
        if (m.n_tris) *source = {m, prim_base, mesh_id};
    }
    if (blockIdx.x * blockDim.x >= m.n_tris) return;  // whole block (only the launch for an empty mesh)
    Box cb = empty_box();
    if (t < m.n_tris) {
        uint32_t v[3];
        float3 p[3];
        load_corners(m, t, v, p);
        const Box b = corners_box(p);
        float c[3];
        for (int k = 0; k < 3; ++k) c[k] = (b.lo[k] + b.hi[k]) * 0.5f;
        cent[prim_base + t] = make_float4(c[0], c[1], c[2], 0.0f);
        cb = unite(cb, {{c[0], c[1], c[2]}, {c[0], c[1], c[2]}});
    }
    cb = wave_unite(cb);
    if ((threadIdx.x & 63) == 0) store_box(wpart[threadIdx.x >> 6], cb);
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < 4; ++w) cb = unite(cb, load_box(wpart[w]));
        store_box(partial + 2 * (uint64_t)blockIdx.x, cb);
    }
}

__global__ void k_mesh_offsets_tail(int32_t* mesh_offsets, uint32_t n_meshes, uint32_t n) {
    if (threadIdx.x == 0 && blockIdx.x == 0) mesh_offsets[n_meshes] = (int32_t)n;
}

RT_DEV uint32_t expand10(uint32_t v) {
    v &= 0x3FFu;
    v = (v | (v << 16)) & 0x030000FFu;
    v = (v | (v << 8)) & 0x0300F00Fu;
    v = (v | (v << 4)) & 0x030C30C3u;
    v = (v | (v << 2)) & 0x09249249u;
    return v;
}

RT_DEV uint32_t quantize10(float c, float lo, float scale) {
    float q = (c - lo) * scale;
    q = fminf(fmaxf(q, 0.0f), 1023.0f);
    return (uint32_t)q;
}

RT_DEV float quantize_scale(float lo, float hi) {
    const float ext = hi - lo;
    return ext > 0.0f ? 1024.0f / ext : 0.0f;
}

RT_DEV uint32_t morton30(float x, float y, float z, const float* lo, const float* scale) {
    return (expand10(quantize10(x, lo[0], scale[0])) << 2) | (expand10(quantize10(y, lo[1], scale[1])) << 1) |
           expand10(quantize10(z, lo[2], scale[2]));
}

// One block folds the gather's bounds of 256 centroids each into (lo.xyz, scale.xyz) for the quantiser.
__global__ void __launch_bounds__(1024) k_bounds_final(const float4* __restrict__ partial, uint32_t nparts,
                                                       float* __restrict__ cb) {
    __shared__ float4 lds[2 * 1024 / 64];
    const Box b = block_unite<1024>(partial, nparts, lds);
    if (threadIdx.x == 0)
        for (int a = 0; a < 3; ++a) {
            cb[a] = b.lo[a];
            cb[4 + a] = quantize_scale(b.lo[a], b.hi[a]);
        }
}

__global__ void __launch_bounds__(256) k_morton(const float4* __restrict__ cent, uint32_t n,
                                                 const float* __restrict__ cb,
                                                 uint32_t* __restrict__ keys,
                                                 uint32_t* __restrict__ vals) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float4 c = cent[i];
    keys[i] = morton30(c.x, c.y, c.z, cb, cb + 4);
    vals[i] = i;
}

// Order of a scene of at most kSmallMax triangles in two launches. k_order_chunks: a workgroup folds
// the gather's bounds for itself, and codes and sorts its kOrderChunk triangles by counting
// smaller keys. k_order_merge: a pair's place is its place in its chunk plus, for every other chunk,
// a binary search in LDS; each of 4 waves takes a quarter of the chunks for the same 64 pairs.
// Equal codes keep their order: they count as smaller in chunks before the pair's own.
// The general path's 14 launches of codes and radix passes run up to 6 workgroups each at 11,560
// triangles and take 58 us of kernel time, these two take 13; one workgroup that held all pairs and made
// the four radix passes in LDS took 44, bound by the ballots of its 16 waves. The limit is the LDS that
// holds all codes: at 32,000 triangles these take 30 us, the general path 59 at 33,620.
constexpr uint32_t kOrderChunk = 256;
constexpr uint32_t kSmallMax = 32 * 1024;

__global__ void __launch_bounds__(kOrderChunk) k_order_chunks(const float4* __restrict__ cent, uint32_t n,
                                                              const float4* __restrict__ partial,
                                                              uint32_t nparts, uint32_t* __restrict__ keys,
                                                              uint32_t* __restrict__ vals) {
    constexpr int kWaves = kOrderChunk / 64;
    __shared__ float4 lds[2 * kWaves];
    __shared__ uint4 sk[kOrderChunk / 4];
    const uint32_t tid = threadIdx.x;
    const int wave = tid >> 6;
    const Box b = block_unite<kOrderChunk>(partial, nparts, lds);
    float scale[3];
    for (int a = 0; a < 3; ++a) scale[a] = quantize_scale(b.lo[a], b.hi[a]);
    const uint32_t i = blockIdx.x * kOrderChunk + tid;
    uint32_t key = 0xFFFFFFFFu;  // past the end: above every code
    if (i < n) {
        const float4 c = cent[i];
        key = morton30(c.x, c.y, c.z, b.lo, scale);
    }
    ((uint32_t*)sk)[tid] = key;
    __syncthreads();
    uint32_t rank = 0;
    // four keys a step; equal ones count before this thread's own
#pragma unroll 8
    for (int j = 0; j < 16 * wave; ++j) {
        const uint4 q = sk[j];
        rank += (uint32_t)(q.x <= key) + (uint32_t)(q.y <= key) + (uint32_t)(q.z <= key) + (uint32_t)(q.w <= key);
    }
#pragma unroll 8
    for (int j = 16 * wave; j < 16 * (wave + 1); ++j) {
        const uint4 q = sk[j];
        const uint32_t j0 = 4 * (uint32_t)j;
        rank += (uint32_t)(q.x < key + (j0 < tid)) + (uint32_t)(q.y < key + (j0 + 1 < tid)) +
                (uint32_t)(q.z < key + (j0 + 2 < tid)) + (uint32_t)(q.w < key + (j0 + 3 < tid));
    }
#pragma unroll 8
    for (int j = 16 * (wave + 1); j < 16 * kWaves; ++j) {
        const uint4 q = sk[j];
        rank += (uint32_t)(q.x < key) + (uint32_t)(q.y < key) + (uint32_t)(q.z < key) + (uint32_t)(q.w < key);
    }
    if (i < n) {
        keys[i - tid + rank] = key;
        vals[i - tid + rank] = i;
    }
}

template <uint32_t kMax>
__global__ void __launch_bounds__(256) k_order_merge(const uint32_t* __restrict__ kin,
                                                     const uint32_t* __restrict__ vin, uint32_t n,
                                                     uint32_t* __restrict__ keys,
                                                     uint32_t* __restrict__ order) {
    __shared__ uint32_t sk[kMax];
    __shared__ uint32_t part[4][64];
    const uint32_t tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const uint32_t chunks = (n + kOrderChunk - 1) / kOrderChunk;
    for (uint32_t i0 = tid; i0 < chunks * kOrderChunk; i0 += 32 * 256) {  // 32 loads in flight
        uint32_t v[32];
#pragma unroll
        for (int q = 0; q < 32; ++q) v[q] = i0 + q * 256 < n ? kin[i0 + q * 256] : 0xFFFFFFFFu;
#pragma unroll
        for (int q = 0; q < 32; ++q) sk[i0 + q * 256] = v[q];  // kMax is a multiple of the 8,192 of a round
    }
    const uint32_t i = blockIdx.x * 64 + lane;
    const uint32_t val = wave == 0 && i < n ? vin[i] : 0u;
    __syncthreads();
    const uint32_t own = blockIdx.x * 64 / kOrderChunk;
    const uint32_t key = sk[i];  // blocks cover whole chunks at most
    uint32_t rank = 0;
    for (uint32_t c0 = wave; c0 < chunks; c0 += 16) {  // four searches at a time hide each other's LDS latency
        uint32_t at[4] = {0, 0, 0, 0}, k[4];
        const uint32_t* a[4];
#pragma unroll
        for (uint32_t q = 0; q < 4; ++q) {
            const uint32_t c = c0 + 4 * q;
            k[q] = c >= chunks || c == own ? 0u : c < own ? key + 1 : key;  // count codes below k (30 bits)
            a[q] = sk + (c < chunks ? c : 0u) * kOrderChunk;
        }
#pragma unroll
        for (uint32_t step = kOrderChunk / 2; step; step >>= 1)
#pragma unroll
            for (int q = 0; q < 4; ++q) at[q] += a[q][at[q] + step - 1] < k[q] ? step : 0u;
#pragma unroll
        for (int q = 0; q < 4; ++q) rank += at[q] + (a[q][at[q]] < k[q] ? 1u : 0u);
    }
    part[wave][lane] = rank;
    __syncthreads();
    if (wave == 0 && i < n) {
        const uint32_t at = part[0][lane] + part[1][lane] + part[2][lane] + part[3][lane] + i % kOrderChunk;
        keys[at] = key;
        order[at] = val;
    }
}

// Whether the LBVH kernels run: always (deep NULL), or where a PLOC tree turned out too deep (*deep set),
// with `order` the Morton order instead of PLOC's slots. The device decides, so a PLOC build does not
// wait for its stream.
struct Fallback {
    const uint32_t* deep;
    const uint32_t* order;
    RT_DEV bool taken() const { return !deep || *deep; }
};

// Store of arrays that no kernel of the build reads again (leaf records, 4-wide nodes). PAST: past the caches, which
// then keep what the next kernels read. That pays where the scene does not fit them: at 1.31 M triangles the emit went
// from 72 to 63 us, the 4-wide nodes from 45 to 39, a build with its first frame from 466 to 434 (256x144) and from
// 1,506 to 1,474 (1280x720). A smaller scene's first calls find these arrays in the caches: build and first frame
// of 256x144 at 450,000 triangles 292 us, past the caches 302, at 251,000 225 and 229, at 648,000 365 and 366.
constexpr uint32_t kPastCaches = 500000;  // triangles

template <bool PAST>
RT_DEV void store_last(float4* p, const float4& v) {
    typedef float vec4 __attribute__((ext_vector_type(4)));
    const vec4 q = {v.x, v.y, v.z, v.w};
    if constexpr (PAST)
        __builtin_nontemporal_store(q, (vec4*)p);
    else
        *(vec4*)p = q;
}

// Copies `per` float4s of each of the block's `rows` records from LDS (record r at
// stage[r * pitch]) to out[0 .. rows*per), one float4 per thread and instruction.
template <bool PAST>
RT_DEV void store_staged(float4* __restrict__ out, const float4* stage, uint32_t rows, uint32_t per,
                         uint32_t pitch) {
    for (uint32_t q = threadIdx.x; q < rows * per; q += blockDim.x) {
        const uint32_t r = q / per;
        store_last<PAST>(out + q, stage[r * pitch + (q - r * per)]);
    }
}

// One thread per slot: the intersection record (p0, e1, e2, primitive id) and the shading record (three
// normals, three uvs, mesh id) of its triangle, from the mesh's vertices; the padded leaf box of the slot
// for an LBVH; the slot of the primitive. The block's records go out through LDS as consecutive
// float4s. Bound by memory: 148 B of stores per triangle, and the vertices, which neighbours in Morton
// order share in L2. At 1.31 M triangles 63 us and 21 for the gather; records written in
// primitive order by the gather and permuted here took 71 and 81.
template <bool PAST>
__global__ void __launch_bounds__(256) k_emit(const uint32_t* __restrict__ slots, Fallback fb, uint32_t n,
                                              const MeshSource* __restrict__ meshes, uint32_t n_sources,
                                              float4* __restrict__ leafbox, float4* __restrict__ tris,
                                              float4* __restrict__ shade, uint32_t* __restrict__ prim_slot) {
    constexpr uint32_t kPitch = 5;  // float4s per staged record (4 used)
    __shared__ float4 stage[256 * kPitch];
    const uint64_t s0 = (uint64_t)blockIdx.x * 256;
    const uint32_t rows = n - s0 < 256 ? (uint32_t)(n - s0) : 256u;
    const bool mine = threadIdx.x < rows, taken = fb.taken();
    const uint32_t* __restrict__ order = fb.deep && taken ? fb.order : slots;
    float4 tri[3], shd[4];
    Box box = empty_box();
    if (mine) {
        const uint32_t prim = order[s0 + threadIdx.x];
        const MeshSource& src = mesh_of(meshes, n_sources, prim);
        const rt_mesh_desc& m = src.d;
        uint32_t v[3];
        float3 p[3], nr[3];
        load_corners(m, prim - src.base, v, p);
        box = padded(corners_box(p));
        prim_slot[prim] = (uint32_t)s0 + threadIdx.x;
        const float e1x = p[1].x - p[0].x, e1y = p[1].y - p[0].y, e1z = p[1].z - p[0].z;
        const float e2x = p[2].x - p[0].x, e2y = p[2].y - p[0].y, e2z = p[2].z - p[0].z;
        tri[0] = make_float4(p[0].x, p[0].y, p[0].z, __int_as_float((int32_t)prim));
        tri[1] = make_float4(e1x, e1y, e1z, 0.0f);
        tri[2] = make_float4(e2x, e2y, e2z, 0.0f);
        if (m.nrm_offset != RT_ABSENT) {
            for (int k = 0; k < 3; ++k) nr[k] = load_f3((const char*)m.vertices, v[k], m.vertex_stride, m.nrm_offset);
        } else {
            const float gx = fmaf(e1y, e2z, -(e1z * e2y));
            const float gy = fmaf(e1z, e2x, -(e1x * e2z));
            const float gz = fmaf(e1x, e2y, -(e1y * e2x));
            const float l2 = fmaf(gx, gx, fmaf(gy, gy, gz * gz));
            const float il = l2 > 0.0f ? 1.0f / sqrtf(l2) : 0.0f;
            nr[0] = nr[1] = nr[2] = make_float3(gx * il, gy * il, gz * il);
        }
        float2 uv[3] = {make_float2(0.0f, 0.0f), make_float2(0.0f, 0.0f), make_float2(0.0f, 0.0f)};
        if (m.uv_offset != RT_ABSENT)
            for (int k = 0; k < 3; ++k) {
                const float* q = (const float*)((const char*)m.vertices + (uint64_t)v[k] * m.vertex_stride + m.uv_offset);
                uv[k] = make_float2(q[0], q[1]);
            }
        shd[0] = make_float4(nr[0].x, nr[0].y, nr[0].z, nr[1].x);
        shd[1] = make_float4(nr[1].y, nr[1].z, nr[2].x, nr[2].y);
        shd[2] = make_float4(nr[2].z, uv[0].x, uv[0].y, uv[1].x);
        shd[3] = make_float4(uv[1].y, uv[2].x, uv[2].y, __int_as_float((int32_t)src.id));
    }
    float4* st = stage + threadIdx.x * kPitch;
    if (mine) { st[0] = shd[0]; st[1] = shd[1]; st[2] = shd[2]; st[3] = shd[3]; }
    __syncthreads();
    store_staged<PAST>(shade + 4 * s0, stage, rows, 4, kPitch);
    __syncthreads();
    if (mine) { st[0] = tri[0]; st[1] = tri[1]; st[2] = tri[2]; }
    __syncthreads();
    store_staged<PAST>(tris + 3 * s0, stage, rows, 3, kPitch);
    if (!taken) return;
    __syncthreads();
    if (mine) store_box(st, box);
    __syncthreads();
    for (uint32_t q = threadIdx.x; q < rows * 2; q += 256) leafbox[2 * s0 + q] = stage[(q >> 1) * kPitch + (q & 1)];
}

// ---- tree ----
// The binary radix tree over the extended keys (code, slot). Boundary P lies between slots P - 1
// and P; diff(P) is the common prefix of the two (-1 at 0 and n). Each boundary inside the range is
// the split of one internal node, whose slots reach to the nearest boundaries on either side with a
// smaller diff; that pair never ties except at the root. A node [lo, hi] is the right child of
// boundary lo if diff(lo) > diff(hi + 1), else the left child of boundary hi + 1, and its id is lo or
// hi accordingly (the root's is 0).
//
// k_tree_local: one workgroup per kTreeBlock slots builds every node that lies inside them in one
// pass, bottom-up in LDS: a node stores its box under its id, the second child to arrive at a
// boundary (LDS counter, workgroup acq_rel) makes the parent and goes on. Left over are the "top"
// boundaries, whose nodes span blocks: the strict prefix and suffix minima of diff, so at most 2 x 64,
// and the block's lower edge. They cut the block into segments, the largest subtrees inside it.
// k_tree_top: one wave per top boundary finds the ends that lie in other blocks by a 64-ary search and
// unites its children's boxes from segments, block suffixes and prefixes at top boundaries and whole
// blocks. No node waits on another workgroup.
//
// What bounds it: LDS round trips per level of a walk (10 to 17 levels), and 64 B per node of stores
// in pieces of 16 B; one slot per thread puts two workgroups on a CU (41 KB of LDS would let in three).
// At 1.31 M triangles 56 us for the local pass and 25 for the top; separate kernels for the hierarchy
// (binary searches in memory, 93 us), a refit over its arrays (142), a sparse table of block unions
// (17) and the top refit (10) took 262. At 11,560 triangles 24 us against 61.
// length of the common prefix of the extended keys (a, i) and (b, j)
RT_DEV int key_prefix(uint32_t a, uint32_t b, int64_t i, int64_t j) {
    return a != b ? __clz(a ^ b) : 32 + __clz((uint32_t)i ^ (uint32_t)j);
}

// common prefix of slots p - 1 and p; -1 at the scene's ends
RT_DEV int diff_at(const uint32_t* __restrict__ keys, int64_t n, int64_t p) {
    return p <= 0 || p >= n ? -1 : key_prefix(keys[p - 1], keys[p], p - 1, p);
}

// Record of node `id` with slots [lo, hi1) split at boundary p; a child of at most kLeafMax slots
// becomes one leaf of them.
RT_DEV void store_tree_node(float4* __restrict__ nodes, uint32_t id, uint32_t lo, uint32_t p, uint32_t hi1,
                            const Box& l, const Box& r) {
    const uint32_t nl = p - lo, nr = hi1 - p;
    const int32_t tl = nl <= (uint32_t)kLeafMax ? leaf_ref(lo, nl) : (int32_t)(p - 1);
    const int32_t tr = nr <= (uint32_t)kLeafMax ? leaf_ref(p, nr) : (int32_t)p;
    float4* nd = nodes + (uint64_t)id * 4;
    nd[0] = make_float4(l.lo[0], l.hi[0], l.lo[1], l.hi[1]);
    nd[1] = make_float4(r.lo[0], r.hi[0], r.lo[1], r.hi[1]);
    nd[2] = make_float4(l.lo[2], l.hi[2], r.lo[2], r.hi[2]);
    nd[3] = make_float4(__int_as_float(tl), __int_as_float(tr), 0.0f, 0.0f);
}

RT_DEV void store_bounds(float* __restrict__ bounds, const Box& b) {
    for (int c = 0; c < 3; ++c) {
        bounds[c] = b.lo[c];
        bounds[4 + c] = b.hi[c];
    }
    bounds[3] = bounds[7] = 0.0f;
}

__global__ void __launch_bounds__(kTreeBlock) k_tree_local(const uint32_t* __restrict__ keys,
                                                             uint32_t n, Fallback fb, const float4* __restrict__ leafbox,
                                                             float4* __restrict__ nodes,
                                                             float* __restrict__ bounds, TopArrays top) {
    __shared__ float box[6][kTreeBlock];  // by local node id: the box of a node whose parent is pending
    __shared__ int32_t other[kTreeBlock];  // and the end of its slots that is not its id
    __shared__ uint32_t arrived[kTreeBlock];
    __shared__ int32_t diff[kTreeBlock + 1];
    __shared__ int32_t seg[kTopMax + 2];   // segment starts, then the block's end
    __shared__ int32_t sdiff[kTopMax + 2];  // diff there
    __shared__ float sbox[kTopMax + 2][6];
    __shared__ int32_t nseg;
    if (!fb.taken()) return;
    const int64_t blo = (int64_t)blockIdx.x * kTreeBlock;
    const int cnt = (int)(n - blo < kTreeBlock ? n - blo : kTreeBlock);
    const int tid = threadIdx.x;
    Box b = empty_box();
    if (tid < cnt) {
        diff[tid] = diff_at(keys, n, blo + tid);
        if (tid == 0) diff[cnt] = diff_at(keys, n, blo + cnt);
        b = load_box(leafbox + 2 * (uint64_t)(blo + tid));
    }
    arrived[tid] = 0;
    __syncthreads();
    auto put = [&](int e, const Box& b) {
        for (int c = 0; c < 3; ++c) {
            box[c][e] = b.lo[c];
            box[3 + c][e] = b.hi[c];
        }
    };
    auto get = [&](int e) {
        Box b;
        for (int c = 0; c < 3; ++c) {
            b.lo[c] = box[c][e];
            b.hi[c] = box[3 + c][e];
        }
        return b;
    };
    if (tid < cnt) {
        Box l = b, r = b;
        int lo = tid, hi = tid, split = tid;
        for (;;) {
            const int dl = diff[lo], dr = diff[hi + 1];
            const bool right = dl > dr, root = dl < 0 && dr < 0;
            const int e = right ? lo : hi;
            if (lo < hi)
                store_tree_node(nodes, root ? 0u : (uint32_t)(blo + e), (uint32_t)(blo + lo),
                                (uint32_t)(blo + split), (uint32_t)(blo + hi + 1), l, r);
            if (root) {
                store_bounds(bounds, b);
                break;
            }
            put(e, b);
            other[e] = right ? hi : lo;
            const int p = right ? lo : hi + 1;
            if (p == 0 || p == cnt) break;  // the boundary to another block
            const uint32_t prev = __hip_atomic_fetch_add(&arrived[p], 1u, __ATOMIC_ACQ_REL,
                                                         __HIP_MEMORY_SCOPE_WORKGROUP);
            if (prev == 0) break;
            const int q = right ? lo - 1 : hi + 1;  // the sibling's id
            const Box o = get(q);
            if (right) {
                l = o;
                r = b;
                lo = other[q];
            } else {
                l = b;
                r = o;
                hi = other[q];
            }
            split = p;
            b = unite(l, r);
        }
    }
    if (gridDim.x == 1) return;
    __syncthreads();
    // the segments' starts: 0 and the boundaries at which fewer than two children arrived
    if (tid < 64) {
        uint32_t m = 0;
#pragma unroll
        for (int k = 0; k < kTreeBlock / 64; ++k) {
            const int p = k * 64 + tid;
            const bool is = p == 0 || (p < cnt && arrived[p] < 2u);
            const uint64_t mask = __ballot(is);
            const uint32_t at = m + __builtin_amdgcn_mbcnt_hi((uint32_t)(mask >> 32),
                                                              __builtin_amdgcn_mbcnt_lo((uint32_t)mask, 0u));
            if (is && at < (uint32_t)kTopMax) seg[at] = p;  // always true: at most 129
            m += (uint32_t)__popcll(mask);
        }
        if (tid == 0) {
            nseg = (int32_t)(m < (uint32_t)kTopMax ? m : (uint32_t)kTopMax);
            seg[nseg] = cnt;
        }
    }
    __syncthreads();
    const int m = nseg;
    const int first = blo == 0 ? 1 : 0;  // boundary 0 of the scene is no node's split
    if (tid == 0) top.count[blockIdx.x] = (uint32_t)(m - first);
    const int j = tid, p = j <= m ? seg[j] : 0, d = diff[p];
    const bool is = j < m;
    Box own = empty_box();
    if (j <= m) sdiff[j] = d;
    if (is) {
        const int end = seg[j + 1], de = diff[end];
        own = get(d > de ? p : end - 1);
        store_box(top.child + 4 * (uint64_t)(d > de ? blo + p : blo + end) + (d > de ? 2 : 0), own);
        for (int c = 0; c < 3; ++c) {
            sbox[j][c] = own.lo[c];
            sbox[j][3 + c] = own.hi[c];
        }
    }
    __syncthreads();
    if (!is) return;
    Box pre = empty_box(), suf = empty_box();
    TopEntry t{(int32_t)(blo + p), -1, -1, d, keys[blo + p], {}};
#pragma unroll 2
    for (int i = 0; i < m; ++i) {
        const Box b = {{sbox[i][0], sbox[i][1], sbox[i][2]}, {sbox[i][3], sbox[i][4], sbox[i][5]}};
        if (i < j)
            pre = unite(pre, b);
        else
            suf = unite(suf, b);
        const bool less = sdiff[i] < d;
        if (i < j && less) t.lo = seg[i];  // the last one before j
        if (i > j && less && t.hi1 < 0) t.hi1 = seg[i];
    }
    if (t.hi1 < 0 && sdiff[m] < d) t.hi1 = cnt;
    if (t.lo >= 0) t.lo += (int32_t)blo;
    if (t.hi1 >= 0) t.hi1 += (int32_t)blo;
    store_box(top.pre + 2 * (uint64_t)(blo + p), pre);
    store_box(top.suf + 2 * (uint64_t)(blo + p), suf);
    if (j == 0) store_box(top.block + 2 * (uint64_t)blockIdx.x, suf);
    if (j >= first) top.list[(uint64_t)blockIdx.x * kTopMax + (j - first)] = t;
}

// The first x in [a, b] for which pred(x) holds, with pred(b) true and pred monotone, by all 64 lanes:
// each round tests 64 evenly spaced positions.
template <typename Pred>
RT_DEV int64_t wave_first(int64_t a, int64_t b, int lane, Pred pred) {
    while (a < b) {
        const int64_t step = (b - a + 63) / 64;
        const int64_t x = a + lane * step;
        const uint64_t yes = __ballot(x >= b || pred(x));
        const int f = yes ? __ffsll((unsigned long long)yes) - 1 : 64;
        const int64_t hit = a + f * step;
        if (f > 0) a = a + (f - 1) * step + 1;
        if (f < 64 && hit < b) b = hit;
    }
    return a;
}

// Box of slots [lo, hi1), which span several blocks: the suffix of lo's block, the prefix of hi1's and
// the whole blocks between, spread over the lanes. (min and max are exact, so the order is free.)
RT_DEV Box wave_range_box(const TopArrays& top, int64_t lo, int64_t hi1, uint32_t n, uint32_t nb, int lane) {
    const int64_t b0 = (lo + kTreeBlock - 1) / kTreeBlock;
    const int64_t b1 = hi1 == (int64_t)n ? (int64_t)nb : hi1 / kTreeBlock;
    Box b = empty_box();
    if (lo % kTreeBlock) b = unite(b, load_box(top.suf + 2 * (uint64_t)lo));
    if (hi1 != (int64_t)n && hi1 % kTreeBlock) b = unite(b, load_box(top.pre + 2 * (uint64_t)hi1));
    if (b0 < b1) {
        for (int64_t k = b0 + lane; k < b1; k += 64) b = unite(b, load_box(top.block + 2 * (uint64_t)k));
        b = wave_unite(b);
    }
    return b;
}

__global__ void __launch_bounds__(kTopThreads) k_tree_top(const uint32_t* __restrict__ keys, uint32_t n, Fallback fb,
                                                  float4* __restrict__ nodes, float* __restrict__ bounds,
                                                  TopArrays top) {
    if (!fb.taken()) return;
    const int lane = threadIdx.x & 63;
    const uint32_t nb = gridDim.x, cnt = top.count[blockIdx.x];
    for (uint32_t i = threadIdx.x >> 6; i < cnt; i += blockDim.x >> 6) {
        const TopEntry t = top.list[(uint64_t)blockIdx.x * kTopMax + i];
        const int64_t p = t.p, edge = (int64_t)blockIdx.x * kTreeBlock;
        int64_t lo = t.lo, hi1 = t.hi1;
        // slots of the node are those that share its d leading bits
        const auto prefix = [&](int64_t x) { return key_prefix(keys[x], t.key, x, p); };
        if (lo < 0) lo = wave_first(0, edge - 1, lane, [&](int64_t x) { return prefix(x) >= t.diff; });
        if (hi1 < 0) hi1 = wave_first(edge + kTreeBlock, n, lane, [&](int64_t x) { return prefix(x) < t.diff; });
        const bool root = lo == 0 && hi1 == (int64_t)n;
        const bool right = diff_at(keys, n, lo) > diff_at(keys, n, hi1);
        const bool l_in = lo / kTreeBlock == (p - 1) / kTreeBlock;
        const bool r_in = p / kTreeBlock == (hi1 - 1) / kTreeBlock;
        const Box l = l_in ? load_box(top.child + 4 * (uint64_t)p) : wave_range_box(top, lo, p, n, nb, lane);
        const Box r = r_in ? load_box(top.child + 4 * (uint64_t)p + 2) : wave_range_box(top, p, hi1, n, nb, lane);
        if (lane == 0) {
            store_tree_node(nodes, root ? 0u : (uint32_t)(right ? lo : hi1 - 1), (uint32_t)lo, (uint32_t)p,
                            (uint32_t)hi1, l, r);
            if (root) store_bounds(bounds, unite(l, r));
        }
    }
}

__global__ void k_zero_word(uint32_t* w) { *w = 0u; }

// Traversals keep pending nodes on stacks sized for trees at most kMaxTreeDepth internal levels
// deep (the Karras tree over 62-bit keys has at most 62). A PLOC tree has no such bound (a chain of
// clusters can nest deeper), so its depth is measured: per triangle, the internal nodes above it
// (leaves of the parent array at ni + primitive), counted up to kMaxTreeDepth + 1.
constexpr uint32_t kMaxTreeDepth = 62;

__global__ void __launch_bounds__(256) k_ploc_depth(uint32_t n, const int32_t* __restrict__ parent,
                                                     uint32_t* __restrict__ depth) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    int32_t x = parent[(uint64_t)(n - 1) + i];
    uint32_t d = 0;
    while (x >= 0 && d <= kMaxTreeDepth) {
        ++d;
        x = parent[x];
    }
    if (d > kMaxTreeDepth) atomicMax(depth, d);
}

// ---- PLOC builder (parallel locally-ordered clustering, Meister & Bittner 2018) ----
// Clusters start as the triangles in Morton order (positions 0..n-1, refs ~prim, padded leaf
// boxes). Each iteration: every cluster i picks its nearest neighbour NN(i) among positions
// [i-R, i+R] (smallest surface area of the union box, ties to the smaller position); mutual pairs
// merge into a new node kept at the lower position, the higher one drops out, survivors keep their
// order. An iteration with no mutual pair (possible only with NaN boxes) merges positions 0 and 1.
// The k-th node created (over iterations, in position order) gets id n-2-k: the root is 0 and
// children have larger ids than their parents. Large iterations run as two grid launches
// (the pairs and their counts per tile; compaction), which take 9 us an iteration of a build of 151,380 triangles
// where four (neighbours, counts, offsets, compaction) took 18; once at most kPlocTail clusters remain,
// one workgroup finishes in a single launch. Subtrees of at most
// kLeafMax triangles whose parent is larger become leaves: leaf roots take consecutive slot ranges
// in the order of their smallest Morton position, their triangles left to right.
constexpr int kPlocRadius = 16;
constexpr int kPlocTile = 256;        // clusters per neighbour-search tile (one per thread)
constexpr int kPlocChunk = 1024;      // values per chunk of the slot scan (4 per thread)
constexpr int kPlocGrid = 1024;       // blocks of the grid-stride iteration kernels
// cluster count handed to the one-workgroup tail: above 2,048 an iteration there (15 to 20 us) costs more than
// two launches (9 us); from 4,096 on a build of 151,380 triangles took 650 us, from 2,048 on 590
constexpr int32_t kPlocTail = 2048;

// state[4 * parity]: clusters m, nodes created, buffer parity of the clusters

RT_DEV float union_area(const float4& alo, const float4& ahi, const float4& blo, const float4& bhi) {
    const float dx = fmaxf(ahi.x, bhi.x) - fminf(alo.x, blo.x);
    const float dy = fmaxf(ahi.y, bhi.y) - fminf(alo.y, blo.y);
    const float dz = fmaxf(ahi.z, bhi.z) - fminf(alo.z, blo.z);
    return dx * dy + dy * dz + dz * dx;
}

RT_DEV int32_t ploc_size(const int32_t* __restrict__ nsize, int32_t c) { return c >= 0 ? nsize[c] : 1; }

__global__ void __launch_bounds__(256) k_ploc_init(const uint32_t* __restrict__ morder, uint32_t n,
                                                    const MeshSource* __restrict__ meshes, uint32_t n_sources,
                                                    int32_t* __restrict__ cid, float4* __restrict__ cbox,
                                                    uint32_t* __restrict__ pos_of,
                                                    int32_t* __restrict__ parent, int32_t* __restrict__ state) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const uint32_t p = morder[i];
    pos_of[p] = i;
    cid[i] = ~(int32_t)p;
    const MeshSource& src = mesh_of(meshes, n_sources, p);
    uint32_t v[3];
    float3 c[3];
    load_corners(src.d, p - src.base, v, c);
    store_box(cbox + 2 * (uint64_t)i, padded(corners_box(c)));
    if (i == 0) {
        parent[0] = -1;
        state[0] = (int32_t)n;
        state[1] = 0;
        state[2] = 0;
    }
}

// nearest neighbour of position i among [i-R, i+R] (m >= 2), reading boxes through `box(j)`
template <typename BoxAt>
RT_DEV int32_t ploc_nn(int32_t i, int32_t m, BoxAt box) {
    const int32_t lo = i - kPlocRadius < 0 ? 0 : i - kPlocRadius;
    const int32_t hi = i + kPlocRadius > m - 1 ? m - 1 : i + kPlocRadius;
    float4 ilo, ihi, jlo, jhi;
    box(i, ilo, ihi);
    int32_t bj = lo == i ? i + 1 : lo;
    box(bj, jlo, jhi);
    float best = union_area(ilo, ihi, jlo, jhi);
    // no branch for j == i, so that the loads of 8 candidates go out together (k_ploc_pairs 5.4 -> 4.8 us on
    // average over the iterations of 151,380 triangles)
#pragma unroll 8
    for (int32_t j = bj + 1; j <= hi; ++j) {
        box(j, jlo, jhi);
        const float a = union_area(ilo, ihi, jlo, jhi);
        const bool take = (a < best) & (j != i);
        best = take ? a : best;
        bj = take ? j : bj;
    }
    return bj;
}

// First kernel of an iteration: the mutual pairs of a tile of kPlocTile positions. The neighbours of the
// kPlocRadius positions on either side are searched again here, so that a pair is known without another
// launch. mate[i] is the position i merges with, or -1; part[tile] = positions kept | merges << 16.
// 33 union boxes per position make it VALU work: 2.4 us for 150,000 positions, behind a launch's latency.
constexpr int kPlocLoad = kPlocTile + 4 * kPlocRadius;  // boxes a tile's searches read, one per thread

__global__ void __launch_bounds__(kPlocLoad) k_ploc_pairs(int it, const int32_t* __restrict__ state,
                                                          const float4* __restrict__ cbox0,
                                                          const float4* __restrict__ cbox1,
                                                          int32_t* __restrict__ mate,
                                                          uint32_t* __restrict__ part) {
    const int32_t m = state[4 * (it & 1)];
    if (m <= kPlocTail) return;
    const float4* __restrict__ B = (it & 1) ? cbox1 : cbox0;
    __shared__ float4 wlo[kPlocLoad], whi[kPlocLoad];
    __shared__ int32_t nn[kPlocTile + 2 * kPlocRadius];
    __shared__ uint32_t wcount[kPlocTile / 64];
    const int32_t t = threadIdx.x, ntile = (m + kPlocTile - 1) / kPlocTile;
    for (int32_t tile = blockIdx.x; tile < ntile; tile += gridDim.x) {
        const int32_t nb = tile * kPlocTile - kPlocRadius, wb = nb - kPlocRadius;
        if (wb + t >= 0 && wb + t < m) {
            wlo[t] = B[2 * (uint64_t)(wb + t)];
            whi[t] = B[2 * (uint64_t)(wb + t) + 1];
        }
        __syncthreads();
        if (t < kPlocTile + 2 * kPlocRadius && nb + t >= 0 && nb + t < m)
            nn[t] = ploc_nn(nb + t, m, [&](int32_t j, float4& lo, float4& hi) {
                lo = wlo[j - wb];
                hi = whi[j - wb];
            });
        __syncthreads();
        if (t < kPlocTile) {
            const int32_t i = tile * kPlocTile + t;
            bool keep = false, merge = false;
            if (i < m) {
                const int32_t j = nn[i - nb];
                const bool mutual = nn[j - nb] == i;
                keep = !mutual || i < j;
                merge = mutual && i < j;
                mate[i] = mutual ? j : -1;
            }
            const uint32_t c = (uint32_t)__popcll(__ballot(keep)) | ((uint32_t)__popcll(__ballot(merge)) << 16);
            if ((t & 63) == 0) wcount[t >> 6] = c;
        }
        __syncthreads();
        if (t == 0) part[tile] = wcount[0] + wcount[1] + wcount[2] + wcount[3];
    }
}

// keep / merge flags of position i from the neighbours nn (forced: the fallback merge of 0 and 1)
RT_DEV void ploc_flags(const int32_t* __restrict__ nn, int32_t i, bool forced, uint32_t& keep,
                       uint32_t& merge) {
    if (forced) {
        keep = i != 1;
        merge = i == 0;
        return;
    }
    const int32_t j = nn[i];
    const bool mutual = nn[j] == i;
    keep = !mutual || i < j;
    merge = mutual && i < j;
}

// Exclusive scan of one value per thread over a block of T threads (T = blockDim.x); `total` is
// the block's sum. The PLOC kernels scan (keep, merge) counts packed as keep | merge << 32.
template <int T>
RT_DEV uint64_t block_exclusive_scan(uint64_t v, uint64_t* lds, uint64_t& total) {
    const int t = threadIdx.x;
    lds[t] = v;
    __syncthreads();
    for (int d = 1; d < T; d <<= 1) {
        const uint64_t x = t >= d ? lds[t - d] : 0;
        __syncthreads();
        lds[t] += x;
        __syncthreads();
    }
    total = lds[T - 1];
    const uint64_t incl = lds[t];
    __syncthreads();
    return incl - v;
}

// writes the merged node `id` from the clusters at positions i < j
RT_DEV void ploc_merge(uint32_t n, int32_t id, int32_t ci, int32_t cj, int32_t size, float4 ilo, float4 ihi,
                       float4 jlo, float4 jhi, int32_t* __restrict__ nleft, int32_t* __restrict__ nright,
                       int32_t* __restrict__ nsize, int32_t* __restrict__ parent, float4* __restrict__ nodes,
                       float* __restrict__ bounds, float4& ulo, float4& uhi) {
    const uint64_t ni = (uint64_t)n - 1;
    nleft[id] = ci;
    nright[id] = cj;
    nsize[id] = size;
    parent[ci >= 0 ? (uint64_t)ci : ni + (uint64_t)(~ci)] = id;
    parent[cj >= 0 ? (uint64_t)cj : ni + (uint64_t)(~cj)] = id;
    float4* nd = nodes + (uint64_t)id * 4;
    nd[0] = make_float4(ilo.x, ihi.x, ilo.y, ihi.y);
    nd[1] = make_float4(jlo.x, jhi.x, jlo.y, jhi.y);
    nd[2] = make_float4(ilo.z, ihi.z, jlo.z, jhi.z);
    ulo = make_float4(fminf(ilo.x, jlo.x), fminf(ilo.y, jlo.y), fminf(ilo.z, jlo.z), 0.0f);
    uhi = make_float4(fmaxf(ihi.x, jhi.x), fmaxf(ihi.y, jhi.y), fmaxf(ihi.z, jhi.z), 0.0f);
    if (id == 0) {
        bounds[0] = ulo.x; bounds[1] = ulo.y; bounds[2] = ulo.z; bounds[3] = 0.0f;
        bounds[4] = uhi.x; bounds[5] = uhi.y; bounds[6] = uhi.z; bounds[7] = 0.0f;
    }
}

// Second kernel of an iteration: survivors to their new positions, merged pairs as new nodes. A workgroup
// takes consecutive tiles and sums the counts of all tiles before its own itself (586 words at 150,000
// positions), so the iteration needs no scan launch; one sum over all says whether any pair merged.
__global__ void __launch_bounds__(kPlocTile) k_ploc_compact(int it, uint32_t n, int32_t* __restrict__ state,
                                                            const int32_t* __restrict__ mate,
                                                            const uint32_t* __restrict__ part,
                                                            int32_t* __restrict__ cid0, int32_t* __restrict__ cid1,
                                                            float4* __restrict__ cbox0, float4* __restrict__ cbox1,
                                                            int32_t* __restrict__ nleft, int32_t* __restrict__ nright,
                                                            int32_t* __restrict__ nsize, int32_t* __restrict__ parent,
                                                            float4* __restrict__ nodes, float* __restrict__ bounds) {
    constexpr int kWaves = kPlocTile / 64;
    const int32_t* cur = state + 4 * (it & 1);
    int32_t* nxt = state + 4 * ((it + 1) & 1);
    const int32_t m = cur[0], created = cur[1];
    const int32_t t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const bool writer = blockIdx.x == 0 && t == 0;
    if (m <= kPlocTail) {
        if (writer) {
            nxt[0] = m;
            nxt[1] = created;
            nxt[2] = cur[2];
        }
        return;
    }
    const int32_t* __restrict__ C = (it & 1) ? cid1 : cid0;
    const float4* __restrict__ B = (it & 1) ? cbox1 : cbox0;
    int32_t* __restrict__ C2 = (it & 1) ? cid0 : cid1;
    float4* __restrict__ B2 = (it & 1) ? cbox0 : cbox1;
    __shared__ uint64_t wsum[2][kWaves];
    __shared__ uint32_t wcount[2][kWaves];
    const int32_t ntile = (m + kPlocTile - 1) / kPlocTile;
    const int32_t per = (ntile + (int32_t)gridDim.x - 1) / (int32_t)gridDim.x;
    const int32_t t0 = (int32_t)blockIdx.x * per, t1 = t0 + per < ntile ? t0 + per : ntile;
    uint64_t before = 0, all = 0;  // kept | merged << 32
#pragma unroll 4
    for (int32_t k = t; k < ntile; k += kPlocTile) {
        const uint64_t v = (uint64_t)(part[k] & 0xFFFFu) | ((uint64_t)(part[k] >> 16) << 32);
        all += v;
        before += k < t0 ? v : 0;
    }
    for (int x = 1; x < 64; x <<= 1) {
        all += __shfl_xor((unsigned long long)all, x);
        before += __shfl_xor((unsigned long long)before, x);
    }
    if (lane == 0) {
        wsum[0][wave] = all;
        wsum[1][wave] = before;
    }
    __syncthreads();
    all = before = 0;
    for (int w = 0; w < kWaves; ++w) {
        all += wsum[0][w];
        before += wsum[1][w];
    }
    const bool forced = (all >> 32) == 0;
    if (writer) {
        nxt[0] = forced ? m - 1 : (int32_t)(uint32_t)all;
        nxt[1] = created + (forced ? 1 : (int32_t)(all >> 32));
        nxt[2] = (it + 1) & 1;
    }
    uint32_t kept = (uint32_t)before, merged = (uint32_t)(before >> 32);
    const uint64_t below = (1ull << lane) - 1;
    for (int32_t tile = t0; tile < t1; ++tile) {
        const int32_t i = tile * kPlocTile + t, j = forced ? 1 : i < m ? mate[i] : -1;
        const bool keep = i < m && (forced ? i != 1 : j < 0 || i < j);
        const bool merge = i < m && (forced ? i == 0 : j > i);
        const uint64_t kb = __ballot(keep), mb = __ballot(merge);
        uint32_t* wc = wcount[(tile - t0) & 1];
        if (lane == 0) wc[wave] = (uint32_t)__popcll(kb) | ((uint32_t)__popcll(mb) << 16);
        __syncthreads();
        uint32_t dst = kept + (uint32_t)__popcll(kb & below), rank = merged + (uint32_t)__popcll(mb & below);
        for (int w = 0; w < kWaves; ++w) {
            const uint32_t c = wc[w];
            if (w < wave) {
                dst += c & 0xFFFFu;
                rank += c >> 16;
            }
            kept += c & 0xFFFFu;
            merged += c >> 16;
        }
        if (!keep) continue;
        if (forced) {
            dst = i == 0 ? 0u : (uint32_t)(i - 1);
            rank = 0;
        }
        float4 lo = B[2 * (uint64_t)i], hi = B[2 * (uint64_t)i + 1];
        int32_t c = C[i];
        if (merge) {
            const int32_t cj = C[j], id = (int32_t)n - 2 - (created + (int32_t)rank);
            float4 ulo, uhi;
            ploc_merge(n, id, c, cj, ploc_size(nsize, c) + ploc_size(nsize, cj), lo, hi, B[2 * (uint64_t)j],
                       B[2 * (uint64_t)j + 1], nleft, nright, nsize, parent, nodes, bounds, ulo, uhi);
            c = id;
            lo = ulo;
            hi = uhi;
        }
        C2[dst] = c;
        B2[2 * (uint64_t)dst] = lo;
        B2[2 * (uint64_t)dst + 1] = hi;
    }
}

// Nearest neighbour of position i among [i - R, i + R] by 2^lg consecutive lanes, lane q
// taking a share of the candidates in order; valid in lane 0. The same as ploc_nn: only the first
// candidate counts before it was compared, so a box of NaN keeps it, and a tie goes to the smaller position.
template <typename AreaTo>
RT_DEV int32_t ploc_nn_lanes(int32_t i, int32_t m, int lg, int q, AreaTo area) {
    const int32_t lo = i - kPlocRadius < 0 ? 0 : i - kPlocRadius;
    const int32_t hi = i + kPlocRadius > m - 1 ? m - 1 : i + kPlocRadius;
    const int32_t count = hi - lo, share = (count + (1 << lg) - 1) >> lg;
    int32_t k = q * share;
    const int32_t end = k + share < count ? k + share : count;
    float best = INFINITY;
    int32_t bj = -1;
    if (q == 0) {
        bj = lo == i ? i + 1 : lo;
        best = area(bj);
        k = 1;
    }
#pragma unroll 4
    for (; k < end; ++k) {
        const int32_t j = lo + k + (lo + k >= i ? 1 : 0);
        const float a = area(j);
        if (a < best) {
            best = a;
            bj = j;
        }
    }
    for (int x = 1; x < 1 << lg; x <<= 1) {
        const float oa = __shfl_down(best, x);
        const int32_t oj = __shfl_down(bj, x);
        if (oa < best) {
            best = oa;
            bj = oj;
        }
    }
    return bj;
}

// The remaining iterations in one workgroup, from the state left in state[4 * slot]: more than kPlocTail
// clusters (only if the launched iterations merged less than expected) through memory, the rest in LDS,
// where a search costs no L2 round trips, sizes need no loads and the compaction counts by ballots.
// From 512 clusters down several lanes share a search. The 65 or so iterations from 4,096 clusters on
// took 499 us through memory, 229 like this; those from 2,048 on take 120.
__global__ void __launch_bounds__(1024) k_ploc_tail(int slot, uint32_t n, int32_t* __restrict__ state,
                                                     int32_t* __restrict__ nn, int32_t* __restrict__ cid0,
                                                     int32_t* __restrict__ cid1, float4* __restrict__ cbox0,
                                                     float4* __restrict__ cbox1, int32_t* __restrict__ nleft,
                                                     int32_t* __restrict__ nright, int32_t* __restrict__ nsize,
                                                     int32_t* __restrict__ parent, float4* __restrict__ nodes,
                                                     float* __restrict__ bounds) {
    __shared__ uint64_t lds[1024];
    __shared__ int32_t sm, screated;
    __shared__ uint32_t smerged;
    __shared__ uint64_t carry;
    if (threadIdx.x == 0) {
        sm = state[4 * slot];
        screated = state[4 * slot + 1];
    }
    int par = state[4 * slot + 2];
    __syncthreads();
    for (;;) {
        const int32_t m = sm, created = screated;
        if (m <= kPlocTail) break;
        const int32_t* __restrict__ C = par ? cid1 : cid0;
        const float4* __restrict__ B = par ? cbox1 : cbox0;
        int32_t* __restrict__ C2 = par ? cid0 : cid1;
        float4* __restrict__ B2 = par ? cbox0 : cbox1;
        for (int32_t i = threadIdx.x; i < m; i += blockDim.x)
            nn[i] = ploc_nn(i, m, [&](int32_t j, float4& lo, float4& hi) {
                lo = B[2 * (uint64_t)j];
                hi = B[2 * (uint64_t)j + 1];
            });
        if (threadIdx.x == 0) smerged = 0;
        __syncthreads();
        uint32_t mine = 0;
        for (int32_t i = threadIdx.x; i < m; i += blockDim.x) {
            uint32_t keep, merge;
            ploc_flags(nn, i, false, keep, merge);
            mine += merge;
        }
        if (mine) atomicAdd(&smerged, mine);
        __syncthreads();
        const bool forced = smerged == 0;
        if (threadIdx.x == 0) carry = 0;
        __syncthreads();
        for (int32_t b = 0; b < m; b += 4 * (int32_t)blockDim.x) {
            uint32_t keep[4], merge[4];
            uint64_t v = 0;
            for (int q = 0; q < 4; ++q) {
                const int32_t i = b + (int32_t)threadIdx.x * 4 + q;
                keep[q] = merge[q] = 0;
                if (i < m) ploc_flags(nn, i, forced, keep[q], merge[q]);
                v += (uint64_t)keep[q] | ((uint64_t)merge[q] << 32);
            }
            uint64_t total;
            const uint64_t ex = block_exclusive_scan<1024>(v, lds, total) + carry;
            uint32_t dst = (uint32_t)ex, rank = (uint32_t)(ex >> 32);
            for (int q = 0; q < 4; ++q) {
                const int32_t i = b + (int32_t)threadIdx.x * 4 + q;
                if (!keep[q]) continue;
                if (forced) dst = i == 0 ? 0u : (uint32_t)(i - 1);
                const float4 ilo = B[2 * (uint64_t)i], ihi = B[2 * (uint64_t)i + 1];
                if (merge[q]) {
                    const int32_t j = forced ? 1 : nn[i];
                    const int32_t id = (int32_t)n - 2 - (created + (int32_t)rank);
                    float4 ulo, uhi;
                    ploc_merge(n, id, C[i], C[j], ploc_size(nsize, C[i]) + ploc_size(nsize, C[j]), ilo, ihi,
                               B[2 * (uint64_t)j], B[2 * (uint64_t)j + 1], nleft, nright, nsize, parent, nodes, bounds, ulo, uhi);
                    C2[dst] = id;
                    B2[2 * (uint64_t)dst] = ulo;
                    B2[2 * (uint64_t)dst + 1] = uhi;
                    ++rank;
                } else {
                    C2[dst] = C[i];
                    B2[2 * (uint64_t)dst] = ilo;
                    B2[2 * (uint64_t)dst + 1] = ihi;
                }
                ++dst;
            }
            __syncthreads();
            if (threadIdx.x == 0) carry += total;
            __syncthreads();
        }
        if (threadIdx.x == 0) {
            sm = forced ? m - 1 : (int32_t)(uint32_t)carry;
            screated = created + (forced ? 1 : (int32_t)(carry >> 32));
        }
        par ^= 1;
        __syncthreads();
    }
    constexpr int kPer = kPlocTail / 1024, kWaves = 16;
    __shared__ float box[6][kPlocTail];
    __shared__ int32_t cid[kPlocTail], csize[kPlocTail];
    __shared__ uint16_t near[kPlocTail];
    __shared__ uint32_t wcount[kPer * kWaves];  // per 64 positions: kept | merged << 16
    int32_t m = sm, created = screated;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    {
        const int32_t* __restrict__ C = par ? cid1 : cid0;
        const float4* __restrict__ B = par ? cbox1 : cbox0;
        for (int32_t i = tid; i < m; i += 1024) {
            const Box b = load_box(B + 2 * (uint64_t)i);
            for (int a = 0; a < 3; ++a) {
                box[a][i] = b.lo[a];
                box[3 + a][i] = b.hi[a];
            }
            cid[i] = C[i];
            csize[i] = ploc_size(nsize, C[i]);
        }
    }
    __syncthreads();
    auto lo_of = [&](int32_t i) { return make_float4(box[0][i], box[1][i], box[2][i], 0.0f); };
    auto hi_of = [&](int32_t i) { return make_float4(box[3][i], box[4][i], box[5][i], 0.0f); };
    while (m > 1) {
        const int lg = m > 512 ? 0 : m > 256 ? 1 : m > 128 ? 2 : m > 64 ? 3 : 4;  // 2^lg lanes per search
        for (int32_t w = tid; w < m << lg; w += 1024) {  // one round where lg > 0
            const int32_t i = w >> lg, q = w & ((1 << lg) - 1);
            const float4 lo = lo_of(i), hi = hi_of(i);
            const int32_t j = ploc_nn_lanes(i, m, lg, q, [&](int32_t j) { return union_area(lo, hi, lo_of(j), hi_of(j)); });
            if (q == 0) near[i] = (uint16_t)j;
        }
        __syncthreads();
        bool keep[kPer], merge[kPer];
        int32_t mate[kPer];
        uint64_t kb[kPer], mb[kPer];
#pragma unroll
        for (int c = 0; c < kPer; ++c) {
            const int32_t i = tid + c * 1024;
            keep[c] = merge[c] = false;
            mate[c] = 0;
            if (i < m) {
                mate[c] = near[i];
                const bool mutual = near[mate[c]] == i;
                keep[c] = !mutual || i < mate[c];
                merge[c] = mutual && i < mate[c];
            }
            kb[c] = __ballot(keep[c]);
            mb[c] = __ballot(merge[c]);
            if (lane == 0) wcount[c * kWaves + wave] = (uint32_t)__popcll(kb[c]) | ((uint32_t)__popcll(mb[c]) << 16);
        }
        __syncthreads();
        const uint32_t own = lane < kPer * kWaves ? wcount[lane] : 0u;  // every wave scans the counts
        uint32_t incl = own;
        for (int x = 1; x < 64; x <<= 1) {
            const uint32_t v = __shfl_up(incl, x);
            if (lane >= x) incl += v;
        }
        const uint32_t total = __shfl(incl, 63);
        const bool forced = (total >> 16) == 0;
        const uint64_t below = (1ull << lane) - 1;
        Box bi[kPer], bj[kPer];
        int32_t ci[kPer], cj[kPer], si[kPer], sj[kPer];
        uint32_t dst[kPer], rank[kPer];
#pragma unroll
        for (int c = 0; c < kPer; ++c) {
            const int32_t i = tid + c * 1024;
            const uint32_t at = __shfl(incl - own, c * kWaves + wave);
            dst[c] = (at & 0xFFFFu) + (uint32_t)__popcll(kb[c] & below);
            rank[c] = (at >> 16) + (uint32_t)__popcll(mb[c] & below);
            if (forced) {
                keep[c] = i < m && i != 1;
                merge[c] = i == 0;
                mate[c] = 1;
                dst[c] = i == 0 ? 0u : (uint32_t)(i - 1);
                rank[c] = 0;
            }
            if (keep[c]) {
                const int32_t j = merge[c] ? mate[c] : i;
                for (int a = 0; a < 3; ++a) {
                    bi[c].lo[a] = box[a][i];
                    bi[c].hi[a] = box[3 + a][i];
                    bj[c].lo[a] = box[a][j];
                    bj[c].hi[a] = box[3 + a][j];
                }
                ci[c] = cid[i];
                cj[c] = cid[j];
                si[c] = csize[i];
                sj[c] = csize[j];
            }
        }
        __syncthreads();
#pragma unroll
        for (int c = 0; c < kPer; ++c) {
            if (!keep[c]) continue;
            float4 ulo = make_float4(bi[c].lo[0], bi[c].lo[1], bi[c].lo[2], 0.0f);
            float4 uhi = make_float4(bi[c].hi[0], bi[c].hi[1], bi[c].hi[2], 0.0f);
            if (merge[c]) {
                const float4 ilo = ulo, ihi = uhi;
                const int32_t id = (int32_t)n - 2 - (created + (int32_t)rank[c]);
                si[c] += sj[c];
                ploc_merge(n, id, ci[c], cj[c], si[c], ilo, ihi,
                           make_float4(bj[c].lo[0], bj[c].lo[1], bj[c].lo[2], 0.0f),
                           make_float4(bj[c].hi[0], bj[c].hi[1], bj[c].hi[2], 0.0f), nleft, nright, nsize, parent,
                           nodes, bounds, ulo, uhi);
                ci[c] = id;
            }
            box[0][dst[c]] = ulo.x; box[1][dst[c]] = ulo.y; box[2][dst[c]] = ulo.z;
            box[3][dst[c]] = uhi.x; box[4][dst[c]] = uhi.y; box[5][dst[c]] = uhi.z;
            cid[dst[c]] = ci[c];
            csize[dst[c]] = si[c];
        }
        m = forced ? m - 1 : (int32_t)(total & 0xFFFFu);
        created += forced ? 1 : (int32_t)(total >> 16);
        __syncthreads();
    }
}

// leaf root of primitive p: walk up while the parent holds at most kLeafMax triangles
RT_DEV int32_t ploc_leaf_root(uint32_t n, const int32_t* __restrict__ parent,
                              const int32_t* __restrict__ nsize, uint32_t p) {
    const uint64_t ni = (uint64_t)n - 1;
    int32_t x = ~(int32_t)p;
    for (;;) {
        const int32_t q = parent[x >= 0 ? (uint64_t)x : ni + (uint64_t)(~x)];
        if (q < 0 || nsize[q] > kLeafMax) return x;
        x = q;
    }
}

// smallest Morton position among the (at most kLeafMax) triangles under x
RT_DEV uint32_t ploc_minpos(int32_t x, const int32_t* __restrict__ nleft, const int32_t* __restrict__ nright,
                            const uint32_t* __restrict__ pos_of) {
    int32_t stk[2 * kLeafMax];
    int sp = 0;
    stk[sp++] = x;
    uint32_t best = 0xFFFFFFFFu;
    while (sp) {
        const int32_t c = stk[--sp];
        if (c < 0) {
            const uint32_t q = pos_of[~c];
            best = q < best ? q : best;
        } else if (sp + 2 <= 2 * kLeafMax) {  // always true for a subtree of <= kLeafMax triangles
            stk[sp++] = nright[c];
            stk[sp++] = nleft[c];
        }
    }
    return best;
}

__global__ void __launch_bounds__(256) k_ploc_leafroots(uint32_t n, const uint32_t* __restrict__ deep,
                                                         const uint32_t* __restrict__ morder,
                                                         const int32_t* __restrict__ parent,
                                                         const int32_t* __restrict__ nsize,
                                                         const int32_t* __restrict__ nleft,
                                                         const int32_t* __restrict__ nright,
                                                         const uint32_t* __restrict__ pos_of,
                                                         uint32_t* __restrict__ scan) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n || *deep) return;
    const int32_t x = ploc_leaf_root(n, parent, nsize, morder[i]);
    scan[i] = ploc_minpos(x, nleft, nright, pos_of) == i ? (uint32_t)ploc_size(nsize, x) : 0u;
}

// exclusive scan of scan[0..n) in place: per-chunk totals, chunk offsets, chunk scans
__global__ void __launch_bounds__(256) k_scan_chunks(uint32_t n, const uint32_t* __restrict__ a,
                                                      uint32_t* __restrict__ part) {
    __shared__ uint64_t lds[256];
    const uint32_t c = blockIdx.x;
    uint64_t v = 0;
    for (int q = 0; q < 4; ++q) {
        const uint64_t i = (uint64_t)c * kPlocChunk + threadIdx.x * 4 + q;
        if (i < n) v += a[i];
    }
    uint64_t total;
    block_exclusive_scan<256>(v, lds, total);
    if (threadIdx.x == 0) part[c] = (uint32_t)total;
}

__global__ void __launch_bounds__(1024) k_scan_top(uint32_t nchunk, uint32_t* __restrict__ part) {
    __shared__ uint64_t lds[1024];
    __shared__ uint64_t carry;
    if (threadIdx.x == 0) carry = 0;
    __syncthreads();
    for (uint32_t b = 0; b < nchunk; b += 1024) {
        const uint32_t c = b + threadIdx.x;
        const uint64_t v = c < nchunk ? part[c] : 0;
        uint64_t total;
        const uint64_t ex = block_exclusive_scan<1024>(v, lds, total) + carry;
        if (c < nchunk) part[c] = (uint32_t)ex;
        __syncthreads();
        if (threadIdx.x == 0) carry += total;
        __syncthreads();
    }
}

__global__ void __launch_bounds__(256) k_scan_apply(uint32_t n, uint32_t* __restrict__ a,
                                                     const uint32_t* __restrict__ part) {
    __shared__ uint64_t lds[256];
    const uint32_t c = blockIdx.x;
    uint32_t x[4];
    uint64_t v = 0;
    for (int q = 0; q < 4; ++q) {
        const uint64_t i = (uint64_t)c * kPlocChunk + threadIdx.x * 4 + q;
        x[q] = i < n ? a[i] : 0u;
        v += x[q];
    }
    uint64_t total;
    uint64_t run = block_exclusive_scan<256>(v, lds, total) + part[c];
    for (int q = 0; q < 4; ++q) {
        const uint64_t i = (uint64_t)c * kPlocChunk + threadIdx.x * 4 + q;
        if (i < n) a[i] = (uint32_t)run;
        run += x[q];
    }
}

// slots of the leaf root whose smallest Morton position is i: its triangles left to right from
// the root's first slot; first slots of its internal nodes
__global__ void __launch_bounds__(256) k_ploc_slots(uint32_t n, const uint32_t* __restrict__ deep,
                                                         const uint32_t* __restrict__ morder,
                                                     const int32_t* __restrict__ parent,
                                                     const int32_t* __restrict__ nsize,
                                                     const int32_t* __restrict__ nleft,
                                                     const int32_t* __restrict__ nright,
                                                     const uint32_t* __restrict__ pos_of,
                                                     const uint32_t* __restrict__ scan,
                                                     uint32_t* __restrict__ slot_order,
                                                     uint32_t* __restrict__ slot_of,
                                                     uint32_t* __restrict__ fslot) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n || *deep) return;
    const int32_t x = ploc_leaf_root(n, parent, nsize, morder[i]);
    if (ploc_minpos(x, nleft, nright, pos_of) != i) return;
    uint32_t next = scan[i];
    int32_t stk[2 * kLeafMax];
    int sp = 0;
    stk[sp++] = x;
    while (sp) {
        const int32_t c = stk[--sp];
        if (c < 0) {
            slot_order[next] = (uint32_t)~c;
            slot_of[~c] = next;
            ++next;
        } else if (sp + 2 <= 2 * kLeafMax) {  // always true for a subtree of <= kLeafMax triangles
            fslot[c] = next;
            stk[sp++] = nright[c];
            stk[sp++] = nleft[c];
        }
    }
}

// traversal refs of every internal node: a child of more than kLeafMax triangles by id, else the
// leaf of its slots
__global__ void __launch_bounds__(256) k_ploc_refs(uint32_t n, const uint32_t* __restrict__ deep,
                                                    const int32_t* __restrict__ nleft,
                                                    const int32_t* __restrict__ nright,
                                                    const int32_t* __restrict__ nsize,
                                                    const uint32_t* __restrict__ slot_of,
                                                    const uint32_t* __restrict__ fslot,
                                                    float4* __restrict__ nodes) {
    const uint32_t x = blockIdx.x * blockDim.x + threadIdx.x;
    if (x >= n - 1 || *deep) return;
    auto tref = [&](int32_t c) -> int32_t {
        if (c < 0) return leaf_ref(slot_of[~c], 1u);
        if (nsize[c] > kLeafMax) return c;
        return leaf_ref(fslot[c], (uint32_t)nsize[c]);
    };
    nodes[(uint64_t)x * 4 + 3] = make_float4(__int_as_float(tref(nleft[x])), __int_as_float(tref(nright[x])),
                                             0.0f, 0.0f);
}

// big PLOC iterations to launch for n clusters: enough for m to fall to kPlocTail at 0.88 per
// iteration (measured ~0.83-0.90), plus margin; the tail finishes whatever remains
inline int ploc_iterations(uint32_t n) {
    if (n <= (uint32_t)kPlocTail) return 0;
    return (int)std::ceil(std::log((double)n / kPlocTail) / std::log(1.0 / 0.88)) + 4;
}


// ---- 4-wide nodes ----
// nodes4[i] (8 x float4, 128 B) lists the grandchildren of binary node i reached through its
// internal children, and its leaf children directly, in the order (left..., right...):
//   [0]=lo.x[4] [1]=hi.x[4] [2]=lo.y[4] [3]=hi.y[4] [4]=lo.z[4] [5]=hi.z[4] [6]=refs[4] [7]=0
// Unused slots hold ref RT_EMPTY_ROOT and an empty box (lo=+inf, hi=-inf). Every binary node gets
// a record (traversal from the root only reaches every other level), so refs stay binary ids.
// 4-wide record of binary node i: the boxes and references of its grandchildren (a child that is a
// leaf stands for itself), empty slots padded. The block's 256 records are staged in LDS (a
// 144-byte stride keeps the per-lane writes off one bank) and stored as consecutive float4s, so
// every store instruction writes 4 KB of the output contiguously. (Loading the block's binary
// records through LDS as well measured slower: they are read once and the child reads hit L2.)
template <bool PAST>
__global__ void __launch_bounds__(256) k_wide(uint32_t n, const float4* __restrict__ nodes,
                                              float4* __restrict__ nodes4) {
    constexpr int kPitch = 9;  // float4s per staged record
    __shared__ float4 stage[256 * kPitch];
    const uint64_t base = (uint64_t)blockIdx.x * blockDim.x;
    const uint64_t i = base + threadIdx.x;
    const uint64_t m = (uint64_t)n - 1;  // internal nodes
    const uint64_t rows = m - base < 256 ? m - base : 256;  // records of this block
    if (i < m) {
        // slot order: the two children of the left child (or the left child itself if it is a
        // leaf), then those of the right child; every index below is a compile-time constant, so
        // the record stays in registers
        const float4* nd = nodes + i * 4;
        const float4 n0 = nd[0], n1 = nd[1], n2 = nd[2], n3 = nd[3];
        const int32_t c0 = __float_as_int(n3.x), c1 = __float_as_int(n3.y);
        struct Slot {
            float lx, ly, lz, hx, hy, hz;
            int32_t ref;
        };
        // the one or two entries a child contributes: its grandchildren, or itself if a leaf
        auto entries = [&](int32_t c, float4 b, float bz0, float bz1, Slot& e0, Slot& e1) {
            if (c >= 0) {
                const float4* cd = nodes + (uint64_t)c * 4;
                const float4 m0 = cd[0], m1 = cd[1], m2 = cd[2], m3 = cd[3];
                e0 = {m0.x, m0.z, m2.x, m0.y, m0.w, m2.y, __float_as_int(m3.x)};
                e1 = {m1.x, m1.z, m2.z, m1.y, m1.w, m2.w, __float_as_int(m3.y)};
            } else {
                e0 = {b.x, b.z, bz0, b.y, b.w, bz1, c};
                e1 = {INFINITY, INFINITY, INFINITY, -INFINITY, -INFINITY, -INFINITY, RT_EMPTY_ROOT};
            }
        };
        Slot a0, a1, b0, b1;
        entries(c0, n0, n2.x, n2.y, a0, a1);
        entries(c1, n1, n2.z, n2.w, b0, b1);
        const bool two = c0 >= 0;  // the left child contributes two entries
        const Slot e[4] = {a0, two ? a1 : b0, two ? b0 : b1, two ? b1 : a1};
        // (with a leaf left child, slot 3 takes a1: the empty entry)
        float4* o = stage + threadIdx.x * kPitch;
        o[0] = make_float4(e[0].lx, e[1].lx, e[2].lx, e[3].lx);
        o[1] = make_float4(e[0].hx, e[1].hx, e[2].hx, e[3].hx);
        o[2] = make_float4(e[0].ly, e[1].ly, e[2].ly, e[3].ly);
        o[3] = make_float4(e[0].hy, e[1].hy, e[2].hy, e[3].hy);
        o[4] = make_float4(e[0].lz, e[1].lz, e[2].lz, e[3].lz);
        o[5] = make_float4(e[0].hz, e[1].hz, e[2].hz, e[3].hz);
        o[6] = make_float4(__int_as_float(e[0].ref), __int_as_float(e[1].ref), __int_as_float(e[2].ref),
                           __int_as_float(e[3].ref));
        o[7] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    }
    __syncthreads();
    float4* out = nodes4 + base * 8;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        const uint32_t q = j * 256 + threadIdx.x;  // float4 q of the block's output
        if (q < rows * 8) store_last<PAST>(out + q, stage[(q >> 3) * kPitch + (q & 7)]);
    }
}

// Scene of one triangle: no internal node; the root is leaf slot 0.
__global__ void k_single_leaf_bounds(const float4* __restrict__ leafbox, float* __restrict__ bounds) {
    if (threadIdx.x != 0 || blockIdx.x != 0) return;
    const float4 a = leafbox[0], b = leafbox[1];
    bounds[0] = a.x; bounds[1] = a.y; bounds[2] = a.z; bounds[3] = 0.0f;
    bounds[4] = b.x; bounds[5] = b.y; bounds[6] = b.z; bounds[7] = 0.0f;
}

__global__ void k_empty_bounds(float* __restrict__ bounds) {
    if (threadIdx.x != 0 || blockIdx.x != 0) return;
    bounds[0] = bounds[1] = bounds[2] = INFINITY;
    bounds[4] = bounds[5] = bounds[6] = -INFINITY;
    bounds[3] = bounds[7] = 0.0f;
}

__global__ void __launch_bounds__(256) k_copy_if(const uint32_t* __restrict__ deep,
                                                  const uint32_t* __restrict__ a, uint32_t* __restrict__ b,
                                                  uint32_t n) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n && *deep) b[i] = a[i];
}

inline uint32_t blocks_for(uint64_t n, uint32_t per) { return (uint32_t)((n + per - 1) / per); }

// ---- export in the reference's record types (rendering/_raycaster.py:8-22) ----
// BVH_AABB (48 B) as 3 float4: (min.xyz, 0), (max.xyz, 0), (count, elements, 0, 0) as int bits.
RT_DEV void put_aabb(float4* out, uint32_t j, float lx, float ly, float lz, float hx, float hy,
                     float hz, int32_t count, int32_t elements) {
    out[3 * (uint64_t)j] = make_float4(lx, ly, lz, 0.0f);
    out[3 * (uint64_t)j + 1] = make_float4(hx, hy, hz, 0.0f);
    out[3 * (uint64_t)j + 2] = make_float4(__int_as_float(count), __int_as_float(elements), 0.0f, 0.0f);
}

// Breadth-first numbering of the traversal tree in one workgroup: node 0 is the root; the
// children of the internal nodes of one level are appended as pairs in the order of their parents
// (an exclusive scan over each chunk of 1024 nodes of the level), so the numbering is a fixed
// function of the tree. A node's record is written by its parent (box, and its traversal ref
// parked in `elements` with count -1) and completed when its own level is processed (count and
// elements). 2 L - 1 records for L leaves.
__global__ void __launch_bounds__(1024) k_export_nodes(const float4* __restrict__ nodes, int32_t root,
                                                       const float* __restrict__ bounds,
                                                       float4* __restrict__ out,
                                                       uint32_t* __restrict__ n_out) {
    __shared__ uint32_t scan[1024];
    const uint32_t tid = threadIdx.x;
    if (tid == 0)
        put_aabb(out, 0, bounds[0], bounds[1], bounds[2], bounds[4], bounds[5], bounds[6], -1, root);
    __syncthreads();
    uint32_t lo = 0, hi = 1, next = 1;
    while (lo < hi) {
        for (uint32_t base = lo; base < hi; base += 1024) {
            const uint32_t j = base + tid;
            const bool in = j < hi;
            const int32_t ref = in ? __float_as_int(out[3 * (uint64_t)j + 2].y) : 0;
            const uint32_t internal = (in && ref >= 0) ? 1u : 0u;
            scan[tid] = internal;
            __syncthreads();
            for (uint32_t off = 1; off < 1024; off <<= 1) {  // inclusive Hillis-Steele scan
                const uint32_t v = tid >= off ? scan[tid - off] : 0u;
                __syncthreads();
                scan[tid] += v;
                __syncthreads();
            }
            const uint32_t before = scan[tid] - internal, total = scan[1023];
            if (internal) {
                const uint32_t cb = next + 2u * before;
                const float4* nd = nodes + (uint64_t)ref * 4;
                const float4 n0 = nd[0], n1 = nd[1], n2 = nd[2], n3 = nd[3];
                put_aabb(out, cb, n0.x, n0.z, n2.x, n0.y, n0.w, n2.y, -1, __float_as_int(n3.x));
                put_aabb(out, cb + 1, n1.x, n1.z, n2.z, n1.y, n1.w, n2.w, -1, __float_as_int(n3.y));
                out[3 * (uint64_t)j + 2] = make_float4(__int_as_float(0), __int_as_float((int32_t)cb), 0.0f, 0.0f);
            } else if (in) {
                out[3 * (uint64_t)j + 2] = make_float4(__int_as_float((int32_t)leaf_count(ref)),
                                                       __int_as_float((int32_t)leaf_first(ref)), 0.0f, 0.0f);
            }
            next += 2u * total;
            __syncthreads();
        }
        lo = hi;
        hi = next;
    }
    if (tid == 0 && n_out) *n_out = next;
}

__global__ void k_export_empty(float4* __restrict__ out, uint32_t* __restrict__ n_out) {
    if (threadIdx.x == 0 && blockIdx.x == 0) {
        put_aabb(out, 0, INFINITY, INFINITY, INFINITY, -INFINITY, -INFINITY, -INFINITY, 0, -1);
        if (n_out) *n_out = 1;
    }
}

// BVH_Triangle records (64 B as 4 float4: v0, v1, v2, (index, mesh, 0, 0)) of mesh m, written at
// the slot of each triangle; vertex indices are clamped to n_vertices - 1 as the build does.
__global__ void __launch_bounds__(256) k_export_tris(rt_mesh_desc d, uint32_t m, uint32_t base,
                                                     const uint32_t* __restrict__ inv,
                                                     float4* __restrict__ out) {
    const uint32_t t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= d.n_tris) return;
    const uint64_t s = inv[base + t];
    float4* o = out + 4 * s;
    for (int k = 0; k < 3; ++k) {
        uint32_t vi = d.indices ? (uint32_t)d.indices[3 * (uint64_t)t + k] : 3 * t + k;
        vi = vi < d.n_vertices ? vi : d.n_vertices - 1;
        const float* P = (const float*)((const char*)d.vertices + (uint64_t)vi * d.vertex_stride + d.pos_offset);
        o[k] = make_float4(P[0], P[1], P[2], 0.0f);
    }
    o[3] = make_float4(__int_as_float((int32_t)t), __int_as_float((int32_t)m), 0.0f, 0.0f);
}

}  // namespace
}  // namespace rt

using namespace rt;

extern "C" int rt_scene_sizes_for(uint32_t n_tris, rt_scene_sizes* out) {
    if (!out) return set_error(RT_EINVAL, "rt_scene_sizes_for: out is NULL");
    if (n_tris > kMaxTris) return set_error(RT_ECAPACITY, "rt_scene_sizes_for: too many triangles");
    const uint64_t n = n_tris;
    out->nodes_bytes = 64 * (n > 1 ? n - 1 : 1);
    out->nodes4_bytes = 128 * (n > 1 ? n - 1 : 1);
    out->tris_bytes = 48 * (n ? n : 1);
    out->shade_bytes = 64 * (n ? n : 1);
    out->bounds_bytes = 32;
    out->workspace_bytes = carve(nullptr, n ? n : 1).bytes;
    out->prim_slot_bytes = 4 * (n ? n : 1);
    return RT_OK;
}

extern "C" int rt_scene_build(const rt_mesh_desc* meshes, uint32_t n_meshes, rt_scene* sc,
                              void* workspace, uint64_t ws_bytes, uint32_t* keys_out,
                              uint32_t* order_out, const rt_tuning* tuning, void* stream) {
    if (!sc) return set_error(RT_EINVAL, "rt_scene_build: scene is NULL");
    rt_tuning tu;
    if (int e = resolve_tuning(tuning, tu, "rt_scene_build")) return e;
    if (n_meshes && !meshes) return set_error(RT_EINVAL, "rt_scene_build: meshes is NULL");
    uint64_t n64 = 0;
    for (uint32_t m = 0; m < n_meshes; ++m) {
        const rt_mesh_desc& d = meshes[m];
        if (d.n_tris && !d.vertices) return set_error(RT_EINVAL, "rt_scene_build: mesh vertices NULL");
        if (d.n_tris && d.n_vertices == 0) return set_error(RT_EINVAL, "rt_scene_build: mesh has no vertices");
        if (!d.indices && (uint64_t)d.n_tris * 3 > d.n_vertices)
            return set_error(RT_EINVAL, "rt_scene_build: non-indexed mesh needs 3 vertices per triangle");
        if (d.vertex_stride < 12 || (d.vertex_stride & 3) || (d.pos_offset & 3) ||
            d.pos_offset + 12 > d.vertex_stride)
            return set_error(RT_EINVAL, "rt_scene_build: bad vertex stride/position offset");
        if (d.nrm_offset != RT_ABSENT && ((d.nrm_offset & 3) || d.nrm_offset + 12 > d.vertex_stride))
            return set_error(RT_EINVAL, "rt_scene_build: bad normal offset");
        if (d.uv_offset != RT_ABSENT && ((d.uv_offset & 3) || d.uv_offset + 8 > d.vertex_stride))
            return set_error(RT_EINVAL, "rt_scene_build: bad uv offset");
        n64 += d.n_tris;
    }
    if (n64 > kMaxTris) return set_error(RT_ECAPACITY, "rt_scene_build: too many triangles");
    const uint32_t n = (uint32_t)n64;
    if (sc->n_tris != n || sc->n_meshes != n_meshes)
        return set_error(RT_EINVAL, "rt_scene_build: scene n_tris/n_meshes do not match the meshes");
    if (!sc->nodes || !sc->nodes4 || !sc->tris || !sc->shade || !sc->mesh_offsets || !sc->bounds ||
        !sc->prim_slot)
        return set_error(RT_EINVAL, "rt_scene_build: scene arrays must be allocated");
    if (((uintptr_t)sc->nodes | (uintptr_t)sc->nodes4 | (uintptr_t)sc->tris | (uintptr_t)sc->shade) & 15)
        return set_error(RT_EINVAL, "rt_scene_build: scene arrays must be 16-byte aligned");
    hipStream_t s = (hipStream_t)stream;

    if (n == 0) {
        sc->root = RT_EMPTY_ROOT;
        hipLaunchKernelGGL(k_empty_bounds, dim3(1), dim3(1), 0, s, sc->bounds);
        hipLaunchKernelGGL(k_mesh_offsets_tail, dim3(1), dim3(1), 0, s, sc->mesh_offsets, 0u, 0u);
        for (uint32_t m = 0; m < n_meshes; ++m)
            hipLaunchKernelGGL(k_mesh_offsets_tail, dim3(1), dim3(1), 0, s, sc->mesh_offsets, m, 0u);
        hipLaunchKernelGGL(k_mesh_offsets_tail, dim3(1), dim3(1), 0, s, sc->mesh_offsets, n_meshes, 0u);
        return check_launch("rt_scene_build(empty)");
    }
    const Workspace need = carve(nullptr, n);
    if (!workspace || ws_bytes < need.bytes)
        return set_error(RT_EINVAL, "rt_scene_build: workspace too small (need " +
                                        std::to_string(need.bytes) + " bytes)");
    if ((uintptr_t)workspace & 255)
        return set_error(RT_EINVAL, "rt_scene_build: workspace must be 256-byte aligned");
    Workspace w = carve((char*)workspace, n);

    // 1. gather (one launch per mesh; the descriptor travels as a kernel argument)
    uint32_t base = 0, nparts = 0, nsrc = 0;
    for (uint32_t m = 0; m < n_meshes; ++m) {
        const rt_mesh_desc& d = meshes[m];
        hipLaunchKernelGGL(k_gather, dim3(d.n_tris ? blocks_for(d.n_tris, 256) : 1), dim3(256), 0, s,
                           d, m, n_meshes, base, w.cent, sc->mesh_offsets, w.partial + 2 * (uint64_t)nparts,
                           w.meshes + nsrc);
        nsrc += d.n_tris ? 1 : 0;
        base += d.n_tris;
        nparts += blocks_for(d.n_tris, 256);
    }
    // 2. - 4. centroid bounds, Morton codes and their sort, into the caller's arrays where it wants them
    // (PLOC writes the order of its own slots there)
    const bool ploc = n > 1 && tu.builder == RT_BUILD_PLOC;
    uint32_t* ki = keys_out ? keys_out : w.keys0;
    uint32_t* vi = order_out && !ploc ? order_out : w.vals0;
    if (n <= kSmallMax) {
        hipLaunchKernelGGL(k_order_chunks, dim3(blocks_for(n, kOrderChunk)), dim3(kOrderChunk), 0, s, w.cent, n,
                           w.partial, nparts, w.keys1, w.vals1);
        hipLaunchKernelGGL(n <= kSmallMax / 2 ? k_order_merge<kSmallMax / 2> : k_order_merge<kSmallMax>,
                           dim3(blocks_for(n, 64)), dim3(256), 0, s, w.keys1, w.vals1, n, ki, vi);
    } else {
        hipLaunchKernelGGL(k_bounds_final, dim3(1), dim3(1024), 0, s, w.partial, nparts, w.cbounds);
        hipLaunchKernelGGL(k_morton, dim3(blocks_for(n, 256)), dim3(256), 0, s, w.cent, n, w.cbounds,
                           w.keys0, w.vals0);
        sort_pairs(w.keys0, w.vals0, w.keys1, w.vals1, ki, vi, n, 30, w.hist, w.totals, s);
    }
    float4* nodes = (float4*)sc->nodes;
    const uint32_t nchunk = blocks_for(n, kPlocChunk);
    uint32_t* slots = vi;       // primitive of each slot
    Fallback fb{nullptr, nullptr};
    if (ploc) {
        // 5. PLOC hierarchy (node boxes as it merges, scene bounds at the root)
        hipLaunchKernelGGL(k_ploc_init, dim3(blocks_for(n, 256)), dim3(256), 0, s, vi, n, w.meshes, nsrc,
                           w.cid[0], w.cbox[0], w.pos_of, w.parent, w.state);
        const int iters = ploc_iterations(n);
        const uint32_t grid = std::min<uint32_t>(kPlocGrid, blocks_for(n, kPlocTile));
        for (int it = 0; it < iters; ++it) {
            hipLaunchKernelGGL(k_ploc_pairs, dim3(grid), dim3(kPlocLoad), 0, s, it, w.state, w.cbox[0],
                               w.cbox[1], w.nn, w.part);
            hipLaunchKernelGGL(k_ploc_compact, dim3(grid), dim3(kPlocTile), 0, s, it, n, w.state, w.nn, w.part,
                               w.cid[0], w.cid[1], w.cbox[0], w.cbox[1], w.nleft, w.nright, w.nsize,
                               w.parent, nodes, sc->bounds);
        }
        hipLaunchKernelGGL(k_ploc_tail, dim3(1), dim3(1024), 0, s, iters & 1, n, w.state, w.nn, w.cid[0],
                           w.cid[1], w.cbox[0], w.cbox[1], w.nleft, w.nright, w.nsize, w.parent, nodes,
                           sc->bounds);
        // a tree deeper than the traversal stacks allow is replaced by the LBVH of the same keys
        hipLaunchKernelGGL(k_zero_word, dim3(1), dim3(1), 0, s, w.depth);
        hipLaunchKernelGGL(k_ploc_depth, dim3(blocks_for(n, 256)), dim3(256), 0, s, n, w.parent, w.depth);
        // 6. leaf slots and traversal refs
        slots = order_out ? order_out : w.slot_order;
        fb = {w.depth, vi};
        hipLaunchKernelGGL(k_ploc_leafroots, dim3(blocks_for(n, 256)), dim3(256), 0, s, n, w.depth, vi, w.parent,
                           w.nsize, w.nleft, w.nright, w.pos_of, w.scan);
        hipLaunchKernelGGL(k_scan_chunks, dim3(nchunk), dim3(256), 0, s, n, w.scan, w.part);
        hipLaunchKernelGGL(k_scan_top, dim3(1), dim3(1024), 0, s, nchunk, w.part);
        hipLaunchKernelGGL(k_scan_apply, dim3(nchunk), dim3(256), 0, s, n, w.scan, w.part);
        hipLaunchKernelGGL(k_ploc_slots, dim3(blocks_for(n, 256)), dim3(256), 0, s, n, w.depth, vi, w.parent,
                           w.nsize, w.nleft, w.nright, w.pos_of, w.scan, slots, w.slot_of, w.fslot);
        hipLaunchKernelGGL(k_ploc_refs, dim3(blocks_for(n - 1, 256)), dim3(256), 0, s, n, w.depth, w.nleft,
                           w.nright, w.nsize, w.slot_of, w.fslot, nodes);
    }
    // leaf records; the LBVH tree, or the one in place of a PLOC tree found too deep; 4-wide records
    const bool past = n >= kPastCaches;
    hipLaunchKernelGGL(past ? k_emit<true> : k_emit<false>, dim3(blocks_for(n, 256)), dim3(256), 0, s, slots, fb, n, w.meshes, nsrc, w.leafbox,
                       (float4*)sc->tris, (float4*)sc->shade, (uint32_t*)sc->prim_slot);
    if (ploc && order_out)
        hipLaunchKernelGGL(k_copy_if, dim3(blocks_for(n, 256)), dim3(256), 0, s, w.depth, vi, order_out, n);
    if (n > 1) {
        const uint32_t nb = blocks_for(n, kTreeBlock);
        hipLaunchKernelGGL(k_tree_local, dim3(nb), dim3(kTreeBlock), 0, s, ki, n, fb, w.leafbox, nodes,
                           sc->bounds, w.top);
        if (nb > 1)
            hipLaunchKernelGGL(k_tree_top, dim3(nb), dim3(kTopThreads), 0, s, ki, n, fb, nodes, sc->bounds, w.top);
        hipLaunchKernelGGL(past ? k_wide<true> : k_wide<false>, dim3(blocks_for(n - 1, 256)), dim3(256), 0, s, n,
                           (const float4*)nodes, (float4*)sc->nodes4);
        sc->root = n <= (uint32_t)kLeafMax ? leaf_ref(0, n) : 0;
    } else {
        hipLaunchKernelGGL(k_single_leaf_bounds, dim3(1), dim3(1), 0, s, w.leafbox, sc->bounds);
        sc->root = ~0;
    }
    return check_launch("rt_scene_build");
}

extern "C" int rt_scene_export(const rt_scene* sc, const rt_mesh_desc* meshes, uint32_t n_meshes,
                               void* aabb_out, void* tris_out, uint32_t* n_nodes_out, void* stream) {
    if (!sc || !aabb_out) return set_error(RT_EINVAL, "rt_scene_export: NULL argument");
    if (((uintptr_t)aabb_out | (uintptr_t)tris_out) & 15)
        return set_error(RT_EINVAL, "rt_scene_export: outputs must be 16-byte aligned");
    hipStream_t s = (hipStream_t)stream;
    float4* aabb = (float4*)aabb_out;
    const uint32_t n = sc->n_tris;
    if (sc->root == RT_EMPTY_ROOT || n == 0) {
        hipLaunchKernelGGL(k_export_empty, dim3(1), dim3(1), 0, s, aabb, n_nodes_out);
        return check_launch("rt_scene_export");
    }
    if (!tris_out || !sc->prim_slot || !sc->bounds || (sc->root >= 0 && !sc->nodes))
        return set_error(RT_EINVAL, "rt_scene_export: NULL argument");
    if (n_meshes != sc->n_meshes || (n_meshes && !meshes))
        return set_error(RT_EINVAL, "rt_scene_export: the meshes must be those the scene was built from");
    uint64_t total = 0;
    for (uint32_t m = 0; m < n_meshes; ++m) {
        if (meshes[m].n_tris && (!meshes[m].vertices || !meshes[m].n_vertices))
            return set_error(RT_EINVAL, "rt_scene_export: mesh vertices NULL");
        total += meshes[m].n_tris;
    }
    if (total != n) return set_error(RT_EINVAL, "rt_scene_export: mesh triangle counts do not match the scene");
    const uint32_t* inv = (const uint32_t*)sc->prim_slot;
    uint32_t base = 0;
    for (uint32_t m = 0; m < n_meshes; ++m) {
        if (meshes[m].n_tris)
            hipLaunchKernelGGL(k_export_tris, dim3(blocks_for(meshes[m].n_tris, 256)), dim3(256), 0, s,
                               meshes[m], m, base, inv, (float4*)tris_out);
        base += meshes[m].n_tris;
    }
    hipLaunchKernelGGL(k_export_nodes, dim3(1), dim3(1024), 0, s, (const float4*)sc->nodes, sc->root,
                       sc->bounds, aabb, n_nodes_out);
    return check_launch("rt_scene_export");
}
