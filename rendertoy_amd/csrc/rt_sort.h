// rt_sort.h — stable LSD radix sort of (uint32 key, uint32 value) pairs on the device, used by the
// scene build (Morton codes). Each pass of 8 bits is a per-tile histogram -> per-digit row scan ->
// scatter; the scatter block scans the 256 digit totals itself, ranks keys with wave64 ballot/mbcnt
// multi-split so equal digits keep input order, groups its tile by digit in LDS and writes each
// digit's run of the tile contiguously.
#pragma once

#include "rt_common.h"

namespace rt {
namespace {

constexpr int kSortThreads = 256;
constexpr int kSortItems = 8;                       // items per thread per tile
constexpr int kSortTile = kSortThreads * kSortItems;  // 2048 keys per block
constexpr int kRadixBits = 8;
constexpr int kRadix = 1 << kRadixBits;

__global__ void __launch_bounds__(kSortThreads) k_sort_hist(const uint32_t* __restrict__ keys,
                                                            uint32_t n, int shift,
                                                            uint32_t* __restrict__ hist,
                                                            uint32_t nblk) {
    __shared__ uint32_t h[kRadix];
    h[threadIdx.x] = 0;
    __syncthreads();
    const uint64_t base = (uint64_t)blockIdx.x * kSortTile;
    for (int r = 0; r < kSortItems; ++r) {
        const uint64_t i = base + (uint64_t)r * kSortThreads + threadIdx.x;
        if (i < n) atomicAdd(&h[(keys[i] >> shift) & (kRadix - 1)], 1u);
    }
    __syncthreads();
    hist[(uint64_t)threadIdx.x * nblk + blockIdx.x] = h[threadIdx.x];
}

// Row scan: block d turns row d of the digit-major histogram (counts of digit d in tiles
// 0..nblk-1) into its exclusive prefix sums, in place, and writes the row total to totals[d].
// Thread t takes a contiguous run of the row: its sum, one workgroup scan of the 256 sums, then
// the run's prefixes from its offset.
__global__ void __launch_bounds__(kSortThreads) k_sort_rowscan(uint32_t* __restrict__ hist,
                                                               uint32_t nblk,
                                                               uint32_t* __restrict__ totals) {
    __shared__ uint32_t s[kSortThreads];
    uint32_t* row = hist + (uint64_t)blockIdx.x * nblk;
    const uint32_t per = (nblk + kSortThreads - 1) / kSortThreads;
    const uint32_t b = threadIdx.x * per;
    const uint32_t e = b + per < nblk ? b + per : nblk;  // run [b, e), empty past the row's end
    uint32_t sum = 0;
    for (uint32_t i = b; i < e; ++i) sum += row[i];
    s[threadIdx.x] = sum;
    __syncthreads();
    for (int off = 1; off < kSortThreads; off <<= 1) {  // inclusive scan of the run sums
        const uint32_t x = threadIdx.x >= (uint32_t)off ? s[threadIdx.x - off] : 0u;
        __syncthreads();
        s[threadIdx.x] += x;
        __syncthreads();
    }
    uint32_t run = s[threadIdx.x] - sum;
    for (uint32_t i = b; i < e; ++i) {
        const uint32_t v = row[i];
        row[i] = run;
        run += v;
    }
    if (threadIdx.x == kSortThreads - 1) totals[blockIdx.x] = s[kSortThreads - 1];
}
// Rank of each valid lane's digit among the wave's items so far, and the wave's counts advanced: `count`
// is this wave's own row of LDS, cleared before its first round.
template <int kBits>
RT_DEV uint32_t wave_digit_rank(uint32_t d, bool valid, int lane, uint32_t* count) {
    uint64_t peers = __ballot(valid);
#pragma unroll
    for (int b = 0; b < kBits; ++b) {
        const bool bit = (d >> b) & 1u;
        const uint64_t mb = __ballot(bit);
        peers &= bit ? mb : ~mb;
    }
    const uint32_t rank = __builtin_amdgcn_mbcnt_hi((uint32_t)(peers >> 32),
                                                    __builtin_amdgcn_mbcnt_lo((uint32_t)peers, 0u));
    const uint32_t before = __hip_atomic_load(&count[d], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
    if (valid && rank == 0)
        __hip_atomic_store(&count[d], before + (uint32_t)__popcll(peers), __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_WAVEFRONT);
    return before + rank;
}

// Stable scatter of one tile of kSortTile items, wave w holding items [w, w + 1) * 64 * kSortItems.
// Each wave ranks its items alone, 64 at a time: 8 ballots give the lanes that share a lane's digit, and
// the wave's own count of the digit in LDS goes on from the items before (a wave's LDS accesses stay
// in order, so this takes no barrier; one round of all waves at a time, with three barriers each, took
// 17.2 us a pass at 1.31 M pairs and 11.8 at 11,560, this takes 11.5 and 6.1). After one scan over digits and waves the tile goes to LDS in (digit, input order) and is
// written out with consecutive threads taking consecutive items: each digit's run of the tile lands in
// one contiguous span of the output.
__global__ void __launch_bounds__(kSortThreads) k_sort_scatter(
    const uint32_t* __restrict__ kin, const uint32_t* __restrict__ vin, uint32_t n, int shift,
    const uint32_t* __restrict__ hist, const uint32_t* __restrict__ totals, uint32_t nblk,
    uint32_t* __restrict__ kout,
    uint32_t* __restrict__ vout) {
    constexpr int kWaves = kSortThreads / 64;
    __shared__ uint32_t wcount[kWaves][kRadix];  // a wave's count of digit d, then its LDS position
    __shared__ uint32_t base[kRadix];            // output position minus LDS position of digit d
    __shared__ uint64_t wsum[kWaves];
    __shared__ uint32_t sk[kSortTile];
    __shared__ uint32_t sv[kSortTile];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const uint32_t blk = blockIdx.x;
    const uint64_t tile = (uint64_t)blk * kSortTile;
    const uint32_t m = (uint32_t)(n - tile < (uint64_t)kSortTile ? n - tile : (uint64_t)kSortTile);
    const uint32_t first = wave * (64 * kSortItems) + lane;
    uint32_t key[kSortItems], val[kSortItems], rank[kSortItems];
#pragma unroll
    for (int r = 0; r < kSortItems; ++r) {
        const uint32_t i = first + r * 64;
        key[r] = i < m ? kin[tile + i] : 0u;
        val[r] = i < m ? vin[tile + i] : 0u;
    }
    const uint32_t total = totals[tid], before = hist[(uint64_t)tid * nblk + blk];
    for (int w = 0; w < kWaves; ++w) wcount[w][tid] = 0;
    __syncthreads();
#pragma unroll
    for (int r = 0; r < kSortItems; ++r)
        rank[r] = wave_digit_rank<kRadixBits>((key[r] >> shift) & (kRadix - 1), first + r * 64 < m, lane, wcount[wave]);
    __syncthreads();
    uint32_t cnt = 0;
    for (int w = 0; w < kWaves; ++w) cnt += wcount[w][tid];
    // exclusive scans over the digits of the totals (high half) and the tile's counts (low half)
    uint64_t incl = ((uint64_t)total << 32) | cnt;
    for (int off = 1; off < 64; off <<= 1) {
        const uint64_t x = __shfl_up((unsigned long long)incl, off);
        if (lane >= off) incl += x;
    }
    if (lane == 63) wsum[wave] = incl;
    __syncthreads();
    for (int w = 0; w < wave; ++w) incl += wsum[w];
    uint32_t at = (uint32_t)incl - cnt;  // the digit's first LDS position
    base[tid] = (uint32_t)(incl >> 32) - total + before - at;
    for (int w = 0; w < kWaves; ++w) {
        const uint32_t c = wcount[w][tid];
        wcount[w][tid] = at;
        at += c;
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < kSortItems; ++r) {
        if (first + r * 64 < m) {
            const uint32_t off = wcount[wave][(key[r] >> shift) & (kRadix - 1)] + rank[r];
            sk[off] = key[r];
            sv[off] = val[r];
        }
    }
    __syncthreads();
    for (uint32_t j = tid; j < m; j += kSortThreads) {
        const uint32_t k = sk[j];
        const uint32_t off = base[(k >> shift) & (kRadix - 1)] + j;
        if (off < n) {  // always true for a consistent histogram; keeps writes in bounds
            kout[off] = k;
            vout[off] = sv[j];
        }
    }
}

// Bytes of the histogram scratch for n keys.
inline uint64_t sort_hist_bytes(uint64_t n) {
    const uint64_t nblk = (n + kSortTile - 1) / kSortTile;
    return 4ull * kRadix * (nblk ? nblk : 1);
}

// Sorts n pairs (k0, v0) by the low `bits` bits of the keys in an even number of passes, ceil(bits / 8),
// ping-ponging over (k1, v1); the last pass writes (kout, vout), which may be (k0, v0). hist:
// sort_hist_bytes(n), totals: kRadix words.
inline void sort_pairs(uint32_t* k0, uint32_t* v0, uint32_t* k1, uint32_t* v1, uint32_t* kout, uint32_t* vout,
                       uint32_t n, int bits, uint32_t* hist, uint32_t* totals, hipStream_t s) {
    const uint32_t nblk = (uint32_t)((n + kSortTile - 1) / kSortTile);
    for (int shift = 0; shift < bits; shift += kRadixBits) {
        const bool odd = (shift / kRadixBits) & 1, last = shift + kRadixBits >= bits;
        const uint32_t *ki = odd ? k1 : k0, *vi = odd ? v1 : v0;
        uint32_t* ko = last ? kout : odd ? k0 : k1;
        uint32_t* vo = last ? vout : odd ? v0 : v1;
        hipLaunchKernelGGL(k_sort_hist, dim3(nblk), dim3(kSortThreads), 0, s, ki, n, shift, hist, nblk);
        hipLaunchKernelGGL(k_sort_rowscan, dim3(kRadix), dim3(kSortThreads), 0, s, hist, nblk, totals);
        hipLaunchKernelGGL(k_sort_scatter, dim3(nblk), dim3(kSortThreads), 0, s, ki, vi, n, shift, hist,
                           totals, nblk, ko, vo);
    }
}

}  // namespace
}  // namespace rt
