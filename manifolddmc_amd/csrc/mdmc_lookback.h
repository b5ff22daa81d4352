// mdmc_lookback.h -- single-pass ordered compaction: a block selects elements of its tile of
// R * kLbBlock consecutive elements (element base + r * kLbBlock + threadIdx.x in round r) and
// learns the tile's first output slot by decoupled look-back over the tiles before it (the
// scheme of the prefix sum in mdmc_scan.hip).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace mdmc {

constexpr int kLbBlock = 256;
constexpr int kLbSpinLimit = 1 << 22;

// look-back words (one per tile): flag (2 bits: 1 aggregate, 2 inclusive), the launch's epoch
// (16 bits) and value (46 bits; the sums of int32 counts over fewer than 2^31 elements that
// fit an id range are far below), read and written with relaxed device-scope atomics.  A word of
// another epoch counts as not yet written, so a launch needs no clearing launch before it:
// 3 us of launch time, and 4.5 us on the GPU, per scan of any size.
constexpr uint64_t kLbAgg = 1ULL, kLbInc = 2ULL, kLbValue = (1ULL << 46) - 1;
__device__ __forceinline__ uint64_t lbWord(uint64_t flag, uint32_t epoch, int64_t v) {
    return (flag << 62) | ((uint64_t)(epoch & 0xFFFFu) << 46) | ((uint64_t)v & kLbValue);
}
__device__ __forceinline__ uint64_t lbFlag(uint64_t w, uint32_t epoch) { return ((w >> 46) & 0xFFFFu) == (epoch & 0xFFFFu) ? w >> 62 : 0; }
__device__ __forceinline__ uint64_t lbLoad(const unsigned long long* p) { return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
__device__ __forceinline__ void lbStore(unsigned long long* p, uint64_t v) {
    __hip_atomic_store(p, (unsigned long long)v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Run by the block's first wave: publishes the tile's count, walks back over the earlier
// tiles' words and returns (through *s_off, read after a barrier) the number of selected
// elements before the tile.  A wait past the spin limit does not trust the dispatch order:
// countBefore(lane) (the selected elements among base .. in steps of 64 from lane) gives the
// exact prefix instead, and *directOut (device memory) counts the tile as a diagnostic.
template <class CountBefore>
__device__ __forceinline__ void lbTileOffset(unsigned long long* status, uint32_t epoch, int64_t t, int64_t tileSum, CountBefore countBefore, int64_t* directOut,
                                             long long* s_off) {
    const int lane = threadIdx.x & 63;
    if (t == 0) {
        if (lane == 0) {
            lbStore(&status[0], lbWord(kLbInc, epoch, tileSum));
            *s_off = 0;
        }
        return;
    }
    if (lane == 0) lbStore(&status[t], lbWord(kLbAgg, epoch, tileSum));
    int64_t accum = 0;
    int64_t i = t - 1;
    int spins = 0;
    bool done = false, direct = false;
    while (!done) {
        const int64_t j = i - lane;
        const uint64_t st = j >= 0 ? lbLoad(&status[j]) : lbWord(kLbInc, epoch, 0);
        const uint64_t f = lbFlag(st, epoch);
        const uint64_t incMask = __ballot(f == kLbInc);
        const uint64_t zeroMask = __ballot(f == 0);
        const int firstInc = incMask ? __ffsll((unsigned long long)incMask) - 1 : 64;
        const uint64_t upto = firstInc >= 63 ? ~0ULL : ((1ULL << (firstInc + 1)) - 1ULL);
        if (zeroMask & upto) {
            // the ballots make this branch and the counter uniform over the wave
            if (++spins > kLbSpinLimit) {
                direct = true;
                break;
            }
            __builtin_amdgcn_s_sleep(1);
            continue;
        }
        int64_t val = lane <= firstInc ? (int64_t)(st & kLbValue) : 0;
#pragma unroll
        for (int d = 32; d > 0; d >>= 1) val += __shfl_down(val, d, 64);
        accum += __shfl(val, 0, 64);
        if (firstInc < 64) done = true;
        else i -= 64;
    }
    if (direct) {
        int64_t sum = countBefore(lane);
#pragma unroll
        for (int d = 32; d > 0; d >>= 1) sum += __shfl_down(sum, d, 64);
        accum = __shfl(sum, 0, 64);
        if (lane == 0 && directOut) atomicAdd((unsigned long long*)directOut, 1ULL);
    }
    if (lane == 0) {
        lbStore(&status[t], lbWord(kLbInc, epoch, accum + tileSum));
        *s_off = accum;
    }
}

// Per round r the wave's selection ballot m[r]; on return s_pre[r * 4 + wave] holds the
// number of selected elements of the tile before that wave's 64 elements of round r (index
// order: round, then wave), and the tile's total is returned.  Call from every thread;
// s_cnt holds R * 4 ints, s_pre R * 4 + 1.
template <int R>
__device__ __forceinline__ int lbBlockRanks(const uint64_t m[R], int* s_cnt, int* s_pre) {
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    if (lane == 0)
#pragma unroll
        for (int r = 0; r < R; ++r) s_cnt[r * (kLbBlock / 64) + wid] = __popcll(m[r]);
    __syncthreads();
    constexpr int N = R * (kLbBlock / 64);  // at most 64 counts, one wave scans them
    static_assert(N <= 64, "one wave scans the per-round wave counts");
    if (threadIdx.x < 64) {
        const int v = threadIdx.x < N ? s_cnt[threadIdx.x] : 0;
        int x = v;
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) {
            const int y = __shfl_up(x, d, 64);
            if (lane >= d) x += y;
        }
        if (threadIdx.x < N) s_pre[threadIdx.x] = x - v;
        if (threadIdx.x == N - 1) s_pre[N] = x;
    }
    __syncthreads();
    return s_pre[N];
}

// Stream compaction in the same single pass as the prefix sum (mdmc_scan.hip): the indices i < n with
// (attr[i] & mask) != 0, in increasing order, into idx[0 .. total).  Each tile counts its selected
// elements (16 per thread), scans the counts in the block, gets the tile's first output slot by the
// same look-back (and the same exact fallback: a direct count of the selected elements before the
// tile) and writes its indices; nothing is written per unselected element.  A block of kLbBlock threads
// takes tile t of kListTile elements (tiles in block order).
constexpr int kListItems = 16, kListTile = kLbBlock * kListItems;
struct FlagList {
    const uint32_t* attr;
    int64_t n;
    uint32_t mask;
    int32_t* idx;
    unsigned long long* words;
    uint32_t epoch;
    int64_t *total, *directOut;
};
__device__ __forceinline__ void compactFlaggedTile(const FlagList& a, int64_t t) {
    __shared__ int s_wave[kLbBlock / 64];
    __shared__ long long s_off;
    const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
    const int64_t n = a.n, numTiles = n > 0 ? (n + kListTile - 1) / kListTile : 1;
    if (t >= numTiles) return;
    const int64_t base = t * kListTile;
    const int64_t first = base + (int64_t)tid * kListItems;  // this thread's 16 consecutive elements

    uint32_t bits = 0;
    if (first + kListItems <= n && (((uintptr_t)a.attr) & 15) == 0) {
        const uint4* p = reinterpret_cast<const uint4*>(a.attr + first);
#pragma unroll
        for (int k = 0; k < kListItems / 4; ++k) {
            const uint4 q = p[k];
            bits |= ((q.x & a.mask) ? 1u : 0u) << (4 * k);
            bits |= ((q.y & a.mask) ? 1u : 0u) << (4 * k + 1);
            bits |= ((q.z & a.mask) ? 1u : 0u) << (4 * k + 2);
            bits |= ((q.w & a.mask) ? 1u : 0u) << (4 * k + 3);
        }
    } else {
        for (int k = 0; k < kListItems; ++k)
            if (first + k < n && (a.attr[first + k] & a.mask)) bits |= 1u << k;
    }
    const int cnt = __popc(bits);
    int x = cnt;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const int y = __shfl_up(x, d, 64);
        if (lane >= d) x += y;
    }
    if (lane == 63) s_wave[wid] = x;
    __syncthreads();
    int add = 0, tileSum = 0;
#pragma unroll
    for (int w = 0; w < kLbBlock / 64; ++w) {
        const int sw = s_wave[w];
        if (w < wid) add += sw;
        tileSum += sw;
    }
    const int run = x - cnt + add;  // exclusive prefix of this thread inside the tile

    if (tid < 64)
        lbTileOffset(
            a.words, a.epoch, t, tileSum,
            [&](int l) {
                int64_t sum = 0;
                for (int64_t k = l; k < base; k += 64) sum += (a.attr[k] & a.mask) ? 1 : 0;
                return sum;
            },
            a.directOut, &s_off);
    __syncthreads();
    int64_t o = s_off + run;
    for (uint32_t b = bits; b; b &= b - 1) a.idx[o++] = (int32_t)(first + __ffs(b) - 1);
    if (t == numTiles - 1 && tid == 0) *a.total = s_off + tileSum;
}

}  // namespace mdmc
