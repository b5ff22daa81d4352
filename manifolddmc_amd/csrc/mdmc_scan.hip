// mdmc_scan.hip -- device-wide exclusive prefix sum of int32 counts into int64 offsets,
// in one pass: block b scans tile b of 4096 counts and gets its offset by decoupled
// look-back over the tiles before it.
//
// Tile = block index, not an atomic ticket: the blocks of a launch go to the XCDs
// round-robin and each XCD starts its blocks in increasing order, so every tile below the
// lowest resident one has finished (a lower tile not yet started would sit on an XCD whose
// resident blocks are all lower still), and the lowest resident tile never waits on an
// unstarted one.  The ticket cost one same-address atomic per block: 100 us against 67 us
// for 17 M counts.  That dispatch order is observed behaviour, not a documented
// guarantee, so correctness does not rest on it: a tile whose look-back wait passes its
// spin limit sums every count before it straight from the input instead (exact, only
// slower), then publishes as usual, so a tile that waits on an unstarted one still ends
// and frees its slot.
//
// Look-back words pack flag, the launch's epoch and value (mdmc_lookback.h), so relaxed
// device-scope atomics suffice: a reader needs nothing beyond the word it reads.
#include "mdmc_internal.h"
#include "mdmc_lookback.h"

namespace mdmc {

namespace {
constexpr int kScanBlock = 256;
constexpr int kScanItems = 16;
constexpr int kTile = kScanBlock * kScanItems;
static_assert(kTile == kScanTile, "tile size");
static_assert(kScanBlock == kLbBlock && kListTile == kScanTile, "block size of the look-back, words of a list");

// One launch scans up to kScanJobs arrays: blockIdx.y picks the job, blockIdx.x its tile (a job
// with fewer tiles than the widest leaves the rest of its row idle).
struct ScanJobs {
    ScanJob job[kScanJobs];
    int64_t *stampStart, *stampEnd;
};

__global__ void __launch_bounds__(kScanBlock) kScan(ScanJobs jobs, uint32_t epoch, int64_t* __restrict__ directOut) {
    __shared__ __align__(16) int32_t s_in[kTile];
    __shared__ int64_t s_wave[kScanBlock / 64];
    __shared__ long long s_off;
    const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
    stampClock(jobs.stampStart);
    const ScanJob& job = jobs.job[blockIdx.y];
    const int64_t t = blockIdx.x, n = job.n, numTiles = scanTiles(n);
    if (t >= numTiles) return;
    const int32_t* __restrict__ in = job.in;
    int64_t* __restrict__ out = job.out;
    const int64_t base = t * kTile;

    // 16 consecutive counts per thread: four 16-byte loads each when the tile is full and
    // the input 16-byte aligned, else a coalesced load through LDS
    int32_t v[kScanItems];
    const bool vec = base + kTile <= n && (((uintptr_t)in) & 15) == 0;
    if (vec) {
        const int4* p = reinterpret_cast<const int4*>(in + base) + tid * (kScanItems / 4);
#pragma unroll
        for (int k = 0; k < kScanItems / 4; ++k) {
            const int4 q = p[k];
            v[4 * k] = q.x;
            v[4 * k + 1] = q.y;
            v[4 * k + 2] = q.z;
            v[4 * k + 3] = q.w;
        }
    } else {
        for (int i = tid; i < kTile; i += kScanBlock) {
            const int64_t j = base + i;
            s_in[i] = j < n ? in[j] : 0;
        }
        __syncthreads();
#pragma unroll
        for (int k = 0; k < kScanItems; ++k) v[k] = s_in[tid * kScanItems + k];
    }
    int64_t acc = 0;
#pragma unroll
    for (int k = 0; k < kScanItems; ++k) acc += v[k];
    int64_t x = acc;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const int64_t y = __shfl_up(x, d, 64);
        if (lane >= d) x += y;
    }
    if (lane == 63) s_wave[wid] = x;
    __syncthreads();
    int64_t add = 0, tileSum = 0;
#pragma unroll
    for (int w = 0; w < kScanBlock / 64; ++w) {
        const int64_t s = s_wave[w];
        if (w < wid) add += s;
        tileSum += s;
    }
    int64_t run = x - acc + add;  // exclusive prefix of this thread inside the tile

    if (tid < 64)
        lbTileOffset(
            job.words, epoch, t, tileSum,
            [&](int l) {
                int64_t sum = 0;
                for (int64_t k = l; k < base; k += 64) sum += in[k];
                return sum;
            },
            directOut, &s_off);
    __syncthreads();
    run += s_off;

    // exclusive offsets back through LDS, half a tile at a time, for coalesced int64 stores
    int64_t* s_out = reinterpret_cast<int64_t*>(s_in);  // 4096 int32 slots hold 2048 int64
#pragma unroll
    for (int half = 0; half < 2; ++half) {
        __syncthreads();
        if ((tid >> 7) == half) {
            int64_t r = run;
#pragma unroll
            for (int k = 0; k < kScanItems; ++k) {
                s_out[(tid & 127) * kScanItems + k] = r;
                r += v[k];
            }
        }
        __syncthreads();
        const int64_t o = base + (int64_t)half * (kTile / 2);
        if (vec && (((uintptr_t)out) & 15) == 0) {
            // pairs of offsets as 16-byte stores
            const longlong2* s2 = reinterpret_cast<const longlong2*>(s_out);
            longlong2* o2 = reinterpret_cast<longlong2*>(out + o);
            for (int i = tid; i < kTile / 4; i += kScanBlock) o2[i] = s2[i];
        } else {
            for (int i = tid; i < kTile / 2; i += kScanBlock)
                if (o + i < n) out[o + i] = s_out[i];
        }
    }
    if (t == numTiles - 1 && tid == 0) {
        if (job.total) *job.total = s_off + tileSum;
        if (jobs.stampEnd && blockIdx.y == 0) *jobs.stampEnd = wall_clock64();
    }
}
__global__ void __launch_bounds__(kScanBlock) kCompactFlagged(const uint32_t* __restrict__ attr, int64_t n, uint32_t mask, int32_t* __restrict__ idx,
                                                              unsigned long long* __restrict__ words, uint32_t epoch,
                                                              int64_t* __restrict__ total, int64_t* __restrict__ directOut, int64_t* stamp) {
    stampClock(stamp);
    compactFlaggedTile(FlagList{attr, n, mask, idx, words, epoch, total, directOut}, blockIdx.x);
}
}  // namespace

void scanExclusiveI32(const ScanJob* jobs, int count, uint32_t epoch, hipStream_t s, int64_t* directOut, int64_t* stampStart, int64_t* stampEnd) {
    ScanJobs j{};
    j.stampStart = stampStart;
    j.stampEnd = stampEnd;
    int64_t tiles = 0;
    for (int k = 0; k < count; ++k) {
        j.job[k] = jobs[k];
        tiles = tiles > scanTiles(jobs[k].n) ? tiles : scanTiles(jobs[k].n);
    }
    kScan<<<dim3((unsigned)tiles, (unsigned)count), kScanBlock, 0, s>>>(j, epoch, directOut);
}

void compactFlagged(const uint32_t* attr, int64_t n, uint32_t mask, int32_t* idx, int64_t* total, unsigned long long* words, uint32_t epoch,
                    hipStream_t s, int64_t* directOut, int64_t* stamp) {
    kCompactFlagged<<<(unsigned)scanTiles(n), kScanBlock, 0, s>>>(attr, n, mask, idx, words, epoch, total, directOut, stamp);
}

}  // namespace mdmc
