// mdmc_pipeline.hip -- halfedge mesh, simplifications, non-manifold repair and
// the host-side stage driver.
//
// Restates (MarchingCubes/VisualDMC/src/DMC):
//   HalfedgeMesh::initialize / collectHalfedgeElements / connectHalfedgeTwins /
//     refresh*Flags                                   Halfedges/HalfedgeMesh.cu:14-291, :783-857
//   simplify3X3Y, simplify3X3YOld, simplify3333       Halfedges/HalfedgeMesh.cu:296-683, :859-1048
//   HalfedgeMesh::refreshHashTable                    Halfedges/HalfedgeMesh.cu:1063-1100
//   ManifoldCreator::fixManifoldTwins                 PostProcesses/ManifoldCreator.cu:39-312, :471-486
//   ManifoldSplitter::run and its kernels             PostProcesses/ManifoldSplitter.cu:25-1387
//   ManifoldCreator::detectNonManifoldVertices        PostProcesses/ManifoldCreator.cu:319-536
//
// Where the reference appends with atomics or lets racing threads overwrite a
// value, this code produces the result of one fixed legal schedule: threads of a
// launch taking effect in ascending thread-id order.  Appends become prefix sums,
// "last writer wins" becomes atomicMax, and per-bucket slot order becomes a sort
// by (face, position in face).  The vertex-pair hash table becomes a CSR list of
// outgoing halfedges per vertex: a bucket is the set of halfedges joining the
// same two vertices, found by scanning two short lists.
#include <algorithm>
#include <atomic>
#include <chrono>
#include <cstring>
#include <vector>

#include "mdmc_arena.h"
#include "mdmc_device.h"
#include "mdmc_gridpass.h"
#include "mdmc_internal.h"
#include "mdmc_lookback.h"
#include "mdmc_pipeline.h"

namespace mdmc {

namespace {

constexpr int kMaxBucket = 16;
constexpr int kFanGuard = 4096;

// ---------------------------------------------------------------- counters
enum : int { A_ANOMALY = 0, A_CONFLICT = 1, A_INVALID = 2, A_DIRTY = 3, A_FALLBACK = 4 /* two steps */, A_MERGE_SEQ = 6, A_LB_DIRECT = 7,
             A_NM = 8, A_NSLOW = 9, A_NSLOW_OFF = 10, A_PIN = 11, A_NCOL = 12, A_ADD = 13 /* three */, A_STAMP = 16, A_STATS = A_STAMP + ST_COUNT, A_TICKET = A_STATS + 9, A_NCOUNTERS };
// the slotted non-manifold halfedges the split's working copy marks (markHalfedgesAsNonManifold,
// ManifoldSplitter.cu:527-555, reads the four slots of every full vertex-pair bucket): every
// halfedge of a bucket of 4, and of a larger bucket the ones at ranks 1, 2, 3 and size - 1
__device__ __forceinline__ bool slottedNM(int n, int r) { return n == 4 || (n > 4 && (r == 1 || r == 2 || r == 3 || r == n - 1)); }
// A count summed over a whole launch without one hot address: a block adds its total to one of
// kPartSlots partial sums (by block index, 128 bytes apart), which a later one-wave kernel adds
// up.  Every thread of the block must call it.
constexpr int kPartSlots = 64, kPartStride = 16;
__device__ __forceinline__ void blockAdd(int64_t* parts, int c) {
    __shared__ int s_part[kBlock / 64];
    int x = c;
#pragma unroll
    for (int d = 32; d > 0; d >>= 1) x += __shfl_down(x, d, 64);
    if ((threadIdx.x & 63) == 0) s_part[threadIdx.x >> 6] = x;
    __syncthreads();
    if (threadIdx.x == 0) {
        int t = 0;
        for (int w = 0; w < (int)(blockDim.x + 63) / 64; ++w) t += s_part[w];
        if (t) atomicAdd((unsigned long long*)&parts[(blockIdx.x % kPartSlots) * kPartStride], (unsigned long long)t);
    }
}
// the same from one wave, where few waves have anything to add (no barrier: the block's other
// waves may be done); called by the lanes that are still running
__device__ __forceinline__ void waveAdd(int64_t* parts, bool c) {
    const uint64_t m = __ballot(c);
    if (m && (int)(threadIdx.x & 63) == __ffsll((unsigned long long)m) - 1)
        atomicAdd((unsigned long long*)&parts[(blockIdx.x % kPartSlots) * kPartStride], (unsigned long long)__popcll(m));
}
// and of counts, called by whole waves
__device__ __forceinline__ void waveSum(int64_t* parts, int c) {
    if (__ballot(c != 0) == 0) return;
    int x = c;
#pragma unroll
    for (int d = 32; d > 0; d >>= 1) x += __shfl_down(x, d, 64);
    if ((threadIdx.x & 63) == 0) atomicAdd((unsigned long long*)&parts[(blockIdx.x % kPartSlots) * kPartStride], (unsigned long long)x);
}
__device__ __forceinline__ int64_t sumParts(const int64_t* parts, int lane) {
    int64_t v = parts[lane * kPartStride];
#pragma unroll
    for (int d = 32; d > 0; d >>= 1) v += __shfl_down(v, d, 64);
    return v;
}

// The kernels that end an extraction are launched behind the list of the non-manifold faces
// without waiting for its length (kAwaitSplit): they return at once where faces are left to
// split, or a check failed, and the host then splits and launches them again.  The statistics
// also wait (kAwaitFans) where the fan detection left vertices to its slow pass.  A batch's fan
// detection, which follows its split, waits for the checks alone (kAwaitValid).
enum : int { kAwaitSplit = 1, kAwaitFans = 2, kAwaitValid = 4 };
__device__ __forceinline__ bool notYet(const int64_t* ctr, int guarded) {
    return ((guarded & (kAwaitSplit | kAwaitValid)) && ctr[A_INVALID] != 0) || ((guarded & kAwaitSplit) && ctr[A_NM] != 0) ||
           ((guarded & kAwaitFans) && ctr[A_NSLOW] != 0);
}

// a failed check: counted, and reported through the pinned word whose address the counters hold,
// so that a host that waits anyway sees it without a copy
__device__ __forceinline__ void invalid(int64_t* ctr, int n = 1) {
    atomicAdd((unsigned long long*)&ctr[A_INVALID], (unsigned long long)n);
    *(volatile int64_t*)(intptr_t)ctr[A_PIN] = 1;
}

// A chain of simplifications is launched whole, without waiting for the checks before it or for
// its steps' outcomes: its kernels return at once where the initialize's check failed or one of
// the `before` steps before left merges that need the region rebuild (kLocalMerge); the host
// sees both at the chain's end, runs the rebuild and launches the rest again.
__device__ __forceinline__ bool chainHeld(const int64_t* ctr, int before) {
    return ctr[A_INVALID] != 0 || (before > 0 && ctr[A_FALLBACK] != 0) || (before > 1 && ctr[A_FALLBACK + 1] != 0);
}

__device__ __forceinline__ void anomaly(int64_t* ctr) { atomicAdd((unsigned long long*)&ctr[A_ANOMALY], 1ULL); }

__device__ __forceinline__ int heO(const int4* he, int h) { return ((const int*)he)[4 * (int64_t)h]; }
__device__ __forceinline__ int heF(const int4* he, int h) { return ((const int*)he)[4 * (int64_t)h + 1]; }
__device__ __forceinline__ int heN(const int4* he, int h) { return ((const int*)he)[4 * (int64_t)h + 2]; }
__device__ __forceinline__ int heT(const int4* he, int h) { return ((const int*)he)[4 * (int64_t)h + 3]; }
__device__ __forceinline__ void setT(int4* he, int h, int t) { ((int*)he)[4 * (int64_t)h + 3] = t; }
// the k-th next of h in a face laid out as a halfedge build leaves it (4f .. 4f + 3)
__device__ __forceinline__ int quadNext(int h, int k) { return (h & ~3) | ((h + k) & 3); }
// next of h: from the id where canon marks h as laid out by the build (canon null: all are),
// else from its record (the split rewrites the records of the halfedges it copies back)
__device__ __forceinline__ int nextOf(const int4* he, const uint8_t* canon, int h) { return (!canon || canon[h]) ? quadNext(h, 1) : heN(he, h); }

// bytes [0, head) and [head + body, n) one per thread of the first block, [head, head + body)
// (16-byte aligned) 16 per thread
__global__ void kFillBytes(uint8_t* __restrict__ p, uint8_t byte, size_t head, size_t body, size_t n) {
    const size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (16 * t < body) {
        const uint32_t w = 0x01010101u * byte;
        *reinterpret_cast<uint4*>(p + head + 16 * t) = make_uint4(w, w, w, w);
    }
    if (t < 16) {
        if (t < head) p[t] = byte;
        if (head + body + t < n) p[head + body + t] = byte;
    }
}

// several fills in one launch: block b works on the range j with start[j] <= b < start[j + 1],
// as kFillBytes does on one range
__global__ void kFillMany(FillSet fs) {
    stampClock(fs.stamp);
    int j = 0;
    while (j + 1 < fs.count && (unsigned)blockIdx.x >= fs.start[j + 1]) ++j;
    const size_t t = (size_t)(blockIdx.x - fs.start[j]) * blockDim.x + threadIdx.x;
    uint8_t* p = fs.p[j];
    const uint8_t byte = fs.byte[j];
    if (16 * t < fs.body[j]) {
        const uint32_t w = 0x01010101u * byte;
        *reinterpret_cast<uint4*>(p + fs.head[j] + 16 * t) = make_uint4(w, w, w, w);
    }
    if (t < 16) {
        if (t < fs.head[j]) p[t] = byte;
        if (fs.head[j] + fs.body[j] + t < fs.n[j]) p[fs.head[j] + fs.body[j] + t] = byte;
    }
}

// Elementwise kernels below take four elements per thread: one 16-byte access per array when
// all four are in range and the arrays are 16-byte aligned (the arena's are), else one by one.
__device__ __forceinline__ int64_t firstOfFour() { return 4 * ((int64_t)blockIdx.x * blockDim.x + threadIdx.x); }
__device__ __forceinline__ bool vec4(int64_t i0, int64_t n, const void* a, const void* b) {
    return i0 + 3 < n && ((((uintptr_t)a) | ((uintptr_t)b)) & 15) == 0;
}

// pinned words: the padding pass's "needs the exact blend", the initialize's "inconsistent
// quads", a deferred simplification's "region rebuild needed", the clock ahead of the uploads, the
// copy of the counters at the end
constexpr int kPinSpecial = 3, kPinInvalid = 4, kPinFallback = 5 /* two steps */, kPinUpload = 7, kPinFinal = 16;
// and behind that copy the word that says that it is whole
constexpr int kPinDone = kPinFinal + A_NCOUNTERS;
static_assert(kPinDone < Pipeline::kPinSlots && A_NCOUNTERS < 64, "pinned words, handed over by one wave");

// one wave hands the counters to the host, which may be polling for the word behind them
__device__ __forceinline__ void handOver(const int64_t* ctr, int64_t* pin) {
    volatile int64_t* p = pin;
    const int k = threadIdx.x;
    if (k < A_NCOUNTERS) p[k] = k == A_STAMP + ST_END ? wall_clock64() : __hip_atomic_load(&ctr[k], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    if (k == 0) p[A_NCOUNTERS] = 1;
}
// the clock alone, where no kernel begins or ends a stage
__global__ void kStamp(int64_t* stamp) { *stamp = wall_clock64(); }
__global__ void kReadBack(const int64_t* __restrict__ ctr, int64_t* pin) { handOver(ctr, pin); }

// ---------------------------------------------------------------- halfedge construction
// bucket order after refreshHashTable: (face, position along the face from its first halfedge).
// refreshHashTable's per-face part, ResetFaceFlags (refreshFaceFlagsGPU) ahead of the NM bits the
// bucket pass sets again: the face's first halfedge must be a halfedge id, and
// the pattern / remove / NM bits are cleared (NM is set again from the bucket sizes)
__device__ void clearFaces(int64_t f0, const int32_t* __restrict__ face_he, int64_t F, int64_t H, uint32_t* __restrict__ fattr, int64_t* ctr) {
    if (f0 >= F) return;
    constexpr uint32_t keep = ~(uint32_t)(QA_PATTERN | QA_REMOVE | QA_NM);
    int bad = 0;
    if (vec4(f0, F, face_he, fattr)) {
        const int4 h = reinterpret_cast<const int4*>(face_he)[f0 >> 2];
        uint4 a = reinterpret_cast<const uint4*>(fattr)[f0 >> 2];
        bad = (h.x < 0 || h.x >= H) + (h.y < 0 || h.y >= H) + (h.z < 0 || h.z >= H) + (h.w < 0 || h.w >= H);
        a.x &= keep;
        a.y &= keep;
        a.z &= keep;
        a.w &= keep;
        reinterpret_cast<uint4*>(fattr)[f0 >> 2] = a;
    } else {
        for (int64_t f = f0; f < f0 + 4 && f < F; ++f) {
            const int h = face_he[f];
            bad += (h < 0 || h >= H);
            fattr[f] &= keep;
        }
    }
    if (bad) invalid(ctr, bad);
}

// ---- buckets: the halfedges joining one vertex pair.  They are listed under the
// smaller endpoint m: one short contiguous list per vertex holds every bucket of m.
// A list entry A[i] is (other endpoint | 0x80000000 when the halfedge starts at the
// other endpoint, bucket key); after an initialize the key is the halfedge id, after a
// refresh it is kept in key[h].  A halfedge finds its list from its own endpoints and the
// list offsets; the first list pass leaves only its rank in the list (rank[h]).
__device__ __forceinline__ int pairEntry(int a, int b) { return a <= b ? b : (int)(0x80000000u | (uint32_t)a); }
__device__ __forceinline__ int entryOther(int x) { return x & 0x7FFFFFFF; }

// refreshHashTable's first list pass after a split step.  Each halfedge's ids are checked
// (in range); it is dirty -- its bucket can have changed -- when it was appended or both its
// endpoints were touched.  A bucket changes only through a member that the step wrote back,
// appended or removed, and every such halfedge joins two touched vertices (the working
// copy's, before and after the step), so a halfedge with an untouched endpoint keeps its
// bucket, its members and their keys.  One block checks kDirtyPer (recordsPerLane) * kBlock consecutive halfedges,
// gathers its dirty ones in LDS and appends them to the dirty list with one atomic on
// ctr[A_DIRTY]; the list order is free, since ranks only pick list slots and bucket ranks
// come from the keys.
constexpr int kDirtyBatch = 4;
// records per lane here and in kOutDegreeMoved: 16 where the blocks still fill the chip several times
// over, else 4 (280 k records of the 201x77x131 gyroid: 9.6 us against 24 in kOutDegreeMoved, 19 either
// way here)
inline int recordsPerLane(int64_t H) { return H >= (int64_t)16 * kBlock * 2048 ? 16 : 4; }
// The blocks before quadBlocks take the records the build wrote, quad by quad: where all four keep its
// layout (canon), their origins are the quad's corners, 20 bytes per face instead of 64 and no
// other record's origin to gather; the next recordBlocks take the records appended since, the rest
// clear the faces' bits.  The sizes are those before the step plus
// what it appended, which the host does not know yet (the launch covers the most it can be).
// 512^3 gyroid, 61 M records: 264 us in the first step, 173 in the second; from the records alone 375 and 265.
struct DirtyArgs {
    const int4* he;
    int64_t oldH, oldF, oldV;
    const int4* quads;  // the build's Q quads, records [0, 4Q)
    int64_t Q;
    const uint8_t *canon, *dirtyV;
    int32_t* dlist;
    int64_t quadBlocks, recordBlocks;
    const int32_t* face_he;
    uint32_t* fattr;
    int64_t* ctr;
};
template <int kDirtyPer>
__global__ void __launch_bounds__(kBlock) kDirtyRecords(DirtyArgs a) {
    int64_t* ctr = a.ctr;
    const int64_t V = a.oldV + ctr[A_ADD], H = a.oldH + ctr[A_ADD + 1], F = a.oldF + ctr[A_ADD + 2];
    if ((int64_t)blockIdx.x >= a.quadBlocks + a.recordBlocks) {
        clearFaces(4 * (((int64_t)blockIdx.x - a.quadBlocks - a.recordBlocks) * kBlock + threadIdx.x), a.face_he, F, H, a.fattr, ctr);
        return;
    }
    const int4* __restrict__ he = a.he;
    const uint8_t* __restrict__ dirtyV = a.dirtyV;
    const int64_t oldH = a.oldH;
    __shared__ int s_list[kBlock * kDirtyPer];
    __shared__ int s_face[kBlock * kDirtyPer / 4];
    __shared__ int s_n, s_nf;
    __shared__ long long s_base;
    const int lane = threadIdx.x & 63;
    if (threadIdx.x == 0) s_n = s_nf = 0;
    __syncthreads();
    int nbad = 0;
    auto list = [&](bool hit, int64_t h) {
        const uint64_t m = __ballot(hit);
        if (m == 0) return;
        int at = 0;
        if (lane == 0) at = atomicAdd(&s_n, __popcll(m));
        at = __shfl(at, 0, 64);
        if (hit) s_list[at + __popcll(m & ((1ULL << lane) - 1ULL))] = (int)h;
    };
    if ((int64_t)blockIdx.x < a.quadBlocks) {
        constexpr int kQuads = kDirtyPer / 4;
        const int64_t f0 = (int64_t)blockIdx.x * (kBlock * kQuads) + threadIdx.x;
        int4 q[kQuads];
        uint32_t laid[kQuads];
#pragma unroll
        for (int j = 0; j < kQuads; ++j) {
            const int64_t f = f0 + j * kBlock;
            q[j] = f < a.Q ? a.quads[f] : make_int4(-1, -1, -1, -1);
            laid[j] = f < a.Q ? reinterpret_cast<const uint32_t*>(a.canon)[f] : 0u;
        }
#pragma unroll
        for (int j = 0; j < kQuads; ++j) {
            const int64_t f = f0 + j * kBlock;
            uint32_t hits = 0;
            if (laid[j] == 0x01010101u) {
                const int c[4] = {q[j].x, q[j].y, q[j].z, q[j].w};
                uint32_t d = 0;
                bool bad = false;
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const bool out = c[i] < 0 || c[i] >= V;
                    bad = bad || out;
                    d |= (!out && dirtyV[c[i]] ? 1u : 0u) << i;
                }
                nbad += bad ? 1 : 0;
                hits = d & ((d >> 1) | (d << 3)) & 0xFu;
            }
            const uint64_t other = __ballot(f < a.Q && laid[j] != 0x01010101u);
            if (other) {
                int at = 0;
                if (lane == 0) at = atomicAdd(&s_nf, __popcll(other));
                at = __shfl(at, 0, 64);
                if ((other >> lane) & 1ULL) s_face[at + __popcll(other & ((1ULL << lane) - 1ULL))] = j * kBlock + threadIdx.x;
            }
            if (__ballot(hits != 0) == 0) continue;
#pragma unroll
            for (int i = 0; i < 4; ++i) list((hits >> i) & 1u, 4 * f + i);
        }
        __syncthreads();
        // the quads with records written back: those from their records, on full waves
        const int64_t fb = (int64_t)blockIdx.x * (kBlock * kQuads);
        const int nf = 4 * s_nf;
        for (int k0 = 0; k0 < nf; k0 += kBlock) {
            const int k = k0 + threadIdx.x;
            const int64_t h = k < nf ? 4 * (fb + s_face[k >> 2]) + (k & 3) : 0;
            bool hit = false;
            if (k < nf) {
                const int4 e = he[h];
                bool bad = e.x < 0 || e.x >= V || e.y < 0 || e.y >= F || e.z < 0 || e.z >= H || e.w < -1 || e.w >= H;
                const int b = bad ? 0 : heO(he, e.z);
                bad = bad || b < 0 || b >= V;
                nbad += bad ? 1 : 0;
                hit = !bad && dirtyV[e.x] && dirtyV[b];
            }
            list(hit, h);
        }
    }
    const int64_t b0 = 4 * a.Q + ((int64_t)blockIdx.x - a.quadBlocks) * (kBlock * kDirtyPer) + threadIdx.x;
    for (int k0 = 0; k0 < kDirtyPer && (int64_t)blockIdx.x >= a.quadBlocks; k0 += kDirtyBatch) {
        int4 e[kDirtyBatch];
        int b[kDirtyBatch];
        bool bad[kDirtyBatch], d[kDirtyBatch];
#pragma unroll
        for (int j = 0; j < kDirtyBatch; ++j) {
            const int64_t t = b0 + (int64_t)(k0 + j) * kBlock;
            e[j] = t < H ? he[t] : make_int4(0, 0, 0, -1);
        }
#pragma unroll
        for (int j = 0; j < kDirtyBatch; ++j) {
            const int64_t t = b0 + (int64_t)(k0 + j) * kBlock;
            bad[j] = t < H && (e[j].x < 0 || e[j].x >= V || e[j].y < 0 || e[j].y >= F || e[j].z < 0 || e[j].z >= H || e[j].w < -1 || e[j].w >= H);
            b[j] = (t < H && !bad[j]) ? heO(he, e[j].z) : 0;
        }
#pragma unroll
        for (int j = 0; j < kDirtyBatch; ++j) {
            const int64_t t = b0 + (int64_t)(k0 + j) * kBlock;
            if (t < H && !bad[j]) bad[j] = b[j] < 0 || b[j] >= V;
            d[j] = t < H && !bad[j] && (t >= oldH || (dirtyV[e[j].x] && dirtyV[b[j]]));
            nbad += bad[j] ? 1 : 0;
        }
#pragma unroll
        for (int j = 0; j < kDirtyBatch; ++j) list(d[j], b0 + (int64_t)(k0 + j) * kBlock);
    }
    __syncthreads();
    const int n = s_n;
    if (threadIdx.x == 0 && n > 0) s_base = (long long)atomicAdd((unsigned long long*)&ctr[A_DIRTY], (unsigned long long)n);
    __syncthreads();
    const int64_t base = s_base;
    for (int i = threadIdx.x; i < n; i += kBlock) a.dlist[base + i] = s_list[i];
    if (nbad) invalid(ctr, nbad);
}

// one thread per listed halfedge h (its ids checked by kDirtyRecords): its list vertex
// m = the smaller endpoint, its list entry (other endpoint and direction, bucket key
// 4 * face + position in the face's cycle) and its slot in m's list (an atomic count on
// degM[m]), written in list order so the two passes after the scan read them contiguously.
// A halfedge missing from its face's cycle is counted in ctr[A_INVALID] (the host checks it
// at its next read-back) and still takes a slot, so every later write stays in its list.
// When the four records 4f .. 4f + 3 of h's face f all keep the build's layout (canon: face
// f, next = the quad's next) and the face starts among them, the cycle is that quad's and the
// position is (h - start) mod 4, with no walk.
__global__ void kDirtyKeys(const int4* __restrict__ he, int64_t H, const int32_t* __restrict__ face_he, const uint8_t* __restrict__ canon,
                           const int32_t* __restrict__ dlist, int64_t n, int32_t* __restrict__ degM, int32_t* __restrict__ lm, int2* __restrict__ lent,
                           int32_t* __restrict__ lrank, int64_t* ctr) {
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= n) return;
    const int h = dlist[t];
    const int4 e = he[h];
    const int b = heO(he, e.z);
    int k = face_he[e.y], pos = 0;
    const int f = e.y;
    if (canon && (h >> 2) == f && 4 * (int64_t)f + 3 < H && (k >> 2) == f && reinterpret_cast<const uint32_t*>(canon)[f] == 0x01010101u) {
        pos = (h - k) & 3;
        k = h;
    }
    while (pos < 4 && k != h && k >= 0 && k < H) {
        k = heN(he, k);
        ++pos;
    }
    if (k != h) invalid(ctr);
    const int m = min(e.x, b);
    lm[t] = m;
    lent[t] = make_int2(pairEntry(e.x, b), k == h ? 4 * e.y + pos : 0x7FFFFFFF);
    lrank[t] = atomicAdd(&degM[m], 1);
}

// second list pass, after the scan of the counts: the entry of each listed halfedge goes to
// offM[m] + its slot
__global__ void kPlaceEntries(const int32_t* __restrict__ lm, const int2* __restrict__ lent, const int32_t* __restrict__ lrank, int64_t n,
                              const int64_t* __restrict__ offM, int2* __restrict__ A) {
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= n) return;
    A[offM[lm[t]] + lrank[t]] = lent[t];
}

// the four slots of a bucket: entries beyond the fourth land in slot 0 (glm::ivec4::operator[] default)
__device__ __forceinline__ void bucketSlots(const int mem[kMaxBucket], int n, int s[4]) {
    for (int i = 0; i < 4; ++i) s[i] = (i < n) ? mem[i] : -1;
    for (int k = 4; k < n && k < kMaxBucket; ++k) s[0] = mem[k];
}

__device__ __forceinline__ uint32_t bucketVertexFlag(int n) { return n == 4 ? VF_NM : (n == 3 ? VF_WEIRD : (n == 1 ? VF_BOUNDARY : 0u)); }

// One thread per listed halfedge h of a refresh, reading only the short list of its smaller
// endpoint: the size of its bucket and its rank (position in key order).
__global__ void kBuckets(const int32_t* __restrict__ dlist, const int32_t* __restrict__ lm, const int2* __restrict__ lent, int64_t nList,
                         const int64_t* __restrict__ offM, const int2* __restrict__ A, int32_t* __restrict__ bsize, int32_t* __restrict__ brank) {
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= nList) return;
    const int m = lm[t];
    const int2 own = lent[t];
    const int64_t lo = offM[m], hi = offM[m + 1];
    const int o = entryOther(own.x), key = own.y;
    int n = 0, rk = 0;
    for (int64_t i = lo; i < hi; ++i) {
        const int2 f = A[i];
        if (entryOther(f.x) != o) continue;
        ++n;
        if (f.y < key) ++rk;
    }
    const int h = dlist[t];
    bsize[h] = bucketWord(n, rk);
    if (n >= 4) brank[h] = rk;
}

// vertex flags and face NM bits from the bucket sizes of all halfedges (vflags and the
// faces' NM bits cleared beforehand)
// (four halfedges per thread, their sizes read with one 16-byte load)
__device__ __forceinline__ void sizes4(const int32_t* __restrict__ bsize, int64_t H, int64_t h0, int n[4]) {
    if (h0 + 3 < H) {
        const int4 v = reinterpret_cast<const int4*>(bsize)[h0 >> 2];
        n[0] = bucketSize(v.x);
        n[1] = bucketSize(v.y);
        n[2] = bucketSize(v.z);
        n[3] = bucketSize(v.w);
    } else {
        for (int j = 0; j < 4; ++j) n[j] = h0 + j < H ? bucketSize(bsize[h0 + j]) : 2;
    }
}
__global__ void __launch_bounds__(kBlock) kFlagsFromBuckets(const int4* __restrict__ he, int64_t H, const int32_t* __restrict__ bsize,
                                                            const int32_t* __restrict__ brank, uint32_t* __restrict__ vflags,
                                                            uint32_t* __restrict__ fattr, int64_t* nmParts) {
    const int64_t h0 = 4 * ((int64_t)blockIdx.x * blockDim.x + threadIdx.x);
    int slotted = 0;
    if (h0 < H) {
        int n[4];
        sizes4(bsize, H, h0, n);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            if (n[j] >= 4 && slottedNM(n[j], brank[h0 + j])) ++slotted;
            const uint32_t vf = bucketVertexFlag(n[j]);
            if (!vf) continue;
            const int4 e = he[h0 + j];
            atomicOr(&vflags[e.x], vf);
            if (n[j] == 4) atomicOr(&fattr[e.y], (uint32_t)QA_NM);
        }
    }
    blockAdd(nmParts, slotted);
}

// ---------------------------------------------------------------- halfedge build from outgoing lists
// HalfedgeMesh::initialize (HalfedgeMesh.cu:14-291) from a quad list: halfedge 4f + i runs
// from corner i of quad f to corner i + 1.  The build keeps, per vertex v, the list of the
// halfedges starting at v (out[off[v] .. off[v + 1])).  A bucket -- the halfedges joining
// two vertices a and b -- is read from the list of m = min(a, b): the halfedges x of that
// list that end at o = max(a, b) start at m, and (o != m) the halfedge before such an x in
// its quad starts at o when that quad has o just before m.  Members are ordered by id, as
// the reference's bucket keys are the halfedge ids right after an initialize.
__device__ __forceinline__ int quadCorner(const int4& q, int j) { return j == 0 ? q.x : (j == 1 ? q.y : (j == 2 ? q.z : q.w)); }

struct BucketOf {
    int n, rank, twin;
};
// size and rank of a halfedge's bucket in one word while the simplifications run (both are
// at most the bucket size; a bucket of 65536 or more halfedges saturates)
__device__ __forceinline__ uint32_t packBucket(int n, int rank) { return (uint32_t)min(n, 0xFFFF) | ((uint32_t)min(rank, 0xFFFF) << 16); }

// the twin connectHalfedgeTwins (HalfedgeMesh.cu:173-291) gives the member of rank rk of a
// bucket of n halfedges (mem / dir: its first four members and their directions, in any
// order; partner: the other member of a pair)
__device__ __forceinline__ int bucketTwin(int n, int rk, int partner, int mem[4], int dir[4]) {
    if (n == 2) return partner;
    if (n != 3 && n != 4) return -1;
    for (int i = 1; i < n; ++i) {  // by id
        const int x = mem[i], dx = dir[i];
        int j = i - 1;
        while (j >= 0 && mem[j] > x) {
            mem[j + 1] = mem[j];
            dir[j + 1] = dir[j];
            --j;
        }
        mem[j + 1] = x;
        dir[j + 1] = dx;
    }
    if (n == 3) return mem[(rk + 1) % 3];
    int pr;
    if (dir[0] != dir[1]) pr = rk ^ 1;       // (0,1) (2,3)
    else if (dir[0] != dir[2]) pr = rk ^ 2;  // (0,2) (1,3)
    else pr = 3 - rk;                        // (0,3) (1,2)
    return mem[pr];
}

// bucket size, rank of h and the twin connectHalfedgeTwins (HalfedgeMesh.cu:173-291) gives h:
// the partner of a pair, the next by id of three, the first other-direction member paired
// with the first of four (the same rules kBuckets applies to the bucket lists)
__device__ BucketOf bucketFromOut(int h, int a, int b, const int4* __restrict__ quads, int64_t H, const int64_t* __restrict__ off,
                                  const int32_t* __restrict__ out, int64_t* ctr) {
    const int m = min(a, b), o = max(a, b);
    int mem[4], dir[4];
    int n = 0, rk = 0, partner = -1;
    bool self = false;
    auto add = [&](int id, int d) {
        if (n < 4) {
            mem[n] = id;
            dir[n] = d;
        }
        ++n;
        if (id < h) ++rk;
        if (id != h) partner = id;
        else self = true;
    };
    // the list in groups of four entries, their quads loaded side by side
    const int64_t k0 = off[m], k1 = off[m + 1];
    for (int64_t kb = k0; kb < k1; kb += 4) {
        int xs[4];
        int4 qs[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) xs[i] = kb + i < k1 ? out[kb + i] : 0;
#pragma unroll
        for (int i = 0; i < 4; ++i) qs[i] = (kb + i < k1 && xs[i] >= 0 && xs[i] < H) ? quads[xs[i] >> 2] : make_int4(0, 0, 0, 0);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            if (kb + i >= k1) continue;
            const int x = xs[i];
            if (x < 0 || x >= H) {
                anomaly(ctr);
                continue;
            }
            const int4 q = qs[i];
            const int j = x & 3;
            if (quadCorner(q, j) != m) anomaly(ctr);
            if (quadCorner(q, (j + 1) & 3) == o) add(x, 0);
            if (o != m && quadCorner(q, (j + 3) & 3) == o) add((x & ~3) | ((j + 3) & 3), 1);
        }
    }
    if (!self) anomaly(ctr);
    return BucketOf{n, rk, bucketTwin(n, rk, partner, mem, dir)};
}

// The same for the initialize, from the place kQuadLists gives (code): a pair's other halfedge ends
// where the list's entry starts, as do the halfedges of a face's bucket an odd number of edges on.
// (With a search for the latter, one halfedge in several hundred, kBucketsAll took 690 us at the
// 512^3 gyroid instead of 505: a wave waits for its longest lane.)
__device__ __forceinline__ BucketOf bucketFromPair(int h, int code, const uint32_t* pairFace, const int4* __restrict__ quads, int64_t H,
                                                   const int64_t* __restrict__ off, const int32_t* __restrict__ out, int64_t* ctr) {
    if (code >= 0) {
        const int x = out[code];
        if (x >= 0 && x < H) {
            const int t = quadNext(x, 3);
            return BucketOf{2, t < h ? 1 : 0, t};
        }
    } else if (code == kPairNone) {
        return BucketOf{1, 0, -1};
    } else if (code <= kPairFace) {
        const uint32_t w = pairFace[h];
        const int base = kPairFace - code, own = (int)(w >> 20) & 3;
        int x[4], mem[4], dir[4], n = 0, rk = 0, partner = -1;
        bool bad = false;
#pragma unroll
        for (int p = 0; p < 4; ++p) x[p] = (w >> (16 + p)) & 1u ? out[base + (int)((w >> (4 * p)) & 0xFu)] : -1;
#pragma unroll
        for (int p = 0; p < 4; ++p) {
            if (!((w >> (16 + p)) & 1u)) continue;
            bad = bad || x[p] < 0 || x[p] >= H;
            const int d = (p ^ own) & 1, id = d ? quadNext(x[p], 3) : x[p];
            mem[n] = id;
            dir[n] = d;
            ++n;
            if (id < h) ++rk;
            if (id != h) partner = id;
        }
        if (!bad) return BucketOf{n, rk, bucketTwin(n, rk, partner, mem, dir)};
    }
    const int4 q = quads[h >> 2];
    return bucketFromOut(h, quadCorner(q, h & 3), quadCorner(q, (h + 1) & 3), quads, H, off, out, ctr);
}

// the members of h's bucket sorted by id (first kMaxBucket), returns the true count
__device__ int gatherBucketOut(int h, const int4* __restrict__ quads, int64_t H, const int64_t* __restrict__ off, const int32_t* __restrict__ out,
                               int mem[kMaxBucket]) {
    const int4 qh = quads[h >> 2];
    const int a = quadCorner(qh, h & 3), b = quadCorner(qh, (h + 1) & 3);
    const int m = min(a, b), o = max(a, b);
    int n = 0;
    for (int64_t k = off[m]; k < off[m + 1]; ++k) {
        const int x = out[k];
        if (x < 0 || x >= H) continue;
        const int4 q = quads[x >> 2];
        const int j = x & 3;
        if (quadCorner(q, (j + 1) & 3) == o) {
            if (n < kMaxBucket) mem[n] = x;
            ++n;
        }
        if (o != m && quadCorner(q, (j + 3) & 3) == o) {
            if (n < kMaxBucket) mem[n] = (x & ~3) | ((j + 3) & 3);
            ++n;
        }
    }
    const int cnt = n < kMaxBucket ? n : kMaxBucket;
    for (int i = 1; i < cnt; ++i) {
        const int x = mem[i];
        int j = i - 1;
        while (j >= 0 && mem[j] > x) {
            mem[j + 1] = mem[j];
            --j;
        }
        mem[j + 1] = x;
    }
    return n;
}

// the bucket of halfedge h = 4f + i, and what the bucket pass of an initialize
// derives from it: vertex flags of the origin, the face's NM bit (fattr and the quad
// attributes), an incoming boundary halfedge's share of the destination's valence.  Until the
// simplifications are done a halfedge is its id (origin = corner i of quad f, face f, next
// 4f + (i + 1) % 4) and its twin; the full records are written once after them
// (kRemapRebuild, or kBuildHalfedges where none runs).
__device__ __forceinline__ void storeHalfedge(int h, const int4* __restrict__ quads, const BucketOf& bk, int32_t* __restrict__ twin,
                                              uint32_t* __restrict__ bpack, uint32_t* __restrict__ vflags, uint32_t* __restrict__ fattr,
                                              uint32_t* __restrict__ qattr, int32_t* __restrict__ valence, int32_t* __restrict__ bdin) {
    const int f = h >> 2;
    twin[h] = bk.twin;
    bpack[h] = packBucket(bk.n, bk.rank);
    if (bk.n == 2) return;
    const int4 q = quads[f];
    if (bk.twin == -1) {
        const int b = quadCorner(q, (h + 1) & 3);
        atomicAdd(&valence[b], 1);
        if (bdin) atomicAdd(&bdin[b], 1);
    }
    const uint32_t vf = bucketVertexFlag(bk.n);
    if (vf) atomicOr(&vflags[quadCorner(q, h & 3)], vf);
    if (bk.n == 4) {
        atomicOr(&fattr[f], (uint32_t)QA_NM);
        atomicOr(&qattr[f], (uint32_t)QA_NM);
    }
}

// the same as a finished record with its bucket size and rank (nothing reads ids and twins
// only any more); returns whether the split's working copy would mark it (slottedNM)
__device__ __forceinline__ bool storeRecord(int h, int a, const BucketOf& bk, int4* __restrict__ he, int32_t* __restrict__ bsize,
                                           int32_t* __restrict__ brank, uint32_t* __restrict__ vflags, uint32_t* __restrict__ fattr) {
    const int n = min(bk.n, 0xFFFF), r = min(bk.rank, 0xFFFF);
    he[h] = make_int4(a, h >> 2, quadNext(h, 1), bk.twin);
    bsize[h] = bucketWord(n, r);
    if (n >= 4) brank[h] = r;
    const uint32_t vf = bucketVertexFlag(n);
    if (vf) atomicOr(&vflags[a], vf);
    if (n == 4) atomicOr(&fattr[h >> 2], (uint32_t)QA_NM);
    return slottedNM(n, r);
}

// Every halfedge from its bucket, found where kQuadLists says (in twin and bpack, which then
// take the results).
// Bound by HBM and the gathered list entries: 1.1 GB at least at the 512^3 gyroid's 69 M halfedges
// (240 us), 505 us; searching the lists for every halfedge took 991 us, one thread per quad 789 us.
__global__ void kBucketsAll(const int4* __restrict__ quads, int64_t H, const int64_t* __restrict__ off, const int32_t* __restrict__ out,
                            int32_t* twin, uint32_t* bpack, uint32_t* __restrict__ vflags,
                            uint32_t* __restrict__ fattr, uint32_t* __restrict__ qattr, int32_t* __restrict__ valence, int32_t* __restrict__ bdin,
                            int64_t* ctr) {
    const int64_t hh = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (hh >= H || chainHeld(ctr, 0)) return;
    const int h = (int)hh;
    storeHalfedge(h, quads, bucketFromPair(h, twin[h], bpack, quads, H, off, out, ctr), twin, bpack, vflags, fattr, qattr, valence, bdin);
}

// The same with the records, sizes and ranks written at once, when no simplification (which
// reads ids and twins only) follows: one launch and 24 bytes per halfedge less to move than
// kBucketsAll and a pass that turns its words into records.  The quads are
// checked (kQuadLists) but the host has not looked yet: if any was inconsistent, every record is
// a boundary halfedge of vertex 0, which the kernels launched before the host's next wait can
// follow.
__global__ void __launch_bounds__(kBlock) kBuildHalfedges(const int4* __restrict__ quads, int64_t H, const int64_t* __restrict__ off,
                                                          const int32_t* __restrict__ out, const int32_t* __restrict__ pairAt, const uint32_t* __restrict__ pairFace, int4* __restrict__ he,
                                                          int32_t* __restrict__ bsize, int32_t* __restrict__ brank, uint32_t* __restrict__ vflags,
                                                          uint32_t* __restrict__ fattr, int64_t* nmParts, int64_t* ctr) {
    const int64_t hh = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const bool bad = ctr[A_INVALID] != 0;
    bool slotted = false;
    if (hh < H) {
        const int h = (int)hh;
        int a = 0;
        BucketOf bk{2, 1, -1};
        if (!bad) {
            a = quadCorner(quads[h >> 2], h & 3);
            bk = bucketFromPair(h, pairAt[h], pairFace, quads, H, off, out, ctr);
        }
        slotted = storeRecord(h, a, bk, he, bsize, brank, vflags, fattr);
    }
    waveAdd(nmParts, slotted);
}

// ---- rebuild after a simplification's compaction.  New vertex v' = address[v]; a dropped
// vertex u (vtype[u] == dropType) reappears as t' = address[vtarget[u]] in the faces that
// kCompactQuads relabels; every such t' is touched.  Every edge of a removed quad has a
// dropped or a target endpoint: (x, y, z, w) of a P3X3Y merge drops z into x, and the four
// neighbours (v', v, c, c') of a P3333 centre drop v, v' (into c, c').  So a bucket whose
// two endpoints are untouched has the same members as before (no relabelled vertex maps
// onto either endpoint and no member lay in a removed quad), renumbered in the same order,
// and its halfedges keep size, rank and (renumbered) twin; the others are recomputed from
// the new outgoing lists.  qnew[f] is the new id of old quad f (-1: removed).
//
// Most P3333 merges need no list.  The centre f becomes the quad of the four targets, and its halfedge i
// takes the place of e_i, the outer halfedge of the removed neighbour across its edge i: same ends,
// same direction.  A regular centre (kMark3333: each neighbour's twin is mutual and opposite, its outer
// corners are the targets of the two inner ones) loses
// no other halfedge between kept vertices.  Its corners' three outgoing halfedges lie in itself and two
// neighbours, and a neighbour is no centre nor has it a second regular one: either would have
// a target among its corners, whose valence is not 3.  So every bucket away from the
// targets of irregular centres keeps its size, and one of one or two halfedges its members, with e_i
// replaced by 4f + i; from e_i, that is the twin of the halfedge across its quad.  Only the targets of
// irregular centres are touched then, and larger buckets, whose order may change, are recomputed.
// (At the 512^3 gyroid a third of the halfedges start or end at a target, 0.8% are recomputed now.)
//
// Source chains (by old vertex id): the outgoing halfedges of vertex t are the entries of the
// lists of t and of every vertex on its chain head[t], next[head[t]], ...  A dropped vertex u
// joins its target's chain together with its own chain (vertices dropped into u by earlier
// steps of a deferred chain of simplifications).  Entries of removed or dead quads stay in the
// lists and are skipped by their quad.
__device__ __forceinline__ void spliceChain(int u, int t, int32_t* __restrict__ head, int32_t* __restrict__ next) {
    int last = u;
    const int h0 = head[u];
    if (h0 >= 0) {
        next[u] = h0;
        last = h0;
        while (next[last] >= 0) last = next[last];
    }
    next[last] = atomicExch(&head[t], u);
}

// Sparse work whose every item is a chain of dependent loads: a block takes kSparsePer *
// kBlock consecutive items, calls pred(i) once for each (i < n), gathers the flagged ones in
// LDS (in no particular order) and returns their number; the block then works through the
// list on all its lanes, so one block overlaps many chains instead of a few.
constexpr int kSparsePer = 8;
template <class Pred>
__device__ __forceinline__ int gatherSparse(int64_t n, Pred pred, int* s_list, int* s_n) {
    if (threadIdx.x == 0) *s_n = 0;
    __syncthreads();
    const int lane = threadIdx.x & 63;
    const int64_t b0 = (int64_t)blockIdx.x * (kSparsePer * kBlock) + threadIdx.x;
#pragma unroll
    for (int k = 0; k < kSparsePer; ++k) {
        const int64_t i = b0 + (int64_t)k * kBlock;
        const bool f = i < n && pred(i);
        const uint64_t m = __ballot(f);
        int at = 0;
        if (lane == 0 && m) at = atomicAdd(s_n, __popcll(m));
        at = __shfl(at, 0, 64);
        if (f) s_list[at + __popcll(m & ((1ULL << lane) - 1ULL))] = (int)i;
    }
    __syncthreads();
    return *s_n;
}
inline unsigned sparseBlocks(int64_t n) { return (unsigned)((n + kSparsePer * kBlock - 1) / (kSparsePer * kBlock)); }

__global__ void __launch_bounds__(kBlock) kSources(const uint8_t* __restrict__ vtype, const int32_t* __restrict__ vtarget,
                                                   const int32_t* __restrict__ address, int64_t V, int dropType, uint8_t* __restrict__ touched,
                                                   int32_t* __restrict__ srcHead, int32_t* __restrict__ srcNext, int32_t* __restrict__ outdeg,
                                                   bool touch) {
    // the block's dropped vertices gathered in LDS and handled on consecutive lanes
    __shared__ int s_list[kSparsePer * kBlock];
    __shared__ int s_n;
    const int total = gatherSparse(V, [&](int64_t i) { return vtype[i] == dropType; }, s_list, &s_n);
    for (int j = threadIdx.x; j < total; j += kBlock) {
        const int u = s_list[j];
        const int t = vtarget[u];
        if (t < 0 || t >= V) continue;
        const int tn = address[t];
        if (tn < 0) continue;  // the relabelled quads then hold -1 and fail validation
        if (touch) touched[tn] = 1;
        spliceChain(u, t, srcHead, srcNext);
        if (outdeg) {
            atomicAdd(&outdeg[t], outdeg[u]);
            outdeg[u] = 0;
        }
    }
}

// new vertex v': the halfedges of kept quads in the lists of its old vertex and of the
// vertices on that vertex's chain, counted (every list by current corner: list lengths less the
// halfedges of removed quads, removedAt; after deferred steps: the out-degree kept through the
// chain's removals and drops), then written with their new ids (the bucket pass checks every
// entry it reads against the quad's corner).  The counting pass also moves the vertex's
// position and normal (each new vertex gathers its old one's: 173 us at the 512^3 gyroid with the
// count; scattered by old vertex instead 252 us alone, inside kNumber's rounds 255 us)
__global__ void kOutCount(const int32_t* __restrict__ oldV, int64_t Vn, const int64_t* __restrict__ off, const int32_t* __restrict__ removedAt,
                          const int32_t* __restrict__ srcHead, const int32_t* __restrict__ srcNext, const int32_t* __restrict__ outdeg,
                          int32_t* __restrict__ cnt, const float* __restrict__ pos, const float* __restrict__ nrm, float* __restrict__ npos,
                          float* __restrict__ nnrm) {
    const int64_t vn = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (vn >= Vn) return;
    int u = oldV[vn];
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        npos[3 * vn + k] = pos[3 * (int64_t)u + k];
        nnrm[3 * vn + k] = nrm[3 * (int64_t)u + k];
    }
    if (outdeg) {
        cnt[vn] = outdeg[u];
        return;
    }
    int64_t c = 0;
    int s = srcHead[u];
    for (;;) {
        c += off[u + 1] - off[u] - removedAt[u];
        if (s < 0) break;
        u = s;
        s = srcNext[s];
    }
    cnt[vn] = (int32_t)c;
}

__global__ void kOutFill(const int32_t* __restrict__ oldV, int64_t Vn, const int64_t* __restrict__ off, const int32_t* __restrict__ out,
                         const int32_t* __restrict__ qnew, const int32_t* __restrict__ srcHead,
                         const int32_t* __restrict__ srcNext, const int64_t* __restrict__ off2, int32_t* __restrict__ out2, int64_t cap,
                         int64_t* ctr) {
    const int64_t vn = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (vn >= Vn) return;
    int64_t w = off2[vn];
    int u = oldV[vn];
    int s = srcHead[u];
    for (;;) {
        // groups of four list entries, their new quad ids loaded side by side
        const int64_t k1 = off[u + 1];
        for (int64_t kb = off[u]; kb < k1; kb += 4) {
            int xs[4], fns[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) xs[i] = kb + i < k1 ? out[kb + i] : 0;
#pragma unroll
            for (int i = 0; i < 4; ++i) fns[i] = kb + i < k1 ? qnew[xs[i] >> 2] : -1;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                if (fns[i] < 0) continue;
                if (w < cap) out2[w++] = 4 * fns[i] + (xs[i] & 3);
                else anomaly(ctr);
            }
        }
        if (s < 0) break;
        u = s;
        s = srcNext[s];
    }
}

constexpr int kRebuilt = INT32_MIN;  // in place of a twin: the halfedge is recomputed
constexpr int kOldCentre = 1 << 30;  // in oldQ: the old quad is the centre of a P3333 merge (4 Q < 2^31)
// A halfedge with two untouched endpoints takes size, rank and renumbered twin from its old
// halfedge; the block's other halfedges are gathered in LDS and recomputed from their
// buckets afterwards on full waves.  The chain ends here, so the finished records are written.  A thread
// takes a quad's four halfedges, so that the loads behind the old quad's id are in flight together, and
// the records go through LDS, in order across lanes (stored by quad, every line is written
// back in parts: 2.7 GB instead of 1.4).  Bound by HBM: 2.3 GB moved at the 512^3 gyroid in 579 us
// (616 with the records stored through the caches, and the twin repair behind it 214 instead of 203); a
// thread per halfedge 944 us, the records stored by quad 839 us.
// The compaction checks the quads' new corners, but the host may go on before it has looked (it waits for
// the numbering's totals only): with a bad one, every record is a boundary halfedge of vertex 0, as in
// kBuildHalfedges, no corner is followed, and the next read-back reports it.
__global__ void __launch_bounds__(kBlock) kRemapRebuild(const int4* __restrict__ quads2, int64_t H2, const uint8_t* __restrict__ touched,
                                                        const int32_t* __restrict__ oldQ, const int32_t* __restrict__ twinOld, int64_t Hold,
                                                        const uint32_t* __restrict__ bpackOld,
                                                        const int32_t* __restrict__ qnew, const int64_t* __restrict__ off2,
                                                        const int32_t* __restrict__ out2, int4* __restrict__ he, int32_t* __restrict__ bsize,
                                                        int32_t* __restrict__ brank, uint32_t* __restrict__ vflags, uint32_t* __restrict__ fattr,
                                                        int64_t* nmParts, bool replace, int64_t* ctr) {
    __shared__ __align__(16) int s_v[4 * kBlock], s_t[4 * kBlock];
    __shared__ int s_list[4 * kBlock];
    __shared__ int s_n;
    const int64_t f = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (ctr[A_INVALID] != 0) {
        for (int i = 0; i < 4 && f < H2 / 4; ++i) storeRecord((int)(4 * f + i), 0, BucketOf{2, 1, -1}, he, bsize, brank, vflags, fattr);
        return;
    }
    if (threadIdx.x == 0) s_n = 0;
    __syncthreads();
    int slotted = 0;
    if (f < H2 / 4) {
        const int4 q = quads2[f];
        const int oq = oldQ[f];
        const int fo = oq & ~kOldCentre;
        const int4 t4 = reinterpret_cast<const int4*>(twinOld)[fo];
        const uint4 b4 = reinterpret_cast<const uint4*>(bpackOld)[fo];
        const int v[4] = {q.x, q.y, q.z, q.w};
        int tt[4] = {t4.x, t4.y, t4.z, t4.w};
        uint32_t bo[4] = {b4.x, b4.y, b4.z, b4.w};
        uint8_t tc[4];
        bool later[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) tc[i] = touched[v[i]];
#pragma unroll
        for (int i = 0; i < 4; ++i) later[i] = (tc[i] | tc[(i + 1) & 3]) != 0;
        if (replace && (oq & kOldCentre)) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                if (later[i]) continue;
                if (tt[i] >= 0 && tt[i] < Hold) {  // (a centre has four neighbours)
                    const int e = quadNext(tt[i], 2);
                    tt[i] = twinOld[e];
                    bo[i] = bpackOld[e];
                } else {
                    later[i] = true;
                }
            }
        }
        int fn[4], nb[4], rk[4], tn[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) fn[i] = tt[i] >= 0 && tt[i] < Hold ? qnew[tt[i] >> 2] : 0;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int h = (int)(4 * f + i);
            nb[i] = (int)(bo[i] & 0xFFFFu);
            rk[i] = (int)(bo[i] >> 16);
            if (replace && nb[i] > 2) later[i] = true;
            if (later[i]) {
                s_list[atomicAdd(&s_n, 1)] = h;
                tn[i] = kRebuilt;
                continue;
            }
            int t = -1;
            if (tt[i] >= Hold) {
                anomaly(ctr);
            } else if (tt[i] >= 0) {
                int fo2 = fn[i];
                if (replace && fo2 < 0) {  // an outer halfedge of a removed neighbour
                    const int opposite = quadNext(tt[i], 2), c = twinOld[opposite];
                    if (c >= 0 && c < Hold && twinOld[c] == opposite) {
                        tt[i] = c;
                        fo2 = qnew[c >> 2];
                    }
                }
                if (fo2 < 0) anomaly(ctr);
                else t = 4 * fo2 + (tt[i] & 3);
            }
            if (replace) rk[i] = t >= 0 && t < h ? 1 : 0;
            tn[i] = t;
            const uint32_t vf = bucketVertexFlag(nb[i]);
            if (vf) atomicOr(&vflags[v[i]], vf);
            if (nb[i] == 4) atomicOr(&fattr[f], (uint32_t)QA_NM);
            slotted += slottedNM(nb[i], rk[i]) ? 1 : 0;
            if (nb[i] >= 4) brank[h] = rk[i];
        }
        reinterpret_cast<int4*>(bsize)[f] =
            make_int4(bucketWord(nb[0], rk[0]), bucketWord(nb[1], rk[1]), bucketWord(nb[2], rk[2]), bucketWord(nb[3], rk[3]));
        reinterpret_cast<int4*>(s_v)[threadIdx.x] = q;
        reinterpret_cast<int4*>(s_t)[threadIdx.x] = make_int4(tn[0], tn[1], tn[2], tn[3]);
    }
    waveSum(nmParts, slotted);
    __syncthreads();
    // the records from LDS, in order across lanes
    const int64_t h0 = (int64_t)blockIdx.x * (4 * kBlock);
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const int l = k * kBlock + threadIdx.x;
        const int h = (int)(h0 + l);
        if (h0 + l < H2 && s_t[l] != kRebuilt) storeStreaming(he + h, make_int4(s_v[l], h >> 2, quadNext(h, 1), s_t[l]));
    }
    const int total = s_n;
    for (int k = threadIdx.x; k < total; k += kBlock) {
        const int h = s_list[k];
        const int4 q = quads2[h >> 2];
        const int a = quadCorner(q, h & 3), b = quadCorner(q, (h + 1) & 3);
        waveAdd(nmParts, storeRecord(h, a, bucketFromOut(h, a, b, quads2, H2, off2, out2, ctr), he, bsize, brank, vflags, fattr));
    }
}

// the P3X3Y valence patterns (markElementsP3X3Y, HalfedgeMesh.cu:317-339)
__device__ __forceinline__ bool pattern1(const int v[4]) { return v[0] == 3 && v[1] >= 5 && v[2] == 3 && v[3] >= 5; }
__device__ __forceinline__ bool pattern2(const int v[4]) { return v[0] >= 5 && v[1] == 3 && v[2] >= 5 && v[3] == 3; }

// ---- a chain of simplifications with its compaction deferred to the chain's last step.
// Between the steps every id stays as the halfedge initialize numbered it: a removed quad
// becomes dead (QA_DEAD in qattr and fattr, skipped by every later kernel), a dropped vertex
// becomes dead (vdead) after splicing itself and its chain onto its target's chain, and the
// surviving quads have their corners relabelled in place.  Twins and bucket words are
// recomputed in place for the halfedges with a touched endpoint (the targets) only; the
// others keep theirs (the same argument as for the compacting rebuild above).  The chain's
// last step compacts vertices and quads once, renumbering everything, which gives the arrays
// the step-by-step compactions give (stable compactions compose, and bucket ranks and the
// twin rules only compare ids, whose order every compaction keeps).

// P3X3Y merge (x, a1, z, a3) -> x whose neighbourhood is a plain patch: the four edges of the
// removed quad Q are pairs, x and z each have a closed fan of three quads (Q, N_X, N_B and Q,
// N_A, N_Z) with third neighbours d and c, and after every merge of the step is applied (a
// dropped vertex stands for its target, rep) rep(c) and rep(d) differ from each other and
// from the quad's corners.  Then x's and z's edges to a1 and a3 become two new pairs -- the
// halfedge across a1-x with the one across z-a1, the one across a3-z with the one across x-a3
// -- every other bucket keeps its members (the edge z-c is renamed x-rep(c), x-d is x-rep(d),
// neither meeting another), and no flag or boundary count moves, so the four twins and bucket
// words are written here.  (Q's neighbours are not removed: two merges never share a quad,
// and no other merge writes or reads the halfedges read or written here.)  Any other merge
// marks its target touched for the region rebuild below and is counted in ctr[A_FALLBACK + step].  The block's
// merges are gathered in LDS first: each is a chain of dependent loads.
// The same launch applies removeQuadrilateralsP3X3Y in place: every kept quad gets the
// compaction's attributes (colour unset, NM and boundary kept: no REMOVE or DEAD bit before or
// after, so the neighbour tests read the same either way), and the lane of each removed quad,
// after reading it, takes one outgoing halfedge off each of its corners, sets its corners to
// -1 and marks it dead.  For a local merge the two corners holding z in N_A and N_Z are
// recorded (zslot) for kDropVertices; a fallback merge's target relabels through z's lists.
__global__ void __launch_bounds__(kBlock) kLocalMerge(int4* __restrict__ quads, uint32_t* qattr, uint32_t* fattr, int64_t Q,
                                                      const int32_t* __restrict__ valence, const uint8_t* __restrict__ vtype,
                                                      const int32_t* __restrict__ vtarget, int32_t* __restrict__ twin, uint32_t* __restrict__ bpack,
                                                      int32_t* __restrict__ outdeg, int2* __restrict__ zslot, int64_t V, uint8_t* __restrict__ touched,
                                                      int allowLocal, int step, int64_t* ctr) {
    if (chainHeld(ctr, step)) return;
    __shared__ int s_list[kSparsePer * kBlock];
    __shared__ int s_n;
    const int total = gatherSparse(
        Q,
        [&](int64_t qq) {
            const uint32_t a = qattr[qq];
            const bool merging = !(a & QA_DEAD) && (a & QA_REMOVE);
            if (!(a & QA_DEAD) && !merging) {
                uint32_t na = QA_COLOR;
                if (a & QA_NM) na |= QA_NM;
                if (a & QA_BOUNDARY) na |= QA_BOUNDARY;
                qattr[qq] = na;
                fattr[qq] = na;
            }
            return merging;
        },
        s_list, &s_n);
    int nfallback = 0;
    for (int j = threadIdx.x; j < total; j += kBlock) {
        const int q = s_list[j];
        const int4 v4 = quads[q];
        const int v[4] = {v4.x, v4.y, v4.z, v4.w};
        const int val[4] = {valence[v[0]], valence[v[1]], valence[v[2]], valence[v[3]]};
        const int X = pattern1(val) ? 0 : 1;  // the merge used pattern 1 (x = corner 0) or 2 (x = corner 1)
        const int Z = X + 2;
        const int x = v[X], a1 = v[X + 1], z = v[Z], a3 = v[(X + 3) & 3];
        const int4 tw4 = reinterpret_cast<const int4*>(twin)[q];
        const int t[4] = {tw4.x, tw4.y, tw4.z, tw4.w};
        const int tX = t[X], tA = t[X + 1], tZ = t[Z], tB = t[(X + 3) & 3];  // across x-a1, a1-z, z-a3, a3-x
        const uint4 bp = reinterpret_cast<const uint4*>(bpack)[q];
        bool ok = allowLocal && x != a1 && x != z && x != a3 && a1 != z && a1 != a3 && z != a3;
        ok = ok && (bp.x & 0xFFFFu) == 2 && (bp.y & 0xFFFFu) == 2 && (bp.z & 0xFFFFu) == 2 && (bp.w & 0xFFFFu) == 2;
        ok = ok && tX >= 0 && tA >= 0 && tZ >= 0 && tB >= 0;
        if (ok) {
            const int nX = tX >> 2, nA = tA >> 2, nZ = tZ >> 2, nB = tB >> 2;
            ok = nX != q && nA != q && nZ != q && nB != q;
            constexpr uint32_t gone = QA_REMOVE | QA_DEAD;
            ok = ok && !((qattr[nX] | qattr[nA] | qattr[nZ] | qattr[nB]) & gone);
            if (ok) {
                const int4 NX = quads[nX], NA = quads[nA], NZ = quads[nZ], NB = quads[nB];
                // x's fan: after tX (a1 -> x) in N_X comes x -> d1; before tB (x -> a3) in N_B comes d2 -> x
                const int hXn = (tX & ~3) | ((tX + 1) & 3), hBp = (tB & ~3) | ((tB + 3) & 3);
                const int d1 = quadCorner(NX, (tX + 2) & 3), d2 = quadCorner(NB, (tB + 3) & 3);
                // z's fan: before tA (z -> a1) in N_A comes c1 -> z; after tZ (a3 -> z) in N_Z comes z -> c2
                const int hAp = (tA & ~3) | ((tA + 3) & 3), hZn = (tZ & ~3) | ((tZ + 1) & 3);
                const int c1 = quadCorner(NA, (tA + 3) & 3), c2 = quadCorner(NZ, (tZ + 2) & 3);
                ok = quadCorner(NX, tX & 3) == a1 && quadCorner(NA, tA & 3) == z && quadCorner(NZ, tZ & 3) == a3 && quadCorner(NB, tB & 3) == x;
                ok = ok && d1 == d2 && c1 == c2 && d1 >= 0 && c1 >= 0;
                ok = ok && twin[hXn] == hBp && twin[hBp] == hXn && twin[hAp] == hZn && twin[hZn] == hAp;
                ok = ok && (bpack[hXn] & 0xFFFFu) == 2 && (bpack[hAp] & 0xFFFFu) == 2;
                if (ok) {
                    const int rc = vtype[c1] == 3 ? vtarget[c1] : c1, rd = vtype[d1] == 3 ? vtarget[d1] : d1;
                    ok = rc >= 0 && rd >= 0 && rc != rd && rc != x && rc != z && rc != a1 && rc != a3 && rd != x && rd != z && rd != a1 &&
                         rd != a3;
                }
            }
        }
        if (ok) {
            twin[tX] = tA;
            twin[tA] = tX;
            bpack[tX] = packBucket(2, tX < tA ? 0 : 1);
            bpack[tA] = packBucket(2, tA < tX ? 0 : 1);
            twin[tZ] = tB;
            twin[tB] = tZ;
            bpack[tZ] = packBucket(2, tZ < tB ? 0 : 1);
            bpack[tB] = packBucket(2, tB < tZ ? 0 : 1);
            // z is the origin of tA (corner tA & 3 of N_A) and the destination of tZ
            if (z >= 0 && z < V) zslot[z] = make_int2(tA, (tZ & ~3) | ((tZ + 1) & 3));
        } else {
            touched[x] = 1;
            ++nfallback;
            if (z >= 0 && z < V) zslot[z] = make_int2(-1, -1);
        }
        // the removal
#pragma unroll
        for (int i = 0; i < 4; ++i)
            if (v[i] >= 0 && v[i] < V) atomicSub(&outdeg[v[i]], 1);
        quads[q] = make_int4(-1, -1, -1, -1);
        qattr[q] = QA_DEAD;
        fattr[q] = QA_DEAD;
    }
    if (nfallback) {
        atomicAdd((unsigned long long*)&ctr[A_FALLBACK + step], (unsigned long long)nfallback);
        ((volatile int64_t*)(intptr_t)ctr[A_PIN])[kPinFallback - kPinInvalid + step] = 1;
    }
}

// the end of a deferred step: valence = out-degree + incoming boundary halfedges, and the next
// step's start (types, touched flags, the old rule's counts when that is next)
__global__ void kStepEnd(const int32_t* __restrict__ outdeg, const int32_t* __restrict__ bdin, int64_t V, int32_t* __restrict__ valence,
                         uint8_t* __restrict__ vtype, uint8_t* __restrict__ touched, int32_t* __restrict__ count, int step,
                         const int64_t* ctr) {
    const int64_t v = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (v >= V || chainHeld(ctr, step + 1)) return;
    valence[v] = outdeg[v] + bdin[v];
    vtype[v] = 0;
    touched[v] = 0;
    if (count) count[v] = 0;
}

// a dropped vertex u (P3X3Y: vtype == dropType) dies: the corners its live outgoing
// halfedges start at become its target (the two recorded by kLocalMerge, or -- after a
// fallback -- one per quad around it, found through its lists); it and its chain join the
// target's chain; its out-degree (after kLocalMerge took the removed quads' halfedges off)
// goes to the target.  A target that is out of range or dropped itself is invalid, as in the
// compacting path.
// (the dropped vertices of a block are gathered in LDS and handled on consecutive lanes: each
// one's work is a chain of dependent loads, which sparse lanes would spread over every wave)
__device__ __forceinline__ void dropVertex(int u, const uint8_t* __restrict__ vtype, const int32_t* __restrict__ vtarget, int64_t V, int dropType,
                                           int4* __restrict__ quads, int64_t H, const int64_t* __restrict__ off, const int32_t* __restrict__ out,
                                           uint8_t* __restrict__ vdead, int32_t* __restrict__ head, int32_t* __restrict__ next,
                                           int32_t* __restrict__ outdeg, const int2* __restrict__ zslot, int64_t* ctr) {
    const int t = vtarget[u];
    if (t < 0 || t >= V || vtype[t] == dropType) {
        invalid(ctr);
        return;
    }
    int* qc = reinterpret_cast<int*>(quads);
    const int2 zs = zslot[u];
    if (zs.x >= 0) {  // a local merge: u's two live quads and its corners in them are known
        qc[zs.x] = t;
        qc[zs.y] = t;
    } else {
        int w = u, sn = head[u];
        for (;;) {
            for (int64_t k = off[w]; k < off[w + 1]; ++k) {
                const int x = out[k];
                if (x < 0 || x >= H) continue;
                if (qc[x] == u) qc[x] = t;  // corner x & 3 of quad x >> 2 (dead quads hold -1)
            }
            if (sn < 0) break;
            w = sn;
            sn = next[sn];
        }
    }
    vdead[u] = 1;
    spliceChain(u, t, head, next);
    atomicAdd(&outdeg[t], outdeg[u]);
    outdeg[u] = 0;
}

__global__ void __launch_bounds__(kBlock) kDropVertices(const uint8_t* __restrict__ vtype, const int32_t* __restrict__ vtarget, int64_t V,
                                                        int dropType, int4* __restrict__ quads, int64_t H, const int64_t* __restrict__ off,
                                                        const int32_t* __restrict__ out, uint8_t* __restrict__ vdead, int32_t* __restrict__ head,
                                                        int32_t* __restrict__ next, int32_t* __restrict__ outdeg, const int2* __restrict__ zslot,
                                                        int step, int64_t* ctr) {
    // (as one block: another may count an invalid target between two waves' looks)
    if (__syncthreads_or(chainHeld(ctr, step) ? 1 : 0)) return;
    __shared__ int s_list[kSparsePer * kBlock];
    __shared__ int s_n;
    const int total = gatherSparse(V, [&](int64_t i) { return vtype[i] == dropType; }, s_list, &s_n);
    for (int j = threadIdx.x; j < total; j += kBlock) dropVertex(s_list[j], vtype, vtarget, V, dropType, quads, H, off, out, vdead, head, next, outdeg, zslot, ctr);
}

// bucketFromOut over the chain lists: the entries of m's list and of its chain's lists, those
// of dead quads (corners -1) skipped
__device__ BucketOf bucketFromChains(int h, int a, int b, const int4* __restrict__ quads, int64_t H,
                                     const int64_t* __restrict__ off, const int32_t* __restrict__ out, const int32_t* __restrict__ head,
                                     const int32_t* __restrict__ next, int64_t* ctr) {
    const int m = min(a, b), o = max(a, b);
    int mem[4], dir[4];
    int n = 0, rk = 0, partner = -1;
    bool self = false;
    auto add = [&](int id, int d) {
        if (n < 4) {
            mem[n] = id;
            dir[n] = d;
        }
        ++n;
        if (id < h) ++rk;
        if (id != h) partner = id;
        else self = true;
    };
    int u = m, s = head[m];
    for (;;) {
        const int64_t k0 = off[u], k1 = off[u + 1];
        for (int64_t kb = k0; kb < k1; kb += 4) {
            int xs[4];
            int4 qs[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) xs[i] = kb + i < k1 ? out[kb + i] : -1;
#pragma unroll
            for (int i = 0; i < 4; ++i) qs[i] = (xs[i] >= 0 && xs[i] < H) ? quads[xs[i] >> 2] : make_int4(0, 0, 0, 0);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                if (kb + i >= k1) continue;
                const int x = xs[i];
                if (x < 0 || x >= H) {
                    anomaly(ctr);
                    continue;
                }
                const int4 q = qs[i];
                const int j = x & 3;
                if (quadCorner(q, j) == -1) continue;  // a dead quad
                if (quadCorner(q, j) != m) anomaly(ctr);
                if (quadCorner(q, (j + 1) & 3) == o) add(x, 0);
                if (o != m && quadCorner(q, (j + 3) & 3) == o) add((x & ~3) | ((j + 3) & 3), 1);
            }
        }
        if (s < 0) break;
        u = s;
        s = next[s];
    }
    if (!self) anomaly(ctr);
    return BucketOf{n, rk, bucketTwin(n, rk, partner, mem, dir)};
}

// ---- the fallback of a deferred step, limited to the region of the merges kLocalMerge left:
// the halfedges at a touched vertex (its live outgoing ones and the ones before them in their
// quads, which end at it) are marked dirty, their endpoints affected; the dirty ones get their
// buckets recomputed; the affected vertices their flags and incoming boundary count (a
// vertex's flags come from the buckets of its outgoing halfedges, its boundary count from the
// twinless halfedges ending at it: both are read off its chain lists).
__device__ __forceinline__ int gatherFlagged(const uint8_t* __restrict__ flag, int64_t n, int* s_list, int* s_wave) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const bool on = i < n && flag[i];
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    const uint64_t m = __ballot(on);
    if (lane == 0) s_wave[wid] = __popcll(m);
    __syncthreads();
    int base = 0, total = 0;
    for (int w = 0; w < kBlock / 64; ++w) {
        if (w < wid) base += s_wave[w];
        total += s_wave[w];
    }
    if (on) s_list[base + __popcll(m & ((1ULL << lane) - 1ULL))] = (int)i;
    __syncthreads();
    return total;
}

__global__ void __launch_bounds__(kBlock) kMarkDirtyRegion(const uint8_t* __restrict__ touched, int64_t V, const int4* __restrict__ quads, int64_t H,
                                                           const int64_t* __restrict__ off, const int32_t* __restrict__ out,
                                                           const int32_t* __restrict__ head, const int32_t* __restrict__ next,
                                                           uint8_t* __restrict__ hdirty, uint8_t* __restrict__ aff) {
    __shared__ int s_list[kBlock];
    __shared__ int s_wave[kBlock / 64];
    const int total = gatherFlagged(touched, V, s_list, s_wave);
    if ((int)threadIdx.x >= total) return;
    const int t = s_list[threadIdx.x];
    const int* qc = reinterpret_cast<const int*>(quads);
    aff[t] = 1;
    int w = t, sn = head[t];
    for (;;) {
        for (int64_t k = off[w]; k < off[w + 1]; ++k) {
            const int h = out[k];
            if (h < 0 || h >= H || qc[h] != t) continue;  // dead, or not t's any more
            const int pr = (h & ~3) | ((h + 3) & 3);
            hdirty[h] = 1;
            hdirty[pr] = 1;
            aff[qc[(h & ~3) | ((h + 1) & 3)]] = 1;
            aff[qc[pr]] = 1;
        }
        if (sn < 0) break;
        w = sn;
        sn = next[sn];
    }
}

// the dirty halfedges' buckets (gathered per block in LDS): twin, bucket word and NM face bits
__global__ void __launch_bounds__(kBlock) kRebuildDirty(const int4* __restrict__ quads, int64_t H, const uint8_t* __restrict__ hdirty,
                                                        const int64_t* __restrict__ off, const int32_t* __restrict__ out,
                                                        const int32_t* __restrict__ head, const int32_t* __restrict__ next,
                                                        int32_t* __restrict__ twin, uint32_t* __restrict__ bpack, uint32_t* __restrict__ fattr,
                                                        uint32_t* __restrict__ qattr, int64_t* ctr) {
    __shared__ int s_list[kBlock];
    __shared__ int s_wave[kBlock / 64];
    const int total = gatherFlagged(hdirty, H, s_list, s_wave);
    if ((int)threadIdx.x >= total) return;
    const int h = s_list[threadIdx.x];
    const int4 q = quads[h >> 2];
    const int a = quadCorner(q, h & 3), b = quadCorner(q, (h + 1) & 3);
    const BucketOf bk = bucketFromChains(h, a, b, quads, H, off, out, head, next, ctr);
    twin[h] = bk.twin;
    bpack[h] = packBucket(bk.n, bk.rank);
    if (bk.n == 4) {
        atomicOr(&fattr[h >> 2], (uint32_t)QA_NM);
        atomicOr(&qattr[h >> 2], (uint32_t)QA_NM);
    }
}

// an affected vertex's flags and incoming boundary count, from its chain lists
__global__ void __launch_bounds__(kBlock) kAffectedFlags(const uint8_t* __restrict__ aff, int64_t V, const int4* __restrict__ quads, int64_t H,
                                                         const int64_t* __restrict__ off, const int32_t* __restrict__ out,
                                                         const int32_t* __restrict__ head, const int32_t* __restrict__ next,
                                                         const int32_t* __restrict__ twin, const uint32_t* __restrict__ bpack,
                                                         uint32_t* __restrict__ vflags, int32_t* __restrict__ bdin) {
    __shared__ int s_list[kBlock];
    __shared__ int s_wave[kBlock / 64];
    const int total = gatherFlagged(aff, V, s_list, s_wave);
    if ((int)threadIdx.x >= total) return;
    const int v = s_list[threadIdx.x];
    const int* qc = reinterpret_cast<const int*>(quads);
    uint32_t f = 0;
    int bd = 0;
    int w = v, sn = head[v];
    for (;;) {
        for (int64_t k = off[w]; k < off[w + 1]; ++k) {
            const int h = out[k];
            if (h < 0 || h >= H || qc[h] != v) continue;
            f |= bucketVertexFlag((int)(bpack[h] & 0xFFFFu));
            if (twin[(h & ~3) | ((h + 3) & 3)] == -1) ++bd;
        }
        if (sn < 0) break;
        w = sn;
        sn = next[sn];
    }
    vflags[v] = f;
    bdin[v] = bd;
}

// list lengths of the fan detection's slow vertices: their out-degree (the halfedges
// kOutFromLists and kOutDegreeMoved counted per origin), 0 for the others
// (outdeg null: the build's list lengths)
__global__ void kSlowDegree(const uint8_t* __restrict__ slow, const int32_t* __restrict__ outdeg, const int64_t* __restrict__ listOff, int64_t V,
                            int32_t* __restrict__ deg) {
    const int64_t v = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (v > V) return;
    deg[v] = (v < V && slow[v]) ? (outdeg ? outdeg[v] : (int32_t)(listOff[v + 1] - listOff[v])) : 0;
}

// outgoing-halfedge lists (by origin) for the fan detection, of the vertices in `only`
// (all when null)
// the lists of slow vertices the build's outgoing lists still describe, copied from them
__global__ void kCopySlowLists(const uint8_t* __restrict__ slow, int64_t V, const int64_t* __restrict__ outOff, const int32_t* __restrict__ outList,
                               const int64_t* __restrict__ off, int32_t* __restrict__ list) {
    const int64_t v = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (v >= V || !slow[v]) return;
    const int64_t o = off[v], d = off[v + 1] - o, src = outOff[v];
    for (int64_t k = 0; k < d; ++k) list[o + k] = outList[src + k];
}

// (deg counts down to 0; a vertex whose count does not end at 0 is skipped by kDetectFans)
__global__ void kFillLists(const int4* __restrict__ he, int64_t H, int64_t V, const uint8_t* __restrict__ only, const int64_t* __restrict__ off,
                           int32_t* __restrict__ deg, int32_t* __restrict__ list, int64_t* ctr) {
    const int64_t h = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (h >= H) return;
    const int o = heO(he, (int)h);
    if (o < 0 || o >= V) return;
    if (only && !only[o]) return;
    const int slot = atomicSub(&deg[o], 1) - 1;
    if (slot >= 0) list[off[o] + slot] = (int32_t)h;
}

// out-degree and one outgoing halfedge from the outgoing lists of the last build, for the
// vertices they still describe: those below listsV that no split step touched (a split
// step rewrites only halfedges whose origin is in its working copy, before and after).
// By the layout flags (canon), a touched vertex counts the entries of its list whose
// records keep the build's layout (never written back, so still starting at it; the
// block's touched vertices are gathered in LDS, their list walks run on full waves) and
// kOutDegreeMoved adds the records the splitter wrote, those of the vertices from listsV on among them.
__global__ void __launch_bounds__(kBlock) kOutFromLists(const int64_t* __restrict__ off, const int32_t* __restrict__ out, int64_t listsV,
                                                        const uint8_t* __restrict__ touched, const uint8_t* __restrict__ canon, int64_t V,
                                                        int32_t* __restrict__ outdeg, int32_t* __restrict__ rep, int64_t* ctr, int guarded) {
    if (notYet(ctr, guarded)) return;
    stampClock(ctr + A_STAMP + ST_DETECT);
    __shared__ int s_list[kSparsePer * kBlock];
    __shared__ int s_n;
    const int total = gatherSparse(
        V,
        [&](int64_t v) {
            if (v < listsV && !(touched && touched[v])) {
                const int64_t o = off[v];
                const int d = (int)(off[v + 1] - o);
                outdeg[v] = d;
                if (d > 0) rep[v] = out[o];
                return false;
            }
            outdeg[v] = 0;
            return v < listsV;
        },
        s_list, &s_n);
    for (int j = threadIdx.x; j < total; j += kBlock) {
        const int v = s_list[j];
        int d = 0, r = -1;
        for (int64_t k = off[v]; k < off[v + 1]; ++k) {
            const int x = out[k];
            if (canon[x]) {
                ++d;
                r = x;
            }
        }
        outdeg[v] = d;
        if (d > 0) rep[v] = r;
    }
}

// the records the splitter wrote back or appended (canon unset): each adds to
// its origin's out-degree, and the first one of a vertex with no other outgoing halfedge
// becomes its walk start.  A lane looks at the layout flags of PER records at once and the block's
// unset ones are added on full waves (512^3 gyroid, 61 M records: 127 us; one per lane 209 us, and 51
// us where the launch is held).
template <int PER>
__global__ void __launch_bounds__(kBlock) kOutDegreeMoved(const int4* __restrict__ he, int64_t H, int64_t V, int64_t listsV, const uint8_t* __restrict__ touched,
                                const uint8_t* __restrict__ canon, int32_t* __restrict__ outdeg, int32_t* __restrict__ rep, int64_t* ctr,
                                int guarded) {
    if (notYet(ctr, guarded)) return;
    __shared__ int s_list[PER * kBlock];
    __shared__ int s_n;
    if (threadIdx.x == 0) s_n = 0;
    __syncthreads();
    const int64_t h0 = PER * ((int64_t)blockIdx.x * blockDim.x + threadIdx.x);
    uint32_t moved = 0;  // bit k: record h0 + k
    if (h0 + PER <= H && (((uintptr_t)canon) & 15) == 0) {
        uint32_t w[PER / 4];
        if (PER == 16) {
            const uint4 c = reinterpret_cast<const uint4*>(canon)[h0 >> 4];
            w[0] = c.x;
            w[PER / 4 > 1 ? 1 : 0] = c.y;
            w[PER / 4 > 2 ? 2 : 0] = c.z;
            w[PER / 4 > 3 ? 3 : 0] = c.w;
        } else {
            w[0] = reinterpret_cast<const uint32_t*>(canon)[h0 >> 2];
        }
#pragma unroll
        for (int k = 0; k < PER; ++k) moved |= ((w[k >> 2] >> (8 * (k & 3))) & 0xFFu ? 0u : 1u) << k;
    } else {
        for (int k = 0; k < PER && h0 + k < H; ++k) moved |= (canon[h0 + k] ? 0u : 1u) << k;
    }
    // (on full waves: a lane has none or many)
    if (moved) {
        int at = atomicAdd(&s_n, __popc(moved));
        for (; moved; moved &= moved - 1) s_list[at++] = (int)(h0 + __ffs(moved) - 1);
    }
    __syncthreads();
    for (int k = threadIdx.x; k < s_n; k += kBlock) {
        const int h = s_list[k];
        const int o = heO(he, h);
        if (o < 0 || o >= V) {
            anomaly(ctr);
            continue;
        }
        if (o >= listsV || (touched && touched[o]))
            if (atomicAdd(&outdeg[o], 1) == 0) rep[o] = h;
    }
}

// A vertex whose outgoing halfedges form one closed clockwise cycle (next(twin(h)) from
// any of them visits all and returns) has a single fan: every fan walk of fanWalk reaches
// the same minimum.  The others are decided by kDetectFans over their outgoing lists.
// Every face around a vertex the splitter never touched lies outside its working copies, so
// the records such a walk visits keep the build's layout and need no layout-flag check
// (touched: the splitter's touched vertices, vertices from listsV on being its additions).
// An open fan is decided here too.  When the clockwise walk stops (no twin, or a step to a
// halfedge of another origin), a counter-clockwise walk (twin of the previous halfedge in
// the quad) runs from the same start; if it stops too and the two chains hold all d outgoing
// halfedges, the vertex has one fan.  Every fan walk of fanWalk from any of them then covers
// both chains: faces are quads, and at a vertex with no bucket of 3 among its edges
// (VF_WEIRD unset) every twin involved is mutual, so each walk direction undoes the other.
// LISTS: nothing was split, so out-degree and start come from the build's lists (off, out) here;
// else outdeg and rep hold them.
template <bool LISTS>
__global__ void kFanFast(const int4* __restrict__ he, int64_t H, int64_t V, const int64_t* __restrict__ off, const int32_t* __restrict__ out,
                         const int32_t* __restrict__ outdeg, const int32_t* __restrict__ rep, uint32_t* __restrict__ vflags, uint8_t* __restrict__ slow,
                         const uint8_t* __restrict__ touched, int64_t listsV, const uint8_t* __restrict__ canon, int64_t* __restrict__ ctr, int guarded) {
    if (notYet(ctr, guarded)) return;
    if (LISTS) stampClock(ctr + A_STAMP + ST_DETECT);
    const int64_t vv = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (vv >= V) return;
    const int v = (int)vv;
    int64_t o = 0;
    int d;
    if (LISTS) {
        o = off[v];
        d = (int)(off[v + 1] - o);
    } else {
        d = outdeg[v];
    }
    bool single = d == 0;  // no outgoing halfedge: no fan, flag cleared
    const bool mayMove = canon && (!touched || v >= listsV || touched[v]);
    if (d > 0) {
        const int start = LISTS ? out[o] : rep[v];
        int cur = start;
        int4 e = he[start];  // the record of cur: one load gives the next step's origin check and twin
        int open = 0;        // the outgoing halfedges the clockwise walk visited before it stopped
        for (int k = 1; k <= d; ++k) {
            const int t = e.w;
            if (t < 0) {
                open = k;
                break;
            }
            // the next record is loaded at the build layout's next of t alongside t's layout
            // flag, and again from t's own next only when the flag says it moved
            const int qn = quadNext(t, 1);
            int4 en = qn < H ? he[qn] : make_int4(-1, -1, -1, -1);
            if (mayMove && !canon[t]) {
                cur = heN(he, t);
                en = he[cur];
            } else {
                cur = qn;
            }
            e = en;
            if (e.x != v) {
                open = k;
                break;
            }
            if (cur == start) {
                single = k == d;
                break;
            }
        }
        if (open > 0 && !(vflags[v] & VF_WEIRD)) {
            int y = start, got = open;
            bool stopped = false;
            while (got <= d) {
                int p;
                if (!mayMove || canon[y]) p = quadNext(y, 3);
                else p = heN(he, heN(he, heN(he, y)));
                const int tp = (p >= 0 && p < H) ? heT(he, p) : -1;
                if (tp < 0 || tp >= H || heO(he, tp) != v) {
                    stopped = true;
                    break;
                }
                ++got;
                y = tp;
            }
            single = stopped && got == d;
        }
    }
    slow[v] = single ? 0 : 1;
    if (single) vflags[v] &= ~(uint32_t)VF_FANS;
    // counts of the vertices left for the outgoing-list pass and of those among them whose
    // outgoing lists are not the build's (one atomic per wave each)
    const uint64_t m = __ballot(!single);
    const uint64_t mt = __ballot(!single && (v >= listsV || (touched && touched[v])));
    const int leader = (int)(threadIdx.x & 63) == __ffsll((unsigned long long)(m ? m : 1ULL)) - 1;
    if (m && leader) atomicAdd((unsigned long long*)&ctr[A_NSLOW], (unsigned long long)__popcll(m));
    if (mt && leader) atomicAdd((unsigned long long*)&ctr[A_NSLOW_OFF], (unsigned long long)__popcll(mt));
}

// ---------------------------------------------------------------- simplifications
__global__ void kMark3x3y(const int4* __restrict__ quads, uint32_t* __restrict__ qattr, int64_t Q, const int32_t* __restrict__ valence, int step,
                          const int64_t* ctr, int64_t* stamp) {
    stampClock(stamp);
    const int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= Q || chainHeld(ctr, step)) return;
    uint32_t a = qattr[q];
    if ((a & QA_NM) || (a & QA_BOUNDARY) || (a & QA_DEAD)) return;
    a &= 0x3F;
    const int4 v = quads[q];
    const int val[4] = {valence[v.x], valence[v.y], valence[v.z], valence[v.w]};
    if (pattern1(val) || pattern2(val)) a |= QA_PATTERN;
    qattr[q] = a;
}

__global__ void kCount3x3yOld(const int4* __restrict__ quads, uint32_t* __restrict__ qattr, int64_t Q, const int32_t* __restrict__ valence,
                              int32_t* __restrict__ count, int step, const int64_t* ctr, int64_t* stamp) {
    stampClock(stamp);
    const int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= Q || chainHeld(ctr, step)) return;
    const uint32_t a0 = qattr[q];
    if (a0 & QA_DEAD) return;
    uint32_t a = a0 & 0x3F;
    const int4 v = quads[q];
    const int val[4] = {valence[v.x], valence[v.y], valence[v.z], valence[v.w]};
    if (pattern1(val)) {
        atomicAdd(&count[v.x], 1);
        atomicAdd(&count[v.z], 1);
        a |= QA_PATTERN;
    } else if (pattern2(val)) {
        atomicAdd(&count[v.y], 1);
        atomicAdd(&count[v.w], 1);
        a |= QA_PATTERN;
    }
    qattr[q] = a;
}

// HalfedgeMesh.cu:368-388 (markTarget: the target gets vtype kTargetType, for the deferred steps'
// local twin update)
constexpr int kTargetType = 4;
__device__ __forceinline__ void handleMerge(float* pos, float* nrm, uint8_t* vtype, int32_t* vtarget, int x, int y, int z, int w,
                                            int markTarget) {
    const int64_t sx = x, sy = y, sw = w;
    f3 p = mk3(pos[3 * sy], pos[3 * sy + 1], pos[3 * sy + 2]);
    const f3 pw = mk3(pos[3 * sw], pos[3 * sw + 1], pos[3 * sw + 2]);
    p = p + scl(0.5f, pw - p);
    f3 n = mk3(nrm[3 * sy], nrm[3 * sy + 1], nrm[3 * sy + 2]);
    const f3 nw = mk3(nrm[3 * sw], nrm[3 * sw + 1], nrm[3 * sw + 2]);
    n = n + scl(0.5f, nw - n);
    n = normalize3(n);
    pos[3 * sx] = p.x; pos[3 * sx + 1] = p.y; pos[3 * sx + 2] = p.z;
    nrm[3 * sx] = n.x; nrm[3 * sx + 1] = n.y; nrm[3 * sx + 2] = n.z;
    vtype[z] = 3;  // VertexType::PatternRemovable
    vtarget[z] = x;
    if (markTarget) vtype[x] = kTargetType;
}

// The simplifications run right after a halfedge build, whose faces are the quads in order:
// halfedge 4f + i is corner i of face f, its next is 4f + (i + 1) % 4 and face_he[f] = 4f.
// So next and face come from the id (quadNext); only twins and origins are read.

// the four edge-neighbour faces of quad q; false when an edge has no twin (the reference
// then reads halfedges[-1], which is undefined; here the quad is left alone)
__device__ __forceinline__ bool neighborFaces(const int32_t* __restrict__ twin, int q, int nb[4]) {
    const int4 tq = *reinterpret_cast<const int4*>(twin + 4 * (int64_t)q);
    const int t[4] = {tq.x, tq.y, tq.z, tq.w};
    bool ok = true;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        ok = ok && t[i] >= 0;
        nb[i] = t[i] >> 2;
    }
    return ok;
}

// mergeVerticesP3X3YColor (colour = 1) and mergeVerticesP3X3Y (colour = 0), HalfedgeMesh.cu:391-498
__global__ void __launch_bounds__(kBlock) kMerge3x3y(const int4* __restrict__ quads, uint32_t* __restrict__ qattr, int64_t Q, const int32_t* __restrict__ twin,
                           const int32_t* __restrict__ valence, const int32_t* __restrict__ count,
                           float* __restrict__ pos, float* __restrict__ nrm, uint8_t* __restrict__ vtype, int32_t* __restrict__ vtarget, int colour,
                           int markTarget, int step, const int64_t* ctr) {
    if (chainHeld(ctr, step)) return;
    // the block's pattern quads gathered in LDS and handled on consecutive lanes (each is a
    // chain of dependent loads; a few per wave would spread it over every wave)
    __shared__ int s_list[kBlock];
    __shared__ int s_wave[kBlock / 64];
    const int64_t qq = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    bool pat = false;
    if (qq < Q) {
        const uint32_t a0 = qattr[qq];
        pat = (a0 & QA_PATTERN) && (colour || !((a0 & QA_NM) || (a0 & QA_BOUNDARY)));
    }
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    const uint64_t mb = __ballot(pat);
    if (lane == 0) s_wave[wid] = __popcll(mb);
    __syncthreads();
    int base = 0, total = 0;
    for (int w = 0; w < kBlock / 64; ++w) {
        if (w < wid) base += s_wave[w];
        total += s_wave[w];
    }
    if (pat) s_list[base + __popcll(mb & ((1ULL << lane) - 1ULL))] = (int)qq;
    __syncthreads();
    if ((int)threadIdx.x >= total) return;
    const int64_t q = s_list[threadIdx.x];
    const uint32_t a = qattr[q];
    const int4 v = quads[q];
    int nb[4];
    if (!neighborFaces(twin, (int)q, nb)) return;
    // the neighbours' attributes and the corner valences loaded side by side before the tests
    // (other faces only add QA_REMOVE meanwhile, which no test reads)
    const uint32_t na[4] = {qattr[nb[0]], qattr[nb[1]], qattr[nb[2]], qattr[nb[3]]};
    const int val[4] = {valence[v.x], valence[v.y], valence[v.z], valence[v.w]};
    for (int i = 0; i < 4; ++i)
        if ((na[i] & QA_NM) || (a & QA_BOUNDARY)) return;
    if (colour) {
        const uint32_t c = a & QA_COLOR;
        for (int i = 0; i < 4; ++i)
            if ((na[i] & QA_PATTERN) && ((na[i] & QA_COLOR) <= c)) return;
    }
    if (pattern1(val) && (colour || (count[v.x] == 1 && count[v.z] == 1))) {
        handleMerge(pos, nrm, vtype, vtarget, v.x, v.y, v.z, v.w, markTarget);
        atomicOr(&qattr[q], (uint32_t)QA_REMOVE);
    } else if (pattern2(val) && (colour || (count[v.y] == 1 && count[v.w] == 1))) {
        handleMerge(pos, nrm, vtype, vtarget, v.y, v.x, v.w, v.z, markTarget);
        atomicOr(&qattr[q], (uint32_t)QA_REMOVE);
    }
}

// markElementsP3333, HalfedgeMesh.cu:547-628.  Its first half, in which every eligible face clears
// its pattern bits before any face marks, has nothing to clear here: an initialize and a
// deferred P3X3Y step leave eligible faces with their colour alone.
// The faces whose four corners have valence 3, one in some thirty, are gathered in LDS and go through
// their neighbours on full waves: 372 us with every lane going on by itself, 267 us now (512^3 gyroid).
__global__ void __launch_bounds__(kBlock) kMark3333(const int4* __restrict__ quads, const int32_t* __restrict__ twin, uint32_t* __restrict__ fattr, int64_t F,
                                                    const int32_t* __restrict__ valence, uint8_t* __restrict__ vtype, int32_t* __restrict__ vtarget, int step,
                                                    const int64_t* ctr, int64_t* stamp) {
    stampClock(stamp);
    __shared__ int s_list[kBlock];
    __shared__ int s_n;
    if (threadIdx.x == 0) s_n = 0;
    __syncthreads();
    const int64_t ff = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (chainHeld(ctr, step)) return;
    {
        const uint32_t a0 = ff < F ? fattr[ff] : (uint32_t)QA_DEAD;
        bool all3 = !(a0 & (QA_NM | QA_BOUNDARY | QA_DEAD));
        if (all3) {
            const int4 q = quads[ff];
            const int val[4] = {valence[q.x], valence[q.y], valence[q.z], valence[q.w]};
            for (int i = 0; i < 4; ++i) all3 = all3 && val[i] == 3;
        }
        const uint64_t m = __ballot(all3);
        const int lane = threadIdx.x & 63;
        int at = 0;
        if (m && lane == 0) at = atomicAdd(&s_n, __popcll(m));
        at = __shfl(at, 0, 64);
        if (all3) s_list[at + __popcll(m & ((1ULL << lane) - 1ULL))] = (int)ff;
    }
    __syncthreads();
    if ((int)threadIdx.x >= s_n) return;
    const int64_t f = s_list[threadIdx.x];
    const int4 qv = quads[f];
    const int org[4] = {qv.x, qv.y, qv.z, qv.w};
    // the four neighbours loaded side by side before any test
    const int4 tw4 = reinterpret_cast<const int4*>(twin)[f];
    const int tw[4] = {tw4.x, tw4.y, tw4.z, tw4.w};
    for (int i = 0; i < 4; ++i)
        if (tw[i] < 0) return;  // no neighbour across a boundary edge
    int nbf[4], nbv[4], nbval[4], back[4];
    uint32_t na[4];
    int4 nq[4];
    for (int i = 0; i < 4; ++i) {
        nbf[i] = tw[i] >> 2;
        na[i] = fattr[nbf[i]];
        nq[i] = quads[nbf[i]];
    }
    for (int i = 0; i < 4; ++i) {
        if ((na[i] & QA_NM) || (na[i] & QA_BOUNDARY)) return;
        nbv[i] = quadCorner(nq[i], (tw[i] + 2) & 3);
    }
    for (int i = 0; i < 4; ++i) nbval[i] = valence[nbv[i]];
    for (int i = 0; i < 4; ++i)
        if (nbval[i] == 3) return;
    bool all4 = true;
    for (int i = 0; i < 4; ++i) all4 = all4 && nbval[i] == 4;
    if (all4) return;
    // whether halfedge i simply takes the place of neighbour i's outer one (see kRemapRebuild)
    bool regular = true;
    for (int i = 0; i < 4; ++i) back[i] = twin[tw[i]];
    for (int i = 0; i < 4; ++i) {
        const int j = (i + 1) & 3;
        regular = regular && back[i] == (int)(4 * f + i) && nbf[i] != f && nbf[i] != nbf[j] && nbf[i] != nbf[(i + 2) & 3];
        regular = regular && quadCorner(nq[i], tw[i] & 3) == org[j] && quadCorner(nq[i], (tw[i] + 1) & 3) == org[i];
        regular = regular && quadCorner(nq[i], (tw[i] + 3) & 3) == nbv[j];
    }
    atomicOr(&fattr[f], (uint32_t)(regular ? QA_PATTERN : QA_PATTERN | QA_ODD));
    for (int i = 0; i < 4; ++i) {
        atomicOr(&fattr[nbf[i]], (uint32_t)QA_REMOVE);
        const int v = org[i];
        vtype[v] = 1;  // VertexType::Pattern3333
        vtarget[v] = nbv[i];
    }
}

// The chain's compaction numbers vertices and quads in one launch: blocks [0, tV) take tiles of
// vertices, the following tQ tiles of quads; kept elements are numbered in order (tile counts,
// block ranks, look-back over the own kind's tiles).
// A vertex is kept unless it is dropped by this step (vtype == dropType) or died in an earlier
// step of the chain; every vertex gets its new address (-1 when dropped) and the kept ones
// their old id and problem.  A quad is kept without remove or dead bit (qnew, -1
// otherwise).  The arrays the following kernels start from (touched, flags, the list lengths' end;
// the chain heads and removal counts of a chain of one) are cleared along the way.
struct NumberArgs {
    const uint8_t* vtype;
    int64_t V;
    int dropType;
    const uint8_t* vdead;
    const int32_t* pid;
    int32_t *npid, *address, *oldV;
    uint8_t* touched;
    uint32_t* vflags;
    int32_t *cnt, *srcHead, *removedAt;
    int64_t tV;
    unsigned long long* wordsV;
    uint32_t epochV;
    const uint32_t* attr;
    int64_t Q;
    int32_t* qnew;
    int64_t tQ;
    unsigned long long* wordsQ;
    uint32_t epochQ;
    int64_t *totalV, *totalQ, *directOut;
    int step;
    const int64_t* ctr;
};
template <int R>
__global__ void __launch_bounds__(kLbBlock) kNumber(NumberArgs a) {
    if (chainHeld(a.ctr, a.step)) return;
    __shared__ int s_cnt[R * (kLbBlock / 64)], s_pre[R * (kLbBlock / 64) + 1];
    __shared__ long long s_off;
    const bool quad = (int64_t)blockIdx.x >= a.tV;
    const int64_t t = quad ? (int64_t)blockIdx.x - a.tV : (int64_t)blockIdx.x, n = quad ? a.Q : a.V;
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    const int64_t base = t * (int64_t)(R * kLbBlock);
    constexpr uint32_t gone = QA_REMOVE | QA_DEAD;
    auto keepOf = [&](int64_t e) {
        if (e >= n) return false;
        if (quad) return !(a.attr[e] & gone);
        return a.vtype[e] != a.dropType && !(a.vdead && a.vdead[e]);
    };
    uint64_t m[R];
    uint32_t kb = 0;
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const bool k = keepOf(base + r * kLbBlock + threadIdx.x);
        m[r] = __ballot(k);
        kb |= (k ? 1u : 0u) << r;
    }
    const int tileSum = lbBlockRanks<R>(m, s_cnt, s_pre);
    if (threadIdx.x < 64)
        lbTileOffset(
            quad ? a.wordsQ : a.wordsV, quad ? a.epochQ : a.epochV, t, tileSum,
            [&](int l) {
                int64_t c = 0;
                for (int64_t e = l; e < base; e += 64) c += keepOf(e) ? 1 : 0;
                return c;
            },
            a.directOut, &s_off);
    __syncthreads();
    const int64_t off = s_off;
    const uint64_t below = (1ULL << lane) - 1ULL;
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const int64_t e = base + r * kLbBlock + threadIdx.x;
        if (e >= n) continue;
        const bool keep = (kb >> r) & 1u;
        const int64_t o = off + s_pre[r * (kLbBlock / 64) + wid] + __popcll(m[r] & below);
        if (quad) {
            a.qnew[e] = keep ? (int32_t)o : -1;
            continue;
        }
        a.address[e] = keep ? (int32_t)o : -1;
        if (a.srcHead) a.srcHead[e] = -1;
        if (a.removedAt) a.removedAt[e] = 0;
        if (!keep) continue;
        a.oldV[o] = (int32_t)e;
        a.touched[o] = 0;
        a.vflags[o] = 0;
        if (a.pid) a.npid[o] = a.pid[e];
    }
    if (t == (quad ? a.tQ : a.tV) - 1 && threadIdx.x == 0) {
        *(quad ? a.totalQ : a.totalV) = off + tileSum;
        if (!quad) a.cnt[off + tileSum] = 0;
    }
}

// removeQuadrilateralsP3X3Y (p3333 = 0) / removeQuadsP3333 (p3333 = 1), HalfedgeMesh.cu:513-538, :657-683
// (touchTargets: the new vertices an irregular or removed P3333 centre's corners move to)
__device__ __forceinline__ void touchTargets(const int4& q, const int32_t* __restrict__ vtarget, const int32_t* __restrict__ address, int64_t V,
                                             uint8_t* __restrict__ touched) {
    for (int i = 0; i < 4; ++i) {
        const int v = quadCorner(q, i);
        const int t = v >= 0 && v < V ? vtarget[v] : -1;
        const int tn = t >= 0 && t < V ? address[t] : -1;
        if (tn >= 0) touched[tn] = 1;
    }
}
// quad q, kept (new id d) or removed (a quad is removed when it has the remove or the dead bit)
__device__ __forceinline__ void compactQuad(int64_t q, bool kept, int64_t d, const int4* __restrict__ quads, const uint32_t* __restrict__ attr,
                                            const int32_t* __restrict__ vtarget, const int32_t* __restrict__ address, int p3333,
                                            int4* __restrict__ nquads, uint32_t* __restrict__ nattr, uint32_t* __restrict__ nfattr,
                                            int32_t* __restrict__ face_he, int32_t* __restrict__ oldQ, int32_t* __restrict__ removedAt, int32_t* __restrict__ outdeg, uint8_t* __restrict__ touched,
                                            const uint8_t* __restrict__ vdead, int64_t V, int64_t* ctr) {
    if (!kept) {
        if (p3333 && (attr[q] & QA_PATTERN)) touchTargets(quads[q], vtarget, address, V, touched);
        // the outgoing halfedges this quad takes from its corners' lists (when the lists are
        // by current corner; a quad dead since an earlier step of the chain takes none)
        if (!(attr[q] & QA_DEAD)) {
            const int4 r = quads[q];
            if (removedAt) {
                atomicAdd(&removedAt[r.x], 1);
                atomicAdd(&removedAt[r.y], 1);
                atomicAdd(&removedAt[r.z], 1);
                atomicAdd(&removedAt[r.w], 1);
            }
            if (outdeg) {  // after deferred steps: the out-degrees kOutCount reads
                atomicSub(&outdeg[r.x], 1);
                atomicSub(&outdeg[r.y], 1);
                atomicSub(&outdeg[r.z], 1);
                atomicSub(&outdeg[r.w], 1);
            }
        }
        return;
    }
    const uint32_t a = attr[q];
    const int4 v4 = quads[q];
    const int v[4] = {v4.x, v4.y, v4.z, v4.w};
    // P3333: the corners of a pattern face move to their targets.  P3X3Y: a corner moves when
    // it is dropped (vtype 3, the drop type), which is when it has no new address -- so the
    // addresses are read first and a target only for the few dropped corners.
    int o[4];
    bool bad = false;
    const bool pat = p3333 && (a & QA_PATTERN) != 0;
    if (pat && (a & QA_ODD)) touchTargets(v4, vtarget, address, V, touched);
#pragma unroll
    for (int i = 0; i < 4; ++i) o[i] = (v[i] >= 0 && v[i] < V && !pat) ? address[v[i]] : -1;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const bool in = v[i] >= 0 && v[i] < V;
        if (in && (pat || (!p3333 && o[i] < 0))) {
            // (a vertex that died in an earlier step has no target)
            const int src = !pat && vdead && vdead[v[i]] ? -1 : vtarget[v[i]];
            o[i] = (src >= 0 && src < V) ? address[src] : -1;
        }
        bad = bad || o[i] < 0;  // a dropped vertex or a missing target: the quad is invalid
    }
    if (bad) invalid(ctr);
    nquads[d] = make_int4(o[0], o[1], o[2], o[3]);
    uint32_t na = QA_COLOR;
    if (a & QA_NM) na |= QA_NM;
    if (a & QA_BOUNDARY) na |= QA_BOUNDARY;
    nattr[d] = na;
    nfattr[d] = na;
    face_he[d] = (int32_t)(4 * d);
    oldQ[d] = (int32_t)q | (pat ? kOldCentre : 0);
}

// removeQuadrilateralsP3X3Y / removeQuadsP3333 from the numbering, one thread per quad
__global__ void kCompactQuads(const int4* __restrict__ quads, const uint32_t* __restrict__ attr, int64_t Q, const int32_t* __restrict__ vtarget,
                              const int32_t* __restrict__ address, int p3333, int4* __restrict__ nquads, uint32_t* __restrict__ nattr,
                              uint32_t* __restrict__ nfattr, int32_t* __restrict__ face_he, int32_t* __restrict__ oldQ, const int32_t* __restrict__ qnew, int32_t* __restrict__ removedAt,
                              int32_t* __restrict__ outdeg, uint8_t* __restrict__ touched, const uint8_t* __restrict__ vdead, int64_t V, int step,
                              int64_t* ctr) {
    const int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= Q || chainHeld(ctr, step)) return;
    const int32_t d = qnew[q];
    compactQuad(q, d >= 0, d, quads, attr, vtarget, address, p3333, nquads, nattr, nfattr, face_he, oldQ, removedAt, outdeg, touched, vdead, V, ctr);
}

// ---------------------------------------------------------------- fixManifoldTwins
// floor of a cell coordinate; a non-finite or huge one (a NaN or Inf sample upstream)
// becomes -2^30, outside every grid, instead of an undefined conversion
__device__ __forceinline__ int cellIndex(float q) { return (q > -1.0e9f && q < 1.0e9f) ? (int)floorf(q) : -(1 << 30); }
__device__ __forceinline__ void cellOf(const GridDev& g, f3 p, int c[3]) {
    const f3 q = (p - mk3(g.ox, g.oy, g.oz)) / mk3(g.dx, g.dy, g.dz);
    c[0] = cellIndex(q.x);
    c[1] = cellIndex(q.y);
    c[2] = cellIndex(q.z);
}
__device__ __forceinline__ f3 nudge(int it) {
    float x = (it & 1) ? 1.f : 0.f, y = (it & 2) ? 1.f : 0.f, z = (it & 4) ? 1.f : 0.f;
    if (it & 8) x = -x;
    if (it & 16) y = -y;
    if (it & 32) z = -z;
    return mk3(x * 0.0001f, y * 0.0001f, z * 0.0001f);
}
__device__ __forceinline__ f3 ld3(const float* p, int i) { return mk3(p[3 * (int64_t)i], p[3 * (int64_t)i + 1], p[3 * (int64_t)i + 2]); }

// reconnectHalfedges, ManifoldCreator.cu:257-312
// the bucket of h, a bucket of four or more whose first member (rank 0) h is
__device__ void fixBucket(int h, int4* __restrict__ he, int64_t H, const int4* __restrict__ quads, const int64_t* __restrict__ off,
                          const int32_t* __restrict__ out, const float* __restrict__ pos, const ProblemDev* __restrict__ probs,
                          const int32_t* __restrict__ pid, int64_t* ctr) {
    int mem[kMaxBucket];
    const int n = gatherBucketOut(h, quads, H, off, out, mem);
    if (n > kMaxBucket) anomaly(ctr);
    int s[4];
    bucketSlots(mem, n, s);
    const int h0 = s[0];
    const ProblemDev& P = probs[pid ? pid[heO(he, h)] : 0];
    const GridDev g = P.g;
    const float iso = P.iso;
    f3 p0 = ld3(pos, heO(he, h0));
    f3 p1 = ld3(pos, heO(he, heN(he, h0)));
    int c0[3], c1[3];
    cellOf(g, p0, c0);
    cellOf(g, p1, c1);
    bool found = false;
    for (int i = 0; i < 64 && !found; ++i) {
        const f3 o0 = nudge(i);
        int a[3];
        cellOf(g, p0 + o0, a);
        for (int k = 0; k < 64; ++k) {
            const f3 o1 = nudge(k);
            int b[3];
            cellOf(g, p1 + o1, b);
            const int sum = abs(a[0] - b[0]) + abs(a[1] - b[1]) + abs(a[2] - b[2]);
            if (sum == 1) {
                p0 = p0 + o0;
                cellOf(g, p0, c0);
                p1 = p1 + o1;
                cellOf(g, p1, c1);
                found = true;
                break;
            }
        }
    }
    const int64_t g0 = (int64_t)c0[2] * g.nx * g.ny + (int64_t)c0[1] * g.nx + c0[0];
    const int64_t g1 = (int64_t)c1[2] * g.nx * g.ny + (int64_t)c1[1] * g.nx + c1[0];
    int ca[3], cb[3];
    for (int i = 0; i < 3; ++i) {
        ca[i] = g0 < g1 ? c0[i] : c1[i];
        cb[i] = g0 < g1 ? c1[i] : c0[i];
    }
    int wn[3], xo[3] = {0, 0, 0}, yo[3] = {0, 0, 0}, mi[3];
    for (int i = 0; i < 3; ++i) {
        wn[i] = max(ca[i], cb[i]) - min(ca[i], cb[i]);
        mi[i] = max(ca[i], cb[i]);
    }
    if (wn[0] == 0) {
        xo[0] = 1;
        if (wn[1] == 0) yo[1] = 1;
        else yo[2] = 1;
    } else {
        xo[1] = 1;
        yo[2] = 1;
    }
    if (mi[0] < 0 || mi[1] < 0 || mi[2] < 0 || mi[0] >= g.nx - 1 || mi[1] >= g.ny - 1 || mi[2] >= g.nz - 1) {
        anomaly(ctr);
        return;
    }
    auto gv = [&](int dx, int dy, int dz) { return g.v[(int64_t)(mi[2] + dz) * g.nx * g.ny + (int64_t)(mi[1] + dy) * g.nx + (mi[0] + dx)]; };
    const float w0 = gv(0, 0, 0), w1 = gv(xo[0], xo[1], xo[2]), w2 = gv(xo[0] + yo[0], xo[1] + yo[1], xo[2] + yo[2]), w3 = gv(yo[0], yo[1], yo[2]);
    const f3 o = mk3(g.ox, g.oy, g.oz), d = mk3(g.dx, g.dy, g.dz);
    const f3 pc0 = o + d * mk3((float)mi[0], (float)mi[1], (float)mi[2]);
    const f3 pc2 = o + d * mk3((float)(mi[0] + xo[0] + yo[0]), (float)(mi[1] + xo[1] + yo[1]), (float)(mi[2] + xo[2] + yo[2]));
    const bool omitX = xo[0] == 0 && yo[0] == 0;
    const bool omitY = xo[1] == 0 && yo[1] == 0;
    auto down = [&](f3 p, float& u, float& v) {
        if (omitX) { u = p.y; v = p.z; }
        else if (omitY) { u = p.x; v = p.z; }
        else { u = p.x; v = p.y; }
    };
    float minU, minV, maxU, maxV;
    down(pc0, minU, minV);
    down(pc2, maxU, maxV);
    int sorted[4] = {-1, -1, -1, -1};
    for (int i = 0; i < 4; ++i) {
        const int hid = s[i];
        const f3 vp = ld3(pos, heO(he, heN(he, heN(he, hid))));
        float u, v;
        down(vp, u, v);
        if (v - minV < 0.f) sorted[0] = hid;
        if (u - maxU > 0.f) sorted[1] = hid;
        if (v - maxV > 0.f) sorted[2] = hid;
        if (u - minU < 0.f) sorted[3] = hid;
    }
    for (int i = 0; i < 4; ++i)
        if (sorted[i] == -1) {
            anomaly(ctr);
            return;
        }
    // AsymptoticDecider2D(w0, w1, w2, w3).quadrant0BelongsTogether(iso), AsymptoticDecider.h:107-164
    const float C = w0 - w1 - w3 + w2;
    const float delta = (w0 * w2 - w1 * w3) / C;
    const bool q0 = (w0 < iso && delta >= iso) || (w0 >= iso && delta < iso);
    if (!q0) {
        setT(he, sorted[0], sorted[1]); setT(he, sorted[1], sorted[0]);
        setT(he, sorted[2], sorted[3]); setT(he, sorted[3], sorted[2]);
    } else {
        setT(he, sorted[0], sorted[3]); setT(he, sorted[3], sorted[0]);
        setT(he, sorted[1], sorted[2]); setT(he, sorted[2], sorted[1]);
    }
}

// Buckets of four or more are rare (one halfedge in several hundred), and repairing one is
// a long dependent chain.  A block takes kFixPer * kBlock consecutive halfedges, reads their
// bucket sizes four at a time (16-byte loads) and the rank only where the size is four or
// more, gathers the rank-0 members in LDS and repairs them on consecutive lanes, so that the
// chains run on full waves.  The blocks from fixBlocks on list the non-manifold faces meanwhile
// (the bits do not change here), which by itself is a launch of 5 us on any small mesh.
constexpr int kFixPer = 16;
__global__ void __launch_bounds__(kBlock) kFixTwins(int4* __restrict__ he, int64_t H, const int4* __restrict__ quads, const int64_t* __restrict__ off,
                                                    const int32_t* __restrict__ out, const int32_t* __restrict__ bsize, const int32_t* __restrict__ brank,
                                                    const float* __restrict__ pos, const ProblemDev* __restrict__ probs, const int32_t* __restrict__ pid,
                                                    FlagList list, unsigned fixBlocks, int64_t* ctr, int64_t* stamp) {
    stampClock(stamp);
    if (blockIdx.x >= fixBlocks) {
        compactFlaggedTile(list, blockIdx.x - fixBlocks);
        return;
    }
    __shared__ int s_list[kFixPer * kBlock];
    __shared__ int s_n;
    const int lane = threadIdx.x & 63;
    if (threadIdx.x == 0) s_n = 0;
    __syncthreads();
    const int64_t g0 = (int64_t)blockIdx.x * (kFixPer / 4 * kBlock) + threadIdx.x;  // groups of four halfedges
#pragma unroll
    for (int k = 0; k < kFixPer / 4; ++k) {
        const int64_t h0 = 4 * (g0 + (int64_t)k * kBlock);
        int n[4];
        sizes4(bsize, H, h0, n);  // past H: size 2, never a hit
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const bool hit = n[j] >= 4 && h0 + j < H && brank[h0 + j] == 0;
            const uint64_t m = __ballot(hit);
            int at = 0;
            if (lane == 0 && m) at = atomicAdd(&s_n, __popcll(m));
            at = __shfl(at, 0, 64);
            if (hit) s_list[at + __popcll(m & ((1ULL << lane) - 1ULL))] = (int)(h0 + j);
        }
    }
    __syncthreads();
    const int total = s_n;
    for (int i = threadIdx.x; i < total; i += kBlock) fixBucket(s_list[i], he, H, quads, off, out, pos, probs, pid, ctr);
}

// ---------------------------------------------------------------- ManifoldSplitter
struct WC {
    // vertices (capacity 8n)
    float *pos, *nrm, *pos0, *nrm0;
    uint32_t* vflags;
    int32_t *v_c2o, *v_o2c;
    // halfedges (capacity 20n)
    int4* he;
    uint32_t* hflags;
    int32_t *h_c2o, *h_o2c;
    // faces (capacity 5n)
    int32_t* f_first;
    uint32_t* f_attr;
    uint32_t* fflags;
    int32_t *f_c2o, *f_o2c;
    int32_t* pid;  // per vertex its problem (several problems), else nullptr
    // the old vertex and halfedge of each corner slot as kWcCopy took them (4n): the entries
    // of the old -> copy maps that the step sets, reset to -1 by kCopyBack at the step's end
    int32_t *v_orig, *h_orig;
    // per old vertex the last copy of it that survives (-1 between steps, as the maps)
    int32_t* v_last;
    int n;
};

// What a split step carries between its launches besides the working copy.  The step was some 50
// launches with three waits; its passes are independent of each other in groups, so each
// group is one launch (blocks take ranges of vertices, halfedges and faces), the arrays are
// grown for the most the step can append (4n vertices, 16n halfedges, 4n faces) before it
// starts, and the host waits once, for the sizes with the refresh's dirty list: 20 launches.
// 128^3 lattice (640 faces, one step): 963 us an extraction before, 811 us now; 201x77x131 gyroid
// (7 k faces) 628 and 493; batch of 16 with few dozen faces 680 and 554.
struct SplitStep {
    WC w;
    int step, vsize, hsize, fsize;
    // merge marks: vertices and halfedges; records in call order, per target a count, a cursor, its
    // offset and its records, then the ivec2 the reference keeps
    int2 *vrec, *hrec;
    int32_t *cntV, *curV, *idxV, *cntH, *curH, *idxH;
    int64_t *offV, *offH;
    int32_t *numV, *exV, *eyV, *numH, *exH, *eyH;
    int32_t *valid, *firstWriter;  // [hsize], [2 hsize]
    int32_t *newV, *newH, *newF;   // 1: the copy back appends this element
    int64_t *addrV, *addrH, *addrF;
    int64_t V0, H0, F0;
    int64_t* ctr;
};
// block b of a launch over ranges of n0, n1, n2 threads: the range and the thread's index in it
__device__ __forceinline__ int rangeOf(int n0, int n1, int n2, int& i) {
    int b = blockIdx.x;
    const int g0 = (n0 + kBlock - 1) / kBlock, g1 = (n1 + kBlock - 1) / kBlock;
    int r = 0;
    if (b >= g0) b -= g0, r = 1;
    if (r == 1 && b >= g1) b -= g1, r = 2;
    i = b * kBlock + threadIdx.x;
    return i < (r == 0 ? n0 : (r == 1 ? n1 : n2)) ? r : 3;
}
inline unsigned rangeBlocks(int64_t n0, int64_t n1, int64_t n2) { return gridFor(n0) + gridFor(n1) + gridFor(n2); }

// copyVerticesToWorkingCopy / copyHalfedgesToWorkingCopy / copyFacesToWorkingCopy (ManifoldSplitter.cu:307-457),
// one thread per face corner: thread 4r + i copies the i-th halfedge of face nm[r] and its
// origin into slot c = 4r + i, so the copies' stores are consecutive across lanes
// (flags start at 0: WorkingCopy ignores its initialFlags argument); the threads also start the
// rest of the step's arrays, 2 vertices, 5 halfedges and up to 2 faces each
__global__ void kWcCopy(const int32_t* __restrict__ nm, int n, const int4* __restrict__ he, const int32_t* __restrict__ face_he,
                        const uint32_t* __restrict__ fattr, const float* __restrict__ pos, const float* __restrict__ nrm,
                        const int32_t* __restrict__ pid, SplitStep s) {
    const WC& w = s.w;
    const int c = blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= 4 * n) return;
    for (int k = 0; k < 2; ++k) {
        const int v = c + 4 * n * k;
        w.vflags[v] = 0;
        if (k) w.v_c2o[v] = -1;
        s.cntV[v] = 0;
        s.curV[v] = 0;
    }
    for (int k = 0; k < 5; ++k) {
        const int h = c + 4 * n * k;
        w.hflags[h] = 0;
        if (k) w.h_c2o[h] = -1;
        s.cntH[h] = 0;
        s.curH[h] = 0;
        s.firstWriter[h] = INT32_MAX;  // atomicMin targets
        s.firstWriter[s.hsize + h] = 0;  // write counts
    }
    w.fflags[c] = 0;
    if (c >= n) w.f_c2o[c] = -1;
    if (c < n) {
        w.fflags[4 * n + c] = 0;
        w.f_c2o[4 * n + c] = -1;
    }
    if (c == 0) s.cntV[8 * n] = s.cntH[20 * n] = 0;
    const int r = c >> 2, i = c & 3;
    const int f = nm[r];
    int h = face_he[f];
    int4 e = he[h];
    for (int k = 0; k < i; ++k) {
        h = e.z;
        e = he[h];
    }
    const int v = e.x;
    for (int k = 0; k < 3; ++k) {
        w.pos[3 * c + k] = pos[3 * (int64_t)v + k];
        w.nrm[3 * c + k] = nrm[3 * (int64_t)v + k];
    }
    w.v_c2o[c] = v;
    w.v_orig[c] = v;
    if (w.pid) w.pid[c] = pid[v];
    atomicMax(&w.v_o2c[v], c);  // racy "last writer" in ascending order
    w.he[c] = e;
    w.h_c2o[c] = h;
    w.h_orig[c] = h;
    w.h_o2c[h] = c;
    if (i == 0) {
        w.f_first[r] = 4 * r;
        w.f_attr[r] = fattr[f];
        w.f_c2o[r] = f;
        w.f_o2c[f] = r;
    }
}

// updateWorkingCopyHalfedges, ManifoldSplitter.cu:463-505, and markHalfedgesAsNonManifold,
// :527-555: the copied halfedges that are slotted non-manifold get the NM flag, as does their
// origin; their count goes to foundParts (nmSlotCheck compares it with the count of all of
// them: the reference would read the copy index of one outside the copy as an invalid id)
__global__ void __launch_bounds__(kBlock) kWcUpdate(int n4, const int32_t* __restrict__ bsize, const int32_t* __restrict__ brank, WC w,
                                                    int64_t* foundParts) {
    const int c = blockIdx.x * blockDim.x + threadIdx.x;
    int found = 0;
    if (c < n4) {
        int4 e = w.he[c];
        e.x = w.v_o2c[e.x];
        e.y = w.f_o2c[e.y];
        e.z = w.h_o2c[e.z];
        if (e.w >= 0) {
            const int m = w.h_o2c[e.w];
            e.w = (m == -1) ? (-e.w - 2) : m;
        }
        w.he[c] = e;
        const int hh = w.h_orig[c];
        const int n = bucketSize(bsize[hh]);
        if (n >= 4 && slottedNM(n, brank[hh])) {
            w.hflags[c] |= VF_NM;
            atomicOr(&w.vflags[e.x], (uint32_t)VF_NM);
            found = 1;
        }
    }
    blockAdd(foundParts, found);
}

// a slotted non-manifold halfedge outside the working copy (its face not marked NM) is an
// anomaly, one per such halfedge and step, as the reference's working copy would not hold it
// (one wave: the partial sums of both counts; the found ones are cleared for the next step)
__device__ __forceinline__ void nmSlotCheck(const int64_t* nmParts, int64_t* foundParts, int64_t* ctr) {
    const int lane = threadIdx.x;
    const int64_t total = sumParts(nmParts, lane), found = sumParts(foundParts, lane);
    foundParts[lane * kPartStride] = 0;
    if (lane == 0 && total > found) ctr[A_ANOMALY] += total - found;
}
__global__ void kNMSlotCheck(const int64_t* nmParts, int64_t* foundParts, int64_t* ctr) { nmSlotCheck(nmParts, foundParts, ctr); }

// performSubdivideQuads, ManifoldSplitter.cu:570-731.  Face r appends 4 vertices at 4n+4r,
// 16 halfedges at 4n+16r and 4 faces at n+4r, which is where the ascending schedule puts them.
// Four threads per face (consecutive lanes of one wave): thread i writes inner vertex i, inner
// halfedge ih[i], the three new halfedges of new face i (with the twins the reference's
// setTwin calls leave on them) and the outer halfedge that joins that face.  Every lane of
// the wave has walked the face before any lane rewrites one of its outer halfedges.
// (the block after the faces' makes the slot check)
__global__ void kSubdivide(const int32_t* __restrict__ nm, WC w, const int64_t* nmParts, int64_t* foundParts, int64_t* ctr) {
    const int n = w.n;
    if (blockIdx.x == gridDim.x - 1) {
        if (threadIdx.x < 64) nmSlotCheck(nmParts, foundParts, ctr);
        return;
    }
    const int c0 = blockIdx.x * blockDim.x + threadIdx.x;
    if (c0 >= 4 * n) return;
    const int r = c0 >> 2, i = c0 & 3;
    const int faceID = w.f_o2c[nm[r]];
    int fh[4], vid[4];
    int cur = w.f_first[faceID];
    for (int k = 0; k < 4; ++k) {
        fh[k] = cur;
        const int4 e = w.he[cur];
        vid[k] = e.x;
        cur = e.z;
    }
    f3 vp[4], vn[4];
    for (int k = 0; k < 4; ++k) {
        vp[k] = ld3(w.pos, vid[k]);
        vn[k] = ld3(w.nrm, vid[k]);
    }
    const float us[4] = {0.33f, 0.67f, 0.67f, 0.33f}, vs[4] = {0.33f, 0.33f, 0.67f, 0.67f};
    const int nx = (i + 1) & 3, pv = (i + 3) & 3;
    const int innerBase = 4 * n + 4 * r;
    {
        const f3 ap = mixv(vp[0], vp[1], us[i]), bp = mixv(vp[3], vp[2], us[i]);
        const f3 an = mixv(vn[0], vn[1], us[i]), bn = mixv(vn[3], vn[2], us[i]);
        const f3 p = mixv(ap, bp, vs[i]), q = mixv(an, bn, vs[i]);
        const int c = innerBase + i;
        w.pos[3 * c] = p.x; w.pos[3 * c + 1] = p.y; w.pos[3 * c + 2] = p.z;
        w.nrm[3 * c] = q.x; w.nrm[3 * c + 1] = q.y; w.nrm[3 * c + 2] = q.z;
        w.vflags[c] &= ~(uint32_t)VF_REMOVE;
        if (w.pid) w.pid[c] = w.pid[vid[0]];
    }
    const int hb = 4 * n + 16 * r;
    auto ih = [&](int k) { return hb + k; };
    auto of = [&](int k, int j) { return hb + 4 + 3 * k + j; };
    const int nf = n + 4 * r + i;
    w.he[ih(i)] = make_int4(innerBase + i, faceID, ih(nx), of(nx, 1));
    if (i == 0) w.f_first[faceID] = ih(0);
    w.he[of(i, 0)] = make_int4(vid[i], nf, of(i, 1), of(nx, 2));
    w.he[of(i, 1)] = make_int4(innerBase + i, nf, of(i, 2), ih(pv));
    w.he[of(i, 2)] = make_int4(innerBase + pv, nf, fh[pv], of(pv, 0));
    int4 e3 = w.he[fh[pv]];
    e3.y = nf;
    e3.z = of(i, 0);
    w.he[fh[pv]] = e3;
    w.f_first[nf] = of(i, 0);
    w.f_attr[nf] = QA_COLOR;  // HalfedgeFace()
    // swapHalfedgeMappings(outer, inner)
    const int a = fh[i], b = ih(i);
    const int ao = w.h_c2o[a], bo = w.h_c2o[b];
    w.h_c2o[a] = bo;
    w.h_c2o[b] = ao;
    if (ao != -1 && bo == -1) w.h_o2c[ao] = b;
}

// performCollapseNonManifoldHalfedges (only copied halfedges, [0, 4n), carry the NM flag) and
// collapseHalfedge, ManifoldSplitter.cu:749-835: remove flags plus the merge marks, recorded in
// call order -- the collapsing halfedges are ranked by a look-back over tiles of 1024 -- and
// counted per target
constexpr int kCollapseRounds = 4;
__device__ void collapseHalfedge(const SplitStep& s, int h, int64_t k) {
    const WC& w = s.w;
    int cf[2][4];
    int4 cur = w.he[h];
    cf[0][0] = h;
    cf[1][0] = cur.w;
    int4 ct = w.he[cur.w];
    for (int i = 1; i < 4; ++i) {
        cf[0][i] = cur.z;
        cf[1][4 - i] = ct.z;
        cur = w.he[cur.z];
        ct = w.he[ct.z];
    }
    for (int fc = 0; fc < 2; ++fc) {
        for (int i = 0; i < 4; ++i) atomicOr(&w.hflags[cf[fc][i]], (uint32_t)VF_REMOVE);
        atomicOr(&w.fflags[heF(w.he, cf[fc][0])], (uint32_t)VF_REMOVE);
    }
    auto mark = [&](int2* rec, int32_t* cnt, int count, int t, int p) {
        *rec = make_int2(t, p);
        if (t < 0 || t >= count) anomaly(s.ctr);
        else atomicAdd(&cnt[t], 1);
    };
    const int a = heO(w.he, cf[0][2]), b = heO(w.he, cf[1][1]);
    const int c = heO(w.he, cf[0][3]), d = heO(w.he, cf[1][2]);
    int2* v = s.vrec + 4 * k;
    mark(v, s.cntV, s.vsize, a, b);
    mark(v + 1, s.cntV, s.vsize, b, a);
    mark(v + 2, s.cntV, s.vsize, c, d);
    mark(v + 3, s.cntV, s.vsize, d, c);
    for (int i = 1; i < 4; ++i) {
        const int ta = heT(w.he, cf[0][i]), tb = heT(w.he, cf[1][i]);
        int2* o = s.hrec + 12 * k + 4 * (i - 1);
        mark(o, s.cntH, s.hsize, cf[0][i], tb);
        mark(o + 1, s.cntH, s.hsize, tb, cf[0][i]);
        mark(o + 2, s.cntH, s.hsize, cf[1][i], ta);
        mark(o + 3, s.cntH, s.hsize, ta, cf[1][i]);
    }
}
__global__ void __launch_bounds__(kLbBlock) kCollapse(SplitStep s, unsigned long long* __restrict__ words, uint32_t epoch, int64_t* __restrict__ directOut) {
    constexpr int R = kCollapseRounds;
    __shared__ int s_cnt[R * (kLbBlock / 64)], s_pre[R * (kLbBlock / 64) + 1];
    __shared__ long long s_off;
    __shared__ int s_list[R * kLbBlock];  // the tile's collapsing halfedges by rank, for full waves
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    const int n = 4 * s.w.n;
    const int64_t t = blockIdx.x, base = t * (int64_t)(R * kLbBlock);
    // (other tiles only add the REMOVE bit meanwhile, and twins do not change)
    auto collapses = [&](int64_t e, bool count) {
        if (e >= n || !(s.w.hflags[e] & VF_NM)) return false;
        const int tw = heT(s.w.he, (int)e);
        if (tw < 0 && count) anomaly(s.ctr);
        return tw >= 0 && tw >= e;
    };
    uint64_t m[R];
    uint32_t kb = 0;
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const bool k = collapses(base + r * kLbBlock + threadIdx.x, true);
        m[r] = __ballot(k);
        kb |= (k ? 1u : 0u) << r;
    }
    const int tileSum = lbBlockRanks<R>(m, s_cnt, s_pre);
    if (threadIdx.x < 64)
        lbTileOffset(
            words, epoch, t, tileSum,
            [&](int l) {
                int64_t c = 0;
                for (int64_t e = l; e < base; e += 64) c += collapses(e, false) ? 1 : 0;
                return c;
            },
            directOut, &s_off);
    const uint64_t below = (1ULL << lane) - 1ULL;
#pragma unroll
    for (int r = 0; r < R; ++r)
        if ((kb >> r) & 1u) s_list[s_pre[r * (kLbBlock / 64) + wid] + __popcll(m[r] & below)] = (int)(base + r * kLbBlock + threadIdx.x);
    __syncthreads();
    for (int j = threadIdx.x; j < tileSum; j += kLbBlock) collapseHalfedge(s, s_list[j], s_off + j);
    if (t == gridDim.x - 1 && threadIdx.x == 0) s.ctr[A_NCOL] = s_off + tileSum;
}

// the records into their targets' lists, and the merge's snapshot of positions and normals
__global__ void kRecScatter(SplitStep s) {
    const int64_t t0 = (int64_t)blockIdx.x * blockDim.x + threadIdx.x, stride = (int64_t)gridDim.x * blockDim.x;
    const int64_t ncol = s.ctr[A_NCOL];
    for (int64_t i = t0; i < 12 * ncol; i += stride) {
        const int t = s.hrec[i].x;
        if (t >= 0 && t < s.hsize) s.idxH[s.offH[t] + atomicAdd(&s.curH[t], 1)] = (int32_t)i;
    }
    for (int64_t i = t0; i < 4 * ncol; i += stride) {
        const int t = s.vrec[i].x;
        if (t >= 0 && t < s.vsize) s.idxV[s.offV[t] + atomicAdd(&s.curV[t], 1)] = (int32_t)i;
    }
    if (s.step >= 3)
        for (int64_t i = t0; i < 3 * (int64_t)s.vsize; i += stride) {
            s.w.pos0[i] = s.w.pos[i];
            s.w.nrm0[i] = s.w.nrm[i];
        }
}
// markVerticesAsMergable / markHalfedgesAsMergeable applied in record order to glm::ivec2
// storage: the counter always advances; the second mark goes to .y, marks 1, 3, 4, 5 to .x,
// later marks are dropped (ManifoldSplitter.cu:749-765)
__device__ void applyRecords(int t, const int2* __restrict__ rec, const int64_t* __restrict__ roff, int32_t* __restrict__ idx,
                             const int32_t* __restrict__ cnt, int32_t* __restrict__ num, int32_t* __restrict__ ex, int32_t* __restrict__ ey) {
    const int m = cnt[t];
    num[t] = 1 + m;
    ex[t] = -1;
    ey[t] = -1;
    if (m == 0) return;
    int32_t* s = idx + roff[t];
    for (int i = 1; i < m; ++i) {  // records in call order
        const int x = s[i];
        int j = i - 1;
        while (j >= 0 && s[j] > x) {
            s[j + 1] = s[j];
            --j;
        }
        s[j + 1] = x;
    }
    for (int j = 0; j < m && j <= 4; ++j) {
        const int p = rec[s[j]].y;
        if (j == 1) ey[t] = p;
        else ex[t] = p;
    }
}
__global__ void kRecApply(SplitStep s) {
    int i;
    const int r = rangeOf(s.vsize, s.hsize, 0, i);
    if (r == 0) applyRecords(i, s.vrec, s.offV, s.idxV, s.cntV, s.numV, s.exV, s.eyV);
    else if (r == 1) applyRecords(i, s.hrec, s.offH, s.idxH, s.cntH, s.numH, s.exH, s.eyH);
}

// a thread's list of merge partners, in LDS (a private array indexed by a variable would lie in
// scratch memory: kMergePlan 390 us at the 512^3 gyroid's first step, 269 us now)
struct Partners {
    int* p;
    __device__ __forceinline__ int& operator[](int i) const { return p[i * kBlock]; }
};
#define MDMC_PARTNERS(name)              \
    __shared__ int s_partners[12 * kBlock]; \
    const Partners name{s_partners + threadIdx.x}

// DeviceMergeList::getAllPartnersOf, ManifoldSplitter.cu:25-62
__device__ int partnersOf(int v, int size, const int32_t* __restrict__ num, const int32_t* __restrict__ ex, const int32_t* __restrict__ ey,
                          const Partners& out, int64_t* ctr) {
    if (v < 0 || v >= size) { anomaly(ctr); return 1; }
    int n = num[v];
    if (n <= 1) return n;  // (out is not read then)
    for (int i = 0; i < 12; ++i) out[i] = -1;
    for (int i = 0; i < n - 1; ++i) {
        if (i >= 12) { anomaly(ctr); break; }
        out[i] = (i == 1) ? ey[v] : ex[v];
    }
    for (int i = 0; i < n - 1 && i < 12; ++i) {
        const int p = out[i];
        if (p < 0 || p >= size) { anomaly(ctr); continue; }
        const int np = num[p];
        for (int k = 0; k < np - 1; ++k) {
            const int pp = (k == 1) ? ey[p] : ex[p];
            bool contained = v == pp;
            for (int z = 0; z < n - 1 && z < 12; ++z) contained = contained || out[z] == pp;
            if (!contained) {
                if (n - 1 >= 12) { anomaly(ctr); continue; }
                out[n - 1] = pp;
                ++n;
            }
        }
    }
    return n;
}

// mergeVertices, ManifoldSplitter.cu:936-990.  A vertex that survives reads partners
// with larger ids only, which no earlier thread writes, so reading the snapshot is the
// ascending schedule's result.  True: v does not survive.
__device__ bool mergeVertex(const WC& w, const Partners& P, int v, int count, const int32_t* __restrict__ num, const int32_t* __restrict__ ex,
                            const int32_t* __restrict__ ey, int64_t* ctr) {
    const int np = partnersOf(v, count, num, ex, ey, P, ctr);
    if (np == 1) return false;
    if (np < 1 || np > 12) { anomaly(ctr); return false; }
    int smallest = v;
    f3 p = ld3(w.pos0, v), nn = ld3(w.nrm0, v);
    bool obsolete = false;
    for (int i = 0; i < np - 1; ++i) {
        const int q = P[i];
        if (q < 0 || q >= count) { anomaly(ctr); continue; }
        p = p + ld3(w.pos0, q);
        nn = nn + ld3(w.nrm0, q);
        if (q < smallest) { obsolete = true; smallest = q; }
    }
    if (obsolete) {
        atomicOr(&w.vflags[v], (uint32_t)VF_REMOVE);
        return true;
    }
    p = divs(p, (float)np);
    w.pos[3 * smallest] = p.x; w.pos[3 * smallest + 1] = p.y; w.pos[3 * smallest + 2] = p.z;
    w.nrm[3 * smallest] = p.x; w.nrm[3 * smallest + 1] = p.y; w.nrm[3 * smallest + 2] = p.z;  // position stored as normal, :989
    return false;
}

// updateHalfedgeVertexIDs, ManifoldSplitter.cu:992-1019
__device__ void updateVertexID(const WC& w, const Partners& P, int h, int vcount, const int32_t* __restrict__ num, const int32_t* __restrict__ ex,
                               const int32_t* __restrict__ ey, int64_t* ctr) {
    const int v = heO(w.he, h);
    const int np = partnersOf(v, vcount, num, ex, ey, P, ctr);
    if (np == 1) return;
    int smallest = v;
    for (int i = 0; i < np - 1; ++i)
        if (P[i] >= 0 && P[i] < smallest) smallest = P[i];
    ((int*)w.he)[4 * (int64_t)h] = smallest;
}

// mergeHalfedges, ManifoldSplitter.cu:1021-1067, planned in parallel on the pre-launch twins.
// valid[h] = new twin or -1.  Flags a conflict when a partner whose twin this launch
// writes is read, or a halfedge would be written twice; then mergeSequential runs instead.
__device__ int planMerge(const WC& w, int h, int count, const int32_t* __restrict__ num, const int32_t* __restrict__ ex, const int32_t* __restrict__ ey,
                         const Partners& P, int& np, int64_t* ctr) {
    np = partnersOf(h, count, num, ex, ey, P, ctr);
    if (np == 1) return -1;
    for (int i = 0; i < np - 1; ++i) {
        if (P[i] < 0 || P[i] >= count) continue;
        const int t = heT(w.he, P[i]);
        if (t < 0 || t >= count) { anomaly(ctr); continue; }
        if (!(w.hflags[t] & VF_REMOVE)) return t;
    }
    return -1;
}

__device__ void planHalfedge(const SplitStep& s, const Partners& P, int h) {
    s.valid[h] = -1;
    if (s.w.hflags[h] & VF_REMOVE) return;
    int np;
    const int t = planMerge(s.w, h, s.hsize, s.numH, s.exH, s.eyH, P, np, s.ctr);
    if (t == -1 || t < h) return;
    s.valid[h] = t;
    atomicMin(&s.firstWriter[h], h);
    atomicMin(&s.firstWriter[t], h);
    if (atomicAdd(&s.firstWriter[s.hsize + h], 1) > 0) atomicAdd((unsigned long long*)&s.ctr[A_CONFLICT], 1ULL);
    if (atomicAdd(&s.firstWriter[s.hsize + t], 1) > 0) atomicAdd((unsigned long long*)&s.ctr[A_CONFLICT], 1ULL);
}

// the merges' first part, and which elements the copy back appends (copyWorkingCopiesBack,
// ManifoldSplitter.cu:1176-1295): vertices (step 3) merge; halfedges take their origins' survivors
// (step 3; a vertex's merge reads no halfedge) and plan their merges (step 4; the plans read
// twins and flags, which no thread here writes)
__global__ void __launch_bounds__(kBlock) kMergePlan(SplitStep s) {
    MDMC_PARTNERS(P);
    int i;
    const int r = rangeOf(s.vsize, s.hsize, s.fsize, i);
    const WC& w = s.w;
    if (r == 0) {
        const bool gone = s.step >= 3 && mergeVertex(w, P, i, s.vsize, s.numV, s.exV, s.eyV, s.ctr);
        s.newV[i] = (!gone && !(w.vflags[i] & VF_REMOVE) && w.v_c2o[i] == -1) ? 1 : 0;
    } else if (r == 1) {
        if (s.step >= 3) updateVertexID(w, P, i, s.vsize, s.numV, s.exV, s.eyV, s.ctr);
        if (s.step >= 4) planHalfedge(s, P, i);
        s.newH[i] = (!(w.hflags[i] & VF_REMOVE) && w.h_c2o[i] == -1) ? 1 : 0;
    } else if (r == 2) {
        s.newF[i] = (!(w.fflags[i] & VF_REMOVE) && w.f_c2o[i] == -1) ? 1 : 0;
    }
}

__global__ void __launch_bounds__(kBlock) kMergeCheck(WC w, int count, const int32_t* __restrict__ num, const int32_t* __restrict__ ex, const int32_t* __restrict__ ey,
                            const int32_t* __restrict__ firstWriter, int64_t* ctr) {
    const int h = blockIdx.x * blockDim.x + threadIdx.x;
    if (h >= count) return;
    if (w.hflags[h] & VF_REMOVE) return;
    MDMC_PARTNERS(P);
    const int np = partnersOf(h, count, num, ex, ey, P, ctr);
    if (np == 1) return;
    for (int i = 0; i < np - 1; ++i) {
        if (P[i] < 0 || P[i] >= count) continue;
        if (firstWriter[P[i]] < h) {  // an earlier thread rewrites a twin this thread reads
            atomicAdd((unsigned long long*)&ctr[A_CONFLICT], 1ULL);
            return;
        }
        const int t = heT(w.he, P[i]);
        if (t < 0 || t >= count) continue;
        if (!(w.hflags[t] & VF_REMOVE)) return;
    }
}

// the planned merges, or -- with a conflict -- the merges in ascending order by one thread.  Its time is one chain
// of loads: with the merge lists as __restrict__ arguments of the kernel, which lets them go through the
// scalar cache, and no address made from the thread's index, 13.2 ms for a step over 24^3 white noise; as
// members of the step, on a lane's own partner list, 16.3 ms.
__device__ __forceinline__ void mergeSequential(const WC& w, int count, const int32_t* __restrict__ num, const int32_t* __restrict__ ex,
                                                const int32_t* __restrict__ ey, const Partners& P, int64_t* ctr) {
    ++ctr[A_MERGE_SEQ];  // the iterations that took this pass (one thread: a plain increment)
    for (int h = 0; h < count; ++h) {
        if (w.hflags[h] & VF_REMOVE) continue;
        int np;
        const int t = planMerge(w, h, count, num, ex, ey, P, np, ctr);
        if (t == -1 || t < h) continue;
        setT(w.he, h, t);
        setT(w.he, t, h);
    }
}

// performMoveVerticesToSurface, ManifoldSplitter.cu:1130-1160
__device__ void moveVertexToSurface(const WC& w, int v, const ProblemDev* __restrict__ probs) {
    if (w.vflags[v] & VF_REMOVE) return;
    const ProblemDev& P = probs[w.pid ? w.pid[v] : 0];
    const GridDev g = P.g;
    const float iso = P.iso;
    f3 point = ld3(w.pos, v);
    int c[3];
    cellOf(g, point, c);
    float s[8];
    for (int k = 0; k < 8; ++k) {
        const int x = min(max(c[0] + (k & 1), 0), g.nx - 1);
        const int y = min(max(c[1] + ((k >> 1) & 1), 0), g.ny - 1);
        const int z = min(max(c[2] + ((k >> 2) & 1), 0), g.nz - 1);
        s[k] = g.v[(int64_t)z * g.nx * g.ny + (int64_t)y * g.nx + x];
    }
    const f3 o = mk3(g.ox, g.oy, g.oz), d = mk3(g.dx, g.dy, g.dz);
    const f3 iv = mk3((float)c[0], (float)c[1], (float)c[2]);
    const f3 iv1 = mk3((float)(c[0] + 1), (float)(c[1] + 1), (float)(c[2] + 1));
    const f3 mn = o + iv * d, mx = o + iv1 * d;
    point = (point - mn) / (mx - mn);
    movePointToSurface(s, iso, point);
    point = o + (iv + point) * d;
    w.pos[3 * v] = point.x;
    w.pos[3 * v + 1] = point.y;
    w.pos[3 * v + 2] = point.z;
}

// the merges' second part (halfedges, step 4) beside the vertices' part of the rest: the last
// surviving copy of an original in ascending order writes it back, and every surviving
// vertex moves to the surface (step 5)
__global__ void __launch_bounds__(kBlock) kMergeApply(SplitStep s, const ProblemDev* __restrict__ probs, const int32_t* __restrict__ numH,
                                                      const int32_t* __restrict__ exH, const int32_t* __restrict__ eyH) {
    __shared__ int s_partners[12 * kBlock];
    int i;
    const int r = rangeOf(s.step >= 4 ? s.hsize : 0, s.vsize, 0, i);
    const WC& w = s.w;
    if (r == 0) {
        if (s.ctr[A_CONFLICT] != 0) {
            if (i == 0) mergeSequential(w, s.hsize, numH, exH, eyH, Partners{s_partners}, s.ctr);
            return;
        }
        const int t = s.valid[i];
        if (t < 0) return;
        setT(w.he, i, t);
        setT(w.he, t, i);
    } else if (r == 1) {
        const int o = w.v_c2o[i];
        if (o >= 0 && !(w.vflags[i] & VF_REMOVE)) atomicMax(&w.v_last[o], i);
        if (s.step >= 5) moveVertexToSurface(w, i, probs);
    }
}

// copyWorkingCopiesBack, ManifoldSplitter.cu:1176-1295, in two parts: every element's id, and the
// vertices; then, with all ids known, the halfedge records and the faces
__global__ void kCopyBackIds(SplitStep s, float* __restrict__ pos, float* __restrict__ nrm, int32_t* __restrict__ pid, uint8_t* __restrict__ canon) {
    int i;
    const int r = rangeOf(s.vsize, s.hsize, s.fsize, i);
    const WC& w = s.w;
    if (r == 0) {
        if (w.vflags[i] & VF_REMOVE) return;
        int64_t o = w.v_c2o[i];
        if (o == -1) {
            o = s.V0 + s.addrV[i];
            w.v_c2o[i] = (int32_t)o;
        } else if (w.v_last[o] != i) {
            return;
        }
        for (int k = 0; k < 3; ++k) {
            pos[3 * o + k] = w.pos[3 * i + k];
            nrm[3 * o + k] = w.nrm[3 * i + k];
        }
        if (pid) pid[o] = w.pid[i];
    } else if (r == 1) {
        if (w.hflags[i] & VF_REMOVE) return;
        int64_t o = w.h_c2o[i];
        if (o == -1) {
            o = s.H0 + s.addrH[i];
            w.h_c2o[i] = (int32_t)o;
        }
        canon[o] = 0;  // this record may leave the build's layout
    } else if (r == 2) {
        if (w.fflags[i] & VF_REMOVE) return;
        if (w.f_c2o[i] == -1) w.f_c2o[i] = (int32_t)(s.F0 + s.addrF[i]);
    }
}

__device__ void copyBackRecord(const WC& w, int h, int4* __restrict__ he) {
    if (w.hflags[h] & VF_REMOVE) return;
    const int64_t me = w.h_c2o[h];
    int4 e = w.he[h];  // the record copied back to me: no other thread writes he[me]
    e.z = w.h_c2o[e.z];
    e.y = w.f_c2o[e.y];
    e.x = w.v_c2o[e.x];
    int t = e.w;
    if (t < 0) {
        t = -t - 2;
        e.w = t;
        if (t != -1) setT(he, t, (int)me);
    } else {
        e.w = w.h_c2o[t];
    }
    he[me] = e;
}
// (the vertices mark what the step touched, by their ids after the copy back, and reset the map
// entries the step set -- kWcCopy's, which kSubdivide only re-points -- so that the maps are all
// -1 again for the next step without a full fill; the first block clears the partial sums
// the refresh counts again)
__global__ void kCopyBack(SplitStep s, const int32_t* __restrict__ nm, int4* __restrict__ he, int32_t* __restrict__ face_he, uint32_t* __restrict__ fattr,
                          uint8_t* __restrict__ dirtyV, uint8_t* __restrict__ touched, int64_t* __restrict__ nmParts) {
    if (blockIdx.x == 0)
        for (int k = threadIdx.x; k < kPartSlots * kPartStride; k += kBlock) nmParts[k] = 0;
    int i;
    const int r = rangeOf(s.vsize, s.hsize, s.fsize, i);
    const WC& w = s.w;
    if (r == 0) {
        const int o = w.v_c2o[i];
        if (o >= 0) {
            dirtyV[o] = 1;
            touched[o] = 1;
        }
        if (i < 4 * w.n) {
            w.v_last[w.v_orig[i]] = -1;
            w.v_o2c[w.v_orig[i]] = -1;
            w.h_o2c[w.h_orig[i]] = -1;
            if ((i & 3) == 0) w.f_o2c[nm[i >> 2]] = -1;
        }
    } else if (r == 1) {
        copyBackRecord(w, i, he);
    } else if (r == 2) {
        if (w.fflags[i] & VF_REMOVE) return;
        const int64_t o = w.f_c2o[i];
        face_he[o] = w.h_c2o[w.f_first[i]];
        fattr[o] = w.f_attr[i];
    }
}

// ---------------------------------------------------------------- detectNonManifoldVertices
__device__ int fanWalk(const int4* __restrict__ he, int start, bool cw, int64_t* ctr) {
    auto step = [&](int h) -> int {
        if (cw) {
            const int t = heT(he, h);
            return (t != -1) ? heN(he, t) : -1;
        }
        const int s = heN(he, heN(he, heN(he, h)));
        const int t = heT(he, s);
        return (t != -1) ? t : -1;
    };
    const int origin = heO(he, start);
    int result = start;
    int cur = step(start);
    int guard = 0;
    while (cur != -1) {
        if (++guard > kFanGuard) { anomaly(ctr); break; }
        if (cur == result) break;
        if (origin != heO(he, cur)) break;
        if (cur < result) result = cur;
        cur = step(cur);
    }
    return result;
}

// One thread per vertex v over its outgoing halfedges: the fan key of each (the smallest
// id reached by fanWalk clockwise and counter-clockwise) and the number of distinct keys.
// Up to kFanLocal halfedges the walks run on successor indices in LDS: a step to a
// halfedge that does not start at v ends the walk, as the origin test of fanWalk does.
constexpr int kFanLocal = 16;
__global__ void __launch_bounds__(kBlock) kDetectFans(const int4* __restrict__ he, int64_t V, const uint8_t* __restrict__ only, const int64_t* __restrict__ off,
                                                      const int32_t* __restrict__ list, const int32_t* __restrict__ left, uint32_t* __restrict__ vflags,
                                                      int32_t* __restrict__ keyScratch, int64_t* ctr) {
    __shared__ int s_h[kFanLocal * kBlock];
    __shared__ int8_t s_cw[kFanLocal * kBlock];
    __shared__ int8_t s_ccw[kFanLocal * kBlock];
    const int64_t vv = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (vv >= V) return;
    if (only && !only[vv]) return;
    if (left && left[vv] != 0) {  // the list and the out-degree disagree
        anomaly(ctr);
        return;
    }
    const int tid = threadIdx.x;
    const int64_t b0 = off[vv];
    const int d = (int)(off[vv + 1] - b0);
    int distinct = 0;
    if (d <= kFanLocal) {
        auto H_ = [&](int k) -> int& { return s_h[k * kBlock + tid]; };
        for (int k = 0; k < d; ++k) H_(k) = list[b0 + k];
        // successor codes: index in the list, -1 = no successor, -2 = a halfedge of another origin
        auto local = [&](int g) -> int {
            if (g == -1) return -1;
            for (int j = 0; j < d; ++j)
                if (H_(j) == g) return j;
            return -2;
        };
        for (int k = 0; k < d; ++k) {
            const int h = H_(k);
            const int t = heT(he, h);
            s_cw[k * kBlock + tid] = (int8_t)local(t != -1 ? heN(he, t) : -1);
            s_ccw[k * kBlock + tid] = (int8_t)local(heT(he, heN(he, heN(he, heN(he, h)))));
        }
        auto walk = [&](int start, const int8_t* succ) -> int {
            int result = H_(start);
            int cur = succ[start * kBlock + tid];
            int guard = 0;
            while (cur != -1) {
                if (++guard > kFanGuard) {
                    anomaly(ctr);
                    break;
                }
                if (cur == -2) break;
                const int hc = H_(cur);
                if (hc == result) break;
                if (hc < result) result = hc;
                cur = succ[cur * kBlock + tid];
            }
            return result;
        };
        int keys[kFanLocal];
        for (int k = 0; k < d; ++k) {
            const int kk = min(walk(k, s_cw), walk(k, s_ccw));
            bool seen = false;
            for (int j = 0; j < k; ++j) seen = seen || keys[j] == kk;
            keys[k] = kk;
            if (!seen) ++distinct;
        }
    } else {
        for (int k = 0; k < d; ++k) {
            const int h = list[b0 + k];
            const int kk = min(h, min(fanWalk(he, h, true, ctr), fanWalk(he, h, false, ctr)));
            bool seen = false;
            for (int j = 0; j < k; ++j) seen = seen || keyScratch[b0 + j] == kk;
            keyScratch[b0 + k] = kk;
            if (!seen) ++distinct;
        }
    }
    if (distinct > 1) vflags[vv] |= VF_FANS;
    else vflags[vv] &= ~(uint32_t)VF_FANS;
}

// ---------------------------------------------------------------- statistics
// counts over the vertex-pair buckets (HalfedgeMesh.cu:1164-1239, ManifoldCreator.cu:545-549)
__global__ void __launch_bounds__(kBlock) kStats(const int4* __restrict__ he, int64_t H, const int32_t* __restrict__ face_he, int64_t F,
                                                 const int32_t* __restrict__ bsize, const uint32_t* __restrict__ vflags, int64_t V, const uint8_t* __restrict__ canon, int64_t* ctr, int64_t* pin, int guarded) {
    if (notYet(ctr, guarded)) {
        if (blockIdx.x == 0 && threadIdx.x < 64) handOver(ctr, pin);
        return;
    }
    stampClock(ctr + A_STAMP + ST_STATS);
    __shared__ unsigned int acc[9];
    __shared__ bool s_last;
    if (threadIdx.x < 9) acc[threadIdx.x] = 0;
    __syncthreads();
    unsigned int loc[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
    const int64_t t0 = (int64_t)blockIdx.x * blockDim.x + threadIdx.x, stride = (int64_t)gridDim.x * blockDim.x;
    auto bucket = [&](int w) {
        if (!bucketFirst(w)) return;
        const int n = bucketSize(w);
        loc[0] += (n == 4);
        loc[1] += (n == 3);
        loc[2] += (n > 0);
    };
    // the number of a face's edges in buckets of three and more
    // (constant indices only: a computed index would put loc in scratch memory)
    auto face = [&](int k) {
        loc[3] += k == 0;
        loc[4] += k == 1;
        loc[5] += k == 2;
        loc[6] += k == 3;
        loc[7] += k == 4;
    };
    auto wide = [&](const int4& w) { return (bucketSize(w.x) > 2) + (bucketSize(w.y) > 2) + (bucketSize(w.z) > 2) + (bucketSize(w.w) > 2); };
    // four halfedges per 16-byte load, then the tail; a face whose four records, the ones of its own
    // id, all keep the build's layout is those four halfedges, counted from the same load (read
    // again by face they cost 245 MB of the 512^3 gyroid's 675)
    const int64_t H4 = H >> 2, n4 = H4 > F ? H4 : F;
#pragma unroll 4
    for (int64_t i = t0; i < n4; i += stride) {
        int4 w = make_int4(0, 0, 0, 0);
        if (i < H4) {
            w = reinterpret_cast<const int4*>(bsize)[i];
            bucket(w.x);
            bucket(w.y);
            bucket(w.z);
            bucket(w.w);
        }
        if (i < F) {
            int h = face_he[i];
            const int64_t q = h >> 2;
            if (4 * q + 3 < H && (!canon || reinterpret_cast<const uint32_t*>(canon)[q] == 0x01010101u)) {
                if (q != i) w = reinterpret_cast<const int4*>(bsize)[q];
                face(wide(w));
            } else {
                int k = 0;
                for (int j = 0; j < 4; ++j) {
                    if (bucketSize(bsize[h]) > 2) ++k;
                    h = nextOf(he, canon, h);
                }
                face(k);
            }
        }
    }
    for (int64_t i = 4 * H4 + t0; i < H; i += stride) bucket(bsize[i]);
    for (int64_t v = t0; v < V; v += stride) loc[8] += (vflags[v] & VF_FANS) ? 1u : 0u;
    for (int k = 0; k < 9; ++k) {
        unsigned int v = loc[k];
        for (int d = 32; d > 0; d >>= 1) v += __shfl_down(v, d, 64);
        if ((threadIdx.x & 63) == 0 && v) atomicAdd(&acc[k], v);
    }
    __syncthreads();
    if (threadIdx.x < 9 && acc[threadIdx.x]) atomicAdd((unsigned long long*)&ctr[A_STATS + threadIdx.x], (unsigned long long)acc[threadIdx.x]);
    // the last block to finish hands the counters over: no copy, no second wait.  The block's
    // sums were added by its first wave, which waits for its own atomics before it takes its
    // ticket; the sums are read back with atomic loads, so no block needs a device-scope fence
    // (each would write its XCD's L2 back: +0.1 ms at 128^3)
    if (threadIdx.x < 64) {
        __builtin_amdgcn_s_waitcnt(0);
        if (threadIdx.x == 0) s_last = atomicAdd((unsigned long long*)&ctr[A_TICKET], 1ULL) == gridDim.x - 1;
    }
    __syncthreads();
    if (!s_last) return;
    if (threadIdx.x < 64) handOver(ctr, pin);
}


// The resident mesh into the caller's device buffers, every array in one launch: block b works
// on the array j with start[j] <= b < start[j + 1], kCopyPer * kBlock of its items (16 bytes of
// an array copied as it is, four faces or vertices of a narrowed one, one vertex of the
// vertex -> halfedge array).
//
// HalfedgeMesh's vertex -> halfedge array as collectHalfedgeElements leaves it holds the highest
// halfedge starting at each vertex of the last initialize ("last writer wins" in ascending
// thread order): the maximum of the vertex's outgoing list, whose entries are consecutive;
// -1 where the list is empty, 0 in the slots a split's resizes added.
//
// Bound by HBM: 2.5 GB moved at the 512^3 gyroid in 587 us (4.3 TB/s).  Nothing here is read twice, so loads
// and stores pass the caches by: 651 us there through them, and 20 us instead of 10 at the 256^3 blobs, whose
// 13 MB of stores waited for older lines to be written back.  The eleven launches this replaces
// took 1.43 ms (700 us of it one atomicMax per halfedge) and 100 us of launch time on a mesh of any size.
constexpr int kCopyPer = 4;
enum : int { CM_POS, CM_NRM, CM_HE, CM_FACE, CM_VHE_COPY, CM_FATTR, CM_VFLAGS, CM_VHE, CM_COUNT };
struct CopyMesh {
    const void* src[CM_COUNT];
    void* dst[CM_COUNT];
    int64_t n[CM_COUNT];  // words copied; faces / vertices of the others
    unsigned start[CM_COUNT + 1];
    const int64_t* off;  // the outgoing lists of the last initialize's listsV vertices (CM_VHE)
    int64_t listsV;
};
__device__ __forceinline__ int64_t cmItems(int j, int64_t n) { return j == CM_VHE ? n : (n + 3) / 4; }
__global__ void __launch_bounds__(kBlock) kCopyMesh(CopyMesh c) {
    int j = 0;
    while (j + 1 < CM_COUNT && blockIdx.x >= c.start[j + 1]) ++j;
    const int64_t n = c.n[j], items = cmItems(j, n);
    const int64_t i0 = (int64_t)(blockIdx.x - c.start[j]) * (kCopyPer * kBlock) + threadIdx.x;
    const bool vec = ((((uintptr_t)c.src[j]) | ((uintptr_t)c.dst[j])) & 15) == 0;
    if (j < CM_FATTR) {
        const uint32_t* src = (const uint32_t*)c.src[j];
        uint32_t* dst = (uint32_t*)c.dst[j];
        uint4 w[kCopyPer];
#pragma unroll
        for (int k = 0; k < kCopyPer; ++k) {
            const int64_t i = i0 + (int64_t)k * kBlock;
            if (vec && 4 * i + 3 < n) w[k] = loadStreaming(reinterpret_cast<const uint4*>(src) + i);
        }
#pragma unroll
        for (int k = 0; k < kCopyPer; ++k) {
            const int64_t i = i0 + (int64_t)k * kBlock;
            if (vec && 4 * i + 3 < n) storeStreaming(reinterpret_cast<uint4*>(dst) + i, w[k]);
            else
                for (int64_t t = 4 * i; t < 4 * i + 4 && t < n; ++t) dst[t] = src[t];
        }
        return;
    }
    for (int k = 0; k < kCopyPer; ++k) {
        const int64_t i = i0 + (int64_t)k * kBlock;
        if (i >= items) return;
        if (j == CM_VHE) {
            const int32_t* list = (const int32_t*)c.src[j];
            int32_t best = 0;
            if (i < c.listsV) {
                best = -1;
                const int64_t e = c.off[i + 1];
                for (int64_t q = c.off[i]; q < e; q += 4) {
                    int h[4];
#pragma unroll
                    for (int t = 0; t < 4; ++t) h[t] = list[q + t < e ? q + t : e - 1];
                    best = max(max(best, max(h[0], h[1])), max(h[2], h[3]));
                }
            }
            storeStreaming((int32_t*)c.dst[j] + i, best);
            continue;
        }
        const uint32_t* src = (const uint32_t*)c.src[j];
        if (vec && 4 * i + 3 < n) {
            const uint4 w = reinterpret_cast<const uint4*>(src)[i];
            if (j == CM_FATTR) storeStreaming((uint64_t*)c.dst[j] + i, (uint64_t)((w.x & 0xFFFFu) | (w.y << 16)) | (uint64_t)((w.z & 0xFFFFu) | (w.w << 16)) << 32);
            else storeStreaming((uint32_t*)c.dst[j] + i, (w.x & 0xFFu) | ((w.y & 0xFFu) << 8) | ((w.z & 0xFFu) << 16) | (w.w << 24));
        } else {
            for (int64_t t = 4 * i; t < 4 * i + 4 && t < n; ++t) {
                if (j == CM_FATTR) ((uint16_t*)c.dst[j])[t] = (uint16_t)src[t];
                else ((uint8_t*)c.dst[j])[t] = (uint8_t)src[t];
            }
        }
    }
}

}  // namespace

// ============================================================================ host driver

Pipeline::Pipeline() {}
Pipeline::~Pipeline() {
    releaseGraphs();
    for (auto& e : kev)
        if (e) (void)hipEventDestroy(e);
    if (pinH_) (void)hipHostFree(pinH_);
    if (pinBatch_) (void)hipHostFree(pinBatch_);
    for (auto& e : upEv_)
        if (e) (void)hipEventSynchronize(e), (void)hipEventDestroy(e);
    for (void* u : up_)
        if (u) (void)hipHostFree(u);
}

void Pipeline::upload(void* dst, const void* src, size_t bytes, int region) {
    if (bytes == 0) return;
    if (!upEv_[region]) MDMC_HIP(hipEventCreateWithFlags(&upEv_[region], hipEventDisableTiming));
    // the last copy out of this region must be done before its bytes change (normally long done)
    MDMC_HIP(hipEventSynchronize(upEv_[region]));
    if (upCap_[region] < bytes) {
        if (up_[region]) MDMC_HIP(hipHostFree(up_[region]));
        up_[region] = nullptr;
        upCap_[region] = 0;
        const size_t want = bytes + bytes / 2 + 4096;
        MDMC_HIP(hipHostMalloc(&up_[region], want, hipHostMallocDefault));
        upCap_[region] = want;
    }
    std::memcpy(up_[region], src, bytes);
    MDMC_HIP(hipMemcpyAsync(dst, up_[region], bytes, hipMemcpyHostToDevice, stream));
    MDMC_HIP(hipEventRecord(upEv_[region], stream));
}

int64_t* Pipeline::pinHost() {
    if (!pinH_) {
        void* h = nullptr;
        MDMC_HIP(hipHostMalloc(&h, kPinSlots * sizeof(int64_t), hipHostMallocMapped | hipHostMallocCoherent));
        pinH_ = (int64_t*)h;
        void* d = nullptr;
        MDMC_HIP(hipHostGetDevicePointer(&d, h, 0));
        pinD_ = (int64_t*)d;
    }
    return pinH_;
}
int64_t* Pipeline::pinDev() {
    pinHost();
    return pinD_;
}

void Pipeline::kernelTimes(double* msGridPass) {
    float a = 0.f, b = 0.f;
    MDMC_HIP(hipEventElapsedTime(&a, kev[0], kev[1]));
    MDMC_HIP(hipEventElapsedTime(&b, kev[2], kev[3]));
    *msGridPass = (double)a + (double)b;
}

int64_t Pipeline::readI64(const int64_t* dev) {
    int64_t* h = pinHost();
    MDMC_HIP(hipMemcpyAsync(h, dev, sizeof(int64_t), hipMemcpyDeviceToHost, stream));
    MDMC_HIP(hipStreamSynchronize(stream));
    return h[0];
}

// Waits until the device has written the pinned words that ready() looks at.  Waking up from a stream
// synchronisation takes some 8 us, and it waits for everything launched behind the words as well;
// polling sees them 1 to 2 us after they are written.  A wait beyond kPollLimit, where that no
// longer counts (or where the words do not come: held launches, an error, a capture), synchronises,
// which reports errors too.  The words' writers run after every kernel before them in the stream
// has ended, so all that was launched before is complete.  64^3 blobs with the simplifications
// 254 us an extraction before and 227 now, 128^3 lattice 811 and 770, batch of 16 554 and 504.
template <class Ready>
void Pipeline::await(Ready ready) {
    constexpr auto kPollLimit = std::chrono::microseconds(2000);
    const auto t0 = std::chrono::steady_clock::now();
    do {
        for (int k = 0; k < 16; ++k) {
            if (ready()) {
                std::atomic_thread_fence(std::memory_order_acquire);
                return;
            }
            __builtin_ia32_pause();
        }
    } while (std::chrono::steady_clock::now() - t0 < kPollLimit);
    MDMC_HIP(hipStreamSynchronize(stream));
}
// the two totals of a scan or numbering, -1 until written
void Pipeline::expectTotals() {
    volatile int64_t* h = pinHost();
    h[1] = h[2] = -1;
}
bool Pipeline::totalsWritten() {
    const volatile int64_t* h = pinHost();
    return h[1] >= 0 && h[2] >= 0;
}

int64_t* Pipeline::counters() { return arena.get<int64_t>("counters", A_NCOUNTERS); }
// partial sums (kPartSlots, kPartStride apart) of the slotted non-manifold halfedges of the
// current buckets, counted where the bucket sizes are written, and of those a split step's
// working copy holds
int64_t* Pipeline::nmSlotParts() { return arena.get<int64_t>("nm_slot_parts", kPartSlots * kPartStride); }
int64_t* Pipeline::nmFoundParts() {
    const bool fresh = arena.capacity<int64_t>("nm_found_parts") < (size_t)(kPartSlots * kPartStride);
    int64_t* p = arena.get<int64_t>("nm_found_parts", kPartSlots * kPartStride);
    if (fresh) zero(p, kPartSlots * kPartStride * sizeof(int64_t));  // kNMSlotCheck clears it after each use
    return p;
}

const uint8_t* Pipeline::canonFlags() { return canonTracked ? arena.ptr<uint8_t>("he_canon") : nullptr; }

Pipeline::Lookback Pipeline::lookback(int64_t words) {
    const size_t before = arena.capacity<unsigned long long>("lb_words");
    unsigned long long* w = arena.get<unsigned long long>("lb_words", (size_t)words);
    const size_t cap = arena.capacity<unsigned long long>("lb_words");
    if (cap != before || lbEpoch_ == 0xFFFFu) {
        launchFill(w, 0x00, cap * sizeof(unsigned long long));
        lbEpoch_ = 0;
    }
    return Lookback{w, ++lbEpoch_};
}

void Pipeline::scan(std::initializer_list<ScanJob> jobs, int64_t* stampStart, int64_t* stampEnd) {
    ScanJob j[kScanJobs];
    int count = 0;
    int64_t words = 0;
    for (const ScanJob& x : jobs) words += scanTiles(x.n);
    const Lookback lb = lookback(words);
    words = 0;
    for (const ScanJob& x : jobs) {
        j[count] = x;
        j[count++].words = lb.words + words;
        words += scanTiles(x.n);
    }
    scanExclusiveI32(j, count, lb.epoch, stream, lookbackDiag(), stampStart, stampEnd);
}

// lists the faces with the NM bit, ascending (countNonManifoldFaces); their number goes to the
// counter A_NM
int32_t* Pipeline::listNM(bool first) {
    int32_t* nm = arena.get<int32_t>("nmlist", (size_t)std::max<int64_t>(F, 1));
    if (first && listed) return nm;  // by the twin repair
    const Lookback lb = lookback(scanTiles(F));
    compactFlagged(arena.ptr<uint32_t>("fattr"), F, (uint32_t)QA_NM, nm, counters() + A_NM, lb.words, lb.epoch, stream, lookbackDiag(),
                   first ? stamp(ST_SPLIT) : nullptr);
    return nm;
}

// the checks and the number of listed faces, from the counters in h
int64_t Pipeline::checkNM(const int64_t* h) {
    if (h[A_INVALID])
        throw HipError(std::string("inconsistent mesh after ") + (refreshUnchecked ? "splitting" : "quad vertex ids") + " (" +
                           std::to_string(h[A_INVALID]) + " bad ids)", -4);
    refreshUnchecked = false;
    const int64_t n = h[A_NM];
    if (n < 0 || n > F) throw HipError("inconsistent NM-face count (" + std::to_string(n) + ")", -4);
    return n;
}

const int64_t* Pipeline::readCounters() {
    pinHost()[kPinDone] = 0;
    kReadBack<<<1, 64, 0, stream>>>(counters(), pinDev() + kPinFinal);
    return waitStats();
}

// fills with one launch (the runtime's memset launches a body and a tail kernel)
void Pipeline::zero(void* p, size_t bytes) { launchFill(p, 0x00, bytes); }
void Pipeline::launchFill(void* p, uint8_t byte, size_t bytes) {
    if (bytes == 0) return;
    const size_t head = std::min<size_t>((16 - ((uintptr_t)p & 15)) & 15, bytes);
    const size_t body = (bytes - head) & ~(size_t)15;
    const size_t vec = body / 16;
    kFillBytes<<<(unsigned)std::max<size_t>((vec + kBlock - 1) / kBlock, 1), kBlock, 0, stream>>>((uint8_t*)p, byte, head, body, bytes);
}

void Pipeline::FillBatch::add(void* p, uint8_t byte, size_t bytes) {
    if (bytes == 0) return;
    if (fs.count == kFillSetMax) flush();
    const int j = fs.count++;
    const size_t head = std::min<size_t>((16 - ((uintptr_t)p & 15)) & 15, bytes);
    const size_t body = (bytes - head) & ~(size_t)15;
    const size_t vec = body / 16;
    fs.p[j] = (uint8_t*)p;
    fs.byte[j] = byte;
    fs.head[j] = head;
    fs.body[j] = body;
    fs.n[j] = bytes;
    fs.start[j] = blocks;
    blocks += (unsigned)std::max<size_t>((vec + kBlock - 1) / kBlock, 1);
}
void Pipeline::FillBatch::flush() {
    if (fs.count == 0) return;
    kFillMany<<<blocks, kBlock, 0, pl.stream>>>(fs);
    fs.stamp = nullptr;
    fs.count = 0;
    blocks = 0;
}

void Pipeline::prepare(const std::vector<ProblemDev>& problems, bool captured) {
    refreshUnchecked = false;
    PrepareSetup su{};
    su.ctr = counters();
    su.nCtr = A_NCOUNTERS;
    su.parts = nmSlotParts();
    su.nParts = kPartSlots * kPartStride;
    if (problems.size() == 1) {
        probsDev = arena.get<ProblemDev>("gp_probs", 1);
        su.probs = probsDev;
        su.prob = problems[0];
    }
    const bool fresh = arena.capacity<int64_t>("prep_gate") == 0;
    su.gate = arena.get<int64_t>("prep_gate", 1);
    if (fresh) zero(su.gate, sizeof(int64_t));
    su.stamp = stamp(ST_PAD);
    su.pin = pinDev() + kPinInvalid;
    su.pinAt = A_PIN;
    su.special = pinDev() + kPinSpecial;
    su.token = captured ? 0 : ++prepToken_;
    pinHost()[kPinSpecial] = 0;
    pinHost()[kPinInvalid] = 0;
    launchPrepareGrids(prep.desc[0], prep.dev, (int)prep.desc.size(), prep.rows, prep.refinement, prep.pad, su, stream);
}

template <class Again>
void Pipeline::finishPrepare(bool totalsBehind, Again again) {
    if (totalsBehind) await([&] { return totalsWritten(); });
    else MDMC_HIP(hipStreamSynchronize(stream));
    int64_t* h = pinHost();
    if (!h[kPinSpecial]) return;
    h[kPinSpecial] = 0;
    launchPrepareExact(prep.desc[0], prep.dev, (int)prep.desc.size(), prep.rows, prep.pad, stream);
    again();
    MDMC_HIP(hipStreamSynchronize(stream));
}

int64_t* Pipeline::lookbackDiag() { return counters() + A_LB_DIRECT; }

int64_t* Pipeline::stamp(int slot) { return counters() + A_STAMP + slot; }
void Pipeline::launchStamp(int64_t* at) { kStamp<<<1, 1, 0, stream>>>(at); }
// the counters are cleared behind the uploads, so this stamp goes to the pinned words
void Pipeline::stampUpload(bool uploads) {
    pinHost()[kPinUpload] = 0;
    if (uploads) launchStamp(pinDev() + kPinUpload);
}

void Pipeline::counterTotals(int64_t* anomalyCount, int64_t* mergeSeq, int64_t* lookbackDirect) {
    const int64_t* h = pinHost() + kPinFinal;
    *anomalyCount = h[A_ANOMALY];
    *mergeSeq = h[A_MERGE_SEQ];
    *lookbackDirect = h[A_LB_DIRECT];
}

void Pipeline::stageTimes(double ms[9]) {
    if (!clockKHz_) {
        int dev = 0, khz = 0;
        MDMC_HIP(hipGetDevice(&dev));
        MDMC_HIP(hipDeviceGetAttribute(&khz, hipDeviceAttributeWallClockRate, dev));
        clockKHz_ = khz > 0 ? khz : 100000;
    }
    // a stage that launched nothing began when the next one did
    int64_t t[ST_COUNT];
    std::memcpy(t, pinHost() + kPinFinal + A_STAMP, sizeof t);
    for (int i = ST_END - 1; i >= 0; --i)
        if (t[i] == 0) t[i] = t[i + 1];
    if (pinHost()[kPinUpload]) t[ST_PAD] = pinHost()[kPinUpload];
    const double k = 1.0 / clockKHz_;
    ms[0] = (double)(t[ST_END] - t[ST_PAD]) * k;
    for (int i = 0; i < 7; ++i) ms[1 + i] = (double)(t[i + 1] - t[i]) * k;
    ms[8] = t[ST_CLASSIFY] ? (double)(t[ST_TOTALS] - t[ST_CLASSIFY] + (t[ST_EMIT] ? t[ST_INIT] - t[ST_EMIT] : 0)) * k : 0.0;
}

// ---- grid pass
// the outputs of the emit part, sized exactly
void Pipeline::emitArgs(GridPassArgs& a, int64_t C, bool recordAdjoint) {
    if (V >= (int64_t)INT32_MAX / 2 || 4 * Q >= (int64_t)INT32_MAX) throw HipError("mesh exceeds the int32 id range", -3);
    if (recordAdjoint && (V >= ((int64_t)1 << 29) || C >= (int64_t)INT32_MAX))
        throw HipError("adjoint recording needs fewer than 2^29 vertices and 2^31 cells", -3);
    a.pos = arena.get<float>("pos", 3 * (size_t)std::max<int64_t>(V, 1));
    a.nrm = arena.get<float>("nrm", 3 * (size_t)std::max<int64_t>(V, 1));
    a.quads = arena.get<int4>("quads", (size_t)std::max<int64_t>(Q, 1));
    a.qattr = arena.get<uint32_t>("qattr", (size_t)std::max<int64_t>(Q, 1));
    a.adjMap = recordAdjoint ? arena.get<int32_t>("adj_map", (size_t)std::max<int64_t>(C, 1)) : nullptr;
    a.vcell = arena.get<int32_t>("gp_vcell", (size_t)std::max<int64_t>(V, 1));
    a.vct = arena.get<uint16_t>("gp_vct", (size_t)std::max<int64_t>(V, 1));
    a.outdeg = arena.get<int32_t>("out_cnt", (size_t)V + 1);  // the halfedge initialize's list lengths
    a.vflags = arena.get<uint32_t>("vflags", (size_t)std::max<int64_t>(V, 1));
    if (!chain.empty()) {
        const size_t nv = (size_t)std::max<int64_t>(V, 1);
        a.chain.vtype = arena.get<uint8_t>("vtype", nv);
        arena.get<int32_t>("vtarget", nv);
        a.chain.valence = arena.get<int32_t>("valence", nv);
        if (std::count(chain.begin(), chain.end(), (int)S_OLD)) a.chain.count = arena.get<int32_t>("vcount", nv);
        if (chain.size() > 1) {
            a.chain.head = arena.get<int32_t>("src_head", nv);
            a.chain.outdeg = arena.get<int32_t>("outdeg", nv);
            a.chain.bdin = arena.get<int32_t>("bdin", nv);
            a.chain.vdead = arena.get<uint8_t>("vdead", nv);
            a.chain.touched = arena.get<uint8_t>("touched", nv);
        }
    }
    a.V = V;
    a.vpid = nProblems > 1 ? arena.get<int32_t>("pid", (size_t)std::max<int64_t>(V, 1)) : nullptr;
}

// Row slabs: bands of at most SLAB_XMAX cells per row, R rows per block, and chunks of slices
// sized so that the launch has about 4096 blocks (a problem gets its share by its cell count;
// at least 8 slices per chunk, each chunk re-reads one slice before it for its quads).
void Pipeline::slabPass(std::vector<ProblemDev>& problems, int64_t C, int shape, bool surfIter, bool recordAdjoint) {
    const int R = gridPassSlabRows(shape);
    int64_t blocks = 0, segs = 0;
    for (ProblemDev& pr : problems) {
        const int CZ = pr.g.nz - 1;
        pr.bands = (pr.CX + SLAB_XMAX - 1) / SLAB_XMAX;
        pr.bandW = (pr.CX + pr.bands - 1) / pr.bands;
        pr.rowBlocks = (pr.CY + R - 1) / R;
        const int64_t cols = (int64_t)pr.bands * pr.rowBlocks;
        const int64_t share = C > 0 ? (int64_t)(4096.0 * (double)pr.cells / (double)C / (double)cols) : 1;
        const int nzc = (int)std::max<int64_t>(1, std::min<int64_t>((CZ + 7) / 8, share));
        pr.zChunk = (CZ + nzc - 1) / nzc;
        pr.zChunks = (CZ + pr.zChunk - 1) / pr.zChunk;
        pr.blockBase = blocks;
        blocks += cols * pr.zChunks;
        pr.segBase = segs;
        segs += (int64_t)CZ * pr.CY * pr.bands;
    }
    if (blocks >= (int64_t)INT32_MAX || segs >= (int64_t)INT32_MAX) throw HipError("grid pass: too many row segments", -3);
    probsDev = arena.get<ProblemDev>("gp_probs", problems.size());
    upload(probsDev, problems.data(), problems.size() * sizeof(ProblemDev), 0);
    GridPassArgs a{};
    a.probs = probsDev;
    a.nProblems = nProblems;
    a.surfIter = surfIter ? 1 : 0;
    a.numBlocks = blocks;
    a.stampFirst = stamp(ST_DMC);
    a.stampRun = stamp(ST_CLASSIFY);
    a.stampEmit = stamp(ST_EMIT);
    a.numSegs = segs;
    a.segV = arena.get<int32_t>("gp_segv", (size_t)segs + 1);
    a.segQ = arena.get<int32_t>("gp_segq", (size_t)segs + 1);
    int64_t* svo = arena.get<int64_t>("gp_segvo", (size_t)segs + 1);
    int64_t* sqo = arena.get<int64_t>("gp_segqo", (size_t)segs + 1);
    a.segVOff = svo;
    a.segQOff = sqo;
    int64_t* h = pinHost();
    int64_t* pd = pinDev();
    expectTotals();
    tuneEvent(0);
    launchSlabCount(shape, a, stream);
    scan({ScanJob{a.segV, svo, segs + 1, pd + 1, nullptr}, ScanJob{a.segQ, sqo, segs + 1, pd + 2, nullptr}}, nullptr, stamp(ST_TOTALS));
    tuneEvent(1);
    await([&] { return totalsWritten(); });
    V = h[1];
    Q = h[2];
    emitArgs(a, C, recordAdjoint);
    gpVOff_ = svo;
    gpQOff_ = sqo;
    gpLast_ = segs;
    tuneEvent(2);
    launchSlabEmit(shape, a, stream);
    tuneEvent(3);
    dmcV = V;
    dmcQ = Q;
}
int64_t Pipeline::dmcSetup(std::vector<ProblemDev>& problems, bool recordAdjoint) {
    vertHeV = vertHeQ = 0;
    batchVertHe = false;
    tuning_ = false;
    nProblems = (int)problems.size();
    if (recordAdjoint && nProblems != 1) throw HipError("adjoint recording needs a single problem", -4);
    int64_t C = 0;
    for (ProblemDev& pr : problems) {
        pr.CX = pr.g.nx - 1;
        pr.CY = pr.g.ny - 1;
        pr.cells = (int64_t)pr.CX * pr.CY * (pr.g.nz - 1);
        pr.cellBase = C;
        C += pr.cells;
        if (pr.cells >= (int64_t)INT32_MAX) throw HipError("a grid has 2^31 cells or more", -3);
        // the grid pass splits tile cell offsets with a float-reciprocal division (exact below 2^24)
        if (pr.CX >= (1 << 23) || pr.CY >= (1 << 23)) throw HipError("a grid has 2^23 cells or more along x or y", -3);
    }
    return C;
}

// the autotuner's workload class: cell count and problem count to the next power of two,
// move-to-surface on / off
int Pipeline::shapeClass(int64_t C, bool surfIter) const {
    int lc = 0, lp = 0;
    while (((int64_t)1 << lc) < C + 1) ++lc;
    while ((1 << lp) < nProblems) ++lp;
    return (lc << 16) | (lp << 1) | (surfIter ? 1 : 0);
}

int Pipeline::resolveShape(int64_t C, bool surfIter) {
    lastShape = tileShape;
    if (lastShape == GP_SHAPE_AUTO) {
        auto it = tuned.find(shapeClass(C, surfIter));
        if (it != tuned.end()) lastShape = it->second;
    }
    return lastShape;
}

void Pipeline::dmc(std::vector<ProblemDev>& problems, bool surfIter, bool recordAdjoint) {
    const int64_t C = dmcSetup(problems, recordAdjoint);
    const bool tune = resolveShape(C, surfIter) == GP_SHAPE_AUTO;
    if (tune || gridPassIsSlab(lastShape)) finishPrepare(false, [] {});
    if (tune) {
        // autotuner: on the first extraction of a workload class, time every shape on this
        // very input and keep the fastest for the class.  The XCD-chunked shapes (1-3, 7, 8)
        // move less data out of L2 (about half for the tiles, measured at 512^3); a
        // launch-order or work-queue shape (4-6, 9) must beat them by 3% to be chosen.
        double best = 1e30;
        if (!kev[0])
            for (auto& e : kev) MDMC_HIP(hipEventCreate(&e));
        tuning_ = true;
        for (int sh = GP_SHAPE_FIRST; sh <= GP_SHAPE_LAST; ++sh) {
            gridPass(problems, C, sh, surfIter, recordAdjoint);
            MDMC_HIP(hipEventSynchronize(kev[3]));
            double ms = 0.0;
            kernelTimes(&ms);
            tuneMs[sh] = ms;
            const double cost = (sh <= 3 || gridPassIsSlab(sh)) ? ms : ms * 1.03;
            if (cost < best) {
                best = cost;
                lastShape = sh;
            }
        }
        tuning_ = false;
        tuned[shapeClass(C, surfIter)] = lastShape;
        if (lastShape == GP_SHAPE_LAST) return;  // the last candidate's output is in place
    }
    gridPass(problems, C, lastShape, surfIter, recordAdjoint);
}

// addresses of every device buffer the front of a tile-shape grid pass touches
std::vector<int64_t> Pipeline::frontBuffers() {
    std::vector<int64_t> b;
    for (const char* n : {"counters", "nm_slot_parts", "prep_gate", "grid", "prep_desc", "gp_probs", "gp_queue", "gp_rec", "gp_tv", "gp_tq", "gp_tna", "gp_map", "gp_tvo", "gp_tqo",
                          "gp_lb", "gp_ticket"})
        b.push_back((int64_t)(intptr_t)arena.ptr<char>(n));
    b.push_back((int64_t)(intptr_t)pinDev());
    return b;
}

void Pipeline::releaseGraphs() {
    if (fg_.exec) (void)hipGraphExecDestroy(fg_.exec);
    fg_.exec = nullptr;
    fg_.sig.clear();
    if (fg_.stage) (void)hipHostFree(fg_.stage);
    fg_.stage = nullptr;
    fg_.stageCap = 0;
}

bool Pipeline::runFrontGraph(const std::vector<int64_t>& shapeSig, std::vector<ProblemDev>& problems, int64_t C, int shape, bool surfIter) {
    if (!stream) return false;  // the default stream cannot be captured
    const size_t prepBytes = prep.desc.size() * sizeof(PrepareDesc);
    std::vector<int64_t> sig = shapeSig;
    const std::vector<int64_t> bufs = frontBuffers();
    sig.insert(sig.end(), bufs.begin(), bufs.end());
    const size_t pbytes = problems.size() * sizeof(ProblemDev);
    const size_t probOff = (prepBytes + 255) & ~(size_t)255;
    if (fg_.exec && fg_.sig == sig) {
        // replay: the descriptors of this call into the graph's staging, then the graph
        assignTiles(problems, shape);
        std::memcpy(fg_.stage, prep.desc.data(), prepBytes);
        std::memcpy((char*)fg_.stage + probOff, problems.data(), pbytes);
        probsDev = arena.ptr<ProblemDev>("gp_probs");
        refreshUnchecked = false;
        pinHost()[kPinSpecial] = 0;
        pinHost()[kPinInvalid] = 0;
        expectTotals();
        ga_ = fgArgs_;
        MDMC_HIP(hipGraphLaunch(fg_.exec, stream));
        ++graphReplays;
        return true;
    }
    if (sig != fgLastEager_) return false;  // first call with these shapes and buffers: run it eagerly
    // second call with the same shapes and no buffer moved since: capture the front once
    releaseGraphs();
    fg_.stageCap = probOff + pbytes;
    MDMC_HIP(hipHostMalloc(&fg_.stage, fg_.stageCap, hipHostMallocDefault));
    std::memcpy(fg_.stage, prep.desc.data(), prepBytes);
    hipGraph_t graph = nullptr;
    MDMC_HIP(hipStreamBeginCapture(stream, hipStreamCaptureModeRelaxed));
    try {
        MDMC_HIP(hipMemcpyAsync(prep.dev, fg_.stage, prepBytes, hipMemcpyHostToDevice, stream));
        prepare(problems, true);
        gridPassFront(problems, C, shape, surfIter, (char*)fg_.stage + probOff);
    } catch (...) {
        (void)hipStreamEndCapture(stream, &graph);
        if (graph) (void)hipGraphDestroy(graph);
        releaseGraphs();
        throw;
    }
    MDMC_HIP(hipStreamEndCapture(stream, &graph));
    hipGraphExec_t exec = nullptr;
    const hipError_t e = hipGraphInstantiate(&exec, graph, nullptr, nullptr, 0);
    (void)hipGraphDestroy(graph);
    MDMC_HIP(e);
    fg_.exec = exec;
    fg_.sig = sig;
    fgArgs_ = ga_;
    MDMC_HIP(hipGraphLaunch(fg_.exec, stream));
    ++graphReplays;
    return true;
}

// classify -> scan of the tile counts -> exact output sizes -> emit
void Pipeline::gridPass(std::vector<ProblemDev>& problems, int64_t C, int shape, bool surfIter, bool recordAdjoint) {
    if (gridPassIsSlab(shape)) {
        slabPass(problems, C, shape, surfIter, recordAdjoint);
        return;
    }
    gridPassFront(problems, C, shape, surfIter, nullptr);
    gridPassBack(problems, C, shape, surfIter, recordAdjoint);
}

int64_t Pipeline::assignTiles(std::vector<ProblemDev>& problems, int shape) {
    const int T = gridPassTile(shape);
    int64_t numTiles = 0;
    for (ProblemDev& pr : problems) {
        pr.tileBase = numTiles;
        numTiles += (pr.cells + T - 1) / T;
    }
    return numTiles;
}

// The part of a tile-shape grid pass that the shapes alone determine: the problems' upload,
// classification and the tile-count scans, with no host synchronisation.  stagedProbs: copy
// the problems from that pinned buffer (a graph capture; the caller fills it before every
// replay) instead of through upload().
void Pipeline::gridPassFront(std::vector<ProblemDev>& problems, int64_t C, int shape, bool surfIter, void* stagedProbs) {
    const int T = gridPassTile(shape);
    const int64_t numTiles = assignTiles(problems, shape);
    probsDev = arena.get<ProblemDev>("gp_probs", problems.size());
    const size_t pbytes = problems.size() * sizeof(ProblemDev);
    if (problems.size() == 1) {
        // stored by prepare()
    } else if (stagedProbs) {
        std::memcpy(stagedProbs, problems.data(), pbytes);
        MDMC_HIP(hipMemcpyAsync(probsDev, stagedProbs, pbytes, hipMemcpyHostToDevice, stream));
    } else {
        upload(probsDev, problems.data(), pbytes, 0);
    }
    GridPassArgs& a = ga_;
    a = GridPassArgs{};
    a.probs = probsDev;
    a.nProblems = nProblems;
    a.surfIter = surfIter ? 1 : 0;
    a.numTiles = numTiles;
    a.stampFirst = stamp(ST_DMC);
    a.stampRun = stamp(ST_CLASSIFY);
    a.stampEmit = stamp(ST_EMIT);
    a.queue = arena.get<int64_t>("gp_queue", 2);
    a.rec = arena.get<uint32_t>("gp_rec", (size_t)std::max<int64_t>(numTiles * T, 1));
    a.tileV = arena.get<int32_t>("gp_tv", (size_t)numTiles + 1);
    a.tileQ = arena.get<int32_t>("gp_tq", (size_t)numTiles + 1);
    a.tileNA = arena.get<int32_t>("gp_tna", (size_t)numTiles + 1);
    a.cellMap = arena.get<uint32_t>("gp_map", (size_t)std::max<int64_t>(C, 1));
    int64_t* tvo = arena.get<int64_t>("gp_tvo", (size_t)numTiles + 1);
    int64_t* tqo = arena.get<int64_t>("gp_tqo", (size_t)numTiles + 1);
    a.tileVOff = tvo;
    a.tileQOff = tqo;
    // look-back words of the two scans of the tile counts, cleared by classify (a captured launch
    // replays its epoch, so this part goes without)
    const int64_t words = scanTiles(numTiles + 1);
    a.lb = arena.get<unsigned long long>("gp_lb", 2 * (size_t)words);
    a.lbWords = 2 * words;
    // totals straight into pinned host memory: [1] V, [2] Q
    int64_t* pd = pinDev();
    expectTotals();
    tuneEvent(0);
    // 512 tiles: the blocks' tickets, on one line and about 14 ns each, then cost what the launch
    // of a scan does (64^3 blobs, 135 tiles: 218 us an extraction with the scan, 205 without; 16^3 110 and 100)
    const bool own = numTiles > 0 && numTiles <= kTotalsTiles && !gridPassIsQueue(shape);
    if (own) {
        const bool fresh = arena.capacity<unsigned long long>("gp_ticket") == 0;
        a.ticket = arena.get<unsigned long long>("gp_ticket", 1);
        if (fresh) zero(a.ticket, sizeof(unsigned long long));
        a.sumV = tvo;
        a.sumQ = tqo;
        a.totalV = pd + 1;
        a.totalQ = pd + 2;
        a.stampTotals = stamp(ST_TOTALS);
    }
    launchGridClassify(shape, a, stream);
    if (own) {
        // by the last block
    } else if (numTiles > 0) {
        const ScanJob jobs[2] = {{a.tileV, tvo, numTiles + 1, pd + 1, a.lb}, {a.tileQ, tqo, numTiles + 1, pd + 2, a.lb + words}};
        scanExclusiveI32(jobs, 2, 0, stream, lookbackDiag(), nullptr, stamp(ST_TOTALS));
    } else {
        zero(pd + 1, 2 * sizeof(int64_t));
    }
    tuneEvent(1);
}

// the rest: read the totals back, size the outputs, emit quads and dual vertices
void Pipeline::gridPassBack(std::vector<ProblemDev>& problems, int64_t C, int shape, bool surfIter, bool recordAdjoint) {
    GridPassArgs& a = ga_;
    int64_t* h = pinHost();
    finishPrepare(true, [&] { gridPassFront(problems, C, shape, surfIter, nullptr); });
    if (!totalsWritten()) throw HipError("grid pass totals missing", -4);
    V = h[1];
    Q = h[2];
    emitArgs(a, C, recordAdjoint);
    gpVOff_ = a.tileVOff;
    gpQOff_ = a.tileQOff;
    gpLast_ = a.numTiles;
    tuneEvent(2);
    launchGridEmit(shape, a, stream);
    tuneEvent(3);
    dmcV = V;
    dmcQ = Q;
}

int32_t* Pipeline::pid() { return nProblems > 1 ? arena.ptr<int32_t>("pid") : nullptr; }

// HalfedgeMesh::initialize from the grid pass's output: outgoing lists (lengths and ranks from
// the vertices' contours), then every halfedge from its bucket
void Pipeline::halfedgeInitialize() {
    H = 4 * Q;
    F = Q;
    int32_t* face_he = arena.get<int32_t>("face_he", (size_t)F);
    uint32_t* fattr = arena.get<uint32_t>("fattr", (size_t)F);
    // (cleared flags, list lengths and valence come from the grid pass's vertex kernel)
    uint32_t* vflags = arena.ptr<uint32_t>("vflags");
    const int32_t* cnt = arena.ptr<int32_t>("out_cnt");
    const int4* quads = arena.ptr<int4>("quads");
    uint32_t* qattr = arena.ptr<uint32_t>("qattr");
    // the vertex -> halfedge array is derived from these quads when it is copied out
    vertHeV = V;
    vertHeQ = Q;
    // the list lengths (out-degrees) come from the grid pass's vertex kernel, the ranks from the
    // corner vertices' contours: no counting atomics
    int64_t* off = arena.get<int64_t>("out_off", (size_t)V + 1);
    scan({ScanJob{cnt, off, V + 1, nullptr, nullptr}}, stamp(ST_INIT));
    int32_t* out = arena.get<int32_t>("out_list", (size_t)std::max<int64_t>(H, 1));
    int32_t* twin = arena.get<int32_t>("twin", (size_t)std::max<int64_t>(H, 1));
    uint32_t* bpack = arena.get<uint32_t>("bpack", (size_t)std::max<int64_t>(H, 1));
    launchQuadLists(quads, qattr, Q, V, arena.ptr<int32_t>("gp_vcell"), arena.ptr<uint16_t>("gp_vct"), pid(), probsDev, off, out, twin, bpack, face_he,
                    fattr,
                    counters() + A_INVALID, pinDev() + kPinInvalid, stream);
    if (!chain.empty()) {
        if (H > 0)
            kBucketsAll<<<gridFor(H), kBlock, 0, stream>>>(quads, H, off, out, twin, bpack, vflags, fattr, qattr, arena.ptr<int32_t>("valence"),
                                                           chain.size() > 1 ? arena.ptr<int32_t>("bdin") : nullptr, counters());
    } else {
        // no simplification reads ids and twins only: the records at once
        int4* he = arena.get<int4>("he", (size_t)std::max<int64_t>(H, 1));
        int32_t* bsize = arena.get<int32_t>("bsize", (size_t)std::max<int64_t>(H, 1));
        int32_t* brank = arena.get<int32_t>("brank", (size_t)std::max<int64_t>(H, 1));
        if (H > 0)
            kBuildHalfedges<<<gridFor(H), kBlock, 0, stream>>>(quads, H, off, out, twin, bpack, he, bsize, brank, vflags, fattr, nmSlotParts(), counters());
    }
    listsV = V;
    splitTouched = false;
    canonTracked = false;
}

void Pipeline::checkValid(const char* what) {
    const int64_t bad = readI64(counters() + A_INVALID);
    if (bad) throw HipError(std::string("inconsistent mesh after ") + what + " (" + std::to_string(bad) + " bad ids)", -4);
}

// refreshHashTable (HalfedgeMesh.cu:1063-1100) after a split step: only the halfedges
// whose bucket can have changed (both endpoints in dirty_v, or appended), which
// kDirtyRecords lists, are re-bucketed; the others keep their sizes and ranks (same
// members, same keys), and the flags are rebuilt from all sizes.  Vm, Hm, Fm bound the new sizes,
// which the host learns here; splitStep cleared the arrays that are counted into.
void Pipeline::refreshHashTable(size_t Vm, size_t Hm, size_t Fm) {
    const int4* he = arena.ptr<int4>("he");
    const int32_t* face_he = arena.ptr<int32_t>("face_he");
    uint32_t* fattr = arena.ptr<uint32_t>("fattr");
    int32_t* degM = arena.ptr<int32_t>("degM");
    int32_t* dlist = arena.ptr<int32_t>("dirty_list");
    const int lanePer = recordsPerLane(H);
    const int64_t per = (int64_t)kBlock * lanePer;
    DirtyArgs a{};
    a.he = he;
    a.oldH = H;
    a.oldF = F;
    a.oldV = V;
    a.quads = arena.ptr<int4>("quads");
    a.Q = Q;
    a.canon = canonFlags();
    a.dirtyV = arena.ptr<uint8_t>("dirty_v");
    a.dlist = dlist;
    a.quadBlocks = (4 * Q + per - 1) / per;
    a.recordBlocks = ((int64_t)Hm - 4 * Q + per - 1) / per;
    a.face_he = face_he;
    a.fattr = fattr;
    a.ctr = counters();
    const unsigned blocks = (unsigned)(a.quadBlocks + a.recordBlocks) + gridFor(((int64_t)Fm + 3) / 4);
    if (lanePer == 4) kDirtyRecords<4><<<blocks, kBlock, 0, stream>>>(a);
    else kDirtyRecords<16><<<blocks, kBlock, 0, stream>>>(a);
    const int64_t* c = readCounters();
    if (c[A_INVALID]) throw HipError("inconsistent mesh after splitting (" + std::to_string(c[A_INVALID]) + " bad ids)", -4);
    V += c[A_ADD];
    H += c[A_ADD + 1];
    F += c[A_ADD + 2];
    const int64_t n = c[A_DIRTY];
    if (n < 0 || n > H || V > (int64_t)Vm || H > (int64_t)Hm || F > (int64_t)Fm)
        throw HipError("inconsistent mesh after splitting (dirty list of " + std::to_string(n) + ")", -4);
    int32_t* bsize = arena.ptr<int32_t>("bsize");
    int32_t* brank = arena.ptr<int32_t>("brank");
    if (n > 0) {
        int32_t* lm = arena.get<int32_t>("bl_m", (size_t)n);
        int2* lent = arena.get<int2>("bl_entry", (size_t)n);
        int32_t* lrank = arena.get<int32_t>("bl_rank", (size_t)n);
        int64_t* offM = arena.get<int64_t>("offM", (size_t)V + 1);
        int2* A = arena.get<int2>("listA", (size_t)n);
        kDirtyKeys<<<gridFor(n), kBlock, 0, stream>>>(he, H, face_he, canonFlags(), dlist, n, degM, lm, lent, lrank, counters());
        scan(degM, offM, V + 1);
        kPlaceEntries<<<gridFor(n), kBlock, 0, stream>>>(lm, lent, lrank, n, offM, A);
        kBuckets<<<gridFor(n), kBlock, 0, stream>>>(dlist, lm, lent, n, offM, A, bsize, brank);
    }
    if (H > 0)
        kFlagsFromBuckets<<<gridFor((H + 3) / 4), kBlock, 0, stream>>>(he, H, bsize, brank, arena.ptr<uint32_t>("vflags"), fattr, nmSlotParts());
    refreshUnchecked = true;  // kDirtyKeys' face-walk check is read back with the next NM-face count
}

// ---- simplifications
void Pipeline::setChain(bool colour, bool old, bool p3333) {
    chain.clear();
    if (colour) chain.push_back(S_COLOUR);
    if (old) chain.push_back(S_OLD);
    if (p3333) chain.push_back(S_3333);
}

// The chain: every step but the last removes and relabels in place (the ids stay the
// initialize's), the last compacts.  All of it is launched at once (see chainHeld) and waited for
// once, at the compaction's totals; a step whose merges need the region rebuild (none on smooth
// or noisy fields of the benchmarks) costs one more round from there on.  Waiting after the
// initialize's check and after every step instead: 337 us for the 64^3 blobs, 258 us now.
void Pipeline::simplify() {
    if (V == 0 || Q == 0 || chain.empty()) return;
    int64_t* h = pinHost();
    h[kPinFallback] = h[kPinFallback + 1] = 0;
    int from = 0;
    bool ended = false;  // step `from` has only its end left
    while (true) {
        launchChain(from, ended);
        const volatile int64_t* hv = h;  // where the totals are written, no kernel before them was held
        await([&] { return totalsWritten() || hv[kPinInvalid] || hv[kPinFallback] || hv[kPinFallback + 1]; });
        if (!totalsWritten()) MDMC_HIP(hipStreamSynchronize(stream));
        if (h[kPinInvalid]) checkValid("quad vertex ids");
        int s = 0;
        while (s < 2 && !h[kPinFallback + s]) ++s;
        if (s == 2) break;
        if (s + 1 >= (int)chain.size()) throw HipError("inconsistent simplification step", -4);
        h[kPinFallback + s] = 0;
        rebuildRegion();
        zero(counters() + A_FALLBACK + s, sizeof(int64_t));
        from = s;
        ended = true;
    }
    finishChain();
}

void Pipeline::launchChain(int from, bool ended) {
    const int4* cquads = arena.ptr<int4>("quads");
    int4* quads = arena.ptr<int4>("quads");
    uint32_t* qattr = arena.ptr<uint32_t>("qattr");
    uint32_t* fattr = arena.ptr<uint32_t>("fattr");
    int32_t* twin = arena.ptr<int32_t>("twin");
    int32_t* valence = arena.ptr<int32_t>("valence");
    int32_t* count = arena.ptr<int32_t>("vcount");
    uint8_t* vtype = arena.ptr<uint8_t>("vtype");
    int32_t* vtarget = arena.ptr<int32_t>("vtarget");
    const size_t nv = (size_t)V;
    for (int k = from; k < (int)chain.size(); ++k) {
        const bool last = k + 1 == (int)chain.size();
        if (!(ended && k == from)) {
            int64_t* st = k == 0 ? stamp(ST_SIMPLIFY) : nullptr;
            if (chain[k] == S_3333) {
                kMark3333<<<gridFor(F), kBlock, 0, stream>>>(cquads, twin, fattr, F, valence, vtype, vtarget, k, counters(), st);
            } else {
                const bool colour = chain[k] == S_COLOUR;
                if (colour) kMark3x3y<<<gridFor(Q), kBlock, 0, stream>>>(cquads, qattr, Q, valence, k, counters(), st);
                else kCount3x3yOld<<<gridFor(Q), kBlock, 0, stream>>>(cquads, qattr, Q, valence, count, k, counters(), st);
                kMerge3x3y<<<gridFor(Q), kBlock, 0, stream>>>(cquads, qattr, Q, twin, valence, count, arena.ptr<float>("pos"), arena.ptr<float>("nrm"), vtype,
                                                              vtarget, colour ? 1 : 0, last ? 0 : 1, k, counters());
            }
            if (!last) {
                // (P3333 ends a chain, so a deferred step is a P3X3Y one: it drops single vertices)
                int32_t* outdeg = arena.ptr<int32_t>("outdeg");
                int2* zslot = arena.get<int2>("zslot", nv);
                kLocalMerge<<<sparseBlocks(Q), kBlock, 0, stream>>>(quads, qattr, fattr, Q, valence, vtype, vtarget, twin, arena.ptr<uint32_t>("bpack"), outdeg,
                                                               zslot, V, arena.ptr<uint8_t>("touched"), localMerges ? 1 : 0, k, counters());
                kDropVertices<<<sparseBlocks(V), kBlock, 0, stream>>>(vtype, vtarget, V, 3, quads, H, arena.ptr<int64_t>("out_off"), arena.ptr<int32_t>("out_list"),
                                                                 arena.ptr<uint8_t>("vdead"), arena.ptr<int32_t>("src_head"),
                                                                 arena.get<int32_t>("src_next", nv), outdeg, zslot, k, counters());
            }
        }
        if (!last)
            kStepEnd<<<gridFor(V), kBlock, 0, stream>>>(arena.ptr<int32_t>("outdeg"), arena.ptr<int32_t>("bdin"), V, valence, vtype,
                                                        arena.ptr<uint8_t>("touched"), chain[k + 1] == S_OLD ? count : nullptr, k, counters());
    }
    launchCompaction();
}

// the merges the local update could not take: their region's buckets, flags and boundary
// counts recomputed
void Pipeline::rebuildRegion() {
    uint8_t* hdirty = arena.get<uint8_t>("hdirty", (size_t)H);
    uint8_t* aff = arena.get<uint8_t>("vaffected", (size_t)V);
    {
        FillBatch fb(*this);
        fb.add(hdirty, 0x00, (size_t)H);
        fb.add(aff, 0x00, (size_t)V);
    }
    const int4* quads = arena.ptr<int4>("quads");
    const int64_t* off = arena.ptr<int64_t>("out_off");
    const int32_t* out = arena.ptr<int32_t>("out_list");
    const int32_t* head = arena.ptr<int32_t>("src_head");
    const int32_t* next = arena.ptr<int32_t>("src_next");
    int32_t* twin = arena.ptr<int32_t>("twin");
    uint32_t* bpack = arena.ptr<uint32_t>("bpack");
    kMarkDirtyRegion<<<gridFor(V), kBlock, 0, stream>>>(arena.ptr<uint8_t>("touched"), V, quads, H, off, out, head, next, hdirty, aff);
    kRebuildDirty<<<gridFor(H), kBlock, 0, stream>>>(quads, H, hdirty, off, out, head, next, twin, bpack, arena.ptr<uint32_t>("fattr"),
                                                     arena.ptr<uint32_t>("qattr"), counters());
    kAffectedFlags<<<gridFor(V), kBlock, 0, stream>>>(aff, V, quads, H, off, out, head, next, twin, bpack, arena.ptr<uint32_t>("vflags"),
                                                      arena.ptr<int32_t>("bdin"));
}

void Pipeline::launchCompaction() {
    const int step = (int)chain.size() - 1;
    const bool p3333 = chain[step] == S_3333, chained = step > 0;
    const int dropType = p3333 ? 1 : 3;
    // the chain's last step: this step's removals and the dead elements of the earlier ones
    uint8_t* vtype = arena.ptr<uint8_t>("vtype");
    int32_t* vtarget = arena.ptr<int32_t>("vtarget");
    const uint32_t* attr = p3333 ? arena.ptr<uint32_t>("fattr") : arena.ptr<uint32_t>("qattr");
    // vertex and quad compaction, each one pass (look-back over tiles), with one read-back of
    // both totals; the outputs are sized for the inputs (at most as many are kept)
    // tiles of 4096 elements, or 1024 where that leaves the chip with fewer than a block per CU
    // (long look-back chains cost more than they give on large meshes: 0.11 / 0.41 -> 0.18 /
    // 0.48 ms at 17 M elements; 110 k vertices and quads: 38 -> 12 us)
    const int R = V + Q < (int64_t)1024 * 16 * kLbBlock ? 4 : 16;
    const int64_t tile = (int64_t)R * kLbBlock, tV = (V + tile - 1) / tile, tQ = (Q + tile - 1) / tile;
    int32_t* address = arena.get<int32_t>("vaddress", (size_t)std::max<int64_t>(V, 1));  // written for every vertex below
    // the compacted arrays go to the second buffers, which then swap with the primary ones;
    // both are sized for the grid pass's output so that later extractions of the same
    // workload reallocate neither
    const size_t capV = (size_t)std::max(V, dmcV), capQ = (size_t)std::max(Q, dmcQ);
    int32_t* npid = pid() ? arena.get<int32_t>("pid2", capV) : nullptr;
    int32_t* oldV = arena.get<int32_t>("oldV", (size_t)std::max<int64_t>(V, 1));
    arena.get<float>("pos2", 3 * capV);
    arena.get<float>("nrm2", 3 * capV);
    int4* quads = arena.ptr<int4>("quads");
    int4* nquads = arena.get<int4>("quads2", capQ);
    uint32_t* nattr = arena.get<uint32_t>("qattr2", capQ);
    int32_t* oldQ = arena.get<int32_t>("oldQ", (size_t)std::max<int64_t>(Q, 1));
    int32_t* qnew = arena.get<int32_t>("qnew", (size_t)std::max<int64_t>(Q, 1));
    // with every list still by current corner the removed quads' entries are counted per
    // corner; after deferred steps the lists are the initialize's and kOutCount checks entries
    int32_t* removedAt = chained ? nullptr : arena.get<int32_t>("removed_at", (size_t)std::max<int64_t>(V, 1));
    int32_t* outdeg = chained ? arena.ptr<int32_t>("outdeg") : nullptr;
    // source chains by old vertex id (kept from the deferred steps of the chain)
    int32_t* srcHead = arena.get<int32_t>("src_head", (size_t)std::max<int64_t>(V, 1));
    int32_t* srcNext = arena.get<int32_t>("src_next", (size_t)std::max<int64_t>(V, 1));
    uint8_t* touched = arena.get<uint8_t>("touched", (size_t)std::max<int64_t>(V, 1));
    uint32_t* vflags = arena.ptr<uint32_t>("vflags");
    int32_t* cnt = arena.get<int32_t>("out_cnt", (size_t)V + 1);
    int32_t* face_he = arena.ptr<int32_t>("face_he");
    uint32_t* nfattr = arena.get<uint32_t>("fattr2", capQ);
    // totals straight into pinned host memory: [1] V, [2] Q
    int64_t* h = pinHost();
    int64_t* pd = pinDev();
    expectTotals();
    {
        NumberArgs na{};
        na.vtype = vtype;
        na.V = V;
        na.dropType = dropType;
        na.vdead = chained ? arena.ptr<uint8_t>("vdead") : nullptr;
        na.pid = pid();
        na.npid = npid;
        na.address = address;
        na.oldV = oldV;
        na.touched = touched;
        na.vflags = vflags;
        na.cnt = cnt;
        na.srcHead = chained ? nullptr : srcHead;
        na.removedAt = removedAt;
        na.tV = tV;
        na.attr = attr;
        na.Q = Q;
        na.qnew = qnew;
        na.tQ = tQ;
        const Lookback lb = lookback(std::max<int64_t>(tV + tQ, 1));
        na.wordsV = lb.words;
        na.wordsQ = lb.words + tV;
        na.epochV = na.epochQ = lb.epoch;
        na.totalV = pd + 1;
        na.totalQ = pd + 2;
        na.directOut = lookbackDiag();
        na.step = step;
        na.ctr = counters();
        if (R == 4) kNumber<4><<<(unsigned)(tV + tQ), kLbBlock, 0, stream>>>(na);
        else kNumber<16><<<(unsigned)(tV + tQ), kLbBlock, 0, stream>>>(na);
    }
    if (Q > 0)
        kCompactQuads<<<gridFor(Q), kBlock, 0, stream>>>(quads, attr, Q, vtarget, address, p3333 ? 1 : 0, nquads, nattr, nfattr, face_he, oldQ, qnew,
                                                         removedAt, outdeg, touched, chained ? arena.ptr<uint8_t>("vdead") : nullptr, V, step, counters());
    if (failCompaction) launchFill(counters() + A_INVALID, 0x01, 1);  // as if a corner was out of range
}

// the compacted mesh's lists and records, once its sizes are known
void Pipeline::finishChain() {
    const int step = (int)chain.size() - 1;
    const bool p3333 = chain[step] == S_3333, chained = step > 0;
    const int dropType = p3333 ? 1 : 3;
    const int64_t* h = pinHost();
    const int64_t nV = h[1], nQ = h[2];
    if (nV < 0 || nV > V || nQ < 0 || nQ > Q) throw HipError("inconsistent compaction counts", -4);
    const size_t capQ = (size_t)std::max(Q, dmcQ);
    const uint8_t* vtype = arena.ptr<uint8_t>("vtype");
    const int32_t* vtarget = arena.ptr<int32_t>("vtarget");
    const int32_t* address = arena.ptr<int32_t>("vaddress");
    const int32_t* oldV = arena.ptr<int32_t>("oldV");
    const int4* nquads = arena.ptr<int4>("quads2");
    const int32_t* oldQ = arena.ptr<int32_t>("oldQ");
    const int32_t* qnew = arena.ptr<int32_t>("qnew");
    int32_t* removedAt = chained ? nullptr : arena.ptr<int32_t>("removed_at");
    int32_t* outdeg = chained ? arena.ptr<int32_t>("outdeg") : nullptr;
    int32_t* srcHead = arena.ptr<int32_t>("src_head");
    int32_t* srcNext = arena.ptr<int32_t>("src_next");
    uint8_t* touched = arena.ptr<uint8_t>("touched");
    uint32_t* vflags = arena.ptr<uint32_t>("vflags");
    int32_t* cnt = arena.ptr<int32_t>("out_cnt");
    uint32_t* nfattr = arena.ptr<uint32_t>("fattr2");
    // HalfedgeMesh::initialize of the compacted quads, from the previous build: the new
    // outgoing lists are the old ones of each new vertex's own and relabelled vertices,
    // renumbered; halfedges with untouched endpoints keep their bucket results
    const int64_t nH = 4 * nQ;
    if (V > 0) kSources<<<sparseBlocks(V), kBlock, 0, stream>>>(vtype, vtarget, address, V, dropType, touched, srcHead, srcNext, outdeg,
                                                              !(p3333 && localMerges));  // else kCompactQuads touched what there is to touch
    const int64_t* off = arena.ptr<int64_t>("out_off");
    const int32_t* out = arena.ptr<int32_t>("out_list");
    if (nV > 0) kOutCount<<<gridFor(nV), kBlock, 0, stream>>>(oldV, nV, off, removedAt, srcHead, srcNext, outdeg, cnt, arena.ptr<float>("pos"),
                                                           arena.ptr<float>("nrm"), arena.ptr<float>("pos2"), arena.ptr<float>("nrm2"));
    int64_t* off2 = arena.get<int64_t>("out_off2", (size_t)std::max<int64_t>(nV, dmcV) + 1);
    scan(cnt, off2, nV + 1);
    int32_t* out2 = arena.get<int32_t>("out_list2", 4 * capQ);
    if (nV > 0)
        kOutFill<<<gridFor(nV), kBlock, 0, stream>>>(oldV, nV, off, out, qnew, srcHead, srcNext, off2, out2, nH, counters());

    int4* he = arena.get<int4>("he", (size_t)std::max<int64_t>(nH, 1));
    int32_t* bsize = arena.get<int32_t>("bsize", (size_t)std::max<int64_t>(nH, 1));
    int32_t* brank = arena.get<int32_t>("brank", (size_t)std::max<int64_t>(nH, 1));
    // (the partial sums of slotted halfedges are clear since the extraction's start)
    if (nH > 0)
        kRemapRebuild<<<gridFor(nQ), kBlock, 0, stream>>>(nquads, nH, touched, oldQ, arena.ptr<int32_t>("twin"), H, arena.ptr<uint32_t>("bpack"),
                                                         qnew, off2, out2, he, bsize, brank, vflags, nfattr, nmSlotParts(), p3333 && localMerges, counters());
    arena.swap("pos", "pos2");
    arena.swap("nrm", "nrm2");
    arena.swap("quads", "quads2");
    arena.swap("qattr", "qattr2");
    arena.swap("fattr", "fattr2");
    if (pid()) arena.swap("pid", "pid2");
    arena.swap("out_off", "out_off2");
    arena.swap("out_list", "out_list2");
    V = nV;
    Q = nQ;
    H = nH;
    F = nQ;
    vertHeV = V;
    vertHeQ = Q;
    listsV = V;
    splitTouched = false;
    canonTracked = false;
}

void Pipeline::fixManifoldTwins(bool list) {
    listed = false;
    if (H == 0) return;
    FlagList fl{};
    if (list && F > 0) {
        const Lookback lb = lookback(scanTiles(F));
        fl = FlagList{arena.ptr<uint32_t>("fattr"), F, (uint32_t)QA_NM, arena.get<int32_t>("nmlist", (size_t)F), lb.words, lb.epoch, counters() + A_NM, lookbackDiag()};
        listed = true;
    }
    const unsigned fixBlocks = (unsigned)((H + kFixPer * kBlock - 1) / (kFixPer * kBlock));
    kFixTwins<<<fixBlocks + (listed ? (unsigned)scanTiles(F) : 0u), kBlock, 0, stream>>>(
        arena.ptr<int4>("he"), H, arena.ptr<int4>("quads"), arena.ptr<int64_t>("out_off"), arena.ptr<int32_t>("out_list"), arena.ptr<int32_t>("bsize"),
        arena.ptr<int32_t>("brank"), arena.ptr<float>("pos"), probsDev, pid(), fl, fixBlocks, counters(), stamp(ST_TWINS));
}

// ---- ManifoldSplitter::run, one problem and all that follows: the last stages are launched
// behind the face list without waiting for its length (see notYet), so a mesh with nothing to
// split waits once, at its end, instead of after the list, the fan detection and the statistics
// (about 12 us of idle GPU each); where faces are split, the launches that returned at once
// cost about 10 us an iteration.
void Pipeline::finishSingle(bool doSplit, int step, int maxIters, bool doDetect, int64_t st9[9]) {
    int iter = 0;
    bool again = doSplit;
    while (true) {
        const int32_t* nm = again ? listNM(iter == 0) : nullptr;
        const int guarded = again || iter == 0 ? kAwaitSplit : 0;
        if (doDetect) launchDetect(guarded);
        launchStats(guarded | kAwaitFans);
        const int64_t* h = waitStats();
        const int64_t n = guarded ? checkNM(h) : 0;
        if (n == 0) break;
        if (iter >= maxIters) {
            // still non-manifold after the allowed iterations (the reference loops until clean)
            extraAnomalies += 1;
            if (doDetect) launchDetect(0);
            launchStats(kAwaitFans);
            waitStats();
            break;
        }
        splitStep(step, n, nm);
        ++iter;
        splitIterations = iter;
        again = step >= 6;
    }
    const int64_t* h = pinHost() + kPinFinal;
    if (doDetect && h[A_NSLOW] != 0) {
        detectSlow(h[A_NSLOW], h[A_NSLOW_OFF]);
        launchStats(0);
        h = waitStats();
    }
    if (h[A_INVALID]) checkNM(h);
    refreshUnchecked = false;
    std::memcpy(st9, h + A_STATS, 9 * sizeof(int64_t));
}

// the splitter alone (a batch, whose regroup follows)
void Pipeline::split(int step, int maxIters) {
    int iter = 0;
    while (true) {
        const int32_t* nm = listNM(iter == 0);
        const int64_t n = checkNM(readCounters());
        if (n == 0) break;
        if (iter >= maxIters) {
            extraAnomalies += 1;
            break;
        }
        splitStep(step, n, nm);
        splitIterations = ++iter;
        if (step < 6) break;
    }
    if (refreshUnchecked) {
        refreshUnchecked = false;
        checkValid("splitting");
    }
}

// one iteration over the n listed faces
void Pipeline::splitStep(int step, int64_t n64, const int32_t* nm) {
    if (20 * n64 >= (int64_t)INT32_MAX / 2) throw HipError("working copy exceeds the int32 id range", -3);
    const int n = (int)n64;
    {
        SplitStep st{};
        WC& w = st.w;
        w.n = n;
        const int nv = 8 * n, nh = 20 * n, nf = 5 * n;
        st.step = step;
        st.vsize = step >= 1 ? nv : 4 * n;
        st.hsize = step >= 1 ? nh : 4 * n;
        st.fsize = step >= 1 ? nf : n;
        st.V0 = V;
        st.H0 = H;
        st.F0 = F;
        st.ctr = counters();
        w.pos = arena.get<float>("wc_pos", 3 * (size_t)nv);
        w.nrm = arena.get<float>("wc_nrm", 3 * (size_t)nv);
        w.pos0 = arena.get<float>("wc_pos0", 3 * (size_t)nv);
        w.nrm0 = arena.get<float>("wc_nrm0", 3 * (size_t)nv);
        w.vflags = arena.get<uint32_t>("wc_vflags", (size_t)nv);
        w.v_c2o = arena.get<int32_t>("wc_v_c2o", (size_t)nv);
        // the old -> copy maps and the last copies are all -1 between steps (kCopyBack), so only a
        // part no step has used yet is filled; a map the arena reallocates holds no -1s: its
        // capacity before the get tells
        static const char* mapName[4] = {"wc_v_o2c", "wc_h_o2c", "wc_f_o2c", "wc_v_last"};
        int32_t* maps[4];
        const int64_t need[4] = {V + nv, H + nh, F + nf, V + 1};
        for (int k = 0; k < 4; ++k) {
            wcMaps[k].cap = (int64_t)arena.capacity<int32_t>(mapName[k]);
            maps[k] = arena.get<int32_t>(mapName[k], (size_t)need[k]);
        }
        w.v_o2c = maps[0];
        w.h_o2c = maps[1];
        w.f_o2c = maps[2];
        w.v_last = maps[3];
        w.he = arena.get<int4>("wc_he", (size_t)nh);
        w.hflags = arena.get<uint32_t>("wc_hflags", (size_t)nh);
        w.h_c2o = arena.get<int32_t>("wc_h_c2o", (size_t)nh);
        w.f_first = arena.get<int32_t>("wc_f_first", (size_t)nf);
        w.f_attr = arena.get<uint32_t>("wc_f_attr", (size_t)nf);
        w.fflags = arena.get<uint32_t>("wc_fflags", (size_t)nf);
        w.f_c2o = arena.get<int32_t>("wc_f_c2o", (size_t)nf);
        w.pid = pid() ? arena.get<int32_t>("wc_pid", (size_t)nv) : nullptr;
        w.v_orig = arena.get<int32_t>("wc_v_orig", 4 * (size_t)n);
        w.h_orig = arena.get<int32_t>("wc_h_orig", 4 * (size_t)n);
        // (only copied halfedges collapse, so at most 4n of them)
        st.vrec = arena.get<int2>("vrec", 16 * (size_t)n);
        st.hrec = arena.get<int2>("hrec", 48 * (size_t)n);
        st.cntV = arena.get<int32_t>("mlv_cnt", (size_t)nv + 1);
        st.curV = arena.get<int32_t>("mlv_cur", (size_t)nv + 1);
        st.offV = arena.get<int64_t>("mlv_off", (size_t)nv + 2);
        st.idxV = arena.get<int32_t>("mlv_idx", 16 * (size_t)n);
        st.numV = arena.get<int32_t>("mlv_num", (size_t)nv);
        st.exV = arena.get<int32_t>("mlv_x", (size_t)nv);
        st.eyV = arena.get<int32_t>("mlv_y", (size_t)nv);
        st.cntH = arena.get<int32_t>("mlh_cnt", (size_t)nh + 1);
        st.curH = arena.get<int32_t>("mlh_cur", (size_t)nh + 1);
        st.offH = arena.get<int64_t>("mlh_off", (size_t)nh + 2);
        st.idxH = arena.get<int32_t>("mlh_idx", 48 * (size_t)n);
        st.numH = arena.get<int32_t>("mlh_num", (size_t)nh);
        st.exH = arena.get<int32_t>("mlh_x", (size_t)nh);
        st.eyH = arena.get<int32_t>("mlh_y", (size_t)nh);
        st.valid = arena.get<int32_t>("mvalid", (size_t)nh);
        st.firstWriter = arena.get<int32_t>("mfirst", 2 * (size_t)nh);
        st.newV = arena.get<int32_t>("cb_pred_v", (size_t)nv);
        st.newH = arena.get<int32_t>("cb_pred_h", (size_t)nh);
        st.newF = arena.get<int32_t>("cb_pred_f", (size_t)nf);
        st.addrV = arena.get<int64_t>("cb_addr_v", (size_t)nv + 1);
        st.addrH = arena.get<int64_t>("cb_addr_h", (size_t)nh + 1);
        st.addrF = arena.get<int64_t>("cb_addr_f", (size_t)nf + 1);
        // the mesh's arrays for the most the step can append
        const size_t Vm = (size_t)V + 4 * (size_t)n, Hm = (size_t)H + 16 * (size_t)n, Fm = (size_t)F + 4 * (size_t)n;
        float* pos = arena.grow<float>("pos", 3 * Vm, 3 * (size_t)V, stream);
        float* nrm = arena.grow<float>("nrm", 3 * Vm, 3 * (size_t)V, stream);
        int32_t* vp = pid() ? arena.grow<int32_t>("pid", Vm, (size_t)V, stream) : nullptr;
        int4* he = arena.grow<int4>("he", Hm, (size_t)H, stream);
        int32_t* face_he = arena.grow<int32_t>("face_he", Fm, (size_t)F, stream);
        uint32_t* fattr = arena.grow<uint32_t>("fattr", Fm, (size_t)F, stream);
        int32_t* bsize = arena.grow<int32_t>("bsize", Hm, (size_t)H, stream);
        int32_t* brank = arena.grow<int32_t>("brank", Hm, (size_t)H, stream);
        uint32_t* vflags = arena.grow<uint32_t>("vflags", Vm, 0, stream);  // rebuilt by the refresh
        uint8_t* dirtyV = arena.get<uint8_t>("dirty_v", Vm);
        int32_t* degM = arena.get<int32_t>("degM", Vm + 1);
        int32_t* dlist = arena.get<int32_t>("dirty_list", Hm);
        // layout flags: all set after the build, cleared for every record written back
        uint8_t* canon = canonTracked ? arena.grow<uint8_t>("he_canon", Hm, (size_t)H, stream) : arena.get<uint8_t>("he_canon", Hm);
        // every vertex any step touches (for the NM-vertex detection's use of the outgoing lists)
        uint8_t* touched = splitTouched ? arena.grow<uint8_t>("split_touched", Vm, (size_t)V, stream) : arena.get<uint8_t>("split_touched", Vm);
        {
            FillBatch fb(*this);
            if (splitIterations == 0 && listed) fb.stampAt(stamp(ST_SPLIT));
            for (int k = 0; k < 4; ++k) {
                WcMap& m = wcMaps[k];
                if (maps[k] != m.ptr || wcMapsDirty || m.cap < need[k]) {
                    fb.add(maps[k], 0xFF, (size_t)need[k] * sizeof(int32_t));
                    m.ptr = maps[k];
                    m.clean = need[k];
                } else if (need[k] > m.clean) {
                    fb.add(maps[k] + m.clean, 0xFF, (size_t)(need[k] - m.clean) * sizeof(int32_t));
                    m.clean = need[k];
                }
            }
            if (splitTouched) fb.add(touched + V, 0x00, Vm - (size_t)V);
            else fb.add(touched, 0x00, Vm);
            if (!canonTracked) fb.add(canon, 0x01, (size_t)H);
            fb.add(canon + H, 0x00, Hm - (size_t)H);
            fb.add(dirtyV, 0x00, Vm);
            fb.add(degM, 0x00, (Vm + 1) * sizeof(int32_t));
            fb.add(vflags, 0x00, Vm * sizeof(uint32_t));
            for (int k : {(int)A_DIRTY, (int)A_CONFLICT}) fb.add(counters() + k, 0x00, sizeof(int64_t));
        }
        splitTouched = canonTracked = true;
        wcMapsDirty = true;  // until kCopyBack has run

        kWcCopy<<<gridFor(4 * (int64_t)n), kBlock, 0, stream>>>(nm, n, he, face_he, fattr, pos, nrm, pid(), st);
        kWcUpdate<<<gridFor(4 * (int64_t)n), kBlock, 0, stream>>>(4 * n, bsize, brank, w, nmFoundParts());
        if (step >= 1) kSubdivide<<<gridFor(4 * (int64_t)n) + 1, kBlock, 0, stream>>>(nm, w, nmSlotParts(), nmFoundParts(), counters());
        else kNMSlotCheck<<<1, 64, 0, stream>>>(nmSlotParts(), nmFoundParts(), counters());
        const unsigned all = rangeBlocks(st.vsize, st.hsize, st.fsize);
        if (step >= 2) {
            const int64_t tiles = (4 * (int64_t)n + kCollapseRounds * kLbBlock - 1) / (kCollapseRounds * kLbBlock);
            const Lookback lb = lookback(tiles);
            kCollapse<<<(unsigned)tiles, kLbBlock, 0, stream>>>(st, lb.words, lb.epoch, lookbackDiag());
            scan({ScanJob{st.cntV, st.offV, st.vsize + 1, nullptr, nullptr}, ScanJob{st.cntH, st.offH, st.hsize + 1, nullptr, nullptr}});
            kRecScatter<<<std::min(gridFor(24 * (int64_t)n), 2048u), kBlock, 0, stream>>>(st);
            kRecApply<<<rangeBlocks(st.vsize, st.hsize, 0), kBlock, 0, stream>>>(st);
        }
        kMergePlan<<<all, kBlock, 0, stream>>>(st);
        if (step >= 4) {
            kMergeCheck<<<gridFor(st.hsize), kBlock, 0, stream>>>(w, st.hsize, st.numH, st.exH, st.eyH, st.firstWriter, counters());
            if (sequentialMerges) launchFill(counters() + A_CONFLICT, 0x01, 1);  // as if a conflict was found
        }
        kMergeApply<<<rangeBlocks(step >= 4 ? st.hsize : 0, st.vsize, 0), kBlock, 0, stream>>>(st, probsDev, st.numH, st.exH, st.eyH);
        // the new vertices, halfedges and faces of the working copy
        int64_t* add = counters() + A_ADD;
        scan({ScanJob{st.newV, st.addrV, st.vsize, add, nullptr}, ScanJob{st.newH, st.addrH, st.hsize, add + 1, nullptr},
              ScanJob{st.newF, st.addrF, st.fsize, add + 2, nullptr}});
        kCopyBackIds<<<all, kBlock, 0, stream>>>(st, pos, nrm, vp, canon);
        kCopyBack<<<all, kBlock, 0, stream>>>(st, nm, he, face_he, fattr, dirtyV, touched, nmSlotParts());
        wcMapsDirty = false;
        refreshHashTable(Vm, Hm, Fm);
    }
}

void Pipeline::launchDetect(int guarded) {
    if (H == 0 || V == 0) return;
    const int4* he = arena.ptr<int4>("he");
    uint32_t* vflags = arena.ptr<uint32_t>("vflags");
    uint8_t* slow = arena.get<uint8_t>("fan_slow", (size_t)V);
    const int64_t *off = arena.ptr<int64_t>("out_off");
    const int32_t* out = arena.ptr<int32_t>("out_list");
    const uint8_t* canon = canonFlags();  // kept since the splitter's first write-back, as its touched flags
    if (!canon) {
        kFanFast<true><<<gridFor(V), kBlock, 0, stream>>>(he, H, V, off, out, nullptr, nullptr, vflags, slow, nullptr, V, nullptr, counters(), guarded);
        return;
    }
    const uint8_t* touched = arena.ptr<uint8_t>("split_touched");
    int32_t* outdeg = arena.get<int32_t>("outdeg", (size_t)V);
    int32_t* rep = arena.get<int32_t>("outrep", (size_t)V);
    // (writes every vertex's out-degree)
    kOutFromLists<<<sparseBlocks(V), kBlock, 0, stream>>>(off, out, listsV, touched, canon, V, outdeg, rep, counters(), guarded);
    if (recordsPerLane(H) == 4) kOutDegreeMoved<4><<<gridFor((H + 3) / 4), kBlock, 0, stream>>>(he, H, V, listsV, touched, canon, outdeg, rep, counters(), guarded);
    else kOutDegreeMoved<16><<<gridFor((H + 15) / 16), kBlock, 0, stream>>>(he, H, V, listsV, touched, canon, outdeg, rep, counters(), guarded);
    kFanFast<false><<<gridFor(V), kBlock, 0, stream>>>(he, H, V, off, out, outdeg, rep, vflags, slow, touched, listsV, canon, counters(), guarded);
}

void Pipeline::detectNonManifoldVertices() {
    launchDetect(kAwaitValid);  // the walks follow the lists
    const int64_t* h = readCounters();
    if (h[A_INVALID]) checkNM(h);
    if (h[A_NSLOW]) detectSlow(h[A_NSLOW], h[A_NSLOW_OFF]);
}

// the vertices launchDetect left, over their outgoing lists (nSlowOff of them with lists that
// are not the build's)
void Pipeline::detectSlow(int64_t nSlow, int64_t nSlowOff) {
    const int4* he = arena.ptr<int4>("he");
    uint32_t* vflags = arena.ptr<uint32_t>("vflags");
    const uint8_t* slow = arena.ptr<uint8_t>("fan_slow");
    const bool fast = listsV == V && !splitTouched && !canonFlags();
    int32_t* outdeg = arena.get<int32_t>("outdeg", (size_t)V);
    int32_t* deg = arena.get<int32_t>("deg", (size_t)V + 1);
    kSlowDegree<<<gridFor(V + 1), kBlock, 0, stream>>>(slow, fast ? nullptr : outdeg, fast ? arena.ptr<int64_t>("out_off") : nullptr, V, deg);
    int64_t* off = arena.get<int64_t>("off", (size_t)V + 1);
    scan(deg, off, V + 1);
    int32_t* list = arena.get<int32_t>("list", (size_t)H);
    const bool copyLists = nSlowOff == 0;  // every slow vertex keeps the build's list
    if (copyLists) kCopySlowLists<<<gridFor(V), kBlock, 0, stream>>>(slow, V, arena.ptr<int64_t>("out_off"), arena.ptr<int32_t>("out_list"), off, list);
    else kFillLists<<<gridFor(H), kBlock, 0, stream>>>(he, H, V, slow, off, deg, list, counters());
    int32_t* key = arena.get<int32_t>("fankey", (size_t)H);
    kDetectFans<<<gridFor(V), kBlock, 0, stream>>>(he, V, slow, off, list, copyLists ? nullptr : deg, vflags, key, counters());
}

void Pipeline::launchStats(int guarded) {
    // Each block ends with up to ten atomics on one line, about 14 ns of them in a row, so a
    // small mesh takes a block per CU (one thread per halfedge and up to 4096 blocks: 33 us at
    // 150 k halfedges, 57 us at 1 M; now 10 and 21 us), a large one as many as the chip holds.
    const int64_t n = std::max<int64_t>(std::max(H, std::max(F, V)), 1);
    pinHost()[kPinDone] = 0;
    const int64_t blocks = std::min<int64_t>(gridFor(n, 4 * kBlock), std::max<int64_t>(256, std::min<int64_t>(n / (16 * kBlock), 2048)));
    kStats<<<(unsigned)blocks, kBlock, 0, stream>>>(
        arena.ptr<int4>("he"), H, arena.ptr<int32_t>("face_he"), F, arena.ptr<int32_t>("bsize"),
        arena.ptr<uint32_t>("vflags"), V, canonFlags(), counters(), pinDev() + kPinFinal, guarded);
}

// waits for the statistics; the counters they handed over.  A launch that failed leaves the word
// behind them unset.  (hipGetLastError behind the launch would also report an error that another call of this
// thread left long before, one that has nothing to do with the extraction.)
const int64_t* Pipeline::waitStats() {
    const volatile int64_t* done = pinHost() + kPinDone;
    await([&] { return *done != 0; });
    if (*done == 0) throw HipError("the extraction's last kernel did not run", (int)hipErrorLaunchFailure);
    return pinHost() + kPinFinal;
}

void Pipeline::finishEmpty() {
    launchStats(0);
    waitStats();
}

// Whether the mesh copy's kernel may store there: memory of the current device.  Another GPU's may not be
// mapped here, and host memory is the copy engine's anyway.
static bool ownMemory(const void* p) {
    hipPointerAttribute_t a{};
    int dev = 0;
    if (hipPointerGetAttributes(&a, p) != hipSuccess) {
        (void)hipGetLastError();  // memory that HIP does not know
        return false;
    }
    return a.type == hipMemoryTypeDevice && hipGetDevice(&dev) == hipSuccess && a.device == dev;
}

void Pipeline::copyOut(float* positions, float* normals, int32_t* halfedges, int32_t* face_halfedge, uint16_t* face_attr, uint8_t* vertex_flags,
                       int32_t* vertex_halfedge, bool dstDevice) {
    // one launch into buffers of this device; for others it makes the three derived arrays in
    // device memory and copies follow
    struct Array {
        int kind;
        const char* name;
        void* dst;
        int64_t n;
        size_t bytes;
        const char* made;  // where a derived array is made for a copy
    };
    const Array arrays[] = {
        {CM_POS, "pos", positions, 3 * V, 3 * (size_t)V * sizeof(float), nullptr},
        {CM_NRM, "nrm", normals, 3 * V, 3 * (size_t)V * sizeof(float), nullptr},
        {CM_HE, "he", halfedges, 4 * H, (size_t)H * sizeof(int4), nullptr},
        {CM_FACE, "face_he", face_halfedge, F, (size_t)F * sizeof(int32_t), nullptr},
        {batchVertHe ? CM_VHE_COPY : CM_VHE, batchVertHe ? "batch_vert_he" : "out_list", vertex_halfedge, V, (size_t)V * sizeof(int32_t),
         batchVertHe ? nullptr : "vert_he"},
        {CM_FATTR, "fattr", face_attr, F, (size_t)F * sizeof(uint16_t), "out_fattr"},
        {CM_VFLAGS, "vflags", vertex_flags, V, (size_t)V, "out_vflags"},
    };
    CopyMesh c{};
    const void* from[CM_COUNT] = {};  // what the copies read
    for (const Array& x : arrays) {
        if (!x.dst || x.n == 0) continue;
        void* dst = x.dst;
        if (!dstDevice || !ownMemory(x.dst)) {
            dst = x.made ? arena.get<char>(x.made, x.bytes) : nullptr;
            from[x.kind] = x.made ? dst : arena.ptr<char>(x.name);
        }
        c.src[x.kind] = arena.ptr<char>(x.name);
        c.dst[x.kind] = dst;
        c.n[x.kind] = dst ? x.n : 0;
    }
    unsigned blocks = 0;
    for (int j = 0; j < CM_COUNT; ++j) {
        const int64_t items = j == CM_VHE ? c.n[j] : (c.n[j] + 3) / 4;
        c.start[j] = blocks;
        blocks += (unsigned)((items + kCopyPer * kBlock - 1) / (kCopyPer * kBlock));
    }
    c.start[CM_COUNT] = blocks;
    c.off = arena.ptr<int64_t>("out_off");
    c.listsV = std::min(vertHeV, V);
    void* args[] = {&c};
    if (blocks > 0) MDMC_HIP(hipLaunchKernel((const void*)kCopyMesh, dim3(blocks), dim3(kBlock), args, 0, stream));
    for (const Array& x : arrays)
        if (from[x.kind]) MDMC_HIP(hipMemcpyAsync(x.dst, from[x.kind], x.bytes, dstDevice ? hipMemcpyDeviceToDevice : hipMemcpyDeviceToHost, stream));
    MDMC_HIP(hipStreamSynchronize(stream));
}

void Pipeline::renderVertices(float* out, bool dstDevice) {
    if (V == 0) return;
    const size_t bytes = 10 * (size_t)V * sizeof(float);
    float* dst = dstDevice ? out : arena.get<float>("out_render", 10 * (size_t)V);
    zero(dst, bytes);
    launchRenderVertices(arena.ptr<int4>("he"), H, arena.ptr<float>("pos"), arena.ptr<float>("nrm"), arena.ptr<uint32_t>("vflags"), dst, stream);
    if (!dstDevice) MDMC_HIP(hipMemcpyAsync(out, dst, bytes, hipMemcpyDeviceToHost, stream));
    MDMC_HIP(hipStreamSynchronize(stream));
}

void Pipeline::faceColours(uint8_t* out, bool dstDevice) {
    if (F == 0) return;
    uint8_t* a = arena.get<uint8_t>("fcol_a", (size_t)F);
    uint8_t* b = arena.get<uint8_t>("fcol_b", (size_t)F);
    uint8_t* res = nullptr;
    launchFaceColouring(arena.ptr<int4>("he"), arena.ptr<int32_t>("face_he"), arena.ptr<uint32_t>("fattr"), F, a, b, &res, stream);
    MDMC_HIP(hipMemcpyAsync(out, res, (size_t)F, dstDevice ? hipMemcpyDeviceToDevice : hipMemcpyDeviceToHost, stream));
    MDMC_HIP(hipStreamSynchronize(stream));
}

void Pipeline::triangulateMaxMin(uint32_t* tri, float* quality, bool dstDevice) {
    if (F == 0) return;
    uint32_t* t = dstDevice ? tri : arena.get<uint32_t>("out_tri", 6 * (size_t)F);
    float* q = quality ? (dstDevice ? quality : arena.get<float>("out_quality", 2 * (size_t)F)) : nullptr;
    launchTriangulateMaxMin(arena.ptr<int4>("he"), arena.ptr<int32_t>("face_he"), F, arena.ptr<float>("pos"), t, q, stream);
    if (!dstDevice) {
        MDMC_HIP(hipMemcpyAsync(tri, t, 6 * (size_t)F * sizeof(uint32_t), hipMemcpyDeviceToHost, stream));
        if (quality) MDMC_HIP(hipMemcpyAsync(quality, q, 2 * (size_t)F * sizeof(float), hipMemcpyDeviceToHost, stream));
    }
    MDMC_HIP(hipStreamSynchronize(stream));
}

void Pipeline::triangles(uint32_t* idx, bool dstDevice) {
    if (F == 0) return;
    if (dstDevice) {
        launchDmcTrianglesFromFaces(arena.ptr<int4>("he"), arena.ptr<int32_t>("face_he"), F, idx, stream);
    } else {
        uint32_t* tmp = arena.get<uint32_t>("out_tri", 6 * (size_t)F);
        launchDmcTrianglesFromFaces(arena.ptr<int4>("he"), arena.ptr<int32_t>("face_he"), F, tmp, stream);
        MDMC_HIP(hipMemcpyAsync(idx, tmp, 6 * (size_t)F * sizeof(uint32_t), hipMemcpyDeviceToHost, stream));
    }
    MDMC_HIP(hipStreamSynchronize(stream));
}

}  // namespace mdmc
