// mdmc_batch.hip -- the batched form: many (grid, iso) problems in one extraction.
//
// No reference counterpart (the reference extracts one grid per call).  The
// problems' meshes are disjoint, so every stage of the pipeline runs once over
// their union: the grid pass walks all problems' tiles in one launch, and the
// halfedge, simplification, twin-repair, split and detection kernels work on
// global ids as they do for one mesh.  Element ids stay grouped by problem
// except where the splitter appends; at the end a stable sort by problem makes
// every problem's vertices, halfedges and faces contiguous (CSR-packed), in the
// order a single extraction of that problem produces.
//
// Until the splitter runs, every array is ordered by problem (the grid pass emits the
// problems in order and every compaction is stable), so each problem's first vertex and quad
// follow from the grid pass's tile offsets and the compaction's numbering: a few loads per
// problem, no pass over the elements.  The splitter only appends, so each array is a sorted
// prefix plus a tail.  A split iteration appends its elements in the order of the faces it
// split, so the tail is a few runs that are each in problem order; run starts are found where
// a key falls, and each tail element's place follows from the runs' counts.  (A tail of more than
// kMaxRuns runs is sorted instead: least-significant-bit-first binary splits, per bit a
// prefix sum of the "bit is 0" flags and a scatter.)
#include <algorithm>
#include <vector>

#include "mdmc_device.h"
#include "mdmc_internal.h"
#include "mdmc_pipeline.h"

namespace mdmc {

namespace {

__device__ __forceinline__ int heO(const int4* he, int h) { return ((const int*)he)[4 * (int64_t)h]; }

__global__ void kIota(int32_t* __restrict__ p, int64_t n) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = (int32_t)i;
}

__global__ void kSplitFlags(const int32_t* __restrict__ perm, const int32_t* __restrict__ key, int64_t n, int bit, int32_t* __restrict__ zero) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) zero[i] = ((key[perm[i]] >> bit) & 1) ? 0 : 1;
}
__global__ void kSplitScatter(const int32_t* __restrict__ perm, const int32_t* __restrict__ zero, const int64_t* __restrict__ pre, int64_t n,
                              const int64_t* __restrict__ zeros, int32_t* __restrict__ out) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const int64_t p = pre[i];
    out[zero[i] ? p : *zeros + (i - p)] = perm[i];
}

// ---- where every element goes
constexpr int kMaxRuns = 32;
enum : int { RG_V = 0, RG_H = 1, RG_F = 2 };

// per problem b in [0, B]: its first vertex and quad as the grid pass numbered them (vOff / qOff at
// its first tile or row segment), and after the simplifications' compaction (the first kept one
// from there on: address / qnew, -1 for removed elements; null: nothing was compacted)
struct StartArgs {
    const ProblemDev* probs;
    int B, slab;
    const int64_t *vOff, *qOff;
    int64_t last;
    const int32_t *address, *qnew;
    int64_t dmcV, dmcQ, V, Q;
    int64_t *dmcStartV, *dmcStartQ, *startV, *startQ;
};
__global__ void kProblemStarts(StartArgs a) {
    const int b = blockIdx.x * blockDim.x + threadIdx.x;
    if (b > a.B) return;
    const int64_t i = b == a.B ? a.last : (a.slab ? a.probs[b].segBase : a.probs[b].tileBase);
    int64_t v = a.vOff[i], q = a.qOff[i];
    a.dmcStartV[b] = v;
    a.dmcStartQ[b] = q;
    if (a.address) {
        while (v < a.dmcV && a.address[v] < 0) ++v;
        v = v < a.dmcV ? a.address[v] : a.V;
        while (q < a.dmcQ && a.qnew[q] < 0) ++q;
        q = q < a.dmcQ ? a.qnew[q] : a.Q;
    }
    a.startV[b] = v;
    a.startQ[b] = q;
}

// the three arrays of the mesh, their prefixes [0, n0) and their ends
struct RegroupArgs {
    const int4* he;
    const int32_t* face_he;
    const int32_t* pid;
    int B;
    int64_t n0[3], n[3];
    int32_t* tailKey[3];  // [n - n0]: the tail elements' problems
    int32_t* tailDst[3];  // [n - n0]: their new ids
    int32_t *runCount, *runList;  // [3], [3 * kMaxRuns]: tail indices where a run starts (unordered)
    const int64_t *startV, *startQ;
    int64_t* shift;  // [3 * B]: new id - old id of a problem's prefix elements
};
__device__ __forceinline__ int64_t prefixStart(const RegroupArgs& r, int arr, int b) {
    return arr == RG_V ? r.startV[b] : (arr == RG_H ? 4 * r.startQ[b] : r.startQ[b]);
}
// one thread per tail element, over the three tails in turn
__device__ __forceinline__ bool tailElement(const RegroupArgs& r, int64_t t, int& arr, int64_t& j) {
    arr = 0;
    while (arr < 3 && t >= r.n[arr] - r.n0[arr]) t -= r.n[arr] - r.n0[arr], ++arr;
    j = t;
    return arr < 3;
}
__device__ __forceinline__ int tailProblem(const RegroupArgs& r, int arr, int64_t i) {
    if (arr == RG_V) return r.pid[i];
    return r.pid[heO(r.he, arr == RG_H ? (int)i : r.face_he[i])];
}
__global__ void kTailKeys(RegroupArgs r) {
    int arr;
    int64_t j;
    if (!tailElement(r, (int64_t)blockIdx.x * blockDim.x + threadIdx.x, arr, j)) return;
    const int k = tailProblem(r, arr, r.n0[arr] + j);
    r.tailKey[arr][j] = k;
    if (j > 0 && k < tailProblem(r, arr, r.n0[arr] + j - 1)) {
        const int c = atomicAdd(&r.runCount[arr], 1);
        if (c < kMaxRuns) r.runList[arr * kMaxRuns + c] = (int32_t)j;
    }
}
// the runs of the three tails: run s of array a covers tail elements [start[a][s], start[a][s + 1])
struct Runs {
    int count[3];
    int32_t start[3][kMaxRuns + 1];
    const int32_t* order[3];  // a sorted tail's permutation (one run), else null
};
__device__ __forceinline__ int runOf(const Runs& u, int arr, int64_t j) {
    int s = 0;
    while (s + 1 < u.count[arr] && j >= u.start[arr][s + 1]) ++s;
    return s;
}
// first[arr][s][b] = the first tail position of run s whose key is b or more (b in [0, B]): the
// element before every boundary writes it, so no count and no atomics
__device__ __forceinline__ int64_t firstAt(int arr, int s, int b, int B) { return ((int64_t)arr * kMaxRuns + s) * (B + 1) + b; }
__global__ void kRunStarts(RegroupArgs r, Runs u, int32_t* __restrict__ first, int* __restrict__ bad) {
    int arr;
    int64_t j;
    if (!tailElement(r, (int64_t)blockIdx.x * blockDim.x + threadIdx.x, arr, j)) return;
    const int s = runOf(u, arr, j), B = r.B;
    const int32_t* key = r.tailKey[arr];
    const int32_t* o = u.order[arr];
    const int k = key[o ? o[j] : j];
    const int kp = j > u.start[arr][s] ? key[o ? o[j - 1] : j - 1] : -1;
    if (k < kp || k < 0 || k >= B) {
        atomicOr(bad, 1);
        return;
    }
    for (int kk = kp + 1; kk <= k; ++kk) first[firstAt(arr, s, kk, B)] = (int32_t)j;
    if (j + 1 == u.start[arr][s + 1])
        for (int kk = k + 1; kk <= B; ++kk) first[firstAt(arr, s, kk, B)] = (int32_t)(j + 1);
}
// one block: the problems' new offsets (off[arr][b], [B + 1] each), the shift of their prefixes and,
// in place of first, the new id of a tail element less its tail position
__global__ void __launch_bounds__(1024) kOffsets(RegroupArgs r, Runs u, int32_t* __restrict__ first, int64_t* __restrict__ off) {
    __shared__ int64_t s_wave[16];
    const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6, B = r.B;
    for (int arr = 0; arr < 3; ++arr) {
        int64_t carry = 0;
        const int runs = r.n[arr] > r.n0[arr] ? u.count[arr] : 0;
        for (int b0 = 0; b0 < B; b0 += 1024) {
            const int b = b0 + tid;
            int64_t c = 0, pre = 0;
            if (b < B) {
                pre = prefixStart(r, arr, b + 1) - prefixStart(r, arr, b);
                c = pre;
                for (int s = 0; s < runs; ++s) c += first[firstAt(arr, s, b + 1, B)] - first[firstAt(arr, s, b, B)];
            }
            int64_t x = c;
#pragma unroll
            for (int d = 1; d < 64; d <<= 1) {
                const int64_t y = __shfl_up(x, d, 64);
                if (lane >= d) x += y;
            }
            if (lane == 63) s_wave[wid] = x;
            __syncthreads();
            int64_t add = 0, total = 0;
            for (int w = 0; w < 16; ++w) {
                if (w < wid) add += s_wave[w];
                total += s_wave[w];
            }
            const int64_t o = carry + add + x - c;
            // (every count of this chunk is read: first may be rewritten, b + 1's by its own thread
            // only after this barrier, the next chunk's b not before its own reads)
            int64_t tail = o + pre;
            int64_t place[kMaxRuns];
            for (int s = 0; s < runs; ++s) {
                if (b < B) {
                    const int64_t f = first[firstAt(arr, s, b, B)], g = first[firstAt(arr, s, b + 1, B)];
                    place[s] = tail - f;
                    tail += g - f;
                }
            }
            __syncthreads();
            if (b < B) {
                off[(int64_t)arr * (B + 1) + b] = o;
                r.shift[(int64_t)arr * B + b] = o - prefixStart(r, arr, b);
                for (int s = 0; s < runs; ++s) first[firstAt(arr, s, b, B)] = (int32_t)place[s];
            }
            carry += total;
        }
        if (tid == 0) off[(int64_t)arr * (B + 1) + B] = carry;
        __syncthreads();
    }
}
__global__ void kTailPlaces(RegroupArgs r, Runs u, const int32_t* __restrict__ place) {
    int arr;
    int64_t j;
    if (!tailElement(r, (int64_t)blockIdx.x * blockDim.x + threadIdx.x, arr, j)) return;
    const int s = runOf(u, arr, j);
    const int64_t e = u.order[arr] ? u.order[arr][j] : j;
    r.tailDst[arr][e] = (int32_t)(place[firstAt(arr, s, r.tailKey[arr][e], r.B)] + j);
}
// the new id of element x of array arr, which belongs to problem b
__device__ __forceinline__ int newId(const RegroupArgs& r, int arr, int b, int x) {
    return x < r.n0[arr] ? (int)(x + r.shift[(int64_t)arr * r.B + b]) : r.tailDst[arr][x - r.n0[arr]];
}
// the problem of prefix halfedge or face: the last b with startQ[b] <= q; the lanes of a wave
// mostly share one, found once for the wave's first lane
__device__ __forceinline__ int problemOfQuad(const int64_t* __restrict__ startQ, int B, int64_t q) {
    int lo = 0, hi = B;
    while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        if (startQ[mid] <= q) lo = mid;
        else hi = mid;
    }
    return lo;
}

// bucket / face / vertex counters of HalfedgeMesh.cu:1164-1239 per problem.  Elements are
// sorted by problem, so a wave usually holds one problem: it then adds its sums once.
// Per-problem statistics of one element kind over its regrouped range [0, n), where every
// problem's elements are contiguous and problems ascend: each block reduces a chunk
// of elements in LDS, one row per problem the chunk touches (up to kStatRows; the
// elements of further ones add to global memory directly), and adds every non-zero row
// entry once.  KIND 0: halfedges (slots 0-2: NM-4 / NM-3 / all edges, counted at the
// bucket's first member), 1: faces (slots 3-7: quads with k NM edges), 2: vertices (slot 8:
// non-manifold vertices).  out[9 * problem + slot].
constexpr int kStatRows = 32;
// elements per block: enough that what a block does once (its problem's search, the global additions)
// does not count, few enough that the chip stays full to the end; down to one per thread while that
// gives fewer than 1024 blocks (110 k vertices: 56 us in 27 blocks, 6 us in 432).  5.4 M vertices 350 us with
// 4096, 246 with 1024, 225 with 512, 222 with 256; as many faces 180, 116, 119 with 4096, 1024, 512; 21.6 M
// halfedges 242 with 2048, 243 with 1024, 292 with 512.
template <int KIND>
inline int64_t statChunk(int64_t n) { return std::min<int64_t>(KIND == RG_V ? 512 : 1024, std::max<int64_t>(kBlock, n / 1024 / kBlock * kBlock)); }

__device__ __forceinline__ void statAdd(unsigned* acc, unsigned long long* out, bool live, int p, int pbase, int slot, int accSlot, bool v) {
    // one LDS atomic per wave when all its live lanes share the problem
    const uint64_t alive = __ballot(live), on = __ballot(live && v);
    if (on == 0) return;
    const int pk = __shfl(p, __ffsll((unsigned long long)alive) - 1, 64);
    if (__ballot(live && p == pk) == alive) {
        if ((threadIdx.x & 63) == 0) {
            const int r = pk - pbase;
            const unsigned sum = (unsigned)__popcll(on);
            if (r >= 0 && r < kStatRows) atomicAdd(&acc[r * 5 + accSlot], sum);
            else atomicAdd(&out[(int64_t)pk * 9 + slot], (unsigned long long)sum);
        }
    } else if (live && v) {
        const int r = p - pbase;
        if (r >= 0 && r < kStatRows) atomicAdd(&acc[r * 5 + accSlot], 1u);
        else atomicAdd(&out[(int64_t)p * 9 + slot], 1ULL);
    }
}

// The regroup's pass over one kind of element, a block per chunk of them: moves every element
// to its place with its ids renumbered (MOVE; without a tail every place is the old one and
// nothing is moved) and takes the problems' statistics on the way.  Vertices also get their
// vertex -> halfedge value as the problem's own extraction leaves it: the highest
// initialize-time halfedge 4q+i starting at the vertex (the maximum of its outgoing list), q
// counted inside the problem; -1 where none; 0 for vertices the splitter added.
//
// Bound by HBM: the permutations, their inverses and a copy back of every array, keys for every
// element and an atomicMax per halfedge came to 3.1 ms of the 64-grid batch's 9.4 ms (5.4 M
// vertices); 0.58 ms now (0.93 with 4096 elements a block and every id's shift loaded by itself).
struct MoveArgs {
    RegroupArgs r;
    const float *pos, *nrm;
    const uint32_t *vflags, *fattr;
    const int32_t* bsize;
    const uint8_t* canon;
    const int64_t* listOff;  // the outgoing lists of the last initialize's vertices (the prefix)
    const int32_t* list;
    float *npos, *nnrm;
    uint32_t *nvflags, *nfattr;
    int32_t *npid, *nface_he, *vh;
    int4* nhe;
    unsigned long long* out;
    int* bad;
};
template <int KIND, bool MOVE>
__global__ void __launch_bounds__(kBlock) kRegroup(MoveArgs a, int64_t chunk) {
    constexpr int nslots = KIND == RG_H ? 3 : (KIND == RG_F ? 5 : 1);
    constexpr int base = KIND == RG_H ? 0 : (KIND == RG_F ? 3 : 8);
    const RegroupArgs& r = a.r;
    __shared__ unsigned acc[kStatRows * 5];
    const int64_t n = r.n[KIND], n0 = r.n0[KIND];
    const int64_t c0 = (int64_t)blockIdx.x * chunk;
    const int64_t c1 = c0 + chunk < n ? c0 + chunk : n;
    for (int t = threadIdx.x; t < kStatRows * 5; t += kBlock) acc[t] = 0;
    auto problemOf = [&](int64_t i) -> int {
        if (KIND == RG_V) return r.pid[i];
        if (i >= n0) return r.tailKey[KIND][i - n0];
        return problemOfQuad(r.startQ, r.B, KIND == RG_H ? i >> 2 : i);
    };
    const int pbase = problemOf(c0);
    // most blocks lie in one problem's prefix: no search per element
    const bool one = KIND != RG_V && c1 <= n0 && problemOf(c1 - 1) == pbase;
    // and most elements in the first one's problem, whose shifts are read once
    int64_t shift[3];
    for (int k = 0; k < 3; ++k) shift[k] = MOVE ? r.shift[(int64_t)k * r.B + pbase] : 0;
    auto idOf = [&](int arr, int p, int x) -> int { return p == pbase && x < r.n0[arr] ? (int)(x + shift[arr]) : newId(r, arr, p, x); };
    __syncthreads();
    // uniform trip count so that every lane takes part in the wave reductions
    for (int64_t i0 = c0; i0 < c1; i0 += kBlock) {
        const int64_t i = i0 + threadIdx.x;
        const bool live = i < c1;
        const int p = !live ? 0 : (one ? pbase : problemOf(i));
        const int64_t d = !live ? 0 : (MOVE ? idOf(KIND, p, (int)i) : i);
        if (KIND == RG_H) {
            int w = 0;
            if (live) {
                w = a.bsize[i];
                if (MOVE) {
                    const int4 e = r.he[i];
                    a.nhe[d] = make_int4(idOf(RG_V, p, e.x), idOf(RG_F, p, e.y), idOf(RG_H, p, e.z), e.w >= 0 ? idOf(RG_H, p, e.w) : e.w);
                }
            }
            const bool count = live && bucketFirst(w);
            const int nb = bucketSize(w);
            statAdd(acc, a.out, count, p, pbase, 0, 0, nb == 4);
            statAdd(acc, a.out, count, p, pbase, 1, 1, nb == 3);
            statAdd(acc, a.out, count, p, pbase, 2, 2, nb > 0);
        } else if (KIND == RG_F) {
            int k = 0;
            if (live) {
                const int h0 = a.r.face_he[i];
                // a face whose four records keep the build's layout: one load of their sizes
                const int q4 = h0 & ~3;
                if (q4 + 3 < r.n[RG_H] && (!a.canon || *reinterpret_cast<const uint32_t*>(a.canon + q4) == 0x01010101u)) {
                    const int4 s = reinterpret_cast<const int4*>(a.bsize)[q4 >> 2];
                    k = (bucketSize(s.x) > 2) + (bucketSize(s.y) > 2) + (bucketSize(s.z) > 2) + (bucketSize(s.w) > 2);
                } else {
                    int h = h0;
                    for (int j = 0; j < 4; ++j) {
                        if (bucketSize(a.bsize[h]) > 2) ++k;
                        h = ((const int*)r.he)[4 * (int64_t)h + 2];
                    }
                }
                if (MOVE) {
                    a.nface_he[d] = idOf(RG_H, p, h0);
                    a.nfattr[d] = a.fattr[i];
                }
            }
            for (int kk = 0; kk < 5; ++kk) statAdd(acc, a.out, live, p, pbase, 3 + kk, kk, k == kk);
        } else {
            uint32_t fl = 0;
            if (live) {
                fl = a.vflags[i];
                int best = 0;
                if (i < n0) {
                    if (p < 0 || p >= r.B || i < r.startV[p] || i >= r.startV[p + 1]) atomicOr(a.bad, 1);
                    best = -1;
                    const int64_t e = a.listOff[i + 1];
                    for (int64_t q = a.listOff[i]; q < e; q += 4) {
                        int h[4];
#pragma unroll
                        for (int k = 0; k < 4; ++k) h[k] = a.list[q + k < e ? q + k : e - 1];
                        best = max(max(best, max(h[0], h[1])), max(h[2], h[3]));
                    }
                    if (best >= 0) best -= (int)(4 * r.startQ[p]);
                }
                a.vh[d] = best;
                if (MOVE) {
                    for (int k = 0; k < 3; ++k) {
                        a.npos[3 * d + k] = a.pos[3 * i + k];
                        a.nnrm[3 * d + k] = a.nrm[3 * i + k];
                    }
                    a.nvflags[d] = fl;
                    a.npid[d] = p;
                }
            }
            statAdd(acc, a.out, live, p, pbase, 8, 0, (fl & VF_FANS) != 0);
        }
    }
    __syncthreads();
    for (int t = threadIdx.x; t < kStatRows * nslots; t += kBlock) {
        const int row = t / nslots, sl = t % nslots;
        const unsigned v = acc[row * 5 + sl];
        if (v) atomicAdd(&a.out[(int64_t)(pbase + row) * 9 + base + sl], (unsigned long long)v);
    }
}

template <int KIND, bool MOVE>
void launchRegroup(const MoveArgs& m, int64_t n, hipStream_t s) {
    const int64_t chunk = statChunk<KIND>(n);
    if (n > 0) kRegroup<KIND, MOVE><<<(unsigned)((n + chunk - 1) / chunk), kBlock, 0, s>>>(m, chunk);
}

}  // namespace

// stable permutation of [0, n) sorting key[] in [0, B)
int32_t* Pipeline::stableSortByKey(const int32_t* key, int64_t n, int B, const std::string& tag) {
    int32_t* a = arena.get<int32_t>(tag + "_perm", (size_t)std::max<int64_t>(n, 1));
    int32_t* b = arena.get<int32_t>(tag + "_perm2", (size_t)std::max<int64_t>(n, 1));
    int32_t* flag = arena.get<int32_t>("sort_flag", (size_t)std::max<int64_t>(n, 1));
    int64_t* pre = arena.get<int64_t>("sort_pre", (size_t)n + 1);
    int64_t* zeros = arena.get<int64_t>("sort_zeros", 1);
    if (n == 0) return a;
    kIota<<<gridFor(n), kBlock, 0, stream>>>(a, n);
    int bits = 0;
    while ((1 << bits) < B) ++bits;
    for (int bit = 0; bit < bits; ++bit) {
        kSplitFlags<<<gridFor(n), kBlock, 0, stream>>>(a, key, n, bit, flag);
        scan(flag, pre, n, zeros);
        kSplitScatter<<<gridFor(n), kBlock, 0, stream>>>(a, flag, pre, n, zeros, b);
        std::swap(a, b);
    }
    return a;
}

void Pipeline::regroupBatch(int B) {
    // results the host reads: dmcStart V / Q, offsets V / H / F ([B + 1] each), statistics [9B], bad
    const size_t nb = (size_t)B, words = 5 * (nb + 1) + 9 * nb + 1;
    int64_t* res = arena.get<int64_t>("batch_result", words);
    int64_t* off = res + 2 * (nb + 1);
    unsigned long long* st = (unsigned long long*)(res + 5 * (nb + 1));
    int* bad = (int*)(res + 5 * (nb + 1) + 9 * nb);
    int32_t* runCount = arena.get<int32_t>("rg_runs", 3 * (kMaxRuns + 1));
    {
        FillBatch fb(*this);
        fb.stampAt(stamp(ST_STATS));
        fb.add(st, 0x00, (9 * nb + 1) * sizeof(int64_t));
        fb.add(runCount, 0x00, 3 * sizeof(int32_t));
    }
    StartArgs sa{};
    sa.probs = probsDev;
    sa.B = B;
    sa.slab = gridPassIsSlab(lastShape) ? 1 : 0;
    sa.vOff = gpVOff_;
    sa.qOff = gpQOff_;
    sa.last = gpLast_;
    const bool compacted = !chain.empty() && dmcQ > 0;
    sa.address = compacted ? arena.ptr<int32_t>("vaddress") : nullptr;
    sa.qnew = compacted ? arena.ptr<int32_t>("qnew") : nullptr;
    sa.dmcV = dmcV;
    sa.dmcQ = dmcQ;
    sa.V = vertHeV;
    sa.Q = vertHeQ;
    sa.dmcStartV = res;
    sa.dmcStartQ = res + (nb + 1);
    sa.startV = arena.get<int64_t>("rg_start", 2 * (nb + 1));
    sa.startQ = sa.startV + (nb + 1);
    kProblemStarts<<<gridFor(B + 1), kBlock, 0, stream>>>(sa);

    MoveArgs m{};
    RegroupArgs& r = m.r;
    r.he = arena.ptr<int4>("he");
    r.face_he = arena.ptr<int32_t>("face_he");
    r.pid = pid();
    r.B = B;
    r.n0[RG_V] = std::min(vertHeV, V);
    r.n0[RG_H] = std::min(4 * vertHeQ, H);
    r.n0[RG_F] = std::min(vertHeQ, F);
    r.n[RG_V] = V;
    r.n[RG_H] = H;
    r.n[RG_F] = F;
    r.startV = sa.startV;
    r.startQ = sa.startQ;
    r.shift = arena.get<int64_t>("rg_shift", 3 * nb);
    r.runCount = runCount;
    r.runList = runCount + 3;
    Runs u{};
    int32_t* first = nullptr;
    int64_t tail = 0;
    for (int k = 0; k < 3; ++k) tail += r.n[k] - r.n0[k];
    if (tail > 0) {
        static const char* keyName[3] = {"rg_key_v", "rg_key_h", "rg_key_f"};
        static const char* dstName[3] = {"rg_dst_v", "rg_dst_h", "rg_dst_f"};
        for (int k = 0; k < 3; ++k) {
            r.tailKey[k] = arena.get<int32_t>(keyName[k], (size_t)(r.n[k] - r.n0[k]));
            r.tailDst[k] = arena.get<int32_t>(dstName[k], (size_t)(r.n[k] - r.n0[k]));
        }
        kTailKeys<<<gridFor(tail), kBlock, 0, stream>>>(r);
        int32_t* hr = (int32_t*)pinBatch(3 * (kMaxRuns + 1) * sizeof(int32_t));
        MDMC_HIP(hipMemcpyAsync(hr, runCount, 3 * (kMaxRuns + 1) * sizeof(int32_t), hipMemcpyDeviceToHost, stream));
        MDMC_HIP(hipStreamSynchronize(stream));
        for (int k = 0; k < 3; ++k) {
            const int32_t n = (int32_t)(r.n[k] - r.n0[k]);
            u.count[k] = 1;
            if (hr[k] < kMaxRuns) {
                u.count[k] = hr[k] + 1;
                int32_t* l = hr + 3 + k * kMaxRuns;
                std::sort(l, l + hr[k]);
                for (int s = 0; s < hr[k]; ++s) u.start[k][s + 1] = l[s];
            } else {
                static const char* tag[3] = {"rg_sort_v", "rg_sort_h", "rg_sort_f"};
                u.order[k] = stableSortByKey(r.tailKey[k], n, B, tag[k]);
            }
            u.start[k][u.count[k]] = n;
        }
        first = arena.get<int32_t>("rg_first", (size_t)3 * kMaxRuns * (nb + 1));
        kRunStarts<<<gridFor(tail), kBlock, 0, stream>>>(r, u, first, bad);
    }
    kOffsets<<<1, 1024, 0, stream>>>(r, u, first, off);
    if (tail > 0) kTailPlaces<<<gridFor(tail), kBlock, 0, stream>>>(r, u, first);
    m.pos = arena.ptr<float>("pos");
    m.nrm = arena.ptr<float>("nrm");
    m.vflags = arena.ptr<uint32_t>("vflags");
    m.fattr = arena.ptr<uint32_t>("fattr");
    m.bsize = arena.ptr<int32_t>("bsize");
    m.canon = canonFlags();
    m.listOff = arena.ptr<int64_t>("out_off");
    m.list = arena.ptr<int32_t>("out_list");
    m.out = st;
    m.bad = bad;
    const size_t nv = (size_t)std::max<int64_t>(V, 1), nh = (size_t)std::max<int64_t>(H, 1), nf = (size_t)std::max<int64_t>(F, 1);
    m.vh = arena.get<int32_t>("batch_vert_he", nv);
    if (tail > 0) {
        m.npos = arena.get<float>("pos2", 3 * nv);
        m.nnrm = arena.get<float>("nrm2", 3 * nv);
        m.nvflags = arena.get<uint32_t>("vflags2", nv);
        m.npid = arena.get<int32_t>("pid2", nv);
        m.nhe = arena.get<int4>("he2", nh);
        m.nface_he = arena.get<int32_t>("face_he2", nf);
        m.nfattr = arena.get<uint32_t>("fattr2", nf);
        launchRegroup<RG_H, true>(m, H, stream);
        launchRegroup<RG_F, true>(m, F, stream);
        launchRegroup<RG_V, true>(m, V, stream);
        for (const char* name : {"pos", "nrm", "vflags", "pid", "he", "face_he", "fattr"}) arena.swap(name, std::string(name) + "2");
    } else {
        launchRegroup<RG_H, false>(m, H, stream);
        launchRegroup<RG_F, false>(m, F, stream);
        launchRegroup<RG_V, false>(m, V, stream);
    }
    batchVertHe = true;
    launchStamp(stamp(ST_END));
    const int64_t* h = (const int64_t*)pinBatch(words * sizeof(int64_t));
    MDMC_HIP(hipMemcpyAsync((void*)h, res, words * sizeof(int64_t), hipMemcpyDeviceToHost, stream));
    const int64_t* ctr = readCounters();
    checkNM(ctr);
    if (*(const int*)(h + 5 * (nb + 1) + 9 * nb)) throw HipError("batched form: elements out of problem order", -4);
    batchDmc.resize(2 * nb);
    for (size_t b = 0; b < nb; ++b) {
        batchDmc[2 * b] = h[b + 1] - h[b];
        batchDmc[2 * b + 1] = h[(nb + 1) + b + 1] - h[(nb + 1) + b];
    }
    batchVOff.assign(h + 2 * (nb + 1), h + 3 * (nb + 1));
    batchHOff.assign(h + 3 * (nb + 1), h + 4 * (nb + 1));
    batchFOff.assign(h + 4 * (nb + 1), h + 5 * (nb + 1));
    batchStats.assign(h + 5 * (nb + 1), h + 5 * (nb + 1) + 9 * nb);
}

// pinned host memory for a batch's results
void* Pipeline::pinBatch(size_t bytes) {
    if (pinBatchCap_ < bytes) {
        if (pinBatch_) MDMC_HIP(hipHostFree(pinBatch_));
        pinBatch_ = nullptr;
        pinBatchCap_ = 0;
        MDMC_HIP(hipHostMalloc(&pinBatch_, bytes + bytes / 2, hipHostMallocDefault));
        pinBatchCap_ = bytes + bytes / 2;
    }
    return pinBatch_;
}

}  // namespace mdmc
