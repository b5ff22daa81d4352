// mdmc_internal.h -- host-side declarations shared by the library's translation units.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <string>

namespace mdmc {

constexpr int kBlock = 256;

struct GridDev {
    const float* v;
    int nx, ny, nz;
    float ox, oy, oz;
    float dx, dy, dz;
};

// --- scans (mdmc_scan.hip): exclusive prefix of n int32 values into int64 offsets, the total
// through *total (device or mapped pinned host memory; may be null); up to kScanJobs arrays in
// one launch, each with scanTiles(n) look-back words of its own.  The words are either all zero
// (epoch 0) or hold nothing of this epoch.  The result is exact in every case; a tile whose
// look-back wait passed its spin limit summed its prefix directly and adds 1 to *directOut
// (device memory), a diagnostic only.
constexpr int kScanTile = 4096, kScanJobs = 3;
// at least one tile: an empty array's total is written too
__host__ __device__ inline int64_t scanTiles(int64_t n) { return n > 0 ? (n + kScanTile - 1) / kScanTile : 1; }
struct ScanJob {
    const int32_t* in;
    int64_t* out;
    int64_t n;
    int64_t* total;
    unsigned long long* words;
};
// stampStart / stampEnd (may be null): clock at the launch's start and the first job's end
void scanExclusiveI32(const ScanJob* jobs, int count, uint32_t epoch, hipStream_t s, int64_t* directOut, int64_t* stampStart = nullptr,
                      int64_t* stampEnd = nullptr);
// stream compaction in one pass: the i < n with (attr[i] & mask) != 0, ascending, into
// idx (capacity n); the count through *total
void compactFlagged(const uint32_t* attr, int64_t n, uint32_t mask, int32_t* idx, int64_t* total, unsigned long long* words, uint32_t epoch,
                    hipStream_t s, int64_t* directOut, int64_t* stamp);

// --- stage times: the first block of a stage's first kernel stores the GPU's constant-rate clock
// (null: no stamp).  Timing events instead cost about 5 us of idle GPU at every boundary.
__device__ __forceinline__ void stampClock(int64_t* stamp) {
    // the block first: the others then never wait for the pointer's load (kEmit at 512^3: 5%)
    if (blockIdx.x == 0 && blockIdx.y == 0 && threadIdx.x == 0 && stamp)
        __hip_atomic_store(stamp, (int64_t)wall_clock64(), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// slots: the start of each stage in order (padding, classification, halfedge initialize,
// simplifications, records + twin repair, split, detection, statistics), the end, then the grid
// pass's second part, the end of its first, the start of its last run
enum : int { ST_PAD = 0, ST_DMC, ST_INIT, ST_SIMPLIFY, ST_TWINS, ST_SPLIT, ST_DETECT, ST_STATS, ST_END, ST_EMIT, ST_TOTALS, ST_CLASSIFY, ST_COUNT };

inline unsigned gridFor(int64_t n, int block = kBlock) { return (unsigned)((n + block - 1) / block); }

// --- the reference's synthetic grids (mdmc_generate.hip): implicit surface sc (SurfaceCase
// numbering) at origin + index * delta, and the 4x4x3 edge case ec
void launchFillSurface(float* out, const int dims[3], int surfaceCase, const float origin[3], const float delta[3], hipStream_t s);
void launchFillEdgeCase(float* out, int edgeCase, hipStream_t s);

// --- face exports of OriginalDMC (mdmc_faces.hip): the 5-colouring of the faces' grid-edge
// colours (a, b: F bytes each; *result points at the one holding the colours), and the
// MaxMin-angle triangulation with per-triangle mean ratio (quality may be null)
void launchFaceColouring(const int4* he, const int32_t* face_he, const uint32_t* fattr, int64_t F, uint8_t* a, uint8_t* b, uint8_t** result,
                         hipStream_t s);
void launchTriangulateMaxMin(const int4* he, const int32_t* face_he, int64_t F, const float* pos, uint32_t* tri, float* quality, hipStream_t s);

// --- DMC grid pass (mdmc_dmc.hip)
// padding / refinement (refineGrid) of several grids in one launch: grid g reads in[inx*iny*inz]
// and writes out[onx*ony*onz] with the blocks from base on (prepareBlocks(dims) of them)
struct PrepareDesc {
    const float* in;
    float* out;
    int inx, iny, inz, onx, ony, onz;
    int64_t base;
};
// blocks of the padding / refinement pass over one processed grid of od points: one per row
int64_t prepareBlocks(const int od[3]);
void launchDmcTrianglesFromFaces(const int4* he, const int32_t* face_he, int64_t F, uint32_t* idx, hipStream_t s);
// positions copied from src to positions[3V] and the faces' vertex ids to quads[4F], in one launch
// (either output may be null); the launch's own status
hipError_t launchQuadIds(const int4* he, const int32_t* face_he, int64_t F, const float* src, int64_t V, float* positions, int64_t* quads, hipStream_t s);
// render vertices {position, normal, rgba by vertex flags} of every vertex with an outgoing
// halfedge into out[10 * V] (the caller zero-fills out first)
void launchRenderVertices(const int4* he, int64_t H, const float* pos, const float* nrm, const uint32_t* vflags, float* out, hipStream_t s);

}  // namespace mdmc
