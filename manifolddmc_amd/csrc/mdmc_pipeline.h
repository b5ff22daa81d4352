// mdmc_pipeline.h -- the stage driver behind mdmc_extract.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <initializer_list>
#include <map>
#include <string>
#include <vector>

#include "mdmc_arena.h"
#include "mdmc_gridpass.h"
#include "mdmc_internal.h"

namespace mdmc {

// up to kFillSetMax byte fills for one launch (kFillMany): per range its pointer, the unaligned
// head and tail bytes, the 16-byte aligned body and the range's first block
constexpr int kFillSetMax = 12;
struct FillSet {
    uint8_t* p[kFillSetMax];
    size_t head[kFillSetMax], body[kFillSetMax], n[kFillSetMax];
    unsigned start[kFillSetMax];
    uint8_t byte[kFillSetMax];
    int count = 0;
    int64_t* stamp = nullptr;
};

class Pipeline {
   public:
    Pipeline();
    ~Pipeline();

    hipStream_t stream = nullptr;
    Arena arena;

    // live sizes of the resident mesh
    int64_t V = 0, Q = 0, H = 0, F = 0;
    int64_t dmcV = 0, dmcQ = 0;
    // vertices and quads of the last halfedge initialize (the vertex -> halfedge array)
    int64_t vertHeV = 0, vertHeQ = 0;
    int64_t splitIterations = 0;
    int64_t extraAnomalies = 0;

    // the simplifications of this extraction, in order (set before the grid pass, whose vertex
    // kernel starts their arrays)
    enum : int { S_COLOUR, S_OLD, S_3333 };
    std::vector<int> chain;
    void setChain(bool colour, bool old, bool p3333);
    // vertices the outgoing lists of the last halfedge build describe (-1: none), and
    // whether a split since then keeps the per-vertex "touched" flags
    int64_t listsV = -1;
    bool splitTouched = false;
    // per halfedge whether its record still has the build's layout (next = quadNext, face =
    // id / 4): tracked once a split step writes records back; before that every one has
    bool canonTracked = false;
    const uint8_t* canonFlags();
    // one extraction's padding / refinement: its grids' descriptors (host copy, and the device
    // copy of more than one), and the launch that also clears the counters and stores a
    // single problem (captured: for a graph)
    struct Prepare {
        std::vector<PrepareDesc> desc;
        PrepareDesc* dev = nullptr;
        int64_t rows = 0;
        int refinement = 0, pad = 0;
    } prep;
    void prepare(const std::vector<ProblemDev>& problems, bool captured);
    // waits for the front of the grid pass (totalsBehind: its totals, else all launched so far); where the plain copy met values that need the exact
    // blend, redoes the padding and calls again() (the front over it)
    template <class Again>
    void finishPrepare(bool totalsBehind, Again again);
    // the end of an extraction: with the statistics kernel's last block (one problem), or after a
    // batch's regroup, the counters, statistics and stage clocks go to pinned memory in one
    // read-back; the getters below read that copy
    void finishSingle(bool doSplit, int step, int maxIters, bool doDetect, int64_t st9[9]);
    void finishEmpty();
    void counterTotals(int64_t* anomalyCount, int64_t* mergeSeq, int64_t* lookbackDirect);
    // stage times in ms, from the clock stamps of the stages' first kernels: whole call, then the
    // seven stages of mdmc_stats in order, then the grid pass alone
    void stageTimes(double ms[9]);
    int64_t* stamp(int slot);
    void launchStamp(int64_t* at);
    // before any upload of a field: where the first stage's time then begins
    void stampUpload(bool uploads);
    // device word the single-pass scans and compactions count their direct-sum tiles in
    int64_t* lookbackDiag();

    // the grid pass over one or more (grid, iso) problems (their cellBase / tileBase and
    // cell counts are filled in); recordAdjoint keeps the cell -> vertex map ("adj_map") that
    // the adjoint reads with the vertex -> cell array ("gp_vcell") (one problem only)
    void dmc(std::vector<ProblemDev>& problems, bool surfIter, bool recordAdjoint = false);
    // the grid pass in parts, for the batched form's graph: problem geometry (no GPU work), the
    // tuned or fixed shape (GP_SHAPE_AUTO while a tuning is due), and the shape-determined front
    // (padding, classification, tile-count scans) captured once and replayed for later calls
    // with the same shapes and buffers (false: not replayable yet, run it eagerly), then the rest
    int64_t dmcSetup(std::vector<ProblemDev>& problems, bool recordAdjoint);
    int64_t assignTiles(std::vector<ProblemDev>& problems, int shape);
    void gridPassFront(std::vector<ProblemDev>& problems, int64_t C, int shape, bool surfIter, void* stagedProbs);
    void gridPassBack(std::vector<ProblemDev>& problems, int64_t C, int shape, bool surfIter, bool recordAdjoint);
    int shapeClass(int64_t C, bool surfIter) const;
    int resolveShape(int64_t C, bool surfIter);
    bool runFrontGraph(const std::vector<int64_t>& shapeSig, std::vector<ProblemDev>& problems, int64_t C, int shape, bool surfIter);
    void noteEagerFront(const std::vector<int64_t>& shapeSig) {
        fgLastEager_ = shapeSig;
        const std::vector<int64_t> b = frontBuffers();
        fgLastEager_.insert(fgLastEager_.end(), b.begin(), b.end());
    }
    void releaseGraphs();
    bool useGraphs = true;
    // P3X3Y merges of a deferred chain step with a plain neighbourhood update their twins
    // directly (else every merge's region is rebuilt)
    bool localMerges = true;
    // the splitter's merge phase always in the one-thread ascending pass (a verification switch)
    bool sequentialMerges = false;
    // a chain's compaction counts one quad as inconsistent (a verification switch)
    bool failCompaction = false;
    int64_t graphReplays = 0;
    int nProblems = 1;
    ProblemDev* probsDev = nullptr;
    // per vertex its problem (several problems), else nullptr
    int32_t* pid();

    // batched form (mdmc_batch.hip): the final regroup into contiguous per-problem ranges with
    // offsets, per-problem vertex -> halfedge values, DMC counts and statistics; ends the
    // extraction (one read-back of all of it and the counters)
    void regroupBatch(int B);
    std::vector<int64_t> batchDmc;                     // [2B]: vertices, quads
    std::vector<int64_t> batchVOff, batchHOff, batchFOff;  // [B + 1]
    std::vector<int64_t> batchStats;                   // [9B], as computeStats
    bool batchVertHe = false;
    void halfedgeInitialize();
    void simplify();
    // list: the list of the non-manifold faces with it (the split's first)
    void fixManifoldTwins(bool list);
    bool listed = false;
    void split(int step, int maxIters);
    void detectNonManifoldVertices();

    void copyOut(float* positions, float* normals, int32_t* halfedges, int32_t* face_halfedge, uint16_t* face_attr, uint8_t* vertex_flags,
                 int32_t* vertex_halfedge, bool dstDevice);
    void triangles(uint32_t* idx, bool dstDevice);
    void renderVertices(float* out, bool dstDevice);
    void faceColours(uint8_t* out, bool dstDevice);
    void triangulateMaxMin(uint32_t* tri, float* quality, bool dstDevice);

    int64_t readI64(const int64_t* dev);
    // mapped pinned host words for small read-backs: kernels and copies write them
    // directly, and the host polls for them (slots 0..kPinSlots-1)
    static constexpr int kPinSlots = 64;
    int64_t* pinHost();
    int64_t* pinDev();
    // host -> device copy of a small host array through pinned staging (region 0 or 1, so
    // that two uploads of one stage do not share a buffer); returns after queueing the copy
    void upload(void* dst, const void* src, size_t bytes, int region);
    // while tuning, the duration of a grid pass (classify + scan, then emit) from events on the
    // launch stream; the host read-back of the sizes between them is not counted
    void kernelTimes(double* msGridPass);
    hipEvent_t kev[4] = {nullptr, nullptr, nullptr, nullptr};
    bool tuning_ = false;
    void tuneEvent(int k) {
        if (tuning_) MDMC_HIP(hipEventRecord(kev[k], stream));
    }
    // grid-pass tile shape: GP_SHAPE_AUTO (autotuned per workload class) or a fixed shape;
    // lastShape is the one the last extraction used, tuneMs the last tuning's timings
    int tileShape = GP_SHAPE_AUTO;
    int lastShape = GP_SHAPE_DEFAULT;
    std::map<int, int> tuned;
    double tuneMs[GP_SHAPE_LAST + 1] = {};

   private:
    int64_t* pinH_ = nullptr;
    int64_t* pinD_ = nullptr;
    void* up_[2] = {nullptr, nullptr};
    hipEvent_t upEv_[2] = {nullptr, nullptr};
    size_t upCap_[2] = {0, 0};
    int64_t* counters();
    int64_t* nmSlotParts();
    int64_t* nmFoundParts();
    // exclusive prefix sums in one launch (words of the jobs are set here); total may be null
    void scan(std::initializer_list<ScanJob> jobs, int64_t* stampStart = nullptr, int64_t* stampEnd = nullptr);
    void scan(const int32_t* in, int64_t* out, int64_t n, int64_t* total = nullptr) { scan({ScanJob{in, out, n, total, nullptr}}); }
    // look-back words for one launch over `words` tiles: the launches of a stream run one after
    // the other, so all share one buffer, told apart by the epoch (cleared when the buffer is
    // new and before the 16-bit epochs repeat)
    struct Lookback {
        unsigned long long* words;
        uint32_t epoch;
    };
    Lookback lookback(int64_t words);
    uint32_t lbEpoch_ = 0;
    int64_t prepToken_ = 0;
    int clockKHz_ = 0;
    int32_t* listNM(bool first);
    int64_t checkNM(const int64_t* h);
    const int64_t* readCounters();
    void splitStep(int step, int64_t n64, const int32_t* nm);
    void launchDetect(int guarded);
    void detectSlow(int64_t nSlow, int64_t nSlowOff);
    void launchStats(int guarded);
    const int64_t* waitStats();
    template <class Ready>
    void await(Ready ready);
    void expectTotals();
    bool totalsWritten();
    void zero(void* p, size_t bytes);
    void launchFill(void* p, uint8_t byte, size_t bytes);
    // fills collected and launched together (at flush or at the end of the scope)
    class FillBatch {
       public:
        explicit FillBatch(Pipeline& p) : pl(p) {}
        ~FillBatch() { flush(); }
        void add(void* p, uint8_t byte, size_t bytes);
        void flush();
        void stampAt(int64_t* stamp) { fs.stamp = stamp; }

       private:
        Pipeline& pl;
        FillSet fs;
        unsigned blocks = 0;
    };
    // the splitter's old -> copy maps and last copies: -1 on [0, clean) between steps (each step resets the
    // entries it set); a map the arena reallocated, or one a failed step left dirty, is filled
    struct WcMap {
        void* ptr = nullptr;
        int64_t clean = 0, cap = 0;
    } wcMaps[4];
    bool wcMapsDirty = true;
    void gridPass(std::vector<ProblemDev>& problems, int64_t C, int shape, bool surfIter, bool recordAdjoint);
    void slabPass(std::vector<ProblemDev>& problems, int64_t C, int shape, bool surfIter, bool recordAdjoint);
    GridPassArgs ga_{};
    // the captured front of a batched extraction: the graph, the shapes / options / buffer
    // addresses it was captured with, its pinned descriptor staging, its kernel arguments
    struct FrontGraph {
        hipGraphExec_t exec = nullptr;
        std::vector<int64_t> sig;
        void* stage = nullptr;
        size_t stageCap = 0;
    } fg_;
    GridPassArgs fgArgs_{};
    std::vector<int64_t> fgLastEager_;
    std::vector<int64_t> frontBuffers();
    void refreshHashTable(size_t Vm, size_t Hm, size_t Fm);
    // a refresh ran whose face-walk check (the invalid-record counter) is not read back yet
    bool refreshUnchecked = false;
    void checkValid(const char* what);
    void emitArgs(GridPassArgs& a, int64_t C, bool recordAdjoint);
    void launchChain(int from, bool ended);
    void launchCompaction();
    void rebuildRegion();
    void finishChain();
    int32_t* stableSortByKey(const int32_t* key, int64_t n, int B, const std::string& tag);
    void* pinBatch(size_t bytes);
    void* pinBatch_ = nullptr;
    size_t pinBatchCap_ = 0;
    // the last grid pass's vertex / quad offsets by tile or row segment, and their last index
    const int64_t *gpVOff_ = nullptr, *gpQOff_ = nullptr;
    int64_t gpLast_ = 0;
};

}  // namespace mdmc
