// Host-side internals shared by the C-ABI translation units: error
// reporting, growable device buffers, the context record and stage timing.
#pragma once
#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

#include <initializer_list>
#include <vector>

#include "sbg_internal.h"
#include "sbgpu.h"

namespace sbg {

// records the message for sbg_last_error() and returns `code`
int fail(int code, const char *fmt, ...);

#define HIP_TRY(expr)                                                                                     \
    do {                                                                                                  \
        hipError_t e_ = (expr);                                                                           \
        if (e_ != hipSuccess)                                                                             \
            return fail(SBG_ERR_HIP, "%s failed: %s (%s:%d)", #expr, hipGetErrorString(e_), __FILE__, __LINE__); \
    } while (0)

#define TRY(expr)              \
    do {                       \
        int r_ = (expr);       \
        if (r_ != SBG_OK)      \
            return r_;         \
    } while (0)

// growable device buffer (contents are not preserved on growth)
// page-locked host staging (hipHostMalloc), grown on demand: device-to-host
// copies into it are plain DMA on the stream and never block the host
struct PinnedBuf {
    uint8_t *p = nullptr;
    size_t cap = 0;
    int ensure(size_t n)
    {
        if (n <= cap && p)
            return SBG_OK;
        release();
        const size_t count = n ? n : 1;
        if (hipHostMalloc((void **)&p, count, hipHostMallocDefault) != hipSuccess) {
            p = nullptr;
            (void)hipGetLastError();
            return fail(SBG_ERR_OOM, "hipHostMalloc of %zu bytes failed", count);
        }
        cap = count;
        return SBG_OK;
    }
    void release()
    {
        if (p)
            (void)hipHostFree(p);
        p = nullptr;
        cap = 0;
    }
};

template <typename T>
struct DevBuf {
    T *p = nullptr;
    size_t cap = 0;
    int ensure(size_t n)
    {
        if (n <= cap && p)
            return SBG_OK;
        release();
        const size_t count = n ? n : 1;
        hipError_t e = hipMalloc((void **)&p, count * sizeof(T));
        if (e != hipSuccess) {
            p = nullptr;
            (void)hipGetLastError();
            return fail(SBG_ERR_OOM, "hipMalloc of %zu bytes failed: %s", count * sizeof(T), hipGetErrorString(e));
        }
        cap = count;
        return SBG_OK;
    }
    void release()
    {
        if (p)
            (void)hipFree(p);
        p = nullptr;
        cap = 0;
    }
};

constexpr int kMaxLevels = 256;
constexpr int kComponentsPinned = kMaxLevels + 7;  // sbg_components' repeated-half-edge flag
constexpr int kRayPinned = kMaxLevels + 8;      // 4 words per classification side
constexpr int kPinnedWords = kRayPinned + 8;
constexpr int kExpandGrid = 1024;
constexpr int kLevelsPerSync = 8;
// most breadth-first levels before the persistent depth-first kernel takes the
// frontier, its wave count, and the initial / largest spill region per wave
constexpr int kBfsLevels = 24;
constexpr int kDfsWaves = 512;
// the single-pair search expands levels of at most kTopMax node pairs in one
// workgroup before the depth-first stage
constexpr uint32_t kTopMax = 2048;
// most pairs of tree tiles whose boxes are tested all against all for the
// first frontier (larger trees start from their roots)
constexpr uint64_t kTilePairsMax = (uint64_t)1 << 26;
// longest run of one first triangle that the quick pair sorts order
constexpr uint32_t kSortRunMax = 64;
constexpr uint32_t kSpillInit = 2048, kSpillMax = 1u << 15;
// intersecting pairs and segments up to this size leave through page-locked
// staging (74,898 of them)
constexpr size_t kHitStage = (size_t)4 << 20;
// pair lists whose hit counts share one page-locked block
constexpr size_t kHitSlots = 1024;
// transfers of host arrays (sbg_copy.hip): host threads, the page-locked staging
// (two halves), the piece a thread takes at a time, what is worth a thread, what
// leaves the GPU between two waits, and the arrays of one call
constexpr int kCopyThreads = 8;
constexpr size_t kStageHalf = (size_t)16 << 20;
constexpr size_t kCopyPiece = (size_t)1 << 20;
constexpr size_t kCopyShare = (size_t)1 << 20;
constexpr size_t kOutRound = (size_t)4 << 20;
constexpr int kCopyParts = 4;
struct CopyPool;

}  // namespace sbg

using namespace sbg;

struct sbg_context_s {
    int device = 0;
    hipStream_t stream = nullptr;
    hipStream_t aux = nullptr;        // second stream (default priority): side 1 of sbg_classify_pair
    hipEvent_t auxReady = nullptr;    // orders the aux stream after the main one
    hipStream_t grids = nullptr;      // third stream (default priority): ray grids built at prepare time
    uint32_t *pinned = nullptr;  // host-visible counters (kPinnedWords): search, then two ray sides
    // transfers of host arrays (made on first use): page-locked staging, the
    // event after each half's last copy, the threads, and mesh uploads' stream
    hipStream_t uploads = nullptr;
    PinnedBuf staging;
    hipEvent_t stageDone[2] = {};
    CopyPool *copyPool = nullptr;
    DevBuf<uint2> front[2];
    DevBuf<uint2> spill;              // depth-first spill regions
    uint32_t spillPerWave = kSpillInit;
    bool depthFirst = true;           // false after the spill regions proved too small
    sbg_tuning tune = {kBfsLevels, kDfsWaves, 2, 1, 2, SBG_PRECISION_FP32_FILTERED, 64};
    DevBuf<uint32_t> counters;
    size_t frontCap = 0, candCap = 0;
    // candidates expected from the next search (the last count plus a margin):
    // the pair sort is queued over that many padded slots before the host
    // reads the count, and redone on the exact count if more were found
    size_t sortHint = 0;
    DevBuf<uint32_t> hist;
    DevBuf<GdStats> stats;
    // classification scratch, two sets (side 0 and side 1 of sbg_classify_pair;
    // single calls and other scratch uses take set 0)
    DevBuf<double> pts, pts2;
    DevBuf<uint8_t> flags, bits, votes, flags2, bits2, votes2;
    DevBuf<uint8_t> axes;  // sbg_classify_points' per-axis answers
    DevBuf<uint32_t> ovf, rayList, ovf2, rayList2;
    PinnedBuf votesHost, votesHost2;  // vote readbacks of the two sets
    PinnedBuf hitStage;               // sbg_pairs_hits: kHitStage bytes
    // page-locked words for the hit counts of the live pair lists, in blocks of
    // kHitSlots, and those that no list has
    std::vector<uint32_t *> hitBlocks, hitFree;
    DevBuf<unsigned long long> workCounts;  // sbg_bench_rays
    DevBuf<unsigned long long> ccKeys;      // sbg_half_edges: half-edge table
    DevBuf<uint32_t> ccOwners;
    DevBuf<uint64_t> ccList, ccListAlt;     // sbg_components: half-edges listed by hash
    DevBuf<uint32_t> ccValence, ccMate, ccParent, ccLabels;
    DevBuf<uint8_t> ccBlocked;
    DevBuf<uint32_t> heTris, heOpposite, heQueryOwner, heRepeat;  // sbg_half_edges
    DevBuf<unsigned long long> heQueries;
    DevBuf<double> rawA, rawB, rawSeg;
    DevBuf<uint8_t> rawStatus;
    DevBuf<double> adjXyz, adjAll, adjGradD, adjGall, adjVol;  // sbg_adjoint
    DevBuf<uint32_t> adjSrc, adjFaces;
    int refs = 1;  // the owner + every live mesh / pair list
    bool destroyed = false;
    bool timing = false;
    struct Ev {
        int stage;
        hipEvent_t a, b;
    };
    std::vector<Ev> events;
    double acc[SBG_STAGE_COUNT] = {0};
    // the buffers of the last destroyed pair list and meshes, handed to the
    // next ones
    struct sbg_pairs_s *sparePairs = nullptr;
    std::vector<struct sbg_mesh_s *> spareMeshes;
    // meshes prepared with their ray grid still to be queued on the grid
    // stream (queued after the next prepare of another mesh or at the next
    // pair search, so the host queues both prepares first)
    std::vector<struct sbg_mesh_s *> gridsPending;
    unsigned meshCount = 0;  // meshes made so far: even ones prepare on `stream`, odd ones on `aux`
};

namespace sbg {

// validates the handle and makes its device current
int use(sbg_context ctx);
// Meshes and pair lists hold a reference on their context, so destroying a
// context while they live only marks it; the last release frees it.
void context_release(sbg_context ctx);
void context_free(sbg_context ctx);

// Waits for a stream when a call leaves, whatever path it returns by: for work
// queued there that reads or writes the caller's arrays, or the staging that
// the next call fills.  release(): the call waits by itself from here on.
struct StreamJoin {
    hipStream_t s;
    explicit StreamJoin(hipStream_t stream) : s(stream) {}
    StreamJoin(const StreamJoin &) = delete;
    StreamJoin &operator=(const StreamJoin &) = delete;
    ~StreamJoin()
    {
        if (s)
            (void)hipStreamSynchronize(s);
    }
    void release() { s = nullptr; }
};

// HIP-event bracket of one stage (no-op unless timing is enabled)
struct Stage {
    sbg_context c;
    int stage;
    hipStream_t s;
    hipEvent_t a = nullptr;
    Stage(sbg_context ctx, int st, hipStream_t stream = nullptr) : c(ctx), stage(st), s(stream ? stream : ctx->stream)
    {
        if (c->timing && hipEventCreate(&a) == hipSuccess)
            (void)hipEventRecord(a, s);
        else
            a = nullptr;
    }
    ~Stage()
    {
        if (!a)
            return;
        hipEvent_t b = nullptr;
        if (hipEventCreate(&b) == hipSuccess) {
            (void)hipEventRecord(b, s);
            c->events.push_back({stage, a, b});
        } else {
            (void)hipEventDestroy(a);
        }
    }
};

int check_launch(const char *what);
int ceil_log2(size_t n);

// sbg_copy.hip
struct CopyPart {
    enum Kind { kBytes, kIndices32, kIndices64 };  // uploads: 64-bit ones are narrowed
    void *dev;                                     // on 8 bytes
    void *host;
    size_t bytes;  // on the GPU
    Kind kind = kBytes;
};
inline CopyPart part_in(void *dev, const void *host, size_t bytes) { return {dev, const_cast<void *>(host), bytes}; }
// Up to kCopyParts arrays; parts of 0 bytes are skipped.  copy_in leaves its
// copies queued on the context stream when it succeeds (the caller holds a
// StreamJoin until it waits); a failed copy_in, and copy_out always, have waited.
int copy_in(sbg_context c, std::initializer_list<CopyPart> parts);
int copy_out(sbg_context c, std::initializer_list<CopyPart> parts);
void copy_free(sbg_context c);
// a mesh's vertices and (narrowed) triangle indices; the largest index in *top
template <typename S>
int upload_mesh(sbg_context c, double *dv, uint32_t *dt, const double *xyz, size_t nx, const S *tris, size_t ni,
                uint64_t *top);
// Page-locked host memory (hipHostMalloc, sbg_host_alloc, or registered by the
// caller): a copy to or from it is plain DMA.  *device says
// whether kernels reach it at the same address.
bool page_locked(const void *p, bool *device);

}  // namespace sbg
