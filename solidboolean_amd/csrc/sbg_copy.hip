// Host arrays to and from HBM.
//
// Callers hand over ordinary (pageable) memory.  The runtime pins or stages it on
// the calling thread, copy by copy, each with its own wait.  Here the arrays of a
// call move together: up to kCopyThreads host threads copy pieces of them into
// (out of) page-locked staging, and kernels on the context stream move the staged
// pieces over PCIe, so what follows on the stream needs no wait and first-touch
// page faults of a fresh output array are spread over the threads.  A copy kernel
// rather than the DMA engines: a DMA costs ~15 us to start and end, and pieces
// small enough to overlap (1 MB) would pay that each.
// Arrays that are page-locked already go straight by DMA.
//
// PCIe bounds it: 1 MB pieces arrive at 48 GB/s.  Measured, us per call before /
// after, all host arrays included: 65,536 triangle pairs (9.4 MB in, 3.2 MB out)
// 538 / 454; components of 1.3 M triangles (1.3 MB in, 5.3 MB out) 874 / 756; the
// adjoint of 20,480 faces 460 / 323; two 272 k-triangle meshes created, searched and
// classified 1308 / 1109.  One to eight threads and pieces of 0.5 to 2 MB are within
// 10 % of each other below 10 MB; two 10 MB meshes take 1517 us on two threads.
#include <algorithm>
#include <atomic>
#include <condition_variable>
#include <cstring>
#include <mutex>
#include <new>
#include <thread>

#include "sbg_host.h"

namespace sbg {

// The context's copy threads, started when first wanted and joined with the
// context: run(pieces, wanted, f, arg) calls f(arg, 0) .. f(arg, pieces - 1) on up to
// `wanted` threads, the caller being one, and returns when all are done.
struct CopyPool {
    using Job = void (*)(void *arg, int piece);
    std::mutex m;
    std::condition_variable wake, done;
    std::vector<std::thread> threads;
    Job job = nullptr;
    void *arg = nullptr;
    int pieces = 0;
    std::atomic<int> next{0};
    int seats = 0;  // threads that may still join the job
    int busy = 0;   // threads in it
    bool stop = false;

    void take()
    {
        for (int k; (k = next.fetch_add(1, std::memory_order_relaxed)) < pieces;)
            job(arg, k);
    }
    void serve()
    {
        std::unique_lock<std::mutex> lock(m);
        for (;;) {
            wake.wait(lock, [this] { return stop || seats > 0; });
            if (stop)
                return;
            --seats;
            ++busy;
            lock.unlock();
            take();
            lock.lock();
            if (--busy == 0)
                done.notify_one();
        }
    }
    void run(int n, int wanted, Job f, void *a)
    {
        const int helpers = std::min(n, wanted) - 1;
        if (helpers > 0) {
            std::lock_guard<std::mutex> lock(m);
            while ((int)threads.size() < helpers) {
                try {
                    threads.emplace_back([this] { serve(); });
                } catch (...) {  // no thread to be had: the others take its pieces
                    break;
                }
            }
            job = f;
            arg = a;
            pieces = n;
            next.store(0, std::memory_order_relaxed);
            seats = std::min(helpers, (int)threads.size());
        } else {
            for (int k = 0; k < n; ++k)
                f(a, k);
            return;
        }
        for (int k = 0; k < helpers; ++k)
            wake.notify_one();
        take();
        // a thread that has not woken by now finds no seat
        std::unique_lock<std::mutex> lock(m);
        seats = 0;
        done.wait(lock, [this] { return busy == 0; });
    }
    ~CopyPool()
    {
        {
            std::lock_guard<std::mutex> lock(m);
            stop = true;
        }
        wake.notify_all();
        for (std::thread &t : threads)
            t.join();
    }
};

void copy_free(sbg_context c)
{
    delete c->copyPool;
    c->copyPool = nullptr;
    if (c->uploads) {
        (void)hipStreamSynchronize(c->uploads);
        (void)hipStreamDestroy(c->uploads);
    }
    for (hipEvent_t e : c->stageDone)
        if (e)
            (void)hipEventDestroy(e);
    c->staging.release();
}

// The upload stream, the events after a half of the staging, the pool, and
// staging for `bytes`, in powers of two from 1 MB
static int copy_setup(sbg_context c, size_t bytes)
{
    if (!c->uploads && hipStreamCreateWithFlags(&c->uploads, hipStreamNonBlocking) != hipSuccess) {
        c->uploads = nullptr;
        return fail(SBG_ERR_HIP, "copy stream creation failed");
    }
    for (hipEvent_t &e : c->stageDone)
        if (!e && hipEventCreateWithFlags(&e, hipEventDisableTiming | hipEventReleaseToSystem) != hipSuccess) {
            e = nullptr;
            return fail(SBG_ERR_HIP, "copy event creation failed");
        }
    if (!c->copyPool && !(c->copyPool = new (std::nothrow) CopyPool))
        return fail(SBG_ERR_OOM, "copy threads");
    size_t want = (size_t)1 << 20;
    while (want < bytes)
        want *= 2;
    if (want > c->staging.cap)  // kernels of this call may still read the old one
        HIP_TRY(hipStreamSynchronize(c->stream));
    return c->staging.ensure(want);
}

bool page_locked(const void *p, bool *device)
{
    hipPointerAttribute_t at;
    *device = false;
    if (hipPointerGetAttributes(&at, p) != hipSuccess) {
        (void)hipGetLastError();  // pageable memory is not an error here
        return false;
    }
    *device = at.type == hipMemoryTypeHost && at.devicePointer == p;
    return at.type == hipMemoryTypeHost;
}

static bool pageable(const void *p)
{
    hipPointerAttribute_t at;
    if (hipPointerGetAttributes(&at, p) != hipSuccess) {
        (void)hipGetLastError();
        return true;
    }
    return at.type != hipMemoryTypeHost && at.type != hipMemoryTypeDevice;
}

// What of a call's arrays lies in one piece.  Ranges start on 8 bytes on both
// sides; a workgroup moves kCopyBlock bytes.
struct CopyRanges {
    uint8_t *dst[kCopyParts];
    const uint8_t *src[kCopyParts];
    uint32_t bytes[kCopyParts];
    uint32_t end[kCopyParts];  // workgroups up to this range's last
};
constexpr uint32_t kCopyBlock = 256 * 8 * 4;

__global__ __launch_bounds__(256) void k_copy_ranges(CopyRanges r)
{
    int k = 0;
    uint32_t first = 0;
    while (blockIdx.x >= r.end[k])
        first = r.end[k++];
    const uint32_t base = (blockIdx.x - first) * kCopyBlock, bytes = r.bytes[k];
    const uint64_t *src = reinterpret_cast<const uint64_t *>(r.src[k]);
    uint64_t *dst = reinterpret_cast<uint64_t *>(r.dst[k]);
    const uint32_t words = bytes / 8, w0 = base / 8 + threadIdx.x;
    uint64_t v[4];
#pragma unroll
    for (int j = 0; j < 4; ++j)
        if (w0 + 256 * j < words)
            v[j] = src[w0 + 256 * j];
#pragma unroll
    for (int j = 0; j < 4; ++j)
        if (w0 + 256 * j < words)
            dst[w0 + 256 * j] = v[j];
    // the range's last bytes, by its last workgroup
    if (blockIdx.x + 1 == r.end[k] && threadIdx.x < bytes % 8)
        r.dst[k][8 * (size_t)words + threadIdx.x] = r.src[k][8 * (size_t)words + threadIdx.x];
}

// The arrays of one call end to end, each from a multiple of 64 bytes on.
struct CopyPlan {
    CopyPart part[kCopyParts];
    size_t begin[kCopyParts];
    int n = 0;
    size_t total = 0;

    void add(const CopyPart &p)
    {
        part[n] = p;
        begin[n++] = total;
        total += (p.bytes + 63) & ~(size_t)63;
    }
    // f(part, offset in it, bytes, offset from first) for what of [first, last)
    // lies in each part
    template <typename F>
    void each(size_t first, size_t last, const F &f) const
    {
        for (int i = 0; i < n; ++i) {
            const size_t a = std::max(first, begin[i]), b = std::min(last, begin[i] + part[i].bytes);
            if (a < b)
                f(part[i], a - begin[i], b - a, a - first);
        }
    }
    // the kernel that moves [first, last) between the parts and its staged copy
    hipError_t move(size_t first, size_t last, uint8_t *stage, bool in, hipStream_t s) const
    {
        CopyRanges r = {};
        int k = 0;
        uint32_t blocks = 0;
        each(first, last, [&](const CopyPart &p, size_t o, size_t bytes, size_t at) {
            r.dst[k] = in ? (uint8_t *)p.dev + o : stage + at;
            r.src[k] = in ? stage + at : (const uint8_t *)p.dev + o;
            r.bytes[k] = (uint32_t)bytes;
            r.end[k++] = blocks += (uint32_t)((bytes + kCopyBlock - 1) / kCopyBlock);
        });
        if (!blocks)
            return hipSuccess;
        hipLaunchKernelGGL(k_copy_ranges, dim3(blocks), dim3(256), 0, s, r);
        return hipGetLastError();
    }
};

// the host side of a piece: dst from src, narrowing 64-bit indices and finding
// the largest where the part says so
static uint64_t fill(uint8_t *dst, const CopyPart &p, size_t o, size_t bytes)
{
    uint64_t top = 0;
    if (p.kind == CopyPart::kBytes) {
        std::memcpy(dst, (const uint8_t *)p.host + o, bytes);
    } else if (p.kind == CopyPart::kIndices32) {
        const uint32_t *s = (const uint32_t *)p.host + o / 4;
        uint32_t *d = (uint32_t *)dst, hi = 0;
        for (size_t j = 0; j < bytes / 4; ++j) {
            d[j] = s[j];
            hi = std::max(hi, s[j]);
        }
        top = hi;
    } else {
        const uint64_t *s = (const uint64_t *)p.host + o / 4;
        uint32_t *d = (uint32_t *)dst;
        for (size_t j = 0; j < bytes / 4; ++j) {
            d[j] = (uint32_t)s[j];
            top = std::max(top, s[j]);
        }
    }
    return top;
}

// [first, last) in pieces of kCopyPiece over the pool; f(a, b) returns a
// hipError_t
template <typename F>
static hipError_t over_pieces(sbg_context c, size_t first, size_t last, const F &f)
{
    std::atomic<int> status{hipSuccess};
    auto one = [&](int t) {
        const size_t a = first + t * kCopyPiece;
        hipError_t e = hipSetDevice(c->device);
        if (e == hipSuccess)
            e = f(a, std::min(last, a + kCopyPiece));
        if (e != hipSuccess)
            status = e;
    };
    const size_t bytes = last - first;
    c->copyPool->run((int)((bytes + kCopyPiece - 1) / kCopyPiece), (int)std::min<size_t>(kCopyThreads, bytes / kCopyShare),
                     [](void *f, int t) { (*(decltype(one) *)f)(t); }, &one);
    return (hipError_t)status.load();
}

// Queues the plan's copies to the GPU on s, a half of the staging at a time
static hipError_t queue_in(sbg_context c, const CopyPlan &plan, hipStream_t s, std::atomic<uint64_t> &top)
{
    hipError_t e = hipSuccess;
    int half = 0;
    for (size_t first = 0; first < plan.total && e == hipSuccess; first += kStageHalf, half ^= 1) {
        const size_t last = std::min(plan.total, first + kStageHalf);
        if (first >= 2 * kStageHalf && (e = hipEventSynchronize(c->stageDone[half])) != hipSuccess)
            break;
        uint8_t *stage = c->staging.p + half * kStageHalf;
        e = over_pieces(c, first, last, [&](size_t a, size_t b) {
            uint64_t hi = 0;
            plan.each(a, b, [&](const CopyPart &p, size_t o, size_t bytes, size_t at) {
                hi = std::max(hi, fill(stage + (a - first) + at, p, o, bytes));
            });
            for (uint64_t was = top.load(); was < hi && !top.compare_exchange_weak(was, hi);) {
            }
            return plan.move(a, b, stage + (a - first), true, s);
        });
        if (e == hipSuccess && last < plan.total)
            e = hipEventRecord(c->stageDone[half], s);
    }
    return e;
}

template <typename S>
int upload_mesh(sbg_context c, double *dv, uint32_t *dt, const double *xyz, size_t nx, const S *tris, size_t ni,
                uint64_t *top)
{
    *top = 0;
    if (nx + ni == 0)
        return SBG_OK;
    CopyPlan plan;
    plan.add(part_in(dv, xyz, sizeof(double) * nx));
    CopyPart t = part_in(dt, tris, sizeof(uint32_t) * ni);
    t.kind = sizeof(S) == 8 ? CopyPart::kIndices64 : CopyPart::kIndices32;
    plan.add(t);
    TRY(copy_setup(c, std::min(plan.total, 2 * kStageHalf)));
    std::atomic<uint64_t> hi{0};
    hipError_t e = queue_in(c, plan, c->uploads, hi);
    const hipError_t es = hipStreamSynchronize(c->uploads);
    if (e != hipSuccess || (e = es) != hipSuccess)
        return fail(SBG_ERR_HIP, "mesh upload failed: %s", hipGetErrorString(e));
    *top = hi;
    return SBG_OK;
}
template int upload_mesh<uint32_t>(sbg_context, double *, uint32_t *, const double *, size_t, const uint32_t *, size_t,
                                   uint64_t *);
template int upload_mesh<uint64_t>(sbg_context, double *, uint32_t *, const double *, size_t, const uint64_t *, size_t,
                                   uint64_t *);

// The parts to be staged, the DMA of those that are no pageable memory
// (page-locked, or the GPU's own) queued at once.
static int plan_parts(sbg_context c, std::initializer_list<CopyPart> parts, bool in, CopyPlan &plan)
{
    for (const CopyPart &p : parts) {
        if (!p.bytes)
            continue;
        if (pageable(p.host))
            plan.add(p);
        else if (in)
            HIP_TRY(hipMemcpyAsync(p.dev, p.host, p.bytes, hipMemcpyHostToDevice, c->stream));
        else
            HIP_TRY(hipMemcpyAsync(p.host, p.dev, p.bytes, hipMemcpyDeviceToHost, c->stream));
    }
    return SBG_OK;
}

// Work queued on the context stream after the call sees the data.
int copy_in(sbg_context c, std::initializer_list<CopyPart> parts)
{
    CopyPlan plan;
    StreamJoin join(c->stream);
    TRY(plan_parts(c, parts, true, plan));
    if (plan.total) {
        TRY(copy_setup(c, std::min(plan.total, 2 * kStageHalf)));
        std::atomic<uint64_t> top{0};
        const hipError_t e = queue_in(c, plan, c->stream, top);
        if (e != hipSuccess)
            return fail(SBG_ERR_HIP, "copy to the GPU failed: %s", hipGetErrorString(e));
    }
    join.release();
    return SBG_OK;
}

// Moves the parts out after what the context stream holds; returns when they
// are in place.
int copy_out(sbg_context c, std::initializer_list<CopyPart> parts)
{
    CopyPlan plan;
    StreamJoin join(c->stream);
    TRY(plan_parts(c, parts, false, plan));
    if (!plan.total) {
        join.release();
        HIP_TRY(hipStreamSynchronize(c->stream));
        return SBG_OK;
    }
    TRY(copy_setup(c, std::min(plan.total, 2 * kOutRound)));
    // rounds of kOutRound: one arrives while the threads empty the other
    hipError_t e = hipSuccess;
    auto queue = [&](size_t first, int half) {
        if (first >= plan.total || e != hipSuccess)
            return;
        e = plan.move(first, std::min(plan.total, first + kOutRound), c->staging.p + half * kOutRound, false,
                      c->stream);
        if (e == hipSuccess)
            e = hipEventRecord(c->stageDone[half], c->stream);
    };
    queue(0, 0);
    int half = 0;
    for (size_t first = 0; first < plan.total && e == hipSuccess; first += kOutRound, half ^= 1) {
        const size_t last = std::min(plan.total, first + kOutRound);
        queue(last, half ^ 1);
        if (e != hipSuccess || (e = hipEventSynchronize(c->stageDone[half])) != hipSuccess)
            break;
        const uint8_t *stage = c->staging.p + half * kOutRound;
        e = over_pieces(c, first, last, [&](size_t a, size_t b) {
            plan.each(a, b, [&](const CopyPart &p, size_t o, size_t bytes, size_t at) {
                std::memcpy((uint8_t *)p.host + o, stage + (a - first) + at, bytes);
            });
            return hipSuccess;
        });
    }
    const hipError_t es = hipStreamSynchronize(c->stream);
    join.release();
    if (e != hipSuccess || (e = es) != hipSuccess)
        return fail(SBG_ERR_HIP, "copy from the GPU failed: %s", hipGetErrorString(e));
    return SBG_OK;
}

}  // namespace sbg
