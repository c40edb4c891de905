// A stand-in for the HIP runtime, for tests of libsbgpu.so's host paths on a
// machine without a GPU: memory is host memory, copies happen at once, kernels
// do nothing, and streams only count what was queued on them and what a wait
// has seen done.  Loaded with RTLD_GLOBAL before the library, so that the
// library's calls resolve here; it declares what it needs of the runtime's C
// interface itself.  Tests steer it through the fake_* functions.
#include <cstdint>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <new>
#include <string>
#include <vector>

namespace {

struct Stream;
struct Dep {
    Stream *s;
    uint64_t upTo;
};
struct Stream {
    uint64_t queued = 0, done = 0;
    std::vector<Dep> deps;
};
struct Event {
    Stream *s = nullptr;
    uint64_t at = 0;
};

std::recursive_mutex mu;
using Lock = std::lock_guard<std::recursive_mutex>;
std::vector<Stream *> streams;  // in the order they were made
std::map<const void *, std::string> kernels;
std::map<const void *, std::vector<char>> vars;
std::map<const void *, size_t> varSize;
std::map<const char *, size_t> pinned;
thread_local int lastError = 0;
std::string failKernel;
int failSkip = -1;
int hostAllocs = 0;
const volatile uint8_t *watch = nullptr;
std::string watched;
bool failNew = false;

void finish(Stream *s, uint64_t upTo)
{
    if (upTo > s->done)
        s->done = upTo;
    for (const Dep &d : s->deps)
        if (d.s != s && d.upTo > d.s->done)
            finish(d.s, d.upTo);
}

int index_of(const Stream *s)
{
    for (size_t k = 0; k < streams.size(); ++k)
        if (streams[k] == s)
            return (int)k;
    return -1;
}

}  // namespace

// the library's C++ allocations resolve here too
void *operator new(size_t n)
{
    void *p = failNew ? nullptr : malloc(n ? n : 1);
    if (!p)
        throw std::bad_alloc();
    return p;
}
void operator delete(void *p) noexcept { free(p); }
void operator delete(void *p, size_t) noexcept { free(p); }

extern "C" {

struct dim3 {
    uint32_t x, y, z;
};

// ---- steering ------------------------------------------------------------
// the launch of the (skip + 1)-th kernel from now whose name holds `name` fails
void fake_fail_kernel(const char *name, int skip)
{
    Lock l(mu);
    failKernel = name;
    failSkip = skip;
}
// whether work is queued on the k-th stream that no wait has seen done
int fake_pending(int k)
{
    Lock l(mu);
    return k < (int)streams.size() && streams[k]->queued > streams[k]->done;
}
void fake_drain(void)
{
    Lock l(mu);
    for (Stream *s : streams)
        s->done = s->queued;
}
// C++ allocations throw from now on, or no longer do
void fake_fail_new(int on) { failNew = on != 0; }
int fake_host_allocs(void) { return hostAllocs; }
// from now on every wait for a stream notes the stream's number and *p
void fake_watch(const uint8_t *p)
{
    Lock l(mu);
    watch = p;
    watched.clear();
}
const char *fake_watched(void) { return watched.c_str(); }

// ---- the runtime ------------------------------------------------------------
int hipGetDeviceCount(int *n) { return *n = 1, 0; }
int hipSetDevice(int) { return 0; }
const char *hipGetErrorString(int e) { return e ? "failed" : "no error"; }
int hipGetLastError(void)
{
    const int e = lastError;
    lastError = 0;
    return e;
}
int hipMalloc(void **p, size_t n) { return (*p = calloc(1, n)) ? 0 : 2; }
int hipFree(void *p) { return free(p), 0; }
int hipHostMalloc(void **p, size_t n, unsigned)
{
    Lock l(mu);
    *p = calloc(1, n);
    pinned[(char *)*p] = n;
    ++hostAllocs;
    return 0;
}
int hipHostFree(void *p)
{
    Lock l(mu);
    pinned.erase((char *)p);
    free(p);
    return 0;
}
struct Attributes {  // hipPointerAttribute_t
    int type, device;
    void *devicePointer, *hostPointer;
    int isManaged;
    unsigned allocationFlags;
};
int hipPointerGetAttributes(Attributes *a, const void *p)
{
    Lock l(mu);
    auto it = pinned.upper_bound((const char *)p);
    if (it == pinned.begin() || (--it, (const char *)p >= it->first + it->second))
        return 1;
    memset(a, 0, sizeof(*a));
    a->type = 1;  // host
    a->devicePointer = a->hostPointer = const_cast<void *>(p);
    return 0;
}
int hipStreamCreateWithFlags(void **s, unsigned)
{
    Lock l(mu);
    streams.push_back(new Stream);
    streams.back()->deps.reserve(4096);  // a wait allocates nothing
    *s = streams.back();
    return 0;
}
int hipStreamDestroy(void *) { return 0; }
int hipStreamSynchronize(void *s)
{
    Lock l(mu);
    if (watch)
        watched += std::to_string(index_of((Stream *)s)) + ":" + std::to_string((int)*watch) + " ";
    finish((Stream *)s, ((Stream *)s)->queued);
    return 0;
}
int hipStreamWaitEvent(void *s, void *e, unsigned)
{
    Lock l(mu);
    if (((Event *)e)->s)
        ((Stream *)s)->deps.push_back({((Event *)e)->s, ((Event *)e)->at});
    return 0;
}
int hipEventCreateWithFlags(void **e, unsigned) { return *e = new Event, 0; }
int hipEventCreate(void **e) { return *e = new Event, 0; }
int hipEventDestroy(void *e) { return delete (Event *)e, 0; }
int hipEventRecord(void *e, void *s)
{
    Lock l(mu);
    *(Event *)e = {(Stream *)s, ((Stream *)s)->queued};
    return 0;
}
int hipEventSynchronize(void *e)
{
    Lock l(mu);
    if (((Event *)e)->s)
        finish(((Event *)e)->s, ((Event *)e)->at);
    return 0;
}
int hipEventElapsedTime(float *ms, void *, void *) { return *ms = 0.0f, 0; }
int hipMemcpy(void *d, const void *s, size_t n, int) { return memcpy(d, s, n), 0; }
int hipMemcpyAsync(void *d, const void *s, size_t n, int, void *stream)
{
    Lock l(mu);
    memcpy(d, s, n);
    ++((Stream *)stream)->queued;
    return 0;
}
int hipFuncSetAttribute(const void *, int, int) { return 0; }
int hipLaunchKernel(const void *f, dim3, dim3, void **, size_t, void *stream)
{
    Lock l(mu);
    if (failSkip >= 0 && kernels[f].find(failKernel) != std::string::npos && failSkip-- == 0)
        return lastError = 719;
    ++((Stream *)stream)->queued;
    return 0;
}
int hipGetSymbolAddress(void **p, const void *var)
{
    Lock l(mu);
    vars[var].resize(varSize[var]);
    return *p = vars[var].data(), 0;
}
// capture is not stood in for: a caller that asks for it gets an error
int hipStreamBeginCapture(void *, int) { return 801; }
int hipStreamEndCapture(void *, void **g) { return *g = nullptr, 801; }
int hipGraphInstantiate(void **, void *, void *, char *, size_t) { return 801; }
int hipGraphLaunch(void *, void *) { return 801; }
int hipGraphDestroy(void *) { return 0; }
int hipGraphExecDestroy(void *) { return 0; }

// ---- what the compiler's host code calls ---------------------------------------
thread_local struct {
    dim3 grid, block;
    size_t lds;
    void *stream;
} call;
int __hipPushCallConfiguration(dim3 grid, dim3 block, size_t lds, void *stream)
{
    call = {grid, block, lds, stream};
    return 0;
}
int __hipPopCallConfiguration(dim3 *grid, dim3 *block, size_t *lds, void **stream)
{
    *grid = call.grid;
    *block = call.block;
    *lds = call.lds;
    *stream = call.stream;
    return 0;
}
void **__hipRegisterFatBinary(const void *)
{
    static void *module = nullptr;
    return &module;
}
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterFunction(void **, const void *f, char *, const char *name, unsigned, void *, void *, void *, void *,
                           int *)
{
    Lock l(mu);
    kernels[f] = name;
}
void __hipRegisterVar(void **, void *var, char *, char *, int, size_t size, int, int)
{
    Lock l(mu);
    varSize[var] = size;
}
}
