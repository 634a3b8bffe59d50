// A HIP runtime without a GPU, for tests of the library's host code: memory is
// host memory, kernels are only counted, copies of pinned memory stay pending
// until something waits for them, and the clock advances by 1 ms per launch.
// Loaded before liblcs_hip.so with RTLD_GLOBAL, its symbols are the ones the
// library binds.  rec_* are the tests' own entry points.
#include <hip/hip_runtime.h>

#include <atomic>
#include <chrono>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <set>
#include <string>
#include <thread>
#include <vector>

namespace {
struct Copy {
    void *dst;
    const void *src;
    size_t bytes;
};
std::recursive_mutex mu;
std::vector<Copy> pending;
std::map<char *, size_t> pinned;
std::map<const void *, std::string> names;
std::string launches;   // "name grid.x grid.y\n"
std::map<std::string, std::set<int>> lds_set;
double clock_ms = 0.0;
size_t live = 0;
std::atomic<int> slow_sync{0};
std::map<void *, size_t> device_mem;
thread_local int device = 0;

typedef std::lock_guard<std::recursive_mutex> Lock;

bool is_pinned(const void *p)
{
    auto it = pinned.upper_bound((char *)p);
    if (it == pinned.begin()) return false;
    --it;
    return (char *)p < it->first + it->second;
}

void run_pending()
{
    for (const Copy &c : pending) std::memcpy(c.dst, c.src, c.bytes);
    pending.clear();
}
}  // namespace

extern "C" {

int rec_pending() { Lock l(mu); return (int)pending.size(); }
double rec_clock() { return clock_ms; }
const char *rec_launches() { return launches.c_str(); }
void rec_clear() { Lock l(mu); launches.clear(); }
size_t rec_live() { return live; }
void rec_slow_next_sync(int ms) { slow_sync = ms; }
int rec_lds_devices(const char *name)   // how many devices the kernel's LDS limit was raised on
{
    size_t most = 0;
    for (auto &e : lds_set)
        if (e.first.find(name) != std::string::npos) most = std::max(most, e.second.size());
    return (int)most;
}

hipError_t hipGetDeviceCount(int *n) { *n = 2; return hipSuccess; }
hipError_t hipSetDevice(int d) { device = d; return hipSuccess; }
hipError_t hipGetDevice(int *d) { *d = device; return hipSuccess; }
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600 *p, int)
{
    std::memset(p, 0, sizeof(*p));
    std::strcpy(p->name, "recording");
    std::strcpy(p->gcnArchName, "gfx950");
    p->multiProcessorCount = 256;
    return hipSuccess;
}
hipError_t hipDeviceGetAttribute(int *v, hipDeviceAttribute_t, int) { *v = 256; return hipSuccess; }
hipError_t hipMemGetInfo(size_t *f, size_t *t) { *f = *t = (size_t)64 << 30; return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }

hipError_t hipMalloc(void **p, size_t n)
{
    Lock l(mu);
    *p = std::calloc(1, n ? n : 1);
    device_mem[*p] = n;
    live += n;
    return *p ? hipSuccess : hipErrorOutOfMemory;
}
hipError_t hipFree(void *p)
{
    Lock l(mu);
    run_pending();
    if (p) {
        live -= device_mem[p];
        device_mem.erase(p);
    }
    std::free(p);
    return hipSuccess;
}
hipError_t hipHostMalloc(void **p, size_t n, unsigned)
{
    Lock l(mu);
    *p = std::calloc(1, n ? n : 1);
    pinned[(char *)*p] = n;
    return hipSuccess;
}
hipError_t hipHostFree(void *p)
{
    Lock l(mu);
    pinned.erase((char *)p);
    std::free(p);
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t)
{
    Lock l(mu);
    if (is_pinned(d) || is_pinned(s)) pending.push_back(Copy{d, s, n});
    else std::memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind)
{
    Lock l(mu);
    run_pending();
    std::memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipMemset(void *d, int v, size_t n) { std::memset(d, v, n); return hipSuccess; }

hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) { *s = (hipStream_t)std::malloc(8); return hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t s) { std::free(s); return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t)
{
    if (const int ms = slow_sync.exchange(0)) std::this_thread::sleep_for(std::chrono::milliseconds(ms));
    Lock l(mu);
    run_pending();
    return hipSuccess;
}
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t *e) { *e = (hipEvent_t)std::calloc(1, 8); return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { return hipEventCreate(e); }
hipError_t hipEventDestroy(hipEvent_t e) { std::free(e); return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t) { *(double *)e = clock_ms; return hipSuccess; }
hipError_t hipEventQuery(hipEvent_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { Lock l(mu); run_pending(); return hipSuccess; }
hipError_t hipEventElapsedTime(float *ms, hipEvent_t a, hipEvent_t b)
{
    *ms = (float)(*(double *)b - *(double *)a);
    return hipSuccess;
}

hipError_t hipFuncSetAttribute(const void *f, hipFuncAttribute, int)
{
    Lock l(mu);
    lds_set[names[f]].insert(device);
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void *f, dim3 g, dim3, void **, size_t, hipStream_t)
{
    Lock l(mu);
    clock_ms += 1.0;
    launches += names[f] + " " + std::to_string(g.x) + " " + std::to_string(g.y) + "\n";
    return hipSuccess;
}
hipError_t hipGetSymbolAddress(void **p, const void *) { *p = nullptr; return hipErrorInvalidSymbol; }
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return hipErrorNotSupported; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t *) { return hipErrorNotSupported; }
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }
hipError_t hipGraphExecUpdate(hipGraphExec_t, hipGraph_t, hipGraphNode_t *, hipGraphExecUpdateResult *)
{
    return hipErrorNotSupported;
}
hipError_t hipGraphInstantiate(hipGraphExec_t *, hipGraph_t, hipGraphNode_t *, char *, size_t) { return hipErrorNotSupported; }
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return hipErrorNotSupported; }

struct CallConfig {
    dim3 grid, block;
    size_t lds;
    hipStream_t stream;
};
static thread_local CallConfig config;
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t l, hipStream_t s)
{
    config = CallConfig{g, b, l, s};
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3 *g, dim3 *b, size_t *l, hipStream_t *s)
{
    *g = config.grid;
    *b = config.block;
    *l = config.lds;
    *s = config.stream;
    return hipSuccess;
}
void **__hipRegisterFatBinary(const void *) { static void *h; return &h; }
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterFunction(void **, const void *host, char *, const char *name, unsigned, void *, void *, dim3 *, dim3 *, int *)
{
    names[host] = name;
}
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}
}
