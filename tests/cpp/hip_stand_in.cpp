// A HIP runtime of the CPU: the entry points that libportlbm_hip.so calls, on
// host memory, with kernels recorded and not run.  Loaded before the library
// (RTLD_GLOBAL), it takes the place of libamdhip64 in that process, so that
// what the library does around its kernels -- allocations that fail, which
// kernels a call launches, what it frees -- can be tested without a GPU.
#define __HIP_PLATFORM_AMD__ 1
#include <cxxabi.h>
#include <hip/hip_runtime_api.h>

#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <string>
#include <vector>

namespace
{

std::recursive_mutex g_mutex;
std::map<const void *, std::string> g_kernels;
std::map<std::string, int> g_fail;  // entry point -> calls until the one that fails
std::map<const char *, size_t> g_device, g_host;
size_t g_total = size_t(288) << 30, g_used = 0;
int g_live = 0;  // streams, events and graphs
std::vector<std::string> g_log;
std::string g_text;
hipError_t g_last = hipSuccess;

bool fails(const char *what)
{
    auto it = g_fail.find(what);
    return it != g_fail.end() && --it->second == 0;
}

hipError_t done(hipError_t e)
{
    if (e != hipSuccess)
        g_last = e;
    return e;
}

// [p, p + n) lies in one allocation of `all`
bool inside(const std::map<const char *, size_t> &all, const void *p, size_t n)
{
    const char *c = static_cast<const char *>(p);
    auto it = all.upper_bound(c);
    if (it == all.begin())
        return false;
    --it;
    return c + n <= it->first + it->second;
}

struct Call
{
    dim3 grid, block;
    size_t lds;
    hipStream_t stream;
};
thread_local std::vector<Call> t_calls;

template <class T>
T handle()
{
    ++g_live;
    return reinterpret_cast<T>(std::malloc(16));
}

}  // namespace

#define LOCK std::lock_guard<std::recursive_mutex> lock(g_mutex)

extern "C" {

// ---- controls ---------------------------------------------------------------
// The `after`-th call of `what` from now on fails (0: none does).
void stand_in_fail(const char *what, int after)
{
    LOCK;
    if (after)
        g_fail[what] = after;
    else
        g_fail.erase(what);
}
void stand_in_memory(size_t total)
{
    LOCK;
    g_total = total;
}
// Launches and copies that touch what they should not since the last call, one a line.
const char *stand_in_log(void)
{
    LOCK;
    g_text.clear();
    for (const std::string &l : g_log)
        g_text += l + "\n";
    g_log.clear();
    return g_text.c_str();
}
// Bytes of device and host allocations, streams, events and graphs alive.
void stand_in_live(size_t out[3])
{
    LOCK;
    out[0] = out[1] = 0;
    for (auto &a : g_device)
        out[0] += a.second;
    for (auto &a : g_host)
        out[1] += a.second;
    out[2] = size_t(g_live);
}

// ---- registration and launches ----------------------------------------------
void **__hipRegisterFatBinary(const void *)
{
    static void *handle_of_all[1];
    return handle_of_all;
}
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterFunction(void **, const void *host, char *, const char *name, unsigned, void *, void *, void *,
                           void *, int *)
{
    LOCK;
    int status = 0;
    char *text = abi::__cxa_demangle(name, nullptr, nullptr, &status);
    g_kernels[host] = status == 0 && text ? text : name;
    std::free(text);
}
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}
hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t lds, hipStream_t stream)
{
    t_calls.push_back(Call{grid, block, lds, stream});
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3 *grid, dim3 *block, size_t *lds, hipStream_t *stream)
{
    const Call c = t_calls.back();
    t_calls.pop_back();
    *grid = c.grid;
    *block = c.block;
    *lds = c.lds;
    *stream = c.stream;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void *host, dim3, dim3, void **args, size_t, hipStream_t)
{
    LOCK;
    const std::string name = g_kernels[host];
    g_log.push_back("launch " + name);
    if (name.find("k_copy_frame") != std::string::npos)
    {
        // (const uint4 *from, uint4 *to, size_t n)
        const void *from = *static_cast<void **>(args[0]), *to = *static_cast<void **>(args[1]);
        const size_t bytes = 16u * *static_cast<size_t *>(args[2]);
        if (!inside(g_device, from, bytes) || !inside(g_host, to, bytes))
            g_log.push_back("BAD frame copy out of its arrays");
    }
    return hipSuccess;
}

// ---- memory -------------------------------------------------------------------
hipError_t hipMalloc(void **p, size_t n)
{
    LOCK;
    if (fails("hipMalloc") || g_used + n > g_total)
        return done(hipErrorOutOfMemory);
    *p = std::calloc(1, n + 64);
    g_device[static_cast<char *>(*p)] = n;
    g_used += n;
    return hipSuccess;
}
hipError_t hipFree(void *p)
{
    LOCK;
    if (!p)
        return hipSuccess;
    auto it = g_device.find(static_cast<char *>(p));
    if (it == g_device.end())
    {
        g_log.push_back("BAD hipFree of what is not allocated");
        return done(hipErrorInvalidValue);
    }
    g_used -= it->second;
    g_device.erase(it);
    std::free(p);
    return hipSuccess;
}
hipError_t hipHostMalloc(void **p, size_t n, unsigned)
{
    LOCK;
    if (fails("hipHostMalloc"))
        return done(hipErrorOutOfMemory);
    *p = std::calloc(1, n + 64);
    g_host[static_cast<char *>(*p)] = n;
    return hipSuccess;
}
hipError_t hipHostFree(void *p)
{
    LOCK;
    if (!p)
        return hipSuccess;
    if (!g_host.erase(static_cast<char *>(p)))
    {
        g_log.push_back("BAD hipHostFree of what is not allocated");
        return done(hipErrorInvalidValue);
    }
    std::free(p);
    return hipSuccess;
}
hipError_t hipMemGetInfo(size_t *free_bytes, size_t *total)
{
    LOCK;
    if (fails("hipMemGetInfo"))
        return done(hipErrorUnknown);
    *free_bytes = g_total - g_used;
    *total = g_total;
    return hipSuccess;
}
hipError_t hipMemcpy(void *to, const void *from, size_t n, hipMemcpyKind kind)
{
    LOCK;
    if (fails("hipMemcpy") || !to || !from)
        return done(hipErrorInvalidValue);
    const bool from_device = kind == hipMemcpyDeviceToHost || kind == hipMemcpyDeviceToDevice;
    const bool to_device = kind == hipMemcpyHostToDevice || kind == hipMemcpyDeviceToDevice;
    if ((from_device && !inside(g_device, from, n)) || (to_device && !inside(g_device, to, n)))
    {
        g_log.push_back("BAD copy out of a device allocation");
        return done(hipErrorInvalidValue);
    }
    std::memcpy(to, from, n);
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void *to, const void *from, size_t n, hipMemcpyKind kind, hipStream_t)
{
    {
        LOCK;
        if (fails("hipMemcpyAsync"))
            return done(hipErrorUnknown);
    }
    return hipMemcpy(to, from, n, kind);
}
hipError_t hipMemset(void *p, int, size_t n)  // nothing reads it
{
    LOCK;
    if (!inside(g_device, p, n))
        g_log.push_back("BAD fill out of a device allocation");
    return hipSuccess;
}
hipError_t hipMemsetAsync(void *p, int v, size_t n, hipStream_t) { return hipMemset(p, v, n); }
hipError_t hipGetSymbolAddress(void **p, const void *)
{
    LOCK;
    static void *symbol = nullptr;
    if (!symbol)
        if (hipError_t e = hipMalloc(&symbol, size_t(64) << 20))
            return e;
    *p = symbol;
    return hipSuccess;
}

// ---- device, streams, events, graphs -----------------------------------------
hipError_t hipGetDevice(int *d)
{
    *d = 0;
    return hipSuccess;
}
hipError_t hipDeviceGetAttribute(int *v, hipDeviceAttribute_t a, int)
{
    *v = a == hipDeviceAttributeMultiprocessorCount ? 256 : 1024;
    return hipSuccess;
}
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600 *p, int)
{
    std::memset(p, 0, sizeof(*p));
    std::strcpy(p->name, "stand-in");
    p->multiProcessorCount = 256;
    p->maxThreadsPerBlock = 1024;
    return hipSuccess;
}
hipError_t hipDeviceSynchronize(void) { return hipSuccess; }
hipError_t hipGetLastError(void)
{
    LOCK;
    const hipError_t e = g_last;
    g_last = hipSuccess;
    return e;
}
const char *hipGetErrorString(hipError_t e) { return e == hipErrorOutOfMemory ? "out of memory" : "error"; }
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned)
{
    LOCK;
    if (fails("hipStreamCreateWithFlags"))
        return done(hipErrorOutOfMemory);
    *s = handle<hipStream_t>();
    return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t s)
{
    LOCK;
    --g_live;
    std::free(s);
    return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t e, unsigned) { return done(e ? hipSuccess : hipErrorInvalidHandle); }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned)
{
    LOCK;
    if (fails("hipEventCreateWithFlags"))
        return done(hipErrorOutOfMemory);
    *e = handle<hipEvent_t>();
    return hipSuccess;
}
hipError_t hipEventCreate(hipEvent_t *e) { return hipEventCreateWithFlags(e, 0); }
hipError_t hipEventDestroy(hipEvent_t e)
{
    LOCK;
    --g_live;
    std::free(e);
    return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t e, hipStream_t) { return done(e ? hipSuccess : hipErrorInvalidHandle); }
hipError_t hipEventSynchronize(hipEvent_t e) { return done(e ? hipSuccess : hipErrorInvalidHandle); }
hipError_t hipEventQuery(hipEvent_t e) { return done(e ? hipSuccess : hipErrorInvalidHandle); }
hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t)
{
    *ms = 1.f;
    return hipSuccess;
}
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return hipSuccess; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t *g)
{
    LOCK;
    *g = handle<hipGraph_t>();
    return hipSuccess;
}
hipError_t hipGraphInstantiate(hipGraphExec_t *x, hipGraph_t, hipGraphNode_t *, char *, size_t)
{
    LOCK;
    *x = handle<hipGraphExec_t>();
    return hipSuccess;
}
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return hipSuccess; }
hipError_t hipGraphDestroy(hipGraph_t g)
{
    LOCK;
    --g_live;
    std::free(g);
    return hipSuccess;
}
hipError_t hipGraphExecDestroy(hipGraphExec_t x)
{
    LOCK;
    --g_live;
    std::free(x);
    return hipSuccess;
}

}  // extern "C"
