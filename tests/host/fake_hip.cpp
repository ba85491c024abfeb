// fake_hip.cpp -- a CPU stand-in for the HIP runtime functions that libprocell
// calls, built as libamdhip64.so.7 for the tests of its host code: device
// memory is host memory, streams run at once, kernels are recorded and not
// run.  A simulation kernel leaves its number (1, 2, ...) as the division
// count of each of its sets, so that a test can tell which run a result
// belongs to.
#include <stdlib.h>
#include <string.h>

#include <functional>
#include <map>
#include <set>

#include "fake_hip.hpp"
#include "procell_internal.hpp"

namespace fake {

std::vector<Launch> launches;
uint64_t sim_runs = 0;
int fail_event_record = 0;
uint64_t dead_stream_uses = 0, foreign_stream_uses = 0, streams_alive = 0, memory_alive = 0, memory_bytes = 0;
static float one_ms() { return 1.0f; }
float (*elapsed_ms)() = one_ms;
std::vector<uint32_t> segment_cells;

static std::map<const void *, std::string> names;
static std::map<const void *, void *> symbols;  // static device variables
static std::map<void *, uint64_t> memory;       // and the id of each allocation
static std::set<void *> streams, foreign, freed;  // freed: small allocations, whose addresses come again
static uint64_t next_id = 0;
constexpr uintptr_t kFirstStream = 0x10;
static uintptr_t next_stream = kFirstStream;
static std::map<void *, std::vector<std::function<void()>>> capturing, graphs;
static uintptr_t next_handle = 0x1000;

static hipError_t check(hipStream_t st)
{
    foreign_stream_uses += foreign.count((void *)st);
    if (!st || streams.count((void *)st))
        return hipSuccess;
    ++dead_stream_uses;
    return hipErrorContextIsDestroyed;
}

void device_reset()
{
    for (const auto &m : memory)
        freed.insert(m.first);
    memory.clear();
    streams.clear();
    foreign.clear();
    next_stream = kFirstStream;
    memory_alive = streams_alive = 0;
}

void take_stream()
{
    hipStream_t st;
    (void)hipStreamCreateWithFlags(&st, 0);
    foreign.insert((void *)st);
}

void take_memory()
{
    void *p;
    (void)hipMalloc(&p, 8);
}

static void run(const Launch &l, const procell::RunArgs *a)
{
    launches.push_back(l);
    if (!a)
        return;
    ++sim_runs;
    for (uint32_t i = 0; i < a->n_sets; ++i)
        a->counters[(size_t)i * procell::kCounterCopies * procell::kNumCounters + procell::kDivisions] = sim_runs;
}

}  // namespace fake

using namespace fake;

static struct {
    dim3 grid, block;
    size_t lds;
    hipStream_t stream;
} g_call;

extern "C" {

void **__hipRegisterFatBinary(const void *) { return (void **)&names; }
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterFunction(void **, const void *host, char *, const char *device, unsigned, void *, void *, void *, void *,
                           int *)
{
    names[host] = device;
}
void __hipRegisterVar(void **, void *host, char *, char *, int, size_t size, int, int)
{
    symbols[*(void **)&host] = calloc(1, size);
}
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t lds, hipStream_t st)
{
    g_call = {g, b, lds, st};
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3 *g, dim3 *b, size_t *lds, hipStream_t *st)
{
    *g = g_call.grid, *b = g_call.block, *lds = g_call.lds, *st = g_call.stream;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void *f, dim3 g, dim3 b, void **args, size_t lds, hipStream_t st)
{
    const hipError_t e = check(st);
    if (e != hipSuccess)
        return e;
    const Launch l{names[f], g.x, b.x, lds};
    const bool sim = l.kernel.find("sim_kernel") != std::string::npos || l.kernel.find("sim_filter") != std::string::npos;
    procell::RunArgs a{};
    if (sim)
        memcpy(&a, args[0], sizeof a);
    auto it = capturing.find((void *)st);
    if (it != capturing.end())
        it->second.push_back([=]() { run(l, sim ? &a : nullptr); });
    else
        run(l, sim ? &a : nullptr);
    return hipSuccess;
}
hipError_t hipGetDeviceCount(int *n) { return *n = 1, hipSuccess; }
hipError_t hipSetDevice(int d) { return d == 0 ? hipSuccess : hipErrorInvalidDevice; }
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600 *p, int)
{
    memset(p, 0, sizeof *p);
    strcpy(p->gcnArchName, "gfx950:sramecc+:xnack-");
    p->multiProcessorCount = 256;
    p->maxSharedMemoryPerMultiProcessor = p->sharedMemPerBlock = 163840;
    return hipSuccess;
}
// 160 KB of LDS and 4 (filtered simulation kernel: 6) wavefronts per SIMD
hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int *n, const void *f, int block, size_t lds)
{
    const int waves = names[f].find("sim_filter") != std::string::npos ? 24 : 16;
    *n = waves / ((block + 63) / 64);
    if (lds)
        *n = *n < (int)(163840 / lds) ? *n : (int)(163840 / lds);
    return hipSuccess;
}
hipError_t hipGetSymbolAddress(void **p, const void *host)
{
    return *p = symbols[host], *p ? hipSuccess : hipErrorInvalidSymbol;
}
hipError_t hipMalloc(void **p, size_t n)
{
    if (n <= 64 && !freed.empty()) {
        *p = *freed.begin();
        freed.erase(freed.begin());
    } else {
        *p = calloc(1, n < 64 ? 64 : n);
    }
    memory[*p] = ++next_id;
    memory_bytes = n > memory_bytes ? n : memory_bytes;
    ++memory_alive;
    return *p ? hipSuccess : hipErrorOutOfMemory;
}
hipError_t hipFree(void *p)
{
    if (p && !memory.erase(p))
        return hipErrorInvalidValue;
    memory_alive -= p != nullptr;
    free(p);
    return hipSuccess;
}
hipError_t hipPointerGetAttribute(void *out, hipPointer_attribute what, hipDeviceptr_t p)
{
    if (what != HIP_POINTER_ATTRIBUTE_BUFFER_ID || !memory.count(p))
        return hipErrorInvalidValue;
    memcpy(out, &memory[p], 8);
    return hipSuccess;
}
hipError_t hipHostMalloc(void **p, size_t n, unsigned) { return *p = calloc(1, n), hipSuccess; }
hipError_t hipHostFree(void *p) { return free(p), hipSuccess; }
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind) { return memcpy(d, s, n), hipSuccess; }
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t st)
{
    const hipError_t e = check(st);
    if (e == hipSuccess)
        memcpy(d, s, n);
    return e;
}
hipError_t hipMemset(void *p, int v, size_t n) { return memset(p, v, n), hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t *st, unsigned)
{
    *st = (hipStream_t)(next_stream += 16);
    streams.insert((void *)*st);
    ++streams_alive;
    return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t st)
{
    const hipError_t e = check(st);
    streams_alive -= streams.erase((void *)st);
    return e;
}
hipError_t hipStreamSynchronize(hipStream_t st) { return check(st); }
hipError_t hipStreamBeginCapture(hipStream_t st, hipStreamCaptureMode) { return capturing[(void *)st] = {}, check(st); }
hipError_t hipStreamEndCapture(hipStream_t st, hipGraph_t *g)
{
    *g = (hipGraph_t)(next_handle += 16);
    graphs[*g] = capturing[(void *)st];
    capturing.erase((void *)st);
    return check(st);
}
hipError_t hipGraphInstantiate(hipGraphExec_t *x, hipGraph_t g, hipGraphNode_t *, char *, size_t)
{
    *x = (hipGraphExec_t)(next_handle += 16);
    graphs[*x] = graphs[g];
    return hipSuccess;
}
hipError_t hipGraphLaunch(hipGraphExec_t x, hipStream_t st)
{
    for (auto &f : graphs[x])
        f();
    return check(st);
}
hipError_t hipGraphDestroy(hipGraph_t g) { return graphs.erase(g), hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t x) { return graphs.erase(x), hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { return *e = (hipEvent_t)(next_handle += 16), hipSuccess; }
hipError_t hipEventCreate(hipEvent_t *e) { return hipEventCreateWithFlags(e, 0); }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t st)
{
    if (fail_event_record > 0 && --fail_event_record == 0)
        return hipErrorUnknown;
    return check(st);
}
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t) { return *ms = elapsed_ms(), hipSuccess; }
hipError_t hipDeviceSynchronize() { return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
const char *hipGetErrorString(hipError_t) { return "stand-in"; }

}  // extern "C"
