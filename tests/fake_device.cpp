// A HIP runtime without a GPU, for tests of the host code: it is linked with
// the library's host sources in place of libamdhip64 and of the kernels.
// "Device" memory is mapped, never touched by a kernel, and counted; a launch
// records its engine and its tasks and computes nothing; allocations can be made
// to fail and launches to last.
#include <hip/hip_runtime.h>
#include <sched.h>
#include <sys/mman.h>

#include <algorithm>
#include <atomic>
#include <cstring>
#include <map>
#include <mutex>

#include "../gpumemefficient_amd/csrc/wf_variants.h"
#include "fake_device.h"

namespace {

std::mutex g_mu;
std::map<void *, size_t> g_mem;
size_t g_live = 0, g_peak = 0, g_free = (size_t)288 << 30;
std::atomic<bool> g_hold{false};
std::atomic<int> g_release{0};  // counts fake_release() calls
std::atomic<bool> g_free_hold{false};
std::atomic<int> g_launches{0};
std::atomic<int64_t> g_tasks{0};
std::atomic<int> g_engine{-1};

}  // namespace

extern "C" {

// Device memory that is free to the library; what it holds, and the most it held.
void fake_set_memory(size_t bytes)
{
    std::lock_guard<std::mutex> lk(g_mu);
    g_free = g_live + bytes;
    g_peak = g_live;
}
size_t fake_live() { return g_live; }
size_t fake_peak() { return g_peak; }
// While set, launches begin that do not end before fake_release().
void fake_hold(int on) { g_hold = on != 0; }
void fake_release() { ++g_release; }
// While set, hipFree does not return.
void fake_free_hold(int on) { g_free_hold = on != 0; }
// Engine launches so far; the last one's engine, and the tasks of all.
int fake_launches() { return g_launches; }
int fake_last_engine() { return g_engine; }
int64_t fake_tasks() { return g_tasks.exchange(0); }

hipError_t hipMalloc(void **p, size_t n)
{
    std::lock_guard<std::mutex> lk(g_mu);
    *p = nullptr;
    if (g_live + n > g_free) return hipErrorOutOfMemory;
    void *m = mmap(nullptr, n, PROT_READ | PROT_WRITE, MAP_PRIVATE | MAP_ANONYMOUS | MAP_NORESERVE, -1, 0);
    if (m == MAP_FAILED) return hipErrorOutOfMemory;
    g_mem[m] = n;
    g_live += n;
    g_peak = std::max(g_peak, g_live);
    *p = m;
    return hipSuccess;
}
hipError_t hipFree(void *p)
{
    while (g_free_hold) sched_yield();
    std::lock_guard<std::mutex> lk(g_mu);
    auto it = g_mem.find(p);
    if (it == g_mem.end()) return hipErrorInvalidValue;
    g_live -= it->second;
    munmap(p, it->second);
    g_mem.erase(it);
    return hipSuccess;
}
hipError_t hipHostMalloc(void **p, size_t n, unsigned)
{
    *p = ::operator new(n);
    return hipSuccess;
}
hipError_t hipHostFree(void *p)
{
    ::operator delete(p);
    return hipSuccess;
}
hipError_t hipHostGetDevicePointer(void **d, void *h, unsigned)
{
    *d = h;
    return hipSuccess;
}
hipError_t hipMemGetInfo(size_t *f, size_t *t)
{
    std::lock_guard<std::mutex> lk(g_mu);
    *f = g_free - g_live;
    *t = g_free;
    return hipSuccess;
}
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind)
{
    std::memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind k, hipStream_t) { return hipMemcpy(d, s, n, k); }
hipError_t hipMemcpy2D(void *d, size_t dp, const void *s, size_t sp, size_t w, size_t h, hipMemcpyKind)
{
    for (size_t i = 0; i < h; ++i) std::memcpy((char *)d + i * dp, (const char *)s + i * sp, w);
    return hipSuccess;
}
// (New mappings are zero.)
hipError_t hipMemset(void *, int, size_t) { return hipSuccess; }
hipError_t hipMemsetAsync(void *, int, size_t, hipStream_t) { return hipSuccess; }
hipError_t hipGetDeviceCount(int *n)
{
    *n = 1;
    return hipSuccess;
}
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
hipError_t hipDeviceSynchronize() { return hipSuccess; }
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600 *p, int)
{
    std::memset(p, 0, sizeof(*p));
    std::strcpy(p->gcnArchName, "none");
    p->multiProcessorCount = 256;
    p->warpSize = 64;
    return hipSuccess;
}
hipError_t hipStreamCreate(hipStream_t *s)
{
    *s = (hipStream_t)::operator new(1);
    return hipSuccess;
}
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) { return hipStreamCreate(s); }
hipError_t hipStreamDestroy(hipStream_t s)
{
    ::operator delete((void *)s);
    return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamQuery(hipStream_t) { return hipSuccess; }
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return hipErrorNotSupported; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t *) { return hipErrorNotSupported; }
hipError_t hipGraphInstantiate(hipGraphExec_t *, hipGraph_t, hipGraphNode_t *, char *, size_t) { return hipErrorNotSupported; }
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return hipErrorNotSupported; }
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t *e)
{
    *e = (hipEvent_t) new int(-1);
    return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { return hipEventCreate(e); }
hipError_t hipEventDestroy(hipEvent_t e)
{
    delete (int *)e;
    return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t e, hipStream_t)
{
    *(int *)e = g_hold ? g_release.load() : -1;
    return hipSuccess;
}
hipError_t hipEventQuery(hipEvent_t e) { return *(int *)e == g_release ? hipErrorNotReady : hipSuccess; }
hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t)
{
    *ms = 0.f;
    return hipSuccess;
}
// Two workgroups a CU.
hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int *n, const void *, int, size_t)
{
    *n = 2;
    return hipSuccess;
}

// --- the kernels' entry points ---
#define V(E, R, W, K) {E, R, W, K, 256, nullptr}
const WfVariant wf_variants_async[] = {V(1, 2, 4, 32), V(1, 2, 2, 32), V(1, 2, 1, 32), V(1, 1, 1, 32), V(1, 2, 4, 16)};
const int wf_num_variants_async = 5;
const WfVariant wf_variants_lockstep[] = {V(0, 2, 4, 64), V(0, 2, 4, 32), V(0, 1, 1, 32)};
const int wf_num_variants_lockstep = 3;
const WfVariant wf_variants_bitpar[] = {V(2, 32, 1, 64), V(2, 32, 2, 64), V(3, 32, 1, 64), V(3, 32, 2, 64)};
const int wf_num_variants_bitpar = 4;

hipError_t wf_launch_engine(const WfVariant *v, int, const WfKernelArgs *ka, hipStream_t)
{
    ++g_launches;
    g_engine = v->engine;
    g_tasks += ka->task_end - ka->task_begin;
    return hipSuccess;
}
hipError_t wf_launch_reset(WfResultDev *, int64_t, int32_t *, int64_t, uint32_t *, uint32_t, hipStream_t)
{
    return hipSuccess;
}
hipError_t wf_launch_table(int, const WfKernelArgs *, hipStream_t) { return hipSuccess; }
hipError_t wf_launch_naive(int, int, int, int *, const int32_t *, const int32_t *, int, int, int *, hipStream_t)
{
    return hipSuccess;
}
hipError_t wf_launch_bitpar_combine(const WfSplitDev *, int, const uint32_t *, const WfCutDev *, const uint64_t *,
                                    WfResultDev *, hipStream_t)
{
    return hipSuccess;
}
hipError_t wf_launch_sw_combine(const WfSplitDev *, int, int, const uint32_t *, const WfCutDev *, const uint64_t *,
                                WfResultDev *, hipStream_t)
{
    return hipSuccess;
}
const void *wf_serve_kernel(int *block)
{
    *block = 256;
    return nullptr;
}
hipError_t wf_launch_serve(int, const WfServeArgs *, hipStream_t) { return hipErrorNotSupported; }
hipError_t wf_launch_stencil(int, const WfStencilArgs *, hipStream_t) { return hipSuccess; }
int wf_stencil_resident(int cus) { return 4 * cus; }
hipError_t wf_launch_sat(int, const WfSatArgs *, hipStream_t) { return hipSuccess; }
int wf_sat_resident(int cus) { return cus; }

}  // extern "C"
