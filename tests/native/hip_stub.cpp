// A HIP runtime on the CPU for tests of the host code: memory is the heap's, kernels do not run,
// and every launch is written down.  Loaded with RTLD_GLOBAL ahead of libamb.so, its functions
// take the place of the real runtime's.  Streams and events belong to the device that was current
// when they were made, as on a machine with two GPUs.
#include <hip/hip_runtime_api.h>

#include <cstdlib>
#include <cstring>
#include <ctime>
#include <map>
#include <mutex>
#include <string>
#include <vector>

namespace {
struct Launch {
    std::string name;
    unsigned blocks, threads;
    size_t lds;
};
struct OnDevice {
    int device;
    double at;  // events: the clock when recorded
};
std::mutex g_mutex;
std::map<const void*, std::string> g_kernels;
std::map<const void*, void*> g_symbols;
std::vector<Launch> g_launches;
std::string g_fast;           // kernels whose name holds this take 1 ms, the others 2
double g_clock = 0.0;
std::vector<unsigned long> g_order;  // (thread, launch or copy) in order of the calls
thread_local int t_device = 0;
thread_local unsigned long t_id = 0;
unsigned long g_threads = 0;
thread_local struct { dim3 grid, block; size_t lds; hipStream_t stream; } t_config;

void note(int copy)
{
    const std::lock_guard<std::mutex> lock(g_mutex);
    if (!t_id) t_id = ++g_threads;
    g_order.push_back(2 * t_id + copy);
}
}  // namespace

extern "C" {

// ---- for the tests ---------------------------------------------------------------------
int stub_launches() { return (int)g_launches.size(); }
const char* stub_launch(int i, unsigned* blocks, unsigned* threads, size_t* lds)
{
    *blocks = g_launches[i].blocks;
    *threads = g_launches[i].threads;
    *lds = g_launches[i].lds;
    return g_launches[i].name.c_str();
}
void stub_clear() { g_launches.clear(); g_order.clear(); }
void stub_fast(const char* part) { g_fast = part; }
int stub_order(unsigned long* out, int n)
{
    for (int i = 0; i < n && i < (int)g_order.size(); ++i) out[i] = g_order[i];
    return (int)g_order.size();
}

// ---- registration and launches -----------------------------------------------------------
void** __hipRegisterFatBinary(const void*) { static void* p; return &p; }
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* host, char*, const char* name, unsigned, void*, void*, dim3*, dim3*, int*)
{
    g_kernels[host] = name;
}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t lds, hipStream_t stream)
{
    t_config = {grid, block, lds, stream};
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* grid, dim3* block, size_t* lds, hipStream_t* stream)
{
    *grid = t_config.grid;
    *block = t_config.block;
    *lds = t_config.lds;
    *stream = t_config.stream;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void* f, dim3 grid, dim3 block, void**, size_t lds, hipStream_t)
{
    note(0);
    const std::lock_guard<std::mutex> lock(g_mutex);
    const std::string& name = g_kernels[f];
    g_clock += !g_fast.empty() && name.find(g_fast) != std::string::npos ? 1.0 : 2.0;
    g_launches.push_back({name, grid.x, block.x, lds});
    return hipSuccess;
}
hipError_t hipFuncSetAttribute(const void*, hipFuncAttribute, int) { return hipSuccess; }
hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int* n, const void*, int, size_t) { *n = 2; return hipSuccess; }

// ---- devices ---------------------------------------------------------------------------
hipError_t hipGetDeviceCount(int* n) { *n = 2; return hipSuccess; }
hipError_t hipGetDevice(int* d) { *d = t_device; return hipSuccess; }
hipError_t hipSetDevice(int d) { t_device = d; return hipSuccess; }
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t, int) { *v = 256; return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
const char* hipGetErrorString(hipError_t) { return "stub"; }

// ---- memory ----------------------------------------------------------------------------
hipError_t hipMalloc(void** p, size_t n) { *p = std::calloc(n ? n : 1, 1); return hipSuccess; }
hipError_t hipFree(void* p) { std::free(p); return hipSuccess; }
hipError_t hipHostMalloc(void** p, size_t n, unsigned) { return hipMalloc(p, n); }
hipError_t hipHostFree(void* p) { return hipFree(p); }
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) { note(1); std::memcpy(d, s, n); return hipSuccess; }
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind k, hipStream_t) { return hipMemcpy(d, s, n, k); }
hipError_t hipMemcpyWithStream(void* d, const void* s, size_t n, hipMemcpyKind k, hipStream_t) { return hipMemcpy(d, s, n, k); }
hipError_t hipGetSymbolAddress(void** p, const void* symbol)
{
    void*& m = g_symbols[symbol];
    if (!m) m = std::calloc(4 << 20, 1);
    *p = m;
    return hipSuccess;
}

// ---- streams, events, graphs -------------------------------------------------------------
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) { *s = (hipStream_t) new OnDevice{t_device, 0.0}; return hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t s) { delete (OnDevice*)s; return hipSuccess; }
hipError_t hipStreamGetDevice(hipStream_t s, hipDevice_t* d) { *d = s ? ((OnDevice*)s)->device : t_device; return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t)
{
    const timespec ms{0, 1000000};
    nanosleep(&ms, nullptr);  // other threads run meanwhile
    return hipSuccess;
}
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return hipSuccess; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t* g) { *g = (hipGraph_t)&g_clock; return hipSuccess; }
hipError_t hipGraphInstantiate(hipGraphExec_t* e, hipGraph_t, hipGraphNode_t*, char*, size_t) { *e = (hipGraphExec_t)&g_clock; return hipSuccess; }
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return hipSuccess; }
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { *e = (hipEvent_t) new OnDevice{t_device, 0.0}; return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t* e) { return hipEventCreateWithFlags(e, 0); }
hipError_t hipEventDestroy(hipEvent_t e) { delete (OnDevice*)e; return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s)
{
    OnDevice* ev = (OnDevice*)e;
    if (s && ((OnDevice*)s)->device != ev->device) return hipErrorInvalidHandle;
    ev->at = g_clock;
    return hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t) { return hipStreamSynchronize(nullptr); }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t a, hipEvent_t b) { *ms = (float)(((OnDevice*)b)->at - ((OnDevice*)a)->at); return hipSuccess; }

}  // extern "C"
