// A HIP runtime in host memory, for tests of the library's host side without a
// GPU: allocations come from malloc, copies are memcpy, kernels do not run.
// Loaded with RTLD_GLOBAL before librgrt.so, it answers in libamdhip64's
// place. Copies check that their device side lies in an allocation. fake_fail
// makes the n-th next call of a function fail; fake_log returns what was
// allocated, freed and launched.
#include <hip/hip_runtime_api.h>

#include <cstdlib>
#include <cstring>
#include <map>
#include <string>

namespace {
std::map<const char*, size_t> blocks; // start -> size, device and pinned
std::map<const void*, std::string> kernels, vars;
std::map<const void*, size_t> varSize;
std::map<const void*, void*> varMem;
std::map<std::string, int> failIn;
std::string logged;
int residentBlocks = 5;

hipError_t called(const char* name)
{
    auto it = failIn.find(name);
    if(it == failIn.end() || --it->second > 0) return hipSuccess;
    failIn.erase(it);
    return hipErrorOutOfMemory;
}
void note(const std::string& s) { logged += s + "\n"; }
hipError_t take(const char* name, void** p, size_t n)
{
    *p = nullptr;
    if(hipError_t e = called(name)) return e;
    *p = std::calloc(n ? n : 1, 1);
    blocks[(const char*)*p] = n;
    note(std::string(name) + " " + std::to_string(n));
    return hipSuccess;
}
hipError_t give(const char* name, void* p)
{
    if(!p) return hipSuccess;
    auto it = blocks.find((const char*)p);
    if(it == blocks.end()) return hipErrorInvalidValue;
    note(std::string(name) + " " + std::to_string(it->second));
    blocks.erase(it);
    std::free(p);
    return hipSuccess;
}
bool inside(const void* p, size_t n)
{
    const char* c = (const char*)p;
    for(auto& v: varMem)
        if(c >= (const char*)v.second && c + n <= (const char*)v.second + varSize[v.first]) return true;
    auto it = blocks.upper_bound(c);
    if(it == blocks.begin()) return false;
    --it;
    return c + n <= it->first + it->second;
}
hipError_t copy(void* d, const void* s, size_t n, hipMemcpyKind k)
{
    if((k == hipMemcpyDeviceToHost || k == hipMemcpyDeviceToDevice) && !inside(s, n)) return hipErrorInvalidValue;
    if((k == hipMemcpyHostToDevice || k == hipMemcpyDeviceToDevice) && !inside(d, n)) return hipErrorInvalidValue;
    std::memcpy(d, s, n);
    return hipSuccess;
}
template<typename T>
hipError_t handle(T* h)
{
    *h = (T)(uintptr_t)64;
    return hipSuccess;
}
} // namespace

extern "C" {

void fake_fail(const char* name, int nth) { failIn[name] = nth; }
void fake_occupancy(int blocks) { residentBlocks = blocks; }
const char* fake_log() // since the last call
{
    static std::string out;
    out.swap(logged);
    logged.clear();
    return out.c_str();
}

hipError_t hipMalloc(void** p, size_t n) { return take("hipMalloc", p, n); }
hipError_t hipFree(void* p) { return give("hipFree", p); }
hipError_t hipHostMalloc(void** p, size_t n, unsigned int) { return take("hipHostMalloc", p, n); }
hipError_t hipHostFree(void* p) { return give("hipHostFree", p); }
hipError_t hipHostGetDevicePointer(void** d, void* h, unsigned int)
{
    *d = nullptr;
    if(hipError_t e = called("hipHostGetDevicePointer")) return e;
    *d = h;
    return hipSuccess;
}
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind k) { return copy(d, s, n, k); }
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind k, hipStream_t) { return copy(d, s, n, k); }
hipError_t hipMemset(void* d, int v, size_t n)
{
    if(!inside(d, n)) return hipErrorInvalidValue;
    std::memset(d, v, n);
    return hipSuccess;
}
hipError_t hipMemsetAsync(void* d, int v, size_t n, hipStream_t) { return hipMemset(d, v, n); }
hipError_t hipGetDeviceCount(int* n)
{
    *n = 1;
    return hipSuccess;
}
hipError_t hipGetDeviceProperties(hipDeviceProp_t* p, int) // the header gives it its versioned name
{
    std::memset(p, 0, sizeof(*p));
    p->multiProcessorCount = 2;
    return hipSuccess;
}
hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int* n, const void*, int, size_t)
{
    *n = residentBlocks;
    return hipSuccess;
}
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipDeviceSynchronize() { return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
const char* hipGetErrorString(hipError_t e) { return e == hipErrorOutOfMemory ? "out of memory" : e == hipErrorInvalidValue ? "invalid value" : "error"; }
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned int) { return handle(s); }
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned int) { return hipSuccess; }
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return hipSuccess; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t* g) { return handle(g); }
hipError_t hipGraphInstantiate(hipGraphExec_t* x, hipGraph_t, hipGraphNode_t*, char*, size_t) { return handle(x); }
hipError_t hipGraphExecUpdate(hipGraphExec_t, hipGraph_t, hipGraphNode_t*, hipGraphExecUpdateResult*) { return hipSuccess; }
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return hipSuccess; }
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t* e) { return handle(e); }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { return handle(e); }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t)
{
    *ms = 0.0f;
    return hipSuccess;
}

// What compiled kernels and device variables register, and a launch.
void** __hipRegisterFatBinary(const void*)
{
    static void* h = nullptr;
    return &h;
}
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* f, char*, const char* name, unsigned int, void*, void*, dim3*, dim3*, int*)
{
    kernels[f] = name;
}
void __hipRegisterVar(void**, void* var, char*, char* name, int, size_t size, int, int)
{
    vars[var] = name;
    varSize[var] = size;
}
hipError_t hipGetSymbolAddress(void** p, const void* var)
{
    void*& m = varMem[var];
    if(!m) m = std::aligned_alloc(256, (varSize[var] + 255) / 256 * 256);
    *p = m;
    return hipSuccess;
}
static dim3 launchGrid, launchBlock;
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t, hipStream_t)
{
    launchGrid = g;
    launchBlock = b;
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* g, dim3* b, size_t* shared, hipStream_t* s)
{
    *g = launchGrid;
    *b = launchBlock;
    *shared = 0;
    *s = nullptr;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void* f, dim3 g, dim3 b, void**, size_t, hipStream_t)
{
    note("launch " + kernels[f] + " " + std::to_string(g.x) + " " + std::to_string(b.x));
    return hipSuccess;
}

} // extern "C"
