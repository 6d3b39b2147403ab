// A stand-in for the HIP runtime calls of csrc/g4a.cpp, so that its host code runs
// on a machine without a GPU (tests/hip_standin.py builds it together with the host
// side of g4a.cpp): one gfx950 device of 256 CUs, device addresses that hold no
// memory out of a budget the test sets, and a record of every kernel launch instead
// of the launch. Nothing computes: a test looks at which kernels a call launches
// with which grids, what it allocates and which errors it returns.
#include <hip/hip_ext.h>
#include <hip/hip_runtime_api.h>

#include <cstdlib>
#include <cstring>
#include <map>
#include <set>
#include <sstream>
#include <string>

namespace {
std::map<uintptr_t, size_t> g_live;  // device allocations
uintptr_t g_next = 0x100000000ull;
size_t g_budget = ~size_t(0), g_used = 0;
std::set<std::string> g_names;
std::ostringstream g_launches;  // a line each: kernel name, grid, block
bool g_capturing = false;
hipError_t g_sync = hipSuccess, g_last = hipSuccess;

hipError_t record(hipFunction_t f, unsigned gx, unsigned gy, unsigned gz, unsigned bx) {
    g_launches << reinterpret_cast<const std::string*>(f)->c_str() << ' ' << gx << ' ' << gy << ' ' << gz << ' ' << bx
               << '\n';
    return hipSuccess;
}
template <typename T>
T handle() {
    return reinterpret_cast<T>(std::malloc(1));
}
}  // namespace

extern "C" {

// ---- what a test sets and reads ----
void standin_budget(size_t bytes) { g_budget = bytes; }
size_t standin_used() { return g_used; }
void standin_sync_error(int e) { g_sync = hipError_t(e); }
size_t standin_launches(char* out, size_t cap) {  // the record so far, which it clears
    const std::string s = g_launches.str();
    if (s.size() < cap) {
        std::memcpy(out, s.c_str(), s.size() + 1);
        g_launches.str("");
    }
    return s.size() + 1;
}

// ---- the runtime ----
void** __hipRegisterFatBinary(const void*) { return nullptr; }
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}

hipError_t hipGetDeviceCount(int* n) { return *n = 1, hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600* p, int) {
    std::memset(p, 0, sizeof *p);
    std::strcpy(p->gcnArchName, "gfx950:sramecc+:xnack-");
    p->multiProcessorCount = 256;
    return hipSuccess;
}
hipError_t hipGetLastError() {
    const hipError_t e = g_last;
    return g_last = hipSuccess, e;
}
const char* hipGetErrorString(hipError_t e) { return e == hipErrorOutOfMemory ? "out of memory" : "stand-in error"; }

hipError_t hipMalloc(void** p, size_t n) {
    if (g_capturing) return g_last = hipErrorStreamCaptureUnsupported;
    if (n > g_budget || g_used > g_budget - n) return g_last = hipErrorOutOfMemory;
    *p = reinterpret_cast<void*>(g_next);
    g_live[g_next] = n;
    g_used += n;
    g_next += (n + 511) / 256 * 256;
    return hipSuccess;
}
hipError_t hipFree(void* p) {
    if (!p) return hipSuccess;
    const auto it = g_live.find(reinterpret_cast<uintptr_t>(p));
    if (it == g_live.end()) return hipErrorInvalidValue;
    g_used -= it->second;
    g_live.erase(it);
    return hipSuccess;
}
hipError_t hipHostMalloc(void** p, size_t n, unsigned) { return *p = std::malloc(n), hipSuccess; }
hipError_t hipHostFree(void* p) { return std::free(p), hipSuccess; }
hipError_t hipMemset(void*, int, size_t) { return hipSuccess; }
hipError_t hipMemsetAsync(void*, int, size_t, hipStream_t) { return hipSuccess; }
hipError_t hipMemcpyAsync(void*, const void*, size_t, hipMemcpyKind, hipStream_t) { return hipSuccess; }
hipError_t hipGetSymbolAddress(void** p, const void*) { return *p = reinterpret_cast<void*>(0x10000000), hipSuccess; }

hipError_t hipModuleLoad(hipModule_t* m, const char*) { return *m = handle<hipModule_t>(), hipSuccess; }
hipError_t hipModuleUnload(hipModule_t m) { return std::free(m), hipSuccess; }
hipError_t hipModuleGetFunction(hipFunction_t* f, hipModule_t, const char* name) {
    *f = reinterpret_cast<hipFunction_t>(const_cast<std::string*>(&*g_names.insert(name).first));
    return hipSuccess;
}
hipError_t hipModuleLaunchKernel(hipFunction_t f, unsigned gx, unsigned gy, unsigned gz, unsigned bx, unsigned, unsigned,
                                 unsigned, hipStream_t, void**, void**) {
    return record(f, gx, gy, gz, bx);
}
hipError_t hipExtModuleLaunchKernel(hipFunction_t f, uint32_t x, uint32_t y, uint32_t z, uint32_t bx, uint32_t by,
                                    uint32_t bz, size_t, hipStream_t, void**, void**, hipEvent_t, hipEvent_t, uint32_t) {
    return record(f, x / bx, y / by, z / bz, bx);
}

hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) { return *s = handle<hipStream_t>(), hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t s) { return std::free(s), hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return g_sync; }
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return g_capturing = true, hipSuccess; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t* g) {
    g_capturing = false;
    return *g = handle<hipGraph_t>(), hipSuccess;
}
hipError_t hipGraphInstantiate(hipGraphExec_t* e, hipGraph_t, hipGraphNode_t*, char*, size_t) {
    return *e = handle<hipGraphExec_t>(), hipSuccess;
}
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return hipSuccess; }
hipError_t hipGraphDestroy(hipGraph_t g) { return std::free(g), hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t e) { return std::free(e), hipSuccess; }

hipError_t hipEventCreate(hipEvent_t* e) { return *e = handle<hipEvent_t>(), hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { return *e = handle<hipEvent_t>(), hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t e) { return std::free(e), hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) { return *ms = 0.0f, hipSuccess; }

}  // extern "C"
