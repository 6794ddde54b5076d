// The HIP runtime calls libpkv_hip.so makes, on host memory: kernels do not run,
// allocations are counted and can be made to fail.  Loaded ahead of the runtime by
// the CPU tests of the library's host half.
#include <hip/hip_runtime_api.h>

#include <cstdlib>
#include <cstring>
#include <map>
#include <string>

namespace {
std::map<void*, size_t> g_live;
size_t g_fail_from = ~size_t{0};   // allocations of at least this many bytes fail
hipError_t g_last = hipSuccess;    // hipGetLastError's
std::string g_launched;            // kernels launched, one a line
std::map<const void*, std::string>& names() {   // of the registered kernels
    static std::map<const void*, std::string> n;
    return n;
}
}  // namespace

extern "C" {
void host_hip_fail_from(size_t bytes) { g_fail_from = bytes; }
unsigned host_hip_live(size_t bytes) {
    unsigned n = 0;
    for (auto& [p, size] : g_live) n += size == bytes;
    return n;
}
const char* host_hip_launched() { return g_launched.c_str(); }

hipError_t hipMalloc(void** p, size_t bytes) {
    if (bytes >= g_fail_from) return g_last = hipErrorOutOfMemory;
    *p = std::calloc(1, bytes);
    g_live[*p] = bytes;
    if (bytes == 16) {   // what the device check of the f16 subnormals reads back
        const float want[2] = {0x1p-10f + 0x1p-14f, 0x1p-10f};
        std::memcpy(*p, want, sizeof want);
    }
    return hipSuccess;
}
hipError_t hipFree(void* p) {
    g_live.erase(p);
    std::free(p);
    return hipSuccess;
}
hipError_t hipHostMalloc(void** p, size_t bytes, unsigned) {
    *p = std::calloc(1, bytes);
    return hipSuccess;
}
hipError_t hipHostFree(void* p) {
    std::free(p);
    return hipSuccess;
}
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) {
    std::memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t) {
    std::memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipMemsetAsync(void* d, int v, size_t n, hipStream_t) {
    std::memset(d, v, n);
    return hipSuccess;
}
hipError_t __hipPushCallConfiguration(dim3, dim3, size_t, hipStream_t) { return hipSuccess; }
hipError_t __hipPopCallConfiguration(dim3* grid, dim3* block, size_t* lds, hipStream_t* stream) {
    *grid = *block = dim3(1);
    *lds = 0;
    *stream = nullptr;
    return hipSuccess;
}
void** __hipRegisterFatBinary(const void*) { return nullptr; }
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
void __hipRegisterFunction(void**, const void* f, char*, const char* name, unsigned, void*, void*, dim3*, dim3*, int*) {
    names()[f] = name;
}
hipError_t hipLaunchKernel(const void* f, dim3, dim3, void**, size_t, hipStream_t) {
    g_launched += names()[f] + '\n';
    return hipSuccess;
}
hipError_t hipGetLastError() {
    const hipError_t e = g_last;
    g_last = hipSuccess;
    return e;
}
hipError_t hipGetDeviceCount(int* n) {
    *n = 1;
    return hipSuccess;
}
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600* p, int) {
    std::memset(p, 0, sizeof *p);
    std::strcpy(p->gcnArchName, "gfx950");
    return hipSuccess;
}
hipError_t hipGetSymbolAddress(void** p, const void*) {
    static char symbol[1 << 20];
    *p = symbol;
    return hipSuccess;
}
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipDeviceSynchronize() { return hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) {
    *s = nullptr;
    return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) {
    *e = reinterpret_cast<hipEvent_t>(&g_last);
    return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventQuery(hipEvent_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipFuncSetAttribute(const void*, hipFuncAttribute, int) { return hipSuccess; }
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t, int) {
    *v = 256;
    return hipSuccess;
}
hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int* n, const void*, int, size_t) {
    *n = 1;
    return hipSuccess;
}
}
