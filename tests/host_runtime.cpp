// A HIP runtime without a device, for tests of the library's host code on the
// CPU: memory is host memory, copies are made, a launch is only noted by its
// kernel's name.  Built as libamdhip64.so.7 (host_runtime.map) and loaded
// before the library, which then takes it for the real one.
//
// The test_* functions are the tests' side: which allocation fails, whether
// kernel attributes are refused, and what status integers the device reports.
#include <cxxabi.h>
#include <hip/hip_runtime_api.h>

#include <cstdlib>
#include <cstring>
#include <map>
#include <set>
#include <string>

namespace {
std::map<const void*, std::string> kernels;   // host function -> kernel
std::map<int, int> ints;                      // status integers reported in place of the device's
std::set<const void*> pinned, device;
size_t statusBytes = 0;
std::string launched;
long failIn = 0, allocations = 0;
bool attributesRefused = false;
hipError_t last = hipSuccess;
struct {
    dim3 grid, block;
    size_t shared;
    hipStream_t stream;
} pushed;

hipError_t result(hipError_t e) {
    if (e != hipSuccess) last = e;
    return e;
}
hipError_t copy(void* dst, const void* src, size_t n, hipMemcpyKind kind) {
    std::memcpy(dst, src, n);
    if (kind == hipMemcpyDeviceToHost && n == statusBytes && pinned.count(dst))
        for (auto& [slot, v] : ints) static_cast<int*>(dst)[slot] = v;
    return hipSuccess;
}
int dummy;
}  // namespace

extern "C" {

void test_fail_allocation(long k) { failIn = k; }   // the k-th from now, 0: none
long test_allocations() { return allocations; }     // made so far
long test_live() { return (long)device.size(); }    // not freed
void test_refuse_attributes(int on) { attributesRefused = on != 0; }
void test_status_bytes(size_t n) { statusBytes = n; }
void test_status_int(int slot, int v) { ints[slot] = v; }
void test_status_clear() { ints.clear(); }
const char* test_launched() { return launched.c_str(); }   // kernel names, one per line
void test_forget_launches() { launched.clear(); }

hipError_t hipMalloc(void** p, size_t n) {
    if (failIn > 0 && --failIn == 0) {
        *p = nullptr;
        return result(hipErrorOutOfMemory);
    }
    *p = std::calloc(n ? n : 1, 1);
    device.insert(*p);
    allocations++;
    return hipSuccess;
}
hipError_t hipFree(void* p) {
    device.erase(p);
    std::free(p);
    return hipSuccess;
}
hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
    *p = std::calloc(n ? n : 1, 1);
    pinned.insert(*p);
    return hipSuccess;
}
hipError_t hipHostFree(void* p) {
    pinned.erase(p);
    std::free(p);
    return hipSuccess;
}
hipError_t hipMemcpy(void* dst, const void* src, size_t n, hipMemcpyKind k) { return copy(dst, src, n, k); }
hipError_t hipMemcpyAsync(void* dst, const void* src, size_t n, hipMemcpyKind k, hipStream_t) {
    return copy(dst, src, n, k);
}
hipError_t hipMemsetAsync(void* dst, int v, size_t n, hipStream_t) {
    std::memset(dst, v, n);
    return hipSuccess;
}
hipError_t hipGetLastError() {
    const hipError_t e = last;
    last = hipSuccess;
    return e;
}
const char* hipGetErrorString(hipError_t e) { return e == hipErrorOutOfMemory ? "out of memory" : "error"; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t, int) {
    *v = 256;
    return hipSuccess;
}
hipError_t hipFuncSetAttribute(const void*, hipFuncAttribute, int) {
    return result(attributesRefused ? hipErrorInvalidValue : hipSuccess);
}
hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int* n, const void*, int, size_t) {
    *n = 2;
    return hipSuccess;
}
hipError_t hipGetSymbolAddress(void** p, const void*) {
    static void* area = std::calloc(size_t(64) << 20, 1);
    *p = area;
    return hipSuccess;
}
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) {
    *s = reinterpret_cast<hipStream_t>(&dummy);
    return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t* e) {
    *e = reinterpret_cast<hipEvent_t>(&dummy);
    return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { return hipEventCreate(e); }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) {
    *ms = 1.0f;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void* f, dim3, dim3, void**, size_t, hipStream_t) {
    launched += kernels[f] + "\n";
    return hipSuccess;
}
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t shared, hipStream_t s) {
    pushed = {g, b, shared, s};
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* g, dim3* b, size_t* shared, hipStream_t* s) {
    *g = pushed.grid;
    *b = pushed.block;
    *shared = pushed.shared;
    *s = pushed.stream;
    return hipSuccess;
}
void** __hipRegisterFatBinary(const void*) {
    static void* module;
    return &module;
}
void __hipRegisterFunction(void**, const void* f, char*, const char* name, unsigned, void*, void*, void*, void*,
                           int*) {
    int bad = 0;
    char* d = abi::__cxa_demangle(name, nullptr, nullptr, &bad);
    std::string s = d ? d : name;
    std::free(d);
    s = s.substr(0, s.find('('));
    if (s.rfind("void ", 0) == 0) s = s.substr(5);
    if (s.rfind("mpsgpu::", 0) == 0) s = s.substr(8);
    kernels[f] = s;
}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
void __hipUnregisterFatBinary(void**) {}

}  // extern "C"
