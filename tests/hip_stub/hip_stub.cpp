// A stand-in for the HIP runtime on a machine without a GPU: memory that is reserved but never read or written, one
// device of 256 compute units, and a record of every kernel that would have been launched. Loaded ahead of
// libkernelcore_amd.so (RTLD_GLOBAL), it takes the place of libamdhip64 for the functions the library calls, so that a
// test can call the public entry points and see which kernel each call goes to.
#include <hip/hip_runtime_api.h>
#include <sys/mman.h>

#include <cstdio>
#include <map>
#include <string>

namespace {
struct Config {
    dim3 grid, block;
    size_t shmem;
    hipStream_t stream;
};
std::map<const void*, std::string>& names() {  // (filled by the library's constructors)
    static std::map<const void*, std::string> m;
    return m;
}
Config pending;
std::string record;
bool capturing = false;
std::map<void*, size_t> sizes;
}  // namespace

#define OK(name, ...) hipError_t name(__VA_ARGS__) { return hipSuccess; }
template <class T>
hipError_t handle(T* p) {
    static char dummy[64];
    *p = reinterpret_cast<T>(dummy);
    return hipSuccess;
}

extern "C" {
const char* stub_record() { return record.c_str(); }  // "kernel gridx gridy gridz blockx" a line
void stub_clear() { record.clear(); }
void stub_capturing(int on) { capturing = on; }

void** __hipRegisterFatBinary(const void*) { static void* h; return &h; }
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* host, char*, const char* device, unsigned, void*, void*, void*, void*, int*) {
    names()[host] = device;
}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t shmem, hipStream_t stream) {
    pending = Config{grid, block, shmem, stream};
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* grid, dim3* block, size_t* shmem, hipStream_t* stream) {
    *grid = pending.grid, *block = pending.block, *shmem = pending.shmem, *stream = pending.stream;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void* f, dim3 grid, dim3 block, void**, size_t, hipStream_t) {
    char at[80];
    std::snprintf(at, sizeof at, " %u %u %u %u\n", grid.x, grid.y, grid.z, block.x);
    record += names()[f] + at;
    return hipSuccess;
}
hipError_t hipMalloc(void** p, size_t bytes) {
    *p = mmap(nullptr, bytes, PROT_NONE, MAP_PRIVATE | MAP_ANONYMOUS | MAP_NORESERVE, -1, 0);
    if (*p == MAP_FAILED) return hipErrorOutOfMemory;
    sizes[*p] = bytes;
    return hipSuccess;
}
hipError_t hipFree(void* p) {
    if (p) munmap(p, sizes[p]), sizes.erase(p);
    return hipSuccess;
}
OK(hipMemcpy, void*, const void*, size_t, hipMemcpyKind)
OK(hipMemset, void*, int, size_t)
hipError_t hipMemGetInfo(size_t* f, size_t* t) { *f = *t = size_t(288) << 30; return hipSuccess; }
hipError_t hipGetDeviceCount(int* n) { *n = 1; return hipSuccess; }
hipError_t hipGetDevice(int* d) { *d = 0; return hipSuccess; }
OK(hipSetDevice, int)
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t, int) { *v = 256; return hipSuccess; }
OK(hipDeviceSynchronize)
OK(hipFuncSetAttribute, const void*, hipFuncAttribute, int)
hipError_t hipGetLastError() { return hipSuccess; }
const char* hipGetErrorString(hipError_t) { return "stub"; }
hipError_t hipGetSymbolAddress(void** p, const void*) { return handle(p); }
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) { return handle(s); }
OK(hipStreamDestroy, hipStream_t)
OK(hipStreamSynchronize, hipStream_t)
OK(hipStreamQuery, hipStream_t)
OK(hipStreamWaitEvent, hipStream_t, hipEvent_t, unsigned)
hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus* s) {
    *s = capturing ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone;
    return hipSuccess;
}
OK(hipStreamBeginCapture, hipStream_t, hipStreamCaptureMode)
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t* g) { return handle(g); }
hipError_t hipGraphInstantiate(hipGraphExec_t* e, hipGraph_t, hipGraphNode_t*, char*, size_t) { return handle(e); }
OK(hipGraphLaunch, hipGraphExec_t, hipStream_t)
OK(hipGraphDestroy, hipGraph_t)
OK(hipGraphExecDestroy, hipGraphExec_t)
hipError_t hipEventCreate(hipEvent_t* e) { return handle(e); }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { return handle(e); }
OK(hipEventDestroy, hipEvent_t)
OK(hipEventRecord, hipEvent_t, hipStream_t)
OK(hipEventSynchronize, hipEvent_t)
OK(hipEventQuery, hipEvent_t)
OK(hipEventElapsedTime, float*, hipEvent_t, hipEvent_t)
OK(hipLaunchHostFunc, hipStream_t, hipHostFn_t, void*)
}
