// A HIP runtime without a device (test infrastructure): the calls that
// libsiphon_hip.so makes, recorded instead of carried out, so that the
// library's dispatch, refusals and error paths can be tested on the CPU.
// Device memory is addresses alone; launches run nothing. One thread.
#include <cxxabi.h>
#include <hip/hip_runtime_api.h>

#include <stdlib.h>
#include <string.h>

#include <map>
#include <string>
#include <vector>

namespace {
struct Launch {
    std::string kernel;
    dim3 grid, block;
    size_t lds;
};
std::map<const void *, std::string> names;
std::vector<Launch> launches;
std::string syncs;  // 's' per stream synchronization, 'l' per launch
int calls = 0, fail_at = 0;
bool capture = false;
hipError_t last = hipSuccess;
uintptr_t next_addr = (uintptr_t)1 << 40;
struct { dim3 grid, block; size_t lds; hipStream_t stream; } config;

void *reserve(size_t bytes) {
    void *p = (void *)next_addr;
    next_addr += (bytes + 4095) / 4096 * 4096 + 4096;
    return p;
}
hipError_t result(hipError_t e) {
    if (e != hipSuccess) last = e;
    return e;
}
}  // namespace

extern "C" {

// ---- control ----
// launches since the last call of fake_reset
int fake_launches() { return (int)launches.size(); }
const char *fake_kernel(int i) { return launches[i].kernel.c_str(); }
unsigned fake_grid(int i, int d) { return d == 0 ? launches[i].grid.x : d == 1 ? launches[i].grid.y : launches[i].grid.z; }
unsigned fake_block(int i) { return launches[i].block.x; }
const char *fake_order() { return syncs.c_str(); }
// fail: the launch that fails, counted from here (0: none)
void fake_reset(int fail) { launches.clear(), syncs.clear(), calls = 0, fail_at = fail, last = hipSuccess; }
void fake_capture(int on) { capture = on; }

// ---- registration ----
void **__hipRegisterFatBinary(const void *) { static void *h; return &h; }
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterFunction(void **, const void *host, char *, const char *name, unsigned, void *, void *, void *, void *, int *) {
    int st;
    char *d = abi::__cxa_demangle(name, nullptr, nullptr, &st);
    names[host] = d ? d : name;
    free(d);
}
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t lds, hipStream_t s) {
    config = {g, b, lds, s};
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3 *g, dim3 *b, size_t *lds, hipStream_t *s) {
    *g = config.grid, *b = config.block, *lds = config.lds, *s = config.stream;
    return hipSuccess;
}
// the limits of the runtime: 2^32 work items per dimension, 1024 per
// workgroup, 64 KiB of dynamic LDS
hipError_t hipLaunchKernel(const void *f, dim3 g, dim3 b, void **, size_t lds, hipStream_t) {
    const bool bad = ++calls == fail_at || !g.x || !g.y || !g.z || b.x * b.y * b.z > 1024 || lds > 65536 ||
                     (uint64_t)g.x * b.x >> 32 || (uint64_t)g.y * b.y >> 32 || (uint64_t)g.z * b.z >> 32;
    if (bad) return result(hipErrorInvalidConfiguration);
    launches.push_back({names[f], g, b, lds});
    syncs += 'l';
    return hipSuccess;
}

// ---- the rest ----
hipError_t hipGetDeviceCount(int *n) { *n = 1; return hipSuccess; }
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600 *p, int) {
    memset(p, 0, sizeof *p);
    p->multiProcessorCount = 256;
    p->sharedMemPerBlock = 163840;
    return hipSuccess;
}
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipDeviceSynchronize() { return hipSuccess; }
hipError_t hipGetSymbolAddress(void **p, const void *) { *p = reserve((size_t)32 << 20); return hipSuccess; }
hipError_t hipMalloc(void **p, size_t n) {
    if (capture) return result(hipErrorStreamCaptureUnsupported);
    *p = reserve(n);
    return hipSuccess;
}
hipError_t hipFree(void *) { return hipSuccess; }
hipError_t hipHostMalloc(void **p, size_t n, unsigned) { *p = calloc(1, n); return *p ? hipSuccess : hipErrorOutOfMemory; }
hipError_t hipHostFree(void *p) { free(p); return hipSuccess; }
hipError_t hipHostGetDevicePointer(void **d, void *h, unsigned) { *d = h; return hipSuccess; }
hipError_t hipMemcpy(void *, const void *, size_t, hipMemcpyKind) { return hipSuccess; }
hipError_t hipMemcpyAsync(void *, const void *, size_t, hipMemcpyKind, hipStream_t) { return hipSuccess; }
hipError_t hipMemset(void *, int, size_t) { return hipSuccess; }
hipError_t hipMemsetAsync(void *, int, size_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { *e = (hipEvent_t)1; return hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) { *s = (hipStream_t)1; return hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { syncs += 's'; return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }
hipError_t hipStreamIsCapturing(hipStream_t s, hipStreamCaptureStatus *cs) {
    *cs = capture && s ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone;
    return hipSuccess;
}
const char *hipGetErrorString(hipError_t) { return "fake error"; }
hipError_t hipGetLastError() {
    const hipError_t e = last;
    last = hipSuccess;
    return e;
}
}
