// A stand-in HIP runtime for the CPU: one gfx950 device whose memory is reserved host memory under a
// settable limit, launches that are recorded and not run.  Loaded with RTLD_GLOBAL before
// libimpulse_fft.so, its functions take the place of the runtime's, so that planning, allocation
// failures and the choice of kernels run where there is no GPU.  What a kernel would have written is
// not there: results of a transform mean nothing here.
#define __HIP_PLATFORM_AMD__ 1
#include <hip/hip_runtime_api.h>
#include <sys/mman.h>

#include <cstdio>
#include <cstring>
#include <map>
#include <string>
#include <vector>

namespace {
// kernels by host stub; the library registers them from its constructors, maybe before this file's run
std::map<const void *, std::string> &names()
{
    static auto *m = new std::map<const void *, std::string>();
    return *m;
}
std::map<void *, size_t> blocks;
size_t used = 0, limit = (size_t)-1, peak = 0;
int per_cu = 2;
std::string launches;
struct Config {
    dim3 g, b;
    size_t lds;
    hipStream_t s;
};
std::vector<Config> configs;
}  // namespace

extern "C" {
// ---- what tests set and read
void standin_limit(size_t bytes) { limit = bytes; }
void standin_blocks_per_cu(int n) { per_cu = n; }
size_t standin_used() { return used; }
size_t standin_peak() { return peak; }
// "name grid.x grid.y block lds" of each launch since the last call, a line each
const char *standin_launches()
{
    static std::string last;
    last.swap(launches);
    launches.clear();
    return last.c_str();
}

// ---- registration
void **__hipRegisterFatBinary(const void *)
{
    static void *handle = nullptr;
    return &handle;
}
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterFunction(void **, const void *stub, char *, const char *name, unsigned, void *, void *, dim3 *, dim3 *, int *)
{
    names()[stub] = name;
}
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t lds, hipStream_t s)
{
    configs.push_back({g, b, lds, s});
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3 *g, dim3 *b, size_t *lds, hipStream_t *s)
{
    const Config c = configs.back();
    configs.pop_back();
    *g = c.g;
    *b = c.b;
    *lds = c.lds;
    *s = c.s;
    return hipSuccess;
}

// ---- device
hipError_t hipGetDeviceCount(int *n) { *n = 1; return hipSuccess; }
hipError_t hipGetDevice(int *d) { *d = 0; return hipSuccess; }
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600 *p, int)
{
    std::memset(p, 0, sizeof(*p));
    std::strcpy(p->gcnArchName, "gfx950");
    return hipSuccess;
}
hipError_t hipDeviceGetAttribute(int *v, hipDeviceAttribute_t a, int)
{
    *v = a == hipDeviceAttributeMaxSharedMemoryPerBlock ? 160 * 1024 : a == hipDeviceAttributeMultiprocessorCount ? 256 : 0;
    return hipSuccess;
}
hipError_t hipDeviceSynchronize() { return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
const char *hipGetErrorString(hipError_t) { return "stand-in error"; }
hipError_t hipFuncSetAttribute(const void *, hipFuncAttribute, int) { return hipSuccess; }
hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int *n, const void *, int, size_t) { *n = per_cu; return hipSuccess; }

// ---- memory
hipError_t hipMalloc(void **p, size_t n)
{
    *p = nullptr;
    if (n > limit || used > limit - n) return hipErrorOutOfMemory;
    void *m = mmap(nullptr, n, PROT_READ | PROT_WRITE, MAP_PRIVATE | MAP_ANONYMOUS | MAP_NORESERVE, -1, 0);
    if (m == MAP_FAILED) return hipErrorOutOfMemory;
    blocks[m] = n;
    used += n;
    if (used > peak) peak = used;
    *p = m;
    return hipSuccess;
}
hipError_t hipFree(void *p)
{
    auto it = blocks.find(p);
    if (it == blocks.end()) return p ? hipErrorInvalidValue : hipSuccess;
    munmap(p, it->second);
    used -= it->second;
    blocks.erase(it);
    return hipSuccess;
}
hipError_t hipHostMalloc(void **p, size_t n, unsigned) { return hipMalloc(p, n); }
hipError_t hipHostFree(void *p) { return hipFree(p); }
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind) { std::memcpy(d, s, n); return hipSuccess; }
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t) { std::memcpy(d, s, n); return hipSuccess; }
hipError_t hipGetSymbolAddress(void **p, const void *)
{
    static void *scratch = mmap(nullptr, 64u << 20, PROT_READ | PROT_WRITE, MAP_PRIVATE | MAP_ANONYMOUS | MAP_NORESERVE, -1, 0);
    *p = scratch;
    return hipSuccess;
}

// ---- streams, events, graphs
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) { *s = (hipStream_t)1; return hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return hipSuccess; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t *g) { *g = (hipGraph_t)1; return hipSuccess; }
hipError_t hipGraphInstantiate(hipGraphExec_t *e, hipGraph_t, hipGraphNode_t *, char *, size_t) { *e = (hipGraphExec_t)1; return hipSuccess; }
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return hipSuccess; }
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t *e) { *e = (hipEvent_t)1; return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { *e = (hipEvent_t)1; return hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t) { *ms = 1.0f; return hipSuccess; }

hipError_t hipLaunchKernel(const void *stub, dim3 g, dim3 b, void **, size_t lds, hipStream_t)
{
    char t[96];
    std::snprintf(t, sizeof(t), " %u %u %u %zu\n", g.x, g.y, b.x * b.y * b.z, lds);
    launches += names()[stub] + t;
    return hipSuccess;
}
}
