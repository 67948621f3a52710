// The parts of the HIP runtime that the library calls, on host memory and
// without a GPU, for tests of the host code: allocations come from a budget
// and hold a byte pattern until something writes them, a launch runs no
// kernel but is shown to `fake_on_launch` (grid, block, LDS, arguments), and
// k_fill_u32 is carried out.  A program that names this library before the
// HIP runtime on its link line gets these definitions.
#include "fake_hip.h"

#include <cstdlib>
#include <cstring>
#include <map>
#include <string>

long long fake_free_bytes = (long long)1 << 40;
long long fake_used_bytes = 0;
void (*fake_on_launch)(const FakeLaunch&) = nullptr;

namespace {

std::map<const void*, std::string>& kernels()
{
    static std::map<const void*, std::string> m;
    return m;
}
std::map<void*, size_t>& blocks()
{
    static std::map<void*, size_t> m;
    return m;
}
struct Config {
    dim3 grid, block;
    size_t lds;
    hipStream_t st;
} g_config;
int g_handle;

}  // namespace

extern "C" {

void** __hipRegisterFatBinary(const void*)
{
    static void* module[1];
    return module;
}
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* host, char*, const char* name, unsigned, void*, void*,
                           void*, void*, int*)
{
    kernels()[host] = name;
}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t lds, hipStream_t st)
{
    g_config = Config{grid, block, lds, st};
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* grid, dim3* block, size_t* lds, hipStream_t* st)
{
    *grid = g_config.grid;
    *block = g_config.block;
    *lds = g_config.lds;
    *st = g_config.st;
    return hipSuccess;
}

hipError_t hipLaunchKernel(const void* f, dim3 grid, dim3 block, void** args, size_t lds, hipStream_t)
{
    const FakeLaunch l{kernels()[f].c_str(), grid, block, lds, args};
    // limits of a launch: 1024 work-items per workgroup, 2^32 - 1 per dimension
    const unsigned long long most = 0xFFFFFFFFull;
    if ((unsigned long long)block.x * block.y * block.z > 1024 ||
        (unsigned long long)grid.x * block.x > most || (unsigned long long)grid.y * block.y > most ||
        (unsigned long long)grid.z * block.z > most)
        return hipErrorInvalidConfiguration;
    if (fake_on_launch) fake_on_launch(l);
    if (std::strstr(l.name, "k_fill_u32")) {
        unsigned* p = *(unsigned**)args[0];
        const unsigned v = *(unsigned*)args[1];
        const int64_t n = *(int64_t*)args[2];
        for (int64_t i = 0; i < n; ++i) p[i] = v;
    }
    return hipSuccess;
}

hipError_t hipMalloc(void** p, size_t n)
{
    *p = nullptr;
    if (fake_used_bytes + (long long)n > fake_free_bytes) return hipErrorOutOfMemory;
    *p = std::malloc(n ? n : 1);
    if (!*p) return hipErrorOutOfMemory;
    std::memset(*p, 0xA5, n);
    blocks()[*p] = n;
    fake_used_bytes += (long long)n;
    return hipSuccess;
}
hipError_t hipFree(void* p)
{
    if (!p) return hipSuccess;
    auto it = blocks().find(p);
    if (it == blocks().end()) return hipErrorInvalidValue;
    fake_used_bytes -= (long long)it->second;
    blocks().erase(it);
    std::free(p);
    return hipSuccess;
}
hipError_t hipMemGetInfo(size_t* fr, size_t* tot)
{
    *fr = (size_t)(fake_free_bytes - fake_used_bytes);
    *tot = (size_t)fake_free_bytes;
    return hipSuccess;
}
hipError_t hipHostMalloc(void** p, size_t n, unsigned)
{
    *p = std::calloc(n, 1);
    return *p ? hipSuccess : hipErrorOutOfMemory;
}
hipError_t hipHostFree(void* p)
{
    std::free(p);
    return hipSuccess;
}
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind)
{
    std::memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t)
{
    std::memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipMemset(void* d, int v, size_t n)
{
    std::memset(d, v, n);
    return hipSuccess;
}
hipError_t hipGetSymbolAddress(void**, const void*) { return hipErrorNotSupported; }
hipError_t hipGetDevice(int* d)
{
    *d = 0;
    return hipSuccess;
}
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t, int)
{
    *v = 256;   // compute units: the only attribute asked for
    return hipSuccess;
}
hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int* n, const void*, int, size_t)
{
    *n = 4;
    return hipSuccess;
}
const char* hipGetErrorString(hipError_t) { return "fake HIP error"; }
hipError_t hipGetLastError(void) { return hipSuccess; }

hipError_t hipStreamCreateWithFlags(hipStream_t* st, unsigned)
{
    *st = (hipStream_t)&g_handle;
    return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t* e)
{
    *e = (hipEvent_t)&g_handle;
    return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { return hipEventCreate(e); }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t)
{
    *ms = 0.f;
    return hipSuccess;
}
// no graphs: a plan whose capture fails launches step by step
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return hipErrorNotSupported; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t*) { return hipErrorNotSupported; }
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }
hipError_t hipGraphInstantiate(hipGraphExec_t*, hipGraph_t, hipGraphNode_t*, char*, size_t)
{
    return hipErrorNotSupported;
}
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return hipErrorNotSupported; }

}  // extern "C"
