// launch_record.cpp -- the library's host side without a GPU: libemel_hip's
// own objects linked to these stand-ins for the HIP runtime, which record
// each kernel launch (name, grid, block, LDS) and run nothing.  A launch of
// 2^32 or more work-items in a dimension, which HIP does not support, is
// refused as the runtime does.  Tests ask which kernels a call takes, and
// whether extents too large to allocate are still accepted
// (tests/launch_recorder.py).
#include <cxxabi.h>
#include <hip/hip_runtime_api.h>

#include <cstdlib>
#include <cstring>
#include <map>
#include <string>
#include <vector>

namespace {

struct Launch {
    std::string name;
    uint64_t grid, block, lds;
};

std::map<const void *, std::string> &names()
{
    static std::map<const void *, std::string> m;
    return m;
}

std::vector<Launch> g_launches;
hipError_t g_last = hipSuccess;

struct Config {
    dim3 grid, block;
    size_t lds;
    hipStream_t stream;
};
std::vector<Config> g_configs;

} // namespace

extern "C" {

uint64_t record_count() { return g_launches.size(); }
void record_clear() { g_launches.clear(); }
const char *record_name(uint64_t i) { return g_launches[i].name.c_str(); }
uint64_t record_grid(uint64_t i) { return g_launches[i].grid; }
uint64_t record_block(uint64_t i) { return g_launches[i].block; }
uint64_t record_lds(uint64_t i) { return g_launches[i].lds; }

void **__hipRegisterFatBinary(const void *)
{
    static void *handle;
    return &handle;
}
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}
void __hipRegisterFunction(void **, const void *host, char *, const char *device, unsigned, void *, void *, void *, void *, int *)
{
    int status = 0;
    char *plain = abi::__cxa_demangle(device, nullptr, nullptr, &status);
    names()[host] = status == 0 ? plain : device;
    std::free(plain);
}

hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t lds, hipStream_t stream)
{
    g_configs.push_back({grid, block, lds, stream});
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3 *grid, dim3 *block, size_t *lds, hipStream_t *stream)
{
    const Config c = g_configs.back();
    g_configs.pop_back();
    *grid = c.grid;
    *block = c.block;
    *lds = c.lds;
    *stream = c.stream;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void *fn, dim3 grid, dim3 block, void **, size_t lds, hipStream_t)
{
    const uint64_t items[3] = {uint64_t{grid.x} * block.x, uint64_t{grid.y} * block.y, uint64_t{grid.z} * block.z};
    for (uint64_t n : items)
        if (n == 0 || n >> 32) return g_last = hipErrorInvalidConfiguration;
    g_launches.push_back({names()[fn], uint64_t{grid.x} * grid.y * grid.z, uint64_t{block.x} * block.y * block.z, lds});
    return hipSuccess;
}
hipError_t hipGetLastError()
{
    const hipError_t e = g_last;
    g_last = hipSuccess;
    return e;
}
const char *hipGetErrorString(hipError_t) { return "recorded error"; }

hipError_t hipGetDevice(int *dev)
{
    *dev = 0;
    return hipSuccess;
}
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDeviceCount(int *n)
{
    *n = 1;
    return hipSuccess;
}
#undef hipGetDeviceProperties
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600 *p, int)
{
    std::memset(static_cast<void *>(p), 0, sizeof *p);
    std::strcpy(p->gcnArchName, "gfx950");
    p->multiProcessorCount = 256;
    return hipSuccess;
}
hipError_t hipDeviceGetAttribute(int *value, hipDeviceAttribute_t, int)
{
    *value = 256; // compute units
    return hipSuccess;
}
hipError_t hipDeviceSynchronize() { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t *, unsigned) { return hipErrorNotSupported; }
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus *status)
{
    *status = hipStreamCaptureStatusNone;
    return hipSuccess;
}
hipError_t hipMalloc(void **p, size_t bytes)
{
    *p = std::aligned_alloc(256, (bytes + 255) / 256 * 256);
    return *p ? hipSuccess : hipErrorOutOfMemory;
}
hipError_t hipFree(void *p)
{
    std::free(p);
    return hipSuccess;
}
hipError_t hipHostMalloc(void **p, size_t bytes, unsigned) { return hipMalloc(p, bytes); }
hipError_t hipHostFree(void *p) { return hipFree(p); }
hipError_t hipMemcpyAsync(void *, const void *, size_t, hipMemcpyKind, hipStream_t) { return hipSuccess; }
hipError_t hipMemsetAsync(void *, int, size_t, hipStream_t) { return hipSuccess; }
hipError_t hipGetSymbolAddress(void **p, const void *)
{
    static char symbol[1 << 20];
    *p = symbol;
    return hipSuccess;
}

} // extern "C"
