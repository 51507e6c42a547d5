// A stand-in for the parts of the HIP runtime that liblgx's host code calls,
// so that its rules (which kernel, which grid, how much memory) run without a
// device: allocations are numbers, launches are recorded and checked against
// the runtime's launch limits.  Loaded with RTLD_GLOBAL before liblgx.so.
#define __HIP_PLATFORM_AMD__
#include <hip/hip_runtime.h>

#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <string>

static std::string g_log;
static size_t g_next = (size_t)1 << 40;

extern "C" {

const char* stub_log() { return g_log.c_str(); }
void stub_reset() { g_log.clear(); }

hipError_t hipGetDeviceCount(int* n) { *n = 1; return hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDeviceProperties(hipDeviceProp_t* p, int) {   // the header's name for the R0600 symbol
    std::memset(p, 0, sizeof *p);
    std::strcpy(p->gcnArchName, "gfx950:sramecc+:xnack-");
    return hipSuccess;
}
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t a, int) {
    *v = a == hipDeviceAttributeMultiprocessorCount ? 256 : a == hipDeviceAttributeMaxSharedMemoryPerBlock ? 65536 : 0;
    return hipSuccess;
}
hipError_t hipModuleLoad(hipModule_t* m, const char*) { *m = (hipModule_t)1; return hipSuccess; }
hipError_t hipModuleUnload(hipModule_t) { return hipSuccess; }
hipError_t hipModuleGetFunction(hipFunction_t* f, hipModule_t, const char* name) {
    *f = (hipFunction_t)strdup(name);
    return hipSuccess;
}
hipError_t hipGetSymbolAddress(void** p, const void*) { *p = (void*)((size_t)1 << 39); return hipSuccess; }
hipError_t hipMalloc(void** p, size_t bytes) {
    if (bytes > (size_t)288 << 30) return hipErrorOutOfMemory;   // the device's memory
    *p = (void*)g_next;
    g_next += (bytes + 4095) / 4096 * 4096;
    g_log += "malloc " + std::to_string(bytes) + "\n";
    return hipSuccess;
}
hipError_t hipFree(void*) { return hipSuccess; }
hipError_t hipModuleLaunchKernel(hipFunction_t f, unsigned gx, unsigned gy, unsigned gz, unsigned bx, unsigned by,
                                 unsigned bz, unsigned, hipStream_t, void**, void**) {
    // threads of each dimension below 2^32, at most 65535 workgroups along y and z
    if (!gx || !gy || !gz || (uint64_t)gx * bx > UINT32_MAX || (uint64_t)gy * by > UINT32_MAX ||
        (uint64_t)gz * bz > UINT32_MAX || gy > 65535 || gz > 65535)
        return hipErrorInvalidConfiguration;
    char line[256];
    std::snprintf(line, sizeof line, "%s %u %u %u %u\n", (const char*)f, gx, gy, gz, bx);
    g_log += line;
    return hipSuccess;
}
const char* hipGetErrorString(hipError_t) { return "stub error"; }

}  // extern "C"
