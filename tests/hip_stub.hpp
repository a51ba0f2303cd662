// A HIP runtime for the CPU, as far as the library's host code needs one: memory is the host's, a launch is recorded by its
// kernel's name and does nothing.  (The kernels themselves are not compiled: tests/host_library.py.)
#pragma once

#include <cxxabi.h>
#include <hip/hip_runtime.h>

#include <cstdlib>
#include <cstring>
#include <map>
#include <string>
#include <vector>

struct HipStub {
    std::map<const void *, std::string> names;  // of the kernels' host handles
    std::vector<std::string> launched;
    bool capturing = false;  // what hipStreamIsCapturing says
    static HipStub &get() {
        static HipStub stub;
        return stub;
    }
    // the launches since the last call: kernels and their template arguments, without parameters
    std::string take() {
        std::string all;
        for (const std::string &name : launched) all += (all.empty() ? "" : " ") + name;
        launched.clear();
        return all.empty() ? "-" : all;
    }
};
extern "C" {
hipError_t __hipPushCallConfiguration(dim3, dim3, size_t, hipStream_t) { return hipSuccess; }
hipError_t __hipPopCallConfiguration(dim3 *g, dim3 *b, size_t *lds, hipStream_t *s) { return *g = *b = dim3(1), *lds = 0, *s = nullptr, hipSuccess; }
void **__hipRegisterFatBinary(const void *) { static void *handle; return &handle; }
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterFunction(void **, const void *host, char *, const char *mangled, unsigned, void *, void *, void *, void *, int *) {
    int status = 0;
    char *plain = abi::__cxa_demangle(mangled, nullptr, nullptr, &status);
    std::string name = plain ? plain : mangled;
    free(plain);
    if (name.compare(0, 5, "void ") == 0) name = name.substr(5);
    name = name.substr(0, name.find('('));  // (no template argument has a parenthesis)
    std::string out;
    for (size_t i = 0; i < name.size(); i++) {
        if (name.compare(i, 5, "frk::") == 0) i += 4;
        else if (name[i] != ' ') out += name[i];
    }
    HipStub::get().names[host] = out;
}
hipError_t hipLaunchKernel(const void *f, dim3, dim3, void **, size_t, hipStream_t) { return HipStub::get().launched.push_back(HipStub::get().names[f]), hipSuccess; }
hipError_t hipMalloc(void **p, size_t n) { return (*p = calloc(1, n)) ? hipSuccess : hipErrorOutOfMemory; }
hipError_t hipHostMalloc(void **p, size_t n, unsigned) { return hipMalloc(p, n); }
hipError_t hipFree(void *p) { return free(p), hipSuccess; }
hipError_t hipMemcpy(void *to, const void *from, size_t n, hipMemcpyKind) { return memcpy(to, from, n), hipSuccess; }
hipError_t hipMemcpyAsync(void *to, const void *from, size_t n, hipMemcpyKind, hipStream_t) { return memcpy(to, from, n), hipSuccess; }
hipError_t hipMemsetAsync(void *to, int v, size_t n, hipStream_t) { return memset(to, v, n), hipSuccess; }
hipError_t hipMemGetInfo(size_t *f, size_t *t) { return *f = *t = (size_t)288 << 30, hipSuccess; }
hipError_t hipGetDevice(int *dev) { return *dev = 0, hipSuccess; }
hipError_t hipGetDeviceCount(int *n) { return *n = 1, hipSuccess; }
hipError_t hipDeviceGetAttribute(int *v, hipDeviceAttribute_t, int) { return *v = 256, hipSuccess; }
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600 *p, int) {
    memset(p, 0, sizeof *p);
    strcpy(p->gcnArchName, "gfx950");
    p->multiProcessorCount = 256;
    return hipSuccess;
}
hipError_t hipGetLastError() { return hipSuccess; }
const char *hipGetErrorString(hipError_t) { return "an error"; }
hipError_t hipFuncSetAttribute(const void *, hipFuncAttribute, int) { return hipSuccess; }
hipError_t hipGetSymbolAddress(void **p, const void *) {
    static void *image = calloc(1, (size_t)96 << 20);
    return *p = image, hipSuccess;
}
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) { return *s = (hipStream_t)malloc(1), hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus *cs) {
    return *cs = HipStub::get().capturing ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone, hipSuccess;
}
hipError_t hipThreadExchangeStreamCaptureMode(hipStreamCaptureMode *) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t *e) { return *e = (hipEvent_t)malloc(1), hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { return hipEventCreate(e); }
hipError_t hipEventDestroy(hipEvent_t e) { return free(e), hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventQuery(hipEvent_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t) { return *ms = 1.0f, hipSuccess; }
}
