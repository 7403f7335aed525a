// The HIP calls of the library's host paths on host memory, for CPU tests
// (preloaded in front of the runtime): allocations are malloc's, copies are
// memcpy's, kernels do nothing.  Every call that the tests look at is printed
// on stderr; TQEC_STUB_FAIL names one that fails.
#include <hip/hip_runtime.h>

#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <string>

static std::map<const void *, std::string> &kernels() {
    static std::map<const void *, std::string> m;
    return m;
}
static hipError_t g_last = hipSuccess;

static hipError_t call(const char *name) {
    const char *f = getenv("TQEC_STUB_FAIL");
    const bool bad = f && !strcmp(f, name);
    fprintf(stderr, "stub %s%s\n", name, bad ? " failed" : "");
    return bad ? (g_last = hipErrorUnknown) : hipSuccess;
}

extern "C" {
hipError_t hipGetDevice(int *d) { *d = 0; return hipSuccess; }
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_t *p, int) {
    memset(p, 0, sizeof *p);
    p->sharedMemPerBlock = p->maxSharedMemoryPerMultiProcessor = 160 * 1024;
    p->multiProcessorCount = 256;
    return hipSuccess;
}
hipError_t hipFuncSetAttribute(const void *, hipFuncAttribute, int) { return hipSuccess; }
hipError_t hipMalloc(void **p, size_t n) { *p = malloc(n ? n : 1); return hipSuccess; }
hipError_t hipFree(void *p) { free(p); return hipSuccess; }
hipError_t hipHostMalloc(void **p, size_t n, unsigned) { *p = malloc(n ? n : 1); return hipSuccess; }
hipError_t hipHostFree(void *p) { free(p); return hipSuccess; }
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind) { memcpy(d, s, n); return hipSuccess; }
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind k, hipStream_t) {
    const hipError_t e = call(k == hipMemcpyHostToDevice ? "copy_in" : "copy_out");
    if (!e) memcpy(d, s, n);
    return e;
}
hipError_t hipMemset(void *d, int v, size_t n) { memset(d, v, n); return hipSuccess; }
hipError_t hipDeviceSynchronize() { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t *e) { *e = nullptr; return hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t) {   // everything later is slower
    static float t = 0;
    *ms = t += 1;
    return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t) { return call("wait"); }
hipError_t __hipPushCallConfiguration(dim3, dim3, size_t, hipStream_t) { return hipSuccess; }
hipError_t __hipPopCallConfiguration(dim3 *, dim3 *, size_t *, hipStream_t *) { return hipSuccess; }
void __hipRegisterFunction(void **, const void *host, char *, const char *name, unsigned, void *, void *, void *, void *,
                           int *) {
    kernels()[host] = name;
}
hipError_t hipLaunchKernel(const void *f, dim3, dim3, void **, size_t, hipStream_t) {
    fprintf(stderr, "stub kernel %s\n", kernels()[f].c_str());
    return call("launch");
}
// modules are numbered from 1; TQEC_STUB_OCC: the workgroups per CU of each, a digit apiece
hipError_t hipModuleLoadData(hipModule_t *m, const void *image) {
    static size_t n = 0;
    *m = (hipModule_t)++n;
    // the kernel's LDS, from its metadata (a big-endian 16- or 32-bit number follows the key)
    const char key[] = ".group_segment_fixed_size";
    const unsigned char *p = (const unsigned char *)image;
    while (memcmp(p, key, sizeof key - 1)) ++p;
    p += sizeof key - 1;
    const unsigned lds = *p == 0xcd ? p[1] << 8 | p[2] : *p == 0xce ? p[1] << 24 | p[2] << 16 | p[3] << 8 | p[4] : *p;
    fprintf(stderr, "stub lds %u\n", lds);
    return call("load");
}
hipError_t hipModuleUnload(hipModule_t) { return call("unload"); }
hipError_t hipModuleGetFunction(hipFunction_t *f, hipModule_t m, const char *) {
    *f = (hipFunction_t)m;
    return hipSuccess;
}
hipError_t hipModuleOccupancyMaxActiveBlocksPerMultiprocessor(int *n, hipFunction_t f, int, size_t) {
    const char *occ = getenv("TQEC_STUB_OCC");
    const size_t i = (size_t)f - 1;
    *n = occ && i < strlen(occ) ? occ[i] - '0' : 2;
    return hipSuccess;
}
hipError_t hipModuleLaunchKernel(hipFunction_t f, unsigned, unsigned, unsigned, unsigned, unsigned, unsigned, unsigned,
                                 hipStream_t, void **, void **) {
    fprintf(stderr, "stub module %zu\n", (size_t)f);
    return call("launch");
}
hipError_t hipGetLastError() {
    const hipError_t e = g_last;
    g_last = hipSuccess;
    return e;
}
}
