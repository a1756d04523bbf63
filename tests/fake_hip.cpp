// A HIP runtime of two imaginary GPUs for tests of the engine's host side: device memory is host memory, kernels do
// nothing, and every allocation, launch, event and stream is held against the device that the calling thread has
// current.  Loaded before the engine with RTLD_GLOBAL, it takes the place of the real runtime.
#include <hip/hip_runtime_api.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>
#include <map>
#include <string>

namespace {

thread_local int current = 0;
thread_local hipError_t last_error = hipSuccess;      // until it is asked for
int expected = 0;
int n_checked = 0, n_wrong = 0;
char first_wrong[128];

struct Owned {          // a stream or an event
    int device;
};

void check(const char *what, bool ok) {
    n_checked++;
    if (ok) return;
    if (n_wrong++ == 0) snprintf(first_wrong, sizeof first_wrong, "%s with device %d current", what, current);
}

struct Config {
    dim3 grid, block;
    size_t shared;
    hipStream_t stream;
};
thread_local Config pushed;

std::map<const void *, std::string> kernel_names;
std::map<std::string, std::pair<int, int>> answers;     // by part of a kernel's name
std::map<void *, size_t> sizes;                         // of the device's allocations
size_t held = 0, limit = ~(size_t)0 / 2;
int cus = 256;
std::string launched;       // "name grid;" of every launch since fake_launches was last asked

}  // namespace

extern "C" {

// --- for the test
void fake_thread_device(int device) { current = device; }
void fake_expect(int device) { expected = device; n_checked = n_wrong = 0; first_wrong[0] = 0; }
int fake_checked() { return n_checked; }
const char *fake_wrong() { return n_wrong ? first_wrong : nullptr; }
const char *fake_launches() {
    static std::string out;
    out.swap(launched);
    launched.clear();
    return out.c_str();
}

size_t fake_held() { return held; }
void fake_limit(size_t bytes) { limit = bytes; }
void fake_cus(int n) { cus = n; }
// kernels of this name publish a result: their arguments (by number) are where its sequence number goes, and the number
void fake_answer(const char *name, int host_seq, int seq) { answers[name] = {host_seq, seq}; }

// --- the runtime
hipError_t hipGetDeviceCount(int *n) { *n = 2; return hipSuccess; }
hipError_t hipGetDeviceProperties(hipDeviceProp_t *p, int) {       // (the header's name for the versioned symbol)
    memset(p, 0, sizeof *p);
    strcpy(p->gcnArchName, "gfx950");
    p->multiProcessorCount = cus;
    return hipSuccess;
}
hipError_t hipSetDevice(int d) { current = d; return hipSuccess; }
hipError_t hipGetLastError() {
    const hipError_t e = last_error;
    last_error = hipSuccess;
    return e;
}
hipError_t hipFuncSetAttribute(const void *, hipFuncAttribute, int) { check("hipFuncSetAttribute", current == expected); return hipSuccess; }

hipError_t hipMalloc(void **p, size_t n) {
    check("hipMalloc", current == expected);
    *p = held + n <= limit ? calloc(1, n) : nullptr;
    if (!*p) return last_error = hipErrorOutOfMemory;
    held += sizes[*p] = n;
    return hipSuccess;
}
hipError_t hipHostMalloc(void **p, size_t n, unsigned) { *p = calloc(1, n); return *p ? hipSuccess : hipErrorOutOfMemory; }
hipError_t hipFree(void *p) {
    const auto it = sizes.find(p);
    if (it != sizes.end()) held -= it->second, sizes.erase(it);
    free(p);
    return hipSuccess;
}
hipError_t hipHostFree(void *p) { free(p); return hipSuccess; }
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t) { memcpy(d, s, n); return hipSuccess; }
hipError_t hipGetSymbolAddress(void **p, const void *) {
    static void *image[2];
    check("hipGetSymbolAddress", current == expected);
    if (!image[current]) image[current] = calloc(1, 40u << 20);
    *p = image[current];
    return hipSuccess;
}

hipError_t hipStreamCreate(hipStream_t *s) { check("hipStreamCreate", current == expected); *s = (hipStream_t) new Owned{current}; return hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t s) { delete (Owned *)s; return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t *e) { check("hipEventCreate", current == expected); *e = (hipEvent_t) new Owned{current}; return hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t e) { delete (Owned *)e; return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
    check("hipEventRecord", current == expected && ((Owned *)e)->device == current && (!s || ((Owned *)s)->device == current));
    return hipSuccess;
}
hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t) { *ms = 0.0f; return hipSuccess; }

hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t shared, hipStream_t stream) { pushed = {grid, block, shared, stream}; return hipSuccess; }
hipError_t __hipPopCallConfiguration(dim3 *grid, dim3 *block, size_t *shared, hipStream_t *stream) {
    *grid = pushed.grid;
    *block = pushed.block;
    *shared = pushed.shared;
    *stream = pushed.stream;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void *f, dim3 grid, dim3, void **args, size_t, hipStream_t s) {
    for (const auto &a : answers)
        if (kernel_names[f].find(a.first) != std::string::npos)
            **(unsigned long long **)args[a.second.first] = *(unsigned long long *)args[a.second.second];
    launched += kernel_names[f] + " " + std::to_string(grid.x) + ";";
    check("hipLaunchKernel", current == expected && (!s || ((Owned *)s)->device == current));
    return hipSuccess;
}
void **__hipRegisterFatBinary(const void *) { static void *handle; return &handle; }
void __hipRegisterFunction(void **, const void *f, char *, const char *name, unsigned, void *, void *, dim3 *, dim3 *, int *) { kernel_names[f] = name; }
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}
void __hipUnregisterFatBinary(void **) {}

}  // extern "C"
