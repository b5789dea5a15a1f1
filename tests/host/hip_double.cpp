// A HIP runtime on the host for tests of the renderer's host code: device memory is host memory,
// copies are immediate and kernels do not run.  Loaded before libpathed.so it takes the place of
// the runtime's functions, so that what the host does when an allocation fails, and what it hands
// to a kernel, can be tested without a GPU.
#include <hip/hip_runtime_api.h>

#include <cstdlib>
#include <cstring>
#include <map>
#include <string>
#include <vector>

struct ihipStream_t {
    int device;
};
struct ihipEvent_t {
    int device;
};

namespace {

struct Block {
    size_t bytes;
    bool live;
};
struct Launch {
    std::string name;
    dim3 grid, block;
    std::vector<char> arg;   // the watched argument
};
std::map<char *, Block> blocks;   // freed blocks keep their addresses, so none is taken for another
std::map<const void *, std::string> kernels;
std::vector<Launch> launches;
std::string watchName;
int watchArg = -1;
size_t watchBytes = 0;
int mallocs = 0, failAt = 0;
int deviceCount = 1;
thread_local int device = 0;
thread_local dim3 cfgGrid, cfgBlock;
thread_local size_t cfgShared;
thread_local hipStream_t cfgStream;

}  // namespace

extern "C" {

// --- what a test sets and asks -----------------------------------------------------------------
void double_devices(int n) { deviceCount = n; }
// the n-th allocation from here fails (0: none)
void double_fail_at(int n) {
    mallocs = 0;
    failAt = n;
}
// launches of kernels whose mangled name contains `name` keep their argument `index`
void double_watch(const char *name, int index, size_t bytes) {
    watchName = name;
    watchArg = index;
    watchBytes = bytes;
    launches.clear();
}
int double_launches() { return (int)launches.size(); }
const char *double_name(int k) { return launches[k].name.c_str(); }
void double_grid(int k, unsigned *out) {
    out[0] = launches[k].grid.x;
    out[1] = launches[k].block.x;
}
void double_arg(int k, void *out) { memcpy(out, launches[k].arg.data(), launches[k].arg.size()); }
// bytes from p to the end of the live block that holds it; 0: none does
size_t double_room(void *p) {
    auto it = blocks.upper_bound((char *)p);
    if (it == blocks.begin()) return 0;
    --it;
    const char *end = it->first + it->second.bytes;
    return it->second.live && (char *)p < end ? (size_t)(end - (char *)p) : 0;
}

// --- the runtime ---------------------------------------------------------------------------------
hipError_t hipGetDeviceCount(int *n) { return *n = deviceCount, hipSuccess; }
hipError_t hipGetDevice(int *d) { return *d = device, hipSuccess; }
hipError_t hipSetDevice(int d) {
    if (d < 0 || d >= deviceCount) return hipErrorInvalidDevice;
    device = d;
    return hipSuccess;
}
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600 *p, int) {
    memset(p, 0, sizeof *p);
    p->multiProcessorCount = 256;
    return hipSuccess;
}
hipError_t hipDeviceGetAttribute(int *v, hipDeviceAttribute_t, int) { return *v = 100000, hipSuccess; }
const char *hipGetErrorString(hipError_t e) { return e == hipErrorOutOfMemory ? "out of memory" : "error"; }
hipError_t hipGetLastError() { return hipSuccess; }

hipError_t hipMalloc(void **p, size_t n) {
    if (++mallocs == failAt) return hipErrorOutOfMemory;
    *p = calloc(1, n);
    if (!*p) return hipErrorOutOfMemory;
    blocks[(char *)*p] = Block{n, true};
    return hipSuccess;
}
hipError_t hipFree(void *p) {
    if (!p) return hipSuccess;
    auto it = blocks.find((char *)p);
    if (it == blocks.end() || !it->second.live) return hipErrorInvalidValue;
    it->second.live = false;
    return hipSuccess;
}
hipError_t hipHostMalloc(void **p, size_t n, unsigned) { return *p = calloc(1, n), hipSuccess; }
hipError_t hipHostFree(void *p) { return free(p), hipSuccess; }
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind) {
    if (n == 0) return hipSuccess;
    if (!d || !s) return hipErrorInvalidValue;
    memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind k, hipStream_t) { return hipMemcpy(d, s, n, k); }
hipError_t hipMemsetAsync(void *d, int v, size_t n, hipStream_t) { return memset(d, v, n), hipSuccess; }

hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) { return *s = new ihipStream_t{device}, hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t s) { return delete s, hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamGetDevice(hipStream_t s, hipDevice_t *d) { return *d = s ? s->device : device, hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { return *e = new ihipEvent_t{device}, hipSuccess; }
hipError_t hipEventCreate(hipEvent_t *e) { return hipEventCreateWithFlags(e, 0); }
hipError_t hipEventDestroy(hipEvent_t e) { return delete e, hipSuccess; }
// an event belongs to the device that was current when it was made
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) { return s && s->device != e->device ? hipErrorInvalidHandle : hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventQuery(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t) { return *ms = 1.f, hipSuccess; }

hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return hipSuccess; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t *g) { return *g = nullptr, hipSuccess; }
hipError_t hipGraphInstantiate(hipGraphExec_t *e, hipGraph_t, hipGraphNode_t *, char *, size_t) { return *e = nullptr, hipSuccess; }
hipError_t hipGraphGetNodes(hipGraph_t, hipGraphNode_t *, size_t *n) { return *n = 0, hipSuccess; }
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return hipSuccess; }
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }

void **__hipRegisterFatBinary(const void *) {
    static void *handle;
    return &handle;
}
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterFunction(void **, const void *f, char *, const char *name, unsigned, void *, void *, dim3 *, dim3 *, int *) { kernels[f] = name; }
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}
hipError_t hipGetSymbolAddress(void **p, const void *) { return *p = calloc(1, 1 << 26), hipSuccess; }
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t shared, hipStream_t s) {
    cfgGrid = g;
    cfgBlock = b;
    cfgShared = shared;
    cfgStream = s;
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3 *g, dim3 *b, size_t *shared, hipStream_t *s) {
    *g = cfgGrid;
    *b = cfgBlock;
    *shared = cfgShared;
    *s = cfgStream;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void *f, dim3 g, dim3 b, void **args, size_t, hipStream_t) {
    const std::string &name = kernels[f];
    if (watchArg < 0 || name.find(watchName) == std::string::npos) return hipSuccess;
    const char *a = (const char *)args[watchArg];
    launches.push_back(Launch{name, g, b, std::vector<char>(a, a + watchBytes)});
    return hipSuccess;
}

}  // extern "C"
