// The HIP runtime calls that libplk.so makes, on the CPU: device memory is host memory, copies
// are done at once, and a kernel launch is recorded and not run.  Loaded before libplk.so
// (RTLD_GLOBAL), so that the library's host code, which plans and launches, can be tested
// without a device.  The one-launch Newton solves are played: their exchange places are looked
// at and filled or emptied as dev_newton.h says, and their states finish at the first guess.
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <string>
#include <vector>

#include "engine_common.h"

using namespace plk;

namespace {

struct Launch {
    std::string name;
    dim3 grid, block;
    size_t lds;
};
struct Config {
    dim3 grid, block;
    size_t lds;
    hipStream_t stream;
};
std::vector<Launch> g_launches;
std::vector<Config> g_config;
std::map<const void *, std::string> g_names;
std::map<void *, size_t> g_sizes;
size_t g_bytes = 0;
hipError_t g_last = hipSuccess;
std::string g_fail;       // a launch of a kernel with this in its name fails
int g_finish = 1;         // one-launch solves finish (0: every wait ends)
int g_dirty = 0;          // exchange places found not empty by the launch that uses them
const double *g_hands[2] = {};

bool empty(double v) {
    uint64_t b;
    std::memcpy(&b, &v, 8);
    return b == ~0ull;
}
void play_hand(const HandArea &h, int64_t len) {
    for (int64_t i = 0; i < len; i++) g_dirty += !empty(h.use[i]);
    for (int64_t i = 0; i < len; i++) h.use[i] = 1.0;
    std::memset(h.spare, 0xff, sizeof(double) * h.spare_len);
    g_hands[0] = h.use;
    g_hands[1] = h.spare;
}
void play_state(const NewtonState &start, NewtonState *out) {
    if (!g_finish) return;
    NewtonState s = start;
    s.done = 1;
    s.status = NEWTON_OK;
    s.out = s.x_eval = s.rts;
    s.evals = 1;
    *out = s;
}
hipError_t alloc(void **p, size_t n) {
    *p = std::calloc(1, n ? n : 1);
    if (!*p) return hipErrorOutOfMemory;
    g_sizes[*p] = n;
    g_bytes += n;
    return hipSuccess;
}
hipError_t release(void *p) {
    if (!p) return hipSuccess;
    g_bytes -= g_sizes[p];
    g_sizes.erase(p);
    std::free(p);
    return hipSuccess;
}

}  // namespace

extern "C" {

// ---- the tests' side
int rec_count() { return (int)g_launches.size(); }
const char *rec_name(int i) { return g_launches[i].name.c_str(); }
long rec_lds(int i) { return (long)g_launches[i].lds; }
long rec_blocks(int i) { return (long)g_launches[i].grid.x * g_launches[i].grid.y; }
long rec_threads(int i) { return (long)g_launches[i].block.x; }
void rec_clear() { g_launches.clear(); }
void rec_fail(const char *name) { g_fail = name; }
void rec_finish(int on) { g_finish = on; }
int rec_dirty() { return g_dirty; }
long rec_bytes() { return (long)g_bytes; }

// ---- the runtime's
void **__hipRegisterFatBinary(const void *) {
    static void *one;
    return &one;
}
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}
void __hipRegisterFunction(void **, const void *host, char *, const char *name, unsigned, void *, void *, dim3 *, dim3 *, int *) {
    g_names[host] = name;
}
hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t lds, hipStream_t s) {
    g_config.push_back({grid, block, lds, s});
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3 *grid, dim3 *block, size_t *lds, hipStream_t *s) {
    const Config c = g_config.back();
    g_config.pop_back();
    *grid = c.grid;
    *block = c.block;
    *lds = c.lds;
    *s = c.stream;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void *f, dim3 grid, dim3 block, void **args, size_t lds, hipStream_t) {
    const std::string &name = g_names[f];
    if (!g_fail.empty() && name.find(g_fail) != std::string::npos) return g_last = hipErrorInvalidValue;
    g_launches.push_back({name, grid, block, lds});
    if (name.find("k_newton_solve_multi") != std::string::npos) {
        const int nwg = *(int *)args[1], nbr = (int)grid.x / nwg;
        const NewtonState *start = *(const NewtonState **)args[3];
        play_hand(*(HandArea *)args[4], *(int64_t *)args[2] * nbr);
        for (int i = 0; i < nbr; i++) play_state(start[i], *(NewtonState **)args[5] + i);
    } else if (name.find("k_newton_solve") != std::string::npos) {
        play_hand(*(HandArea *)args[2], (int64_t)newton_hand_len(((KParams *)args[0])->ntiles));
        play_state(*(NewtonState *)args[1], *(NewtonState **)args[3]);
    }
    return hipSuccess;
}
hipError_t hipGetLastError() {
    const hipError_t e = g_last;
    g_last = hipSuccess;
    return e;
}
const char *hipGetErrorString(hipError_t e) { return e == hipErrorInvalidValue ? "invalid value" : "error"; }
hipError_t hipGetDeviceCount(int *n) { return *n = 1, hipSuccess; }
hipError_t hipGetDevice(int *d) { return *d = 0, hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipDeviceGetAttribute(int *v, hipDeviceAttribute_t a, int) {
    *v = a == hipDeviceAttributeMultiprocessorCount ? 256 : 0;
    return hipSuccess;
}
hipError_t hipDeviceGetDefaultMemPool(hipMemPool_t *p, int) { return *p = nullptr, hipSuccess; }
hipError_t hipMemPoolSetAttribute(hipMemPool_t, hipMemPoolAttr, void *) { return hipSuccess; }
hipError_t hipMalloc(void **p, size_t n) { return alloc(p, n); }
hipError_t hipMallocAsync(void **p, size_t n, hipStream_t) { return alloc(p, n); }
hipError_t hipHostMalloc(void **p, size_t n, unsigned) { return alloc(p, n); }
hipError_t hipFree(void *p) { return release(p); }
hipError_t hipFreeAsync(void *p, hipStream_t) { return release(p); }
hipError_t hipHostFree(void *p) { return release(p); }
hipError_t hipHostGetDevicePointer(void **d, void *h, unsigned) { return *d = h, hipSuccess; }
hipError_t hipGetSymbolAddress(void **p, const void *) { return alloc(p, 1 << 20); }
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind) { return std::memcpy(d, s, n), hipSuccess; }
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t) { return std::memcpy(d, s, n), hipSuccess; }
hipError_t hipMemsetAsync(void *d, int v, size_t n, hipStream_t) { return std::memset(d, v, n), hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) { return *s = (hipStream_t)1, hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return hipSuccess; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t *g) { return *g = (hipGraph_t)1, hipSuccess; }
hipError_t hipGraphInstantiate(hipGraphExec_t *e, hipGraph_t, hipGraphNode_t *, char *, size_t) { return *e = (hipGraphExec_t)1, hipSuccess; }
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return hipSuccess; }
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t *e) { return *e = (hipEvent_t)1, hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t) { return *ms = 0.0f, hipSuccess; }

}  // extern "C"
