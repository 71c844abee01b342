// HIP runtime that records instead of running, behind tests/cpu_hip/include/hip/hip_runtime.h -- TEST
// INFRASTRUCTURE ONLY.  Kernels are not executed: a launch is checked against HIP's limits and written to a
// log with its stream, as are event records and waits, so that tests see what the host code would ask of a
// GPU: grids, the order of streams, the life of device memory.  Memory is host memory whose frees are
// tracked.
#include <hip/hip_runtime.h>

#include <dlfcn.h>
#include <map>
#include <set>
#include <string>

namespace emu {
thread_local Idx tid, bid;
Idx bdim, gdim;
thread_local hipStream_t launch_stream = nullptr;
thread_local void *launch_kernel = nullptr;
thread_local size_t launch_bytes = 0;
void *dyn_lds() { return nullptr; }
void sync_block() {}
void sync_wave() {}
void *wave_buf(int) { return nullptr; }
int lane() { return 0; }
}  // namespace emu

namespace {
struct Op {
    char kind;  // 'L' launch, 'R' event record, 'W' wait for an event, 'F' free, 'S' wait of the host
    hipStream_t stream;
    void *what;               // event, address or kernel
    unsigned long long grid;  // workgroups of a launch
    unsigned block;
};
std::mutex mu;
std::condition_variable cv;
hipStream_t held = nullptr;  // launches on this stream ...
std::string held_kernel;     // ... of kernels with this in their name wait ...
int launches_left = 0;       // ... after so many more of them
std::vector<Op> ops;
std::map<void *, size_t> live, freed;  // freed blocks are kept, so that no address is used twice
int errors = 0;            // launches that HIP refuses
int stale = 0;             // launches with an address in a freed block among their arguments
void (*on_instantiate)() = nullptr;
thread_local int last = 0;
long next_handle = 16;
void log(Op o) {
    std::lock_guard<std::mutex> l(mu);
    ops.push_back(o);
}
}  // namespace

extern "C" const char *rec_kernel(void *k) {
    Dl_info i;
    return dladdr(k, &i) && i.dli_sname ? i.dli_sname : "";
}

// HIP takes at most 2^32 - 1 work items in a dimension and 1024 in a workgroup
void emu::run_grid(dim3 g, dim3 b, size_t shm, void (*)(void *), void *args) {
    const bool bad = (unsigned long long)g.x * b.x >= (1ull << 32) || (unsigned long long)g.y * b.y >= (1ull << 32) ||
                     (unsigned long long)g.z * b.z >= (1ull << 32) || g.y > 65535 || g.z > 65535 || g.x == 0 || g.y == 0 ||
                     g.z == 0 || b.x * b.y * b.z > 1024 || shm > 160 * 1024;
    std::unique_lock<std::mutex> l(mu);
    auto mine = [] {
        return held && held == emu::launch_stream && strstr(rec_kernel(emu::launch_kernel), held_kernel.c_str());
    };
    cv.wait(l, [&] { return !mine() || launches_left > 0; });
    if (mine()) --launches_left;
    if (bad) {
        ++errors;
        last = 9;  // invalid configuration
        return;
    }
    for (size_t i = 0; i + 8 <= emu::launch_bytes; i += 8) {
        char *p = *(char **)((char *)args + i);
        auto it = freed.upper_bound(p);
        if (it != freed.begin() && p < (char *)std::prev(it)->first + std::prev(it)->second) {
            ++stale;
            break;
        }
    }
    ops.push_back(Op{'L', emu::launch_stream, emu::launch_kernel, (unsigned long long)g.x * g.y * g.z, b.x});
}

extern "C" {
void rec_reset() {
    std::lock_guard<std::mutex> l(mu);
    ops.clear();
    errors = stale = 0;
}
int rec_stale() { return stale; }
void rec_on_instantiate(void (*f)()) { on_instantiate = f; }
// launches of kernels named *kernel* on `stream` (null: none) wait once `after` more of them have been made, until
// the next call
void rec_hold(void *stream, const char *kernel, int after) {
    std::lock_guard<std::mutex> l(mu);
    held = stream;
    held_kernel = kernel;
    launches_left = after;
    cv.notify_all();
}
int rec_errors() { return errors; }
int rec_count() {
    std::lock_guard<std::mutex> l(mu);
    return (int)ops.size();
}
void rec_op(int i, char *kind, void **stream, void **what, unsigned long long *grid, unsigned *block) {
    std::lock_guard<std::mutex> l(mu);
    *kind = ops[i].kind, *stream = ops[i].stream, *what = ops[i].what, *grid = ops[i].grid, *block = ops[i].block;
}
long long rec_live_bytes() {
    std::lock_guard<std::mutex> l(mu);
    long long n = 0;
    for (auto &kv : live) n += (long long)kv.second;
    return n;
}
}

hipError_t hipGetLastError() {
    const int e = last;
    last = 0;
    return e;
}
const char *hipGetErrorString(hipError_t e) { return e == 9 ? "invalid configuration argument" : "recorded"; }
hipError_t hipMalloc(void **p, size_t n) {
    std::lock_guard<std::mutex> l(mu);
    *p = malloc(n ? n : 1);
    live[*p] = n;
    return hipSuccess;
}
hipError_t hipFree(void *p) {
    std::lock_guard<std::mutex> l(mu);
    auto it = live.find(p);
    if (it == live.end()) return 1;
    freed[p] = it->second;
    live.erase(it);
    ops.push_back(Op{'F', nullptr, p, 0, 0});
    return hipSuccess;
}
hipError_t hipMemGetInfo(size_t *f, size_t *t) {
    *f = *t = (size_t)256 << 30;
    return hipSuccess;
}
hipError_t hipGetDevice(int *d) {
    *d = 0;
    return hipSuccess;
}
hipError_t hipGetDeviceProperties(hipDeviceProp_t *p, int) {
    snprintf(p->gcnArchName, sizeof(p->gcnArchName), "gfx950:recorded");
    p->multiProcessorCount = 256;
    return hipSuccess;
}
hipError_t hipFuncSetAttribute(const void *, int attr, int value) {
    return attr == hipFuncAttributeMaxDynamicSharedMemorySize && value > 160 * 1024;
}
hipError_t hipDeviceGetAttribute(int *v, int, int) {
    *v = 256;
    return hipSuccess;
}
hipError_t hipMemcpy(void *, const void *, size_t, hipMemcpyKind) { return hipSuccess; }
hipError_t hipMemcpyAsync(void *, const void *, size_t, hipMemcpyKind, hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t s) {
    log(Op{'S', s, nullptr, 0, 0});
    return hipSuccess;
}
hipError_t hipDeviceSynchronize() {
    log(Op{'S', nullptr, nullptr, 0, 0});
    return hipSuccess;
}
static hipError_t handle(void **h) {
    std::lock_guard<std::mutex> l(mu);
    *h = (void *)(next_handle += 16);
    return hipSuccess;
}
hipError_t hipEventCreate(hipEvent_t *e) { return handle(e); }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { return handle(e); }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
    log(Op{'R', s, e, 0, 0});
    return hipSuccess;
}
hipError_t hipStreamWaitEvent(hipStream_t s, hipEvent_t e, unsigned) {
    log(Op{'W', s, e, 0, 0});
    return hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t e) {
    log(Op{'S', nullptr, e, 0, 0});
    return hipSuccess;
}
hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t) {
    *ms = 1.0f;
    return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) { return handle(s); }
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return hipSuccess; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t *g) { return handle(g); }
hipError_t hipGraphInstantiate(hipGraphExec_t *x, hipGraph_t, hipGraphNode_t *, char *, size_t) {
    if (on_instantiate) on_instantiate();
    return handle(x);
}
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }
