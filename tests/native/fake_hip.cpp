// A host-only HIP runtime for tests of the engine's host code: device memory is host
// memory, kernels do not run.  It keeps the runtime's error state as HIP 7 does (an
// error stays pending until hipGetLastError takes it, whatever succeeds after it), can
// refuse memory and launches, and watches the order of launches and events.
#include <hip/hip_runtime.h>

#include <cstdlib>
#include <cstring>
#include <map>
#include <vector>

namespace {
hipError_t g_last = hipSuccess;
size_t g_in_use = 0, g_limit = ~(size_t)0;
std::map<void *, size_t> g_mem;
int g_fail_launch = -1;          // launches until one is refused (-1: never)
long g_seq = 0;                  // launches so far
std::map<hipStream_t, long> g_stream_last;   // last launch of a stream not waited for since
struct Event {
    long seq = -1;               // launches when it was recorded (-1: never)
};
int g_stale = 0;                 // stream waits on an event with unfinished launches behind it
struct Launch {
    unsigned gx, gy, gz, bx;
    size_t lds;
};
std::vector<Launch> g_launches;
dim3 g_grid, g_block;
size_t g_shmem;
hipStream_t g_cfg_stream;

hipError_t err(hipError_t e) {
    if (e != hipSuccess) g_last = e;
    return e;
}
}  // namespace

extern "C" {
// control
void fake_reset() {
    g_last = hipSuccess;
    g_limit = ~(size_t)0;
    g_fail_launch = -1;
    g_stale = 0;
    g_launches.clear();
}
void fake_memory_limit(size_t bytes) { g_limit = bytes; }
size_t fake_in_use() { return g_in_use; }
void fake_fail_launch(int after) { g_fail_launch = after; }
int fake_stale_waits() { return g_stale; }
int fake_pending() { return (int)g_last; }
int fake_launch_count() { return (int)g_launches.size(); }
void fake_launch(int i, unsigned *grid, unsigned *block, size_t *lds) {
    grid[0] = g_launches[i].gx; grid[1] = g_launches[i].gy; grid[2] = g_launches[i].gz;
    *block = g_launches[i].bx;
    *lds = g_launches[i].lds;
}

// errors, devices
hipError_t hipGetLastError() {
    const hipError_t e = g_last;
    g_last = hipSuccess;
    return e;
}
hipError_t hipPeekAtLastError() { return g_last; }
const char *hipGetErrorString(hipError_t) { return "fake"; }
hipError_t hipGetDeviceCount(int *n) { *n = 1; return hipSuccess; }
hipError_t hipGetDevice(int *d) { *d = 0; return hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipDeviceSynchronize() { g_stream_last.clear(); return hipSuccess; }
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600 *p, int) {
    memset(p, 0, sizeof *p);
    strcpy(p->gcnArchName, "gfx950");
    return hipSuccess;
}
hipError_t hipGetSymbolAddress(void **p, const void *s) { *p = const_cast<void *>(s); return hipSuccess; }

// memory
hipError_t hipMalloc(void **p, size_t n) {
    *p = nullptr;
    if (g_in_use + n > g_limit) return err(hipErrorOutOfMemory);
    *p = malloc(n);
    g_in_use += n;
    g_mem[*p] = n;
    return hipSuccess;
}
hipError_t hipFree(void *p) {   // waits for the device
    if (!p) return hipSuccess;
    g_stream_last.clear();
    g_in_use -= g_mem[p];
    g_mem.erase(p);
    free(p);
    return hipSuccess;
}
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind) { memcpy(d, s, n); return hipSuccess; }
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t) { memcpy(d, s, n); return hipSuccess; }
hipError_t hipMemsetAsync(void *d, int v, size_t n, hipStream_t) { memset(d, v, n); return hipSuccess; }

// streams, events, graphs
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) { *s = (hipStream_t)malloc(8); return hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t s) { free((void *)s); return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t s) { g_stream_last.erase(s); return hipSuccess; }
hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus *c) { *c = hipStreamCaptureStatusNone; return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t e, unsigned) {
    for (const auto &s : g_stream_last)
        if (s.second > ((Event *)e)->seq) {
            ++g_stale;
            break;
        }
    return hipSuccess;
}
hipError_t hipEventCreate(hipEvent_t *e) { *e = (hipEvent_t) new Event; return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { return hipEventCreate(e); }
hipError_t hipEventDestroy(hipEvent_t e) { delete (Event *)e; return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t) { ((Event *)e)->seq = g_seq; return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t) { *ms = 1.f; return hipSuccess; }
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return hipSuccess; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t *g) { *g = (hipGraph_t)malloc(8); return hipSuccess; }
hipError_t hipGraphInstantiate(hipGraphExec_t *x, hipGraph_t, hipGraphNode_t *, char *, size_t) { *x = (hipGraphExec_t)malloc(8); return hipSuccess; }
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t s) { g_stream_last[s] = ++g_seq; return hipSuccess; }
hipError_t hipGraphDestroy(hipGraph_t g) { free((void *)g); return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t x) { free((void *)x); return hipSuccess; }

// launches
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t shmem, hipStream_t s) {
    g_grid = g; g_block = b; g_shmem = shmem; g_cfg_stream = s;
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3 *g, dim3 *b, size_t *shmem, hipStream_t *s) {
    *g = g_grid; *b = g_block; *shmem = g_shmem; *s = g_cfg_stream;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void *, dim3 g, dim3 b, void **, size_t lds, hipStream_t s) {
    if (g_fail_launch >= 0 && g_fail_launch-- == 0) return err(hipErrorLaunchFailure);
    g_launches.push_back({g.x, g.y, g.z, b.x, lds});
    g_stream_last[s] = ++g_seq;
    return hipSuccess;
}
char fake_fatbin[64];   // stands for the objects' device code
void **__hipRegisterFatBinary(const void *) { static void *h; return &h; }
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterFunction(void **, const void *, char *, const char *, unsigned, void *, void *, void *, void *, int *) {}
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}
}
