/* TEST INFRASTRUCTURE ONLY: the HIP entry points that libtopopt_hip imports, on host
 * memory: allocations are calloc'ed and counted, copies are memcpy, kernels and graphs
 * do nothing.  stub_fail_in(n) makes the n-th allocation from now fail (0: none),
 * stub_fail_graphs(1) every launch of a graph (nothing else ends an iteration here).
 * Memory starts as doubles of 1. */
#include <stddef.h>
#include <stdlib.h>
#include <string.h>

static long g_live, g_bytes, g_count, g_fail_in;
static int g_last;

struct block {
    size_t n;
    char pad[48];
};

static int g_fail_graphs;

void stub_fail_in(long n) { g_fail_in = n; }
void stub_fail_graphs(int f) { g_fail_graphs = f; }
long stub_live(void) { return g_live; }
long stub_bytes(void) { return g_bytes; }
long stub_count(void) { return g_count; }

int hipMalloc(void** p, size_t n) {
    ++g_count;
    if (g_fail_in > 0 && --g_fail_in == 0) return g_last = 2;
    struct block* b = calloc(1, sizeof(struct block) + n);
    if (!b) return g_last = 2;
    b->n = n;
    for (size_t i = 0; i < n / sizeof(double); ++i) ((double*)(b + 1))[i] = 1.0;
    g_live += 1;
    g_bytes += (long)n;
    *p = b + 1;
    return 0;
}
int hipFree(void* p) {
    if (p) {
        struct block* b = (struct block*)p - 1;
        g_live -= 1;
        g_bytes -= (long)b->n;
        free(b);
    }
    return 0;
}
int hipHostMalloc(void** p, size_t n, unsigned f) { return (*p = calloc(1, n)) ? 0 : 2; }
int hipHostFree(void* p) {
    free(p);
    return 0;
}
int hipMemcpy(void* d, const void* s, size_t n, int k) {
    memcpy(d, s, n);
    return 0;
}
int hipMemcpyAsync(void* d, const void* s, size_t n, int k, void* q) {
    memcpy(d, s, n);
    return 0;
}
int hipMemsetAsync(void* d, int v, size_t n, void* q) {
    memset(d, v, n);
    return 0;
}
int hipMemGetInfo(size_t* f, size_t* t) {
    *f = *t = (size_t)1 << 38;
    return 0;
}
int hipGetDevice(int* d) {
    *d = 0;
    return 0;
}
int hipGetDeviceCount(int* n) {
    *n = 1;
    return 0;
}
/* the last error of any call, until it is asked for */
int hipGetLastError(void) {
    int e = g_last;
    g_last = 0;
    return e;
}
const char* hipGetErrorString(int e) { return e == 2 ? "out of memory" : "stub"; }
int hipFuncSetAttribute(const void* f, int a, int v) { return 0; }
int hipGetSymbolAddress(void** p, const void* s) {
    static double scratch[1 << 16];
    *p = scratch;
    return 0;
}
static int handle(void** p) {
    static char h[1];
    *p = h;
    return 0;
}
int hipStreamCreateWithFlags(void** s, unsigned f) { return handle(s); }
int hipStreamDestroy(void* s) { return 0; }
int hipStreamSynchronize(void* s) { return 0; }
int hipStreamWaitEvent(void* s, void* e, unsigned f) { return 0; }
int hipStreamBeginCapture(void* s, int m) { return 0; }
int hipStreamEndCapture(void* s, void** g) { return handle(g); }
int hipGraphInstantiate(void** e, void* g, void** n, char* l, size_t z) { return handle(e); }
int hipGraphDestroy(void* g) { return 0; }
int hipGraphExecDestroy(void* e) { return 0; }
int hipGraphLaunch(void* e, void* s) { return g_fail_graphs ? (g_last = 719) : 0; }
int hipEventCreate(void** e) { return handle(e); }
int hipEventCreateWithFlags(void** e, unsigned f) { return handle(e); }
int hipEventDestroy(void* e) { return 0; }
int hipEventRecord(void* e, void* s) { return 0; }
int hipEventSynchronize(void* e) { return 0; }
int hipEventElapsedTime(float* ms, void* a, void* b) {
    *ms = 0;
    return 0;
}
struct dim {
    unsigned x, y, z;
};
int hipLaunchKernel(const void* f, struct dim g, struct dim b, void** a, size_t l, void* s) {
    return 0;
}
