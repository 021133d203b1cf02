/* Stand-in for the HIP runtime on host memory, for tests of the library's host code without a device: device
 * allocations come from calloc and are counted, a chosen one can be made to fail, kernels do not run, and what
 * they would leave in the counters of the active bricks is given by the test. Built as a shared library with
 * the runtime's soname and loaded before libbnn_flip.so, whose references then bind to it. */
#include <stddef.h>
#include <stdint.h>
#include <stdlib.h>
#include <string.h>

typedef struct {
    unsigned x, y, z;
} dim3;

enum { kMaxBlocks = 4096, kOutOfMemory = 2, kCopyToHost = 2 };
static void*    block[kMaxBlocks];
static size_t   blockBytes[kMaxBlocks];
static size_t   live;
static long     failAt = -1, mallocs;
static uint32_t counts[64];
static size_t   countBytes;

/* the n-th hipMalloc from now fails (0: the next one); -1: none does */
void stub_fail_at(long n) {
    failAt  = n;
    mallocs = 0;
}
long   stub_mallocs(void) { return mallocs; } /* since stub_fail_at */
size_t stub_live_bytes(void) { return live; }
long   stub_live_blocks(void) {
    long n = 0;
    for(int i = 0; i < kMaxBlocks; ++i) n += block[i] != NULL;
    return n;
}
/* what a copy to the host of exactly n words reads (the active bricks' counters) */
void stub_set_counts(const uint32_t* v, uint32_t n) {
    memcpy(counts, v, 4 * (size_t)n);
    countBytes = 4 * (size_t)n;
}

int hipMalloc(void** p, size_t n) {
    *p = NULL;
    if(mallocs++ == failAt) return kOutOfMemory;
    for(int i = 0; i < kMaxBlocks; ++i)
        if(!block[i]) {
            block[i]      = calloc(1, n);
            blockBytes[i] = n;
            live += n;
            *p = block[i];
            return block[i] ? 0 : kOutOfMemory;
        }
    return kOutOfMemory;
}
int hipFree(void* p) {
    for(int i = 0; p && i < kMaxBlocks; ++i)
        if(block[i] == p) {
            live -= blockBytes[i];
            block[i] = NULL;
            free(p);
            return 0;
        }
    return p ? 1 : 0;
}
int hipHostMalloc(void** p, size_t n, unsigned f) {
    (void)f;
    *p = calloc(1, n);
    return *p ? 0 : kOutOfMemory;
}
int hipHostFree(void* p) {
    free(p);
    return 0;
}
int hipMemcpyAsync(void* d, const void* s, size_t n, int kind, void* st) {
    (void)st;
    memcpy(d, kind == kCopyToHost && n == countBytes ? (const void*)counts : s, n);
    return 0;
}
int hipMemsetAsync(void* d, int v, size_t n, void* st) {
    (void)st;
    memset(d, v, n);
    return 0;
}
int hipLaunchKernel(const void* f, dim3 g, dim3 b, void** a, size_t sh, void* st) {
    (void)f, (void)g, (void)b, (void)a, (void)sh, (void)st;
    return 0;
}
int __hipPushCallConfiguration(dim3 g, dim3 b, size_t sh, void* st) {
    (void)g, (void)b, (void)sh, (void)st;
    return 0;
}
int __hipPopCallConfiguration(dim3* g, dim3* b, size_t* sh, void** st) {
    g->x = g->y = g->z = b->x = b->y = b->z = 1;
    *sh = 0;
    *st = NULL;
    return 0;
}
static void* fatBinary;
void** __hipRegisterFatBinary(const void* d) {
    (void)d;
    return &fatBinary;
}
void __hipUnregisterFatBinary(void** m) { (void)m; }
void __hipRegisterFunction(void** m, const void* h, char* d, const char* n, unsigned l, void* a, void* b, void* c, void* e, int* w) {
    (void)m, (void)h, (void)d, (void)n, (void)l, (void)a, (void)b, (void)c, (void)e, (void)w;
}
void __hipRegisterVar(void** m, void* v, char* h, char* d, int e, size_t n, int c, int g) {
    (void)m, (void)v, (void)h, (void)d, (void)e, (void)n, (void)c, (void)g;
}
static int handle;
int hipStreamCreateWithFlags(void** s, unsigned f) {
    (void)f;
    *s = &handle;
    return 0;
}
int hipEventCreate(void** e) {
    *e = &handle;
    return 0;
}
int hipEventElapsedTime(float* ms, void* a, void* b) {
    (void)a, (void)b;
    *ms = 0;
    return 0;
}
int hipGetDevice(int* d) {
    *d = 0;
    return 0;
}
int hipGetSymbolAddress(void** p, const void* s) {
    *p = (void*)s;
    return 0;
}
const char* hipGetErrorString(int e) { return e == kOutOfMemory ? "out of memory" : "error"; }
#define NOTHING(name, ...)       \
    int name(__VA_ARGS__) { return 0; }
NOTHING(hipEventDestroy, void* e)
NOTHING(hipEventRecord, void* e, void* s)
NOTHING(hipGetLastError, void)
NOTHING(hipSetDevice, int d)
NOTHING(hipStreamDestroy, void* s)
NOTHING(hipStreamSynchronize, void* s)
NOTHING(hipStreamBeginCapture, void* s, int m)
NOTHING(hipStreamEndCapture, void* s, void** g)
NOTHING(hipGraphDestroy, void* g)
NOTHING(hipGraphExecDestroy, void* g)
NOTHING(hipGraphInstantiate, void** e, void* g, void* n, char* l, size_t z)
NOTHING(hipGraphLaunch, void* e, void* s)
