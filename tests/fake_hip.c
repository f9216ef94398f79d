/* A HIP runtime of host memory in which kernels do nothing: the C-ABI's host paths on a machine
 * without a GPU, and failures that the real runtime gives only in trouble.  Loaded RTLD_GLOBAL before
 * libmsm_hip.so (tests/test_host_paths.py); fake_* are the test's controls. */
#include <pthread.h>
#include <stddef.h>
#include <stdlib.h>
#include <string.h>

typedef int err_t; /* hipError_t */
typedef struct { unsigned x, y, z; } dim3_t;
enum { OK = 0, OUT_OF_MEMORY = 2, LAUNCH_FAILED = 719 };

static __thread err_t last;
static pthread_mutex_t mu = PTHREAD_MUTEX_INITIALIZER;

/* kernels and their launches */
static struct { const void* host; const char* name; int launches; } fn[4096];
static int nfn;
static char refuse[128];    /* launches of kernels with this in their name are refused */
static long host_limit = -1, dev_limit = -1;    /* allocations beyond this many bytes fail */
static int dev_fail;    /* k > 0: the k-th device allocation from now fails */
static long host_allocs, host_bytes, dev_bytes, memsets;

void fake_refuse(const char* part) { strncpy(refuse, part, sizeof(refuse) - 1); }
void fake_host_limit(long bytes) { host_limit = bytes; }
void fake_dev_limit(long bytes) { dev_limit = bytes; }
static int time_fail;   /* k > 0: the k-th reading of an event pair from now fails */
void fake_time_fail(int k) { time_fail = k; }
void fake_dev_fail(int k) { dev_fail = k; }
long fake_host_bytes(void) { return host_bytes; }
long fake_host_allocs(void) { return host_allocs; }
long fake_dev_bytes(void) { return dev_bytes; }
long fake_memsets(void) { return memsets; }
int fake_launches(const char* part) {
    int n = 0;
    for (int k = 0; k < nfn; ++k)
        if (strstr(fn[k].name, part)) n += fn[k].launches;
    return n;
}

static err_t fail(err_t e) { return last = e; }
err_t hipGetLastError(void) { err_t e = last; last = OK; return e; }
err_t hipPeekAtLastError(void) { return last; }
const char* hipGetErrorString(err_t e) { return e ? "fake error" : "no error"; }

void** __hipRegisterFatBinary(const void* d) { static void* h; (void)d; return &h; }
void __hipUnregisterFatBinary(void** h) { (void)h; }
void __hipRegisterFunction(void** m, const void* host, char* dev, const char* name, unsigned lim,
                           void* a, void* b, void* c, void* d, int* e) {
    (void)m; (void)dev; (void)lim; (void)a; (void)b; (void)c; (void)d; (void)e;
    if (nfn < 4096) { fn[nfn].host = host; fn[nfn].name = name; fn[nfn].launches = 0; ++nfn; }
}
void __hipRegisterVar(void** m, void* var, char* h, char* d, int ext, size_t size, int c, int g) {
    (void)m; (void)var; (void)h; (void)d; (void)ext; (void)size; (void)c; (void)g;
}
err_t hipGetSymbolAddress(void** p, const void* sym) {
    static char* s;
    (void)sym;
    if (!s) s = calloc(1, 4 << 20);
    *p = s;
    return OK;
}

static __thread struct { dim3_t g, b; size_t lds; void* s; } cfg;
err_t __hipPushCallConfiguration(dim3_t g, dim3_t b, size_t lds, void* s) {
    cfg.g = g; cfg.b = b; cfg.lds = lds; cfg.s = s;
    return OK;
}
err_t __hipPopCallConfiguration(dim3_t* g, dim3_t* b, size_t* lds, void** s) {
    *g = cfg.g; *b = cfg.b; *lds = cfg.lds; *s = cfg.s;
    return OK;
}
err_t hipLaunchKernel(const void* f, dim3_t g, dim3_t b, void** args, size_t lds, void* s) {
    (void)g; (void)b; (void)args; (void)lds; (void)s;
    for (int k = 0; k < nfn; ++k)
        if (fn[k].host == f) {
            if (refuse[0] && strstr(fn[k].name, refuse)) return fail(LAUNCH_FAILED);
            ++fn[k].launches;
            return OK;
        }
    return fail(LAUNCH_FAILED);
}

err_t hipGetDeviceCount(int* n) { *n = 1; return OK; }
err_t hipGetDevice(int* d) { *d = 0; return OK; }
err_t hipSetDevice(int d) { (void)d; return OK; }
err_t hipDeviceGetAttribute(int* v, int attr, int dev) { (void)attr; (void)dev; *v = 163840; return OK; }
err_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int* n, const void* f, int b, size_t l) {
    (void)f; (void)b; (void)l;
    *n = 1;
    return OK;
}

/* memory: filled with 0x5a, its size in front */
static err_t take(void** p, size_t n, long limit, long* total) {
    pthread_mutex_lock(&mu);
    if (limit >= 0 && (long)n > limit) { pthread_mutex_unlock(&mu); *p = 0; return fail(OUT_OF_MEMORY); }
    *total += (long)n;
    pthread_mutex_unlock(&mu);
    char* q = malloc(n + 64);
    *(size_t*)q = n;
    memset(q + 64, 0x5a, n);
    *p = q + 64;
    return OK;
}
static err_t give(void* p, long* total) {
    if (!p) return OK;
    pthread_mutex_lock(&mu);
    *total -= (long)*(size_t*)((char*)p - 64);
    pthread_mutex_unlock(&mu);
    free((char*)p - 64);
    return OK;
}
err_t hipMalloc(void** p, size_t n) {
    if (dev_fail && --dev_fail == 0) { *p = 0; return fail(OUT_OF_MEMORY); }
    return take(p, n, dev_limit, &dev_bytes);
}
err_t hipFree(void* p) { return give(p, &dev_bytes); }
err_t hipHostMalloc(void** p, size_t n, unsigned f) {
    (void)f;
    ++host_allocs;
    return take(p, n, host_limit, &host_bytes);
}
err_t hipHostFree(void* p) { return give(p, &host_bytes); }
err_t hipHostGetDevicePointer(void** d, void* h, unsigned f) { (void)f; *d = h; return OK; }
err_t hipMemcpy(void* d, const void* s, size_t n, int k) { (void)k; memcpy(d, s, n); return OK; }
err_t hipMemcpyAsync(void* d, const void* s, size_t n, int k, void* st) {
    (void)k; (void)st;
    memcpy(d, s, n);
    return OK;
}
err_t hipMemset(void* d, int v, size_t n) { ++memsets; memset(d, v, n); return OK; }
err_t hipMemsetAsync(void* d, int v, size_t n, void* s) { (void)s; return hipMemset(d, v, n); }

err_t hipStreamCreateWithFlags(void** s, unsigned f) { (void)f; *s = malloc(8); return OK; }
err_t hipStreamDestroy(void* s) { free(s); return OK; }
err_t hipStreamSynchronize(void* s) { (void)s; return OK; }
err_t hipStreamQuery(void* s) { (void)s; return OK; }
err_t hipStreamBeginCapture(void* s, int m) { (void)s; (void)m; return OK; }
err_t hipStreamEndCapture(void* s, void** g) { (void)s; *g = malloc(8); return OK; }
err_t hipGraphDestroy(void* g) { free(g); return OK; }
err_t hipGraphInstantiate(void** e, void* g, void** n, char* l, size_t z) {
    (void)g; (void)n; (void)l; (void)z;
    *e = malloc(8);
    return OK;
}
err_t hipGraphExecDestroy(void* e) { free(e); return OK; }
err_t hipGraphLaunch(void* e, void* s) { (void)e; (void)s; return OK; }
err_t hipEventCreate(void** e) { *e = malloc(8); return OK; }
err_t hipEventCreateWithFlags(void** e, unsigned f) { (void)f; return hipEventCreate(e); }
err_t hipEventDestroy(void* e) { free(e); return OK; }
err_t hipEventRecord(void* e, void* s) { (void)e; (void)s; return OK; }
err_t hipEventSynchronize(void* e) { (void)e; return OK; }
err_t hipEventElapsedTime(float* ms, void* a, void* b) { 
    (void)a; (void)b;
    *ms = 0.001f;
    return time_fail && --time_fail == 0 ? fail(LAUNCH_FAILED) : OK;
}
