/* The HIP runtime calls of libemerge_amd.so, recorded on the CPU: device memory is host memory within a budget,
 * kernels do nothing, and every call that orders work is written to a log.  Loaded with global symbols
 * before the library (tests/host_calls.py), so that its host code runs here: what it allocates, what it does
 * when memory runs out, and in which order it launches, copies and waits.  Host memory of C++ containers has a
 * limit too (build with -fexceptions). */
#define _GNU_SOURCE
#include <dlfcn.h>
#include <stdarg.h>
#include <stdint.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

enum { SUCCESS = 0, OUT_OF_MEMORY = 2 };

static char *g_log;
static size_t g_len, g_cap;
static size_t g_used, g_budget = (size_t)-1;
static int g_capturing, g_events, g_errors;

static void say(const char *fmt, ...) {
    char line[256];
    va_list ap;
    va_start(ap, fmt);
    const int n = vsnprintf(line, sizeof line - 1, fmt, ap);
    va_end(ap);
    if (g_len + n + 2 > g_cap) g_log = realloc(g_log, g_cap = 2 * g_cap + 4096);
    memcpy(g_log + g_len, line, n);
    g_log[g_len + n] = '\n';
    g_log[g_len += n + 1] = 0;
}
const char *rec_log(void) { return g_log ? g_log : ""; }
void rec_clear(void) { g_len = 0; if (g_log) g_log[0] = 0; }
void rec_budget(size_t bytes) { g_budget = bytes; }
size_t rec_used(void) { return g_used; }
void rec_capturing(int on) { g_capturing = on; }
int rec_last_error(void) { return g_errors; }

/* ---- kernels: names by the host function that stands for them */
struct kernel { const void *host; char name[160]; };
static struct kernel *g_kernel;
static int g_kernels, g_kernel_room;
void **__hipRegisterFatBinary(const void *data) { (void)data; static void *handle; return &handle; }
void __hipUnregisterFatBinary(void **m) { (void)m; }
void __hipRegisterVar(void *m, void *v, char *h, char *d, int e, size_t s, int c, int g) { (void)m; (void)v; (void)h; (void)d; (void)e; (void)s; (void)c; (void)g; }
void __hipRegisterFunction(void **m, const void *host, char *dev, const char *name, unsigned t, void *a, void *b, void *c, void *d, int *w) {
    (void)m; (void)dev; (void)t; (void)a; (void)b; (void)c; (void)d; (void)w;
    if (g_kernels == g_kernel_room) g_kernel = realloc(g_kernel, (g_kernel_room = 2 * g_kernel_room + 4096) * sizeof *g_kernel);
    g_kernel[g_kernels].host = host;
    snprintf(g_kernel[g_kernels++].name, sizeof g_kernel[0].name, "%s", name);
}
/* the function's own name in a mangled one (its length stands before it), or all of it */
static const char *bare(const char *name, int *n) {
    *n = (int)strlen(name);
    for (const char *k = strstr(name, "k_"); k; k = strstr(k + 1, "k_")) {
        const char *d = k;
        while (d > name && d[-1] >= '0' && d[-1] <= '9') d--;
        if (d < k) { *n = atoi(d); return k; }
    }
    return name;
}
typedef struct { unsigned x, y, z; } dim3;
static dim3 g_grid, g_block;
static size_t g_shmem;
static void *g_stream;
int __hipPushCallConfiguration(dim3 g, dim3 b, size_t shmem, void *st) { g_grid = g; g_block = b; g_shmem = shmem; g_stream = st; return SUCCESS; }
int __hipPopCallConfiguration(dim3 *g, dim3 *b, size_t *shmem, void **st) { *g = g_grid; *b = g_block; *shmem = g_shmem; *st = g_stream; return SUCCESS; }
int hipLaunchKernel(const void *host, dim3 g, dim3 b, void **args, size_t shmem, void *st) {
    (void)b; (void)args; (void)shmem;
    for (int i = 0; i < g_kernels; i++)
        if (g_kernel[i].host == host) {
            int n;
            const char *name = bare(g_kernel[i].name, &n);
            say("launch %.*s grid %u,%u stream %zu", n, name, g.x, g.y, (size_t)st);
            return SUCCESS;
        }
    say("launch ? stream %zu", (size_t)st);
    return SUCCESS;
}

/* ---- memory: the size is kept in front of the block */
static int take(void **p, size_t n) {
    if (n > g_budget || g_used > g_budget - n) { *p = NULL; g_errors = OUT_OF_MEMORY; return OUT_OF_MEMORY; }
    char *q = calloc(1, n + 64);
    if (!q) { g_errors = OUT_OF_MEMORY; return OUT_OF_MEMORY; }
    *(size_t *)q = n;
    g_used += n;
    *p = q + 64;
    return SUCCESS;
}
int hipMalloc(void **p, size_t n) { const int rc = take(p, n); say("malloc %zu -> %d", n, rc); return rc; }
int hipMallocAsync(void **p, size_t n, void *st) { (void)st; const int rc = take(p, n); say("malloc %zu -> %d", n, rc); return rc; }
int hipFree(void *p) {
    if (!p) return SUCCESS;
    char *q = (char *)p - 64;
    say("free %zu", *(size_t *)q);
    g_used -= *(size_t *)q;
    free(q);
    return SUCCESS;
}
int hipFreeAsync(void *p, void *st) { (void)st; return hipFree(p); }
int hipHostMalloc(void **p, size_t n, unsigned f) { (void)f; *p = calloc(1, n); return SUCCESS; }
int hipHostFree(void *p) { free(p); return SUCCESS; }
int hipHostGetDevicePointer(void **d, void *h, unsigned f) { (void)f; *d = h; return SUCCESS; }
int hipMemset(void *p, int v, size_t n) { memset(p, v, n); say("memset"); return SUCCESS; }
int hipMemsetAsync(void *p, int v, size_t n, void *st) { memset(p, v, n); say("memset stream %zu", (size_t)st); return SUCCESS; }
int hipMemcpy(void *d, const void *s, size_t n, int k) { (void)k; memcpy(d, s, n); say("memcpy"); return SUCCESS; }
int hipMemcpyAsync(void *d, const void *s, size_t n, int k, void *st) { (void)k; memcpy(d, s, n); say("copy %zu stream %zu", n, (size_t)st); return SUCCESS; }

/* ---- operator new: blocks above a limit are refused as the C++ library refuses them */
static size_t g_host_block = (size_t)-1;
void rec_host_block(size_t bytes) { g_host_block = bytes; }
void *_Znwm(size_t n) {
    void *p = n > g_host_block ? NULL : malloc(n ? n : 1);
    if (!p) ((void (*)(void))dlsym(RTLD_DEFAULT, "_ZSt17__throw_bad_allocv"))();
    return p;
}
void _ZdlPv(void *p) { free(p); }
void _ZdlPvm(void *p, size_t n) { (void)n; free(p); }

/* ---- order: streams, events, graphs */
int hipStreamCreateWithFlags(void **st, unsigned f) { (void)f; *st = (void *)(size_t)1000; return SUCCESS; }
int hipStreamDestroy(void *st) { (void)st; return SUCCESS; }
int hipStreamSynchronize(void *st) { say("wait stream %zu", (size_t)st); return SUCCESS; }
int hipStreamIsCapturing(void *st, int *status) { (void)st; *status = g_capturing; return SUCCESS; }
int hipThreadExchangeStreamCaptureMode(int *mode) { (void)mode; return SUCCESS; }
int hipStreamBeginCapture(void *st, int mode) { (void)mode; say("capture stream %zu", (size_t)st); return SUCCESS; }
int hipStreamEndCapture(void *st, void **graph) { (void)st; *graph = (void *)(size_t)1; return SUCCESS; }
int hipGraphInstantiate(void **e, void *g, void *a, void *b, size_t n) { (void)g; (void)a; (void)b; (void)n; *e = (void *)(size_t)1; return SUCCESS; }
int hipGraphLaunch(void *e, void *st) { (void)e; say("graph stream %zu", (size_t)st); return SUCCESS; }
int hipGraphDestroy(void *g) { (void)g; return SUCCESS; }
int hipGraphExecDestroy(void *e) { (void)e; return SUCCESS; }
int hipEventCreate(void **e) { *e = (void *)(size_t)++g_events; return SUCCESS; }
int hipEventCreateWithFlags(void **e, unsigned f) { (void)f; return hipEventCreate(e); }
int hipEventDestroy(void *e) { (void)e; return SUCCESS; }
int hipEventRecord(void *e, void *st) { say("record event %zu stream %zu", (size_t)e, (size_t)st); return SUCCESS; }
int hipStreamWaitEvent(void *st, void *e, unsigned f) { (void)f; say("stream %zu waits for event %zu", (size_t)st, (size_t)e); return SUCCESS; }
int hipEventSynchronize(void *e) { (void)e; say("wait event"); return SUCCESS; }
int hipEventElapsedTime(float *ms, void *a, void *b) { (void)a; (void)b; *ms = 1.0f; return SUCCESS; }

/* ---- the device */
int hipGetDevice(int *d) { *d = 0; return SUCCESS; }
int hipGetStreamDeviceId(void *st) { (void)st; return 0; }
int hipDeviceGetAttribute(int *v, int a, int d) { (void)a; (void)d; *v = 256; return SUCCESS; }
int hipGetDevicePropertiesR0600(void *p, int d) { (void)d; memset(p, 0, 1024); strcpy(p, "recorder"); return SUCCESS; }
int hipGetSymbolAddress(void **p, const void *s) { *p = (void *)(uintptr_t)s; return SUCCESS; }
int hipGetLastError(void) { const int e = g_errors; g_errors = SUCCESS; return e; }
const char *hipGetErrorString(int e) { return e == OUT_OF_MEMORY ? "out of memory" : e ? "error" : "no error"; }
