/* The HIP runtime calls of libkevernals_amd on host memory, without kernels:
 * for CPU tests of the library's host side (what it allocates, frees, waits
 * for and launches, and in which order).  Loaded before the library, with its
 * symbols global.  Device memory is calloc memory within a budget; a launch
 * only appends the kernel's name to the log. */
#include <stddef.h>
#include <stdint.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

typedef struct { uint32_t x, y, z; } dim3_t;

static size_t budget = (size_t)1 << 40, used;
static int capture, last_error;
static dim3_t last_grid;
static char log_text[1 << 20];
static struct { const void *host; char name[512]; } fn[512];
static int nfn;
static char scratch[1 << 20];

static void note(const char *what)
{
    if (strlen(log_text) + strlen(what) + 2 < sizeof log_text) {
        strcat(log_text, what);
        strcat(log_text, "\n");
    }
}
static int fail(int e) { return last_error = e; }

/* ---- the test's side ---- */
void fake_budget(size_t bytes) { budget = bytes; }
size_t fake_used(void) { return used; }
void fake_capture(int on) { capture = on; }
const char *fake_log(void) { return log_text; }
void fake_log_clear(void) { log_text[0] = 0; }
unsigned fake_grid_z(void) { return last_grid.z; } /* of the last launch */
int fake_kernels(void) { return nfn; }
const char *fake_kernel(int i) { return fn[i].name; }

/* ---- memory ---- */
int hipMalloc(void **p, size_t n)
{
    *p = NULL;
    if (n > budget || used > budget - n)
        return fail(2);
    size_t *q = calloc(1, n + 256);
    if (!q)
        return fail(2);
    *q = n;
    used += n;
    *p = (char *)q + 256;
    return 0;
}
int hipFree(void *p)
{
    if (p) {
        size_t *q = (size_t *)((char *)p - 256);
        used -= *q;
        free(q);
    }
    return 0;
}
int hipMemGetInfo(size_t *avail, size_t *total)
{
    *avail = budget > used ? budget - used : 0;
    *total = budget;
    return 0;
}
int hipMemcpy(void *d, const void *s, size_t n, int k) { (void)k; memcpy(d, s, n); return 0; }
int hipMemcpyAsync(void *d, const void *s, size_t n, int k, void *st) { (void)k; (void)st; memcpy(d, s, n); return 0; }
int hipMemsetAsync(void *d, int v, size_t n, void *st) { (void)st; memset(d, v, n); return 0; }
int hipGetSymbolAddress(void **p, const void *s) { (void)s; *p = scratch; return 0; }

/* ---- device, streams, events, graphs ---- */
int hipGetDeviceCount(int *n) { *n = 1; return 0; }
int hipSetDevice(int d) { (void)d; return 0; }
int hipGetDevicePropertiesR0600(void *p, int d) { (void)p; (void)d; return 0; }
const char *hipGetErrorString(int e) { return e == 2 ? "out of memory" : "error"; }
int hipGetLastError(void) { int e = last_error; last_error = 0; return e; }
int hipStreamCreateWithFlags(void **s, unsigned f) { (void)f; *s = malloc(1); return 0; }
int hipStreamDestroy(void *s) { free(s); return 0; }
int hipStreamSynchronize(void *s) { (void)s; if (capture) return fail(900); note("sync"); return 0; }
int hipStreamIsCapturing(void *s, int *c) { (void)s; *c = capture; return 0; }
int hipStreamBeginCapture(void *s, int m) { (void)s; (void)m; return 0; }
int hipStreamEndCapture(void *s, void **g) { (void)s; *g = NULL; return 0; }
int hipGraphInstantiate(void **x, void *g, void **n, char *b, size_t z) { (void)g; (void)n; (void)b; (void)z; *x = scratch; return 0; }
int hipGraphLaunch(void *x, void *s) { (void)x; (void)s; note("graph"); return 0; }
int hipGraphDestroy(void *g) { (void)g; return 0; }
int hipGraphExecDestroy(void *x) { (void)x; return 0; }
int hipEventCreate(void **e) { *e = malloc(1); return 0; }
int hipEventDestroy(void *e) { free(e); return 0; }
int hipEventRecord(void *e, void *s) { (void)e; (void)s; return 0; }
int hipEventElapsedTime(float *t, void *a, void *b) { (void)a; (void)b; *t = 1.f; return 0; }

/* ---- kernels ---- */
static struct { dim3_t g, b; size_t m; void *s; } pushed;
int __hipPushCallConfiguration(dim3_t g, dim3_t b, size_t m, void *s)
{
    pushed.g = g, pushed.b = b, pushed.m = m, pushed.s = s;
    return 0;
}
int __hipPopCallConfiguration(dim3_t *g, dim3_t *b, size_t *m, void **s)
{
    *g = pushed.g, *b = pushed.b, *m = pushed.m, *s = pushed.s;
    return 0;
}
int hipLaunchKernel(const void *f, dim3_t g, dim3_t b, void **args, size_t m, void *s)
{
    (void)b, (void)args, (void)m, (void)s;
    if (!g.x || !g.y || !g.z)
        return fail(9); /* an empty grid */
    last_grid = g;
    for (int i = 0; i < nfn; ++i)
        if (fn[i].host == f)
            note(fn[i].name);
    return 0;
}
void **__hipRegisterFatBinary(const void *d) { static void *h; (void)d; return &h; }
void __hipUnregisterFatBinary(void **h) { (void)h; }
void __hipRegisterFunction(void **h, const void *host, char *dev, const char *name, unsigned t, void *a, void *b,
                           void *c, void *d, int *e)
{
    (void)h, (void)dev, (void)t, (void)a, (void)b, (void)c, (void)d, (void)e;
    if (nfn < 512) {
        fn[nfn].host = host;
        snprintf(fn[nfn++].name, sizeof fn[0].name, "%s", name);
    }
}
void __hipRegisterVar(void **h, void *v, char *a, const char *n, int e, size_t s, int c, int g)
{
    (void)h, (void)v, (void)a, (void)n, (void)e, (void)s, (void)c, (void)g;
}
