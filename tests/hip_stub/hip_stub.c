/* The HIP runtime calls of the library with host memory in the place of device memory and kernels that do nothing, for
 * CPU tests of its host code.  Loaded with global symbols before the library, whose calls then bind here.  Allocations
 * can be made to fail, and the last error stays until it is asked for, as in the runtime. */
#include <stddef.h>
#include <stdlib.h>
#include <string.h>

enum { OK = 0, OUT_OF_MEMORY = 2, INVALID = 1 };
typedef struct { unsigned x, y, z; } dim;

static int last, skip, fail, launches, unfit;
static size_t live;
static struct { const void *f; char name[256]; } kernels[4096];
static int nkernels, seen[4096];
static unsigned blocks[4096];

/* of the following hipMalloc calls, the first s succeed and the next n fail */
void stub_fail(int s, int n) { skip = s, fail = n; }
size_t stub_live(void) { return live; }
int stub_launches(void) { return launches; }
/* launches of the walking solvers without material, or with factors of the stencils that were never written */
int stub_unfit(void) { return unfit; }
/* kernels of the library: the mangled name of kernel i, and whether it was launched since this was last asked */
int stub_kernels(void) { return nkernels; }
const char *stub_name(int i) { return kernels[i].name; }
int stub_seen(int i) {
    const int v = seen[i];
    seen[i] = 0;
    return v;
}
unsigned stub_blocks(int i) { return blocks[i]; } /* of its last launch */
void **__hipRegisterFatBinary(const void *b) { return (void)b, (void **)kernels; }
void __hipUnregisterFatBinary(void **b) { (void)b; }
void __hipRegisterFunction(void **b, const void *f, char *d, const char *name, unsigned n, void *t, void *bl, void *bd,
                           void *gd, int *w) {
    (void)b, (void)d, (void)n, (void)t, (void)bl, (void)bd, (void)gd, (void)w;
    if (nkernels == 4096) abort();
    kernels[nkernels].f = f;
    strncpy(kernels[nkernels++].name, name, 255);
}
void __hipRegisterVar(void **b, void *v, char *h, char *d, int e, size_t n, int c, int g) {
    (void)b, (void)v, (void)h, (void)d, (void)e, (void)n, (void)c, (void)g;
}

int hipMalloc(void **p, size_t n) {
    *p = NULL;
    if (skip > 0) {
        skip--;
    } else if (fail > 0) {
        fail--;
        return last = OUT_OF_MEMORY;
    }
    size_t *b = malloc(n + 64);
    if (!b) abort();
    memset(b, 0xff, n + 64); /* NaN until written */
    b[0] = n;
    live += n;
    *p = (char *)b + 64;
    return OK;
}
int hipFree(void *p) {
    if (p) {
        size_t *b = (size_t *)((char *)p - 64);
        live -= b[0];
        free(b);
    }
    return OK;
}
int hipLaunchKernel(const void *f, dim g, dim b, void **args, size_t lds, void *st) {
    (void)b, (void)lds, (void)st;
    for (int i = 0; i < nkernels; i++)
        if (kernels[i].f == f) {
            seen[i] = 1;
            blocks[i] = g.x;
            if (strstr(kernels[i].name, "6k_walkI")) { /* WalkMaterial: two orders of the material, the factors */
                const double **m = args[4];
                if (!m[0] || !m[1] || !m[2] || m[2][0] != m[2][0]) unfit++;
            }
        }
    launches++;
    return OK;
}
static dim grid, block; /* of the launch under way */
int __hipPushCallConfiguration(dim g, dim b, size_t lds, void *st) {
    (void)lds, (void)st;
    grid = g, block = b;
    return OK;
}
int __hipPopCallConfiguration(dim *g, dim *b, size_t *lds, void **st) {
    *g = grid, *b = block;
    *lds = 0;
    *st = NULL;
    return OK;
}
int hipGetLastError(void) {
    const int e = last;
    last = OK;
    return e;
}
const char *hipGetErrorString(int e) { return e == OUT_OF_MEMORY ? "out of memory" : "error"; }
int hipMemcpy(void *d, const void *s, size_t n, int k) { return (void)k, memcpy(d, s, n), OK; }
int hipMemcpyAsync(void *d, const void *s, size_t n, int k, void *st) { return (void)k, (void)st, memcpy(d, s, n), OK; }
int hipMemset(void *d, int v, size_t n) { return memset(d, v, n), OK; }
int hipMemsetAsync(void *d, int v, size_t n, void *st) { return (void)st, memset(d, v, n), OK; }
int hipHostMalloc(void **p, size_t n, unsigned fl) { return (void)fl, (*p = malloc(n)) ? OK : OUT_OF_MEMORY; }
int hipMemGetInfo(size_t *f, size_t *t) { return *f = *t = (size_t)1 << 36, OK; }
int hipGetDevice(int *d) { return *d = 0, OK; }
int hipSetDevice(int d) { return d == 0 ? OK : INVALID; }
int hipGetDeviceCount(int *n) { return *n = 1, OK; }
int hipDeviceGetAttribute(int *v, int a, int d) { return (void)a, (void)d, *v = 160 * 1024, OK; }
int hipFuncSetAttribute(const void *f, int a, int v) { return (void)f, (void)a, (void)v, OK; }
int hipGetSymbolAddress(void **p, const void *s) { return (void)s, *p = NULL, INVALID; }
int hipEventCreate(void **e) { return *e = &live, OK; }
int hipEventCreateWithFlags(void **e, unsigned fl) { return (void)fl, *e = &live, OK; }
int hipEventDestroy(void *e) { return (void)e, OK; }
int hipEventElapsedTime(float *t, void *a, void *b) { return (void)a, (void)b, *t = 1, OK; }
int hipEventRecord(void *e, void *st) { return (void)e, (void)st, OK; }
int hipEventSynchronize(void *e) { return (void)e, OK; }
int hipStreamCreateWithFlags(void **s, unsigned fl) { return (void)fl, *s = &live, OK; }
int hipStreamDestroy(void *s) { return (void)s, OK; }
int hipStreamSynchronize(void *s) { return (void)s, OK; }
int hipStreamWaitEvent(void *s, void *e, unsigned fl) { return (void)s, (void)e, (void)fl, OK; }
int hipStreamBeginCapture(void *s, int m) { return (void)s, (void)m, OK; }
int hipStreamEndCapture(void *s, void **g) { return (void)s, *g = &live, OK; }
int hipGraphInstantiate(void **x, void *g, void **n, char *l, size_t sz) {
    return (void)g, (void)n, (void)l, (void)sz, *x = &live, OK;
}
int hipGraphLaunch(void *x, void *s) { return (void)x, (void)s, OK; }
int hipGraphDestroy(void *g) { return (void)g, OK; }
int hipGraphExecDestroy(void *x) { return (void)x, OK; }
