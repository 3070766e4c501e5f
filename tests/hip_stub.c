/* The HIP calls that the library makes, on host memory and without a device:
   kernels do nothing, copies are done at once.  What it keeps is whether work
   has been queued since the last wait for a stream (stub_pending), and it can
   make the n-th call from now on fail (stub_fail_at). */
#include <stdlib.h>
#include <string.h>

typedef int err_t;
typedef struct { unsigned x, y, z; } dim3_t;
enum { OK = 0, OUT_OF_MEMORY = 2, UNKNOWN = 999 };

static long countdown = -1;
static int pending, last;
static void *const STREAM = &pending;

void stub_fail_at(long n)
{
    countdown = n;
    last = OK;
}
long stub_left(void) { return countdown; }
int stub_pending(void) { return pending; }

static err_t step(err_t failure)
{
    if (countdown >= 0 && countdown-- == 0) return last = failure;
    return OK;
}

static err_t queue(void)
{
    err_t e = step(UNKNOWN);
    if (!e) pending = 1;
    return e;
}

err_t hipMalloc(void **p, size_t n)
{
    err_t e = step(OUT_OF_MEMORY);
    if (e) return e;
    return (*p = calloc(n ? n : 1, 1)) ? OK : (last = OUT_OF_MEMORY);
}
err_t hipMallocAsync(void **p, size_t n, void *s) { return hipMalloc(p, n); }
err_t hipFree(void *p) { free(p); return OK; }
err_t hipFreeAsync(void *p, void *s) { free(p); return OK; }
err_t hipMemGetInfo(size_t *f, size_t *t) { *f = *t = (size_t)1 << 34; return OK; }
err_t hipMemcpy(void *d, const void *s, size_t n, int k) { memcpy(d, s, n); return OK; }
err_t hipMemcpyAsync(void *d, const void *s, size_t n, int k, void *st)
{
    err_t e = queue();
    if (!e) memcpy(d, s, n);
    return e;
}
err_t hipMemsetAsync(void *d, int v, size_t n, void *st)
{
    err_t e = queue();
    if (!e) memset(d, v, n);
    return e;
}
err_t hipLaunchKernel(const void *f, dim3_t g, dim3_t b, void **a, size_t l, void *s) { return queue(); }
err_t hipExtLaunchKernel(const void *f, dim3_t g, dim3_t b, void **a, size_t l, void *s, void *e0, void *e1, int fl)
{
    return queue();
}
err_t hipLaunchCooperativeKernel(const void *f, dim3_t g, dim3_t b, void **a, unsigned l, void *s) { return queue(); }

err_t hipStreamCreateWithFlags(void **s, unsigned f) { *s = STREAM; return OK; }
err_t hipStreamDestroy(void *s) { return OK; }
err_t hipStreamSynchronize(void *s) { pending = 0; return OK; }
err_t hipStreamWaitEvent(void *s, void *e, unsigned f) { return OK; }
err_t hipEventCreate(void **e) { *e = STREAM; return OK; }
err_t hipEventCreateWithFlags(void **e, unsigned f) { *e = STREAM; return OK; }
err_t hipEventDestroy(void *e) { return OK; }
err_t hipEventRecord(void *e, void *s) { return OK; }
err_t hipEventSynchronize(void *e) { return OK; }
err_t hipEventElapsedTime(float *ms, void *a, void *b) { *ms = 1; return OK; }

err_t hipGetLastError(void)
{
    err_t e = last;
    last = OK;
    return e;
}
const char *hipGetErrorString(err_t e) { return e == OUT_OF_MEMORY ? "out of memory" : "unknown error"; }
err_t hipGetDevice(int *d) { *d = 0; return OK; }
err_t hipSetDevice(int d) { return OK; }
err_t hipDeviceGetAttribute(int *v, int a, int d) { *v = 1; return OK; }
err_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int *n, const void *f, int b, size_t l) { *n = 1; return OK; }
err_t hipGetSymbolAddress(void **p, const void *s)
{
    static char symbol[1 << 16];
    *p = symbol;
    return OK;
}

err_t __hipPushCallConfiguration(dim3_t g, dim3_t b, size_t l, void *s) { return OK; }
err_t __hipPopCallConfiguration(dim3_t *g, dim3_t *b, size_t *l, void **s)
{
    memset(g, 0, sizeof *g);
    memset(b, 0, sizeof *b);
    *l = 0;
    *s = NULL;
    return OK;
}
void **__hipRegisterFatBinary(const void *d) { static void *h; return &h; }
void __hipUnregisterFatBinary(void **h) {}
void __hipRegisterFunction(void **h, const void *f, char *df, const char *n, unsigned t, void *a, void *b, void *c,
                           void *d, int *e) {}
void __hipRegisterVar(void **h, void *v, char *hv, char *dv, int e, size_t s, int c, int g) {}
