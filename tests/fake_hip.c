/* A HIP runtime without a GPU for host-side tests of libvpmx: device memory is host memory, copies
 * happen at once, kernels do nothing.  Loaded before the library, its functions take the place of the
 * runtime's.  The tests count calls and make the k-th call of one function fail. */
#include <stddef.h>
#include <stdlib.h>
#include <string.h>

enum { MALLOC, MEMCPY, HOSTMALLOC, STREAM, EVENT, LAUNCH, RECORD, ASYNC, NKIND };
static long calls[NKIND], done[NKIND], fail_at[NKIND], held_host, held_dev;
static __thread int last_error;

long fake_calls(int k) { return __sync_fetch_and_add(&calls[k], 0); } /* calls, failed ones among them */
long fake_done(int k) { return __sync_fetch_and_add(&done[k], 0); }   /* calls that succeeded */
long fake_held(int host) { return __sync_fetch_and_add(host ? &held_host : &held_dev, 0); }
/* the n-th call of kind k from now on fails (0: none; -1: every one) */
void fake_fail(int k, long n) { fail_at[k] = n > 0 ? fake_calls(k) + n : n; }
int fake_last_error(void) { return last_error; }

static int enter(int k) {
    const long n = __sync_add_and_fetch(&calls[k], 1);
    if (fail_at[k] == -1 || (fail_at[k] > 0 && n == fail_at[k])) return last_error = 2; /* out of memory */
    __sync_add_and_fetch(&done[k], 1);
    return 0;
}
static int get(void **p, size_t n, long *held) {
    *p = calloc(n ? n : 1, 1);
    if (!*p) return last_error = 2;
    __sync_add_and_fetch(held, 1);
    return 0;
}
static int put(void *p, long *held) {
    if (p) __sync_add_and_fetch(held, -1);
    free(p);
    return 0;
}

int hipGetLastError(void) { int e = last_error; last_error = 0; return e; }
const char *hipGetErrorString(int e) { return e ? "made to fail" : "no error"; }
int hipGetDeviceCount(int *n) { *n = 1; return 0; }
int hipSetDevice(int d) { return d ? (last_error = 101) : 0; }
int hipDeviceGetAttribute(int *v, int a, int d) { return 1; } /* (the context's defaults) */
int hipMalloc(void **p, size_t n) { return enter(MALLOC) ? 2 : get(p, n, &held_dev); }
int hipFree(void *p) { return put(p, &held_dev); }
int hipHostMalloc(void **p, size_t n, unsigned f) { return enter(HOSTMALLOC) ? 2 : get(p, n, &held_host); }
int hipHostFree(void *p) { return put(p, &held_host); }
int hipMemcpy(void *d, const void *s, size_t n, int k) {
    if (enter(MEMCPY)) return 2;
    memcpy(d, s, n);
    return 0;
}
int hipMemcpyAsync(void *d, const void *s, size_t n, int k, void *st) {
    if (!d || !s) return last_error = 1;
    if (enter(ASYNC)) return 2;
    memcpy(d, s, n);
    return 0;
}
int hipPointerGetAttributes(void *a, const void *p) { *(int *)a = 0; return 0; } /* unregistered */
int hipGetSymbolAddress(void **p, const void *s) {
    static double mem[1 << 16];
    *p = mem;
    return 0;
}
int hipStreamCreateWithFlags(void **s, unsigned f) { return enter(STREAM) ? 2 : get(s, 8, &held_dev); }
int hipStreamDestroy(void *s) { return put(s, &held_dev); }
int hipStreamSynchronize(void *s) { return 0; }
int hipStreamWaitEvent(void *s, void *e, unsigned f) { return 0; }
int hipStreamBeginCapture(void *s, int m) { return 0; }
int hipStreamEndCapture(void *s, void **g) { *g = 0; return 0; }
int hipStreamIsCapturing(void *s, int *c) { *c = 0; return 0; }
int hipGraphInstantiate(void **e, void *g, void *n, char *l, size_t b) { *e = 0; return 0; }
int hipGraphLaunch(void *e, void *s) { return 0; }
int hipGraphDestroy(void *g) { return 0; }
int hipGraphExecDestroy(void *g) { return 0; }
int hipEventCreate(void **e) { return enter(EVENT) ? 2 : get(e, 8, &held_dev); }
int hipEventCreateWithFlags(void **e, unsigned f) { return enter(EVENT) ? 2 : get(e, 8, &held_dev); }
int hipEventDestroy(void *e) { return put(e, &held_dev); }
int hipEventRecord(void *e, void *s) { return enter(RECORD) ? 2 : 0; }
int hipEventSynchronize(void *e) { return 0; }
int hipEventElapsedTime(float *ms, void *a, void *b) { *ms = 1.0f; return 0; }
int hipOccupancyMaxActiveBlocksPerMultiprocessor(int *n, const void *f, int t, size_t l) { *n = 1; return 0; }

typedef struct { unsigned x, y, z; } dim3_;
static __thread dim3_ grid_, block_;
static __thread size_t lds_;
static __thread void *stream_;
int hipLaunchKernel(const void *f, dim3_ g, dim3_ b, void **a, size_t l, void *s) {
    if (enter(LAUNCH)) return 2;
    return g.x && g.y && g.z && b.x && b.y && b.z ? 0 : (last_error = 9);
}
int hipExtLaunchKernel(const void *f, dim3_ g, dim3_ b, void **a, size_t l, void *s, void *e0, void *e1, int n) {
    return hipLaunchKernel(f, g, b, a, l, s);
}
int __hipPushCallConfiguration(dim3_ g, dim3_ b, size_t l, void *s) {
    grid_ = g;
    block_ = b;
    lds_ = l;
    stream_ = s;
    return 0;
}
int __hipPopCallConfiguration(dim3_ *g, dim3_ *b, size_t *l, void **s) {
    *g = grid_;
    *b = block_;
    *l = lds_;
    *s = stream_;
    return 0;
}
void **__hipRegisterFatBinary(const void *d) { static void *h; return &h; }
void __hipRegisterFunction(void **m, const void *f, char *d, const char *n, unsigned t, void *a, void *b, void *c, void *e, int *w) {}
void __hipRegisterVar(void **m, void *v, char *h, char *d, int e, size_t s, int c, int g) {}
void __hipUnregisterFatBinary(void **m) {}
