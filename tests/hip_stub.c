/* A HIP runtime without a device, for host-side tests: "device" memory is
 * host memory, kernels are not run, copies are done at once.  What it keeps is
 * the order of the work: each stream counts what was put on it, events and
 * waits carry vector clocks, so a test can ask whether a stream still has work
 * that nobody has waited for.  Allocations are counted and can be made to fail.
 *
 * Built with a version script that names the runtime's symbol versions, and
 * loaded in a process of its own in the runtime's place. */
#include <stddef.h>
#include <stdlib.h>
#include <string.h>

enum { STREAMS = 62, EVENTS = 4096, LOG = 1 << 16 };
typedef struct { unsigned x, y, z; } dim3_t;

static long long clock_of[STREAMS][STREAMS]; /* what a stream's work is ordered behind */
static long long done[STREAMS];              /* work the host has waited for */
static long long events[EVENTS][STREAMS];
static long long n_streams = 1, n_events = 1;
static long long mallocs, fail_from = -1, fail_above = -1, bytes_live, bytes_peak, largest, host_mallocs;
static long long launches, launch_log[LOG], size_log[LOG];
static const char *launch_name[LOG];
static struct { const void *f; const char *name; } functions[4096];
static int n_functions;

/* --- what tests read and set --- */
long long stub_pending(void) {   /* bit s: stream s has work that nobody has waited for */
    long long m = 0;
    for (int s = 0; s < n_streams; s++)
        if (clock_of[s][s] > done[s]) m |= 1ll << s;
    return m;
}
long long stub_mallocs(void) { return mallocs; }
long long stub_largest(void) { const long long v = largest; largest = 0; return v; }
void stub_fail_from(long long k) { fail_from = k < 0 ? -1 : mallocs + k; }   /* device allocations from the k-th on fail */
void stub_fail_above(long long bytes) { fail_above = bytes; }                 /* those larger than this fail */
long long stub_malloc_size(long long i) { return i < mallocs && i < LOG ? size_log[i] : 0; }
long long stub_launches(void) { return launches; }
const char *stub_launch_name(long long i) { return i < launches && i < LOG ? launch_name[i] : ""; }
long long stub_launch_stream(long long i) { return i < launches && i < LOG ? launch_log[i] : -1; }

/* --- the runtime --- */
static int of(void *s) { return (int)(size_t)s; }
static void put(void *s) { clock_of[of(s)][of(s)]++; }

int hipMalloc(void **p, size_t n) {
    if ((long long)n > largest) largest = (long long)n;
    if ((fail_from >= 0 && mallocs >= fail_from) || (fail_above >= 0 && (long long)n > fail_above)) {
        *p = NULL;
        return 2;
    }
    if (mallocs < LOG) size_log[mallocs] = (long long)n;
    mallocs++;
    *p = calloc(1, n);
    return *p ? 0 : 2;
}
int hipFree(void *p) { free(p); return 0; }
int hipHostMalloc(void **p, size_t n, unsigned f) { (void)f; host_mallocs++; *p = calloc(1, n); return *p ? 0 : 2; }
int hipHostFree(void *p) { free(p); return 0; }
int hipGetDeviceCount(int *n) { *n = 1; return 0; }
int hipSetDevice(int d) { (void)d; return 0; }
int hipDeviceGetAttribute(int *v, int a, int d) { (void)a; (void)d; *v = 256; return 0; }
int hipGetLastError(void) { return 0; }
const char *hipGetErrorString(int e) { return e ? "error of the stub" : "no error"; }
int hipGetSymbolAddress(void **p, const void *s) {
    (void)s;
    static void *scratch;
    if (!scratch) scratch = calloc(1, (size_t)64 << 20);
    *p = scratch;
    return 0;
}
int hipStreamCreateWithFlags(void **s, unsigned f) { (void)f; *s = (void *)(size_t)n_streams++; return 0; }
int hipStreamDestroy(void *s) { (void)s; return 0; }
int hipStreamSynchronize(void *s) {
    for (int k = 0; k < STREAMS; k++)
        if (clock_of[of(s)][k] > done[k]) done[k] = clock_of[of(s)][k];
    return 0;
}
int hipEventCreateWithFlags(void **e, unsigned f) { (void)f; *e = (void *)(size_t)n_events++; return 0; }
int hipEventCreate(void **e) { return hipEventCreateWithFlags(e, 0); }
int hipEventDestroy(void *e) { (void)e; return 0; }
int hipEventRecord(void *e, void *s) { memcpy(events[of(e)], clock_of[of(s)], sizeof events[0]); return 0; }
int hipStreamWaitEvent(void *s, void *e, unsigned f) {
    (void)f;
    for (int k = 0; k < STREAMS; k++)
        if (events[of(e)][k] > clock_of[of(s)][k]) clock_of[of(s)][k] = events[of(e)][k];
    return 0;
}
int hipEventElapsedTime(float *ms, void *a, void *b) { (void)a; (void)b; *ms = 0.f; return 0; }
int hipMemcpyAsync(void *d, const void *s, size_t n, int k, void *st) { (void)k; memmove(d, s, n); put(st); return 0; }
int hipMemsetAsync(void *d, int v, size_t n, void *st) { memset(d, v, n); put(st); return 0; }
int hipOccupancyMaxActiveBlocksPerMultiprocessor(int *n, const void *f, int b, size_t l) {
    (void)f; (void)b; (void)l;
    *n = 4;
    return 0;
}
int hipPointerGetAttributes(void *a, const void *p) { (void)a; (void)p; return 1; }

static struct { dim3_t g, b; size_t l; void *s; } call;
int __hipPushCallConfiguration(dim3_t g, dim3_t b, size_t l, void *s) {
    call.g = g; call.b = b; call.l = l; call.s = s;
    return 0;
}
int __hipPopCallConfiguration(dim3_t *g, dim3_t *b, size_t *l, void **s) {
    *g = call.g; *b = call.b; *l = call.l; *s = call.s;
    return 0;
}
int hipLaunchKernel(const void *f, dim3_t g, dim3_t b, void **a, size_t l, void *s) {
    (void)g; (void)b; (void)a; (void)l;
    const char *name = "";
    for (int k = 0; k < n_functions; k++)
        if (functions[k].f == f) name = functions[k].name;
    if (launches < LOG) { launch_name[launches] = name; launch_log[launches] = of(s); }
    launches++;
    put(s);
    return 0;
}
void **__hipRegisterFatBinary(const void *d) { static void *h; (void)d; return &h; }
void __hipRegisterFunction(void **m, const void *f, char *dev, const char *name, unsigned t, void *a, void *b, void *c,
                           void *d, int *w) {
    (void)m; (void)dev; (void)t; (void)a; (void)b; (void)c; (void)d; (void)w;
    functions[n_functions].f = f;
    functions[n_functions++].name = name;
}
void __hipRegisterVar(void **m, void *v, char *h, char *d, int e, size_t s, int c, int g) {
    (void)m; (void)v; (void)h; (void)d; (void)e; (void)s; (void)c; (void)g;
}
void __hipUnregisterFatBinary(void **m) { (void)m; }
int hipStreamBeginCapture(void *s, int m) { (void)s; (void)m; return 0; }
int hipStreamEndCapture(void *s, void **g) { (void)s; *g = (void *)1; return 0; }
int hipGraphInstantiate(void **e, void *g, void **n, char *l, size_t z) { (void)g; (void)n; (void)l; (void)z; *e = (void *)1; return 0; }
int hipGraphDestroy(void *g) { (void)g; return 0; }
int hipGraphExecDestroy(void *e) { (void)e; return 0; }
int hipGraphLaunch(void *e, void *s) { (void)e; put(s); return 0; }
