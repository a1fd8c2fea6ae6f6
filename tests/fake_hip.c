/* A HIP runtime for host-side tests, preloaded over the real one: device memory
 * is host memory, kernels do nothing, and each launch, query and wait is written
 * to the file FAKE_HIP_LOG.  FAKE_HIP: "silent" (streams are idle at once),
 * "count" (k_count_running answers: FP64 systems run for three polls, FP32 ones
 * for eight), "threads" (count, and launches from threads other than the
 * first one fail, with an error that only that thread's hipGetLastError shows). */
#define _GNU_SOURCE
#include <pthread.h>
#include <stdint.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>
#include <sys/syscall.h>
#include <unistd.h>

typedef struct { unsigned x, y, z; } dim3;
enum { kMost = 4096, kFailure = 719 };
static const void *fns[kMost];
static const char *names[kMost];
static int nfns;
static __thread int last_error;
static __thread struct { dim3 g, b; size_t m; void *s; } call;
static pthread_mutex_t lock = PTHREAD_MUTEX_INITIALIZER;

static int mode(const char *m) {
    const char *v = getenv("FAKE_HIP");
    return v && !strcmp(v, m);
}
static void note(const char *fmt, const char *a, const void *p, int x, int y) {
    const char *path = getenv("FAKE_HIP_LOG");
    if (!path) return;
    pthread_mutex_lock(&lock);
    FILE *f = fopen(path, "a");
    if (f) {
        fprintf(f, fmt, a, p, x, y);
        fputc('\n', f);
        fclose(f);
    }
    pthread_mutex_unlock(&lock);
}

void **__hipRegisterFatBinary(const void *d) { return (void **)d; }
void __hipUnregisterFatBinary(void **m) { (void)m; }
void __hipRegisterVar(void **m, void *v, char *h, char *d, int e, size_t s, int c, int g) {
    (void)m, (void)v, (void)h, (void)d, (void)e, (void)s, (void)c, (void)g;
}
void __hipRegisterFunction(void **m, const void *fn, char *d, const char *name, unsigned l, void *t, void *b, void *bd,
                           void *gd, int *w) {
    (void)m, (void)d, (void)l, (void)t, (void)b, (void)bd, (void)gd, (void)w;
    if (nfns < kMost) fns[nfns] = fn, names[nfns++] = name;
}
int __hipPushCallConfiguration(dim3 g, dim3 b, size_t m, void *s) {
    call.g = g, call.b = b, call.m = m, call.s = s;
    return 0;
}
int __hipPopCallConfiguration(dim3 *g, dim3 *b, size_t *m, void **s) {
    *g = call.g, *b = call.b, *m = call.m, *s = call.s;
    return 0;
}
int hipLaunchKernel(const void *fn, dim3 g, dim3 b, void **args, size_t m, void *s) {
    (void)g, (void)b, (void)m, (void)s;
    const char *name = "?";
    for (int k = 0; k < nfns; ++k)
        if (fns[k] == fn) name = names[k];
    if (mode("threads") && syscall(SYS_gettid) != getpid()) return last_error = kFailure;
    if (strstr(name, "k_count_running")) {
        int *out = *(int **)args[3];
        const int nids = *(int *)args[2], poll = *(int *)args[4];
        note("poll %.0s%p %d %d", "", out, nids, poll);
        if (!mode("silent")) {
            const int run = poll <= (strstr(name, "IfE") ? 8 : 3);
            out[0] = run ? nids : 0;
            for (int k = 0; k < nids; ++k) out[2 + k] = run;
            __atomic_store_n(out + 1, poll, __ATOMIC_RELEASE);
        }
        return 0;
    }
    note("launch %s", name, 0, 0, 0);
    return 0;
}
int hipExtLaunchKernel(const void *fn, dim3 g, dim3 b, void **args, size_t m, void *s, void *e0, void *e1, int f) {
    (void)e0, (void)e1, (void)f;
    return hipLaunchKernel(fn, g, b, args, m, s);
}
int hipLaunchCooperativeKernel(const void *fn, dim3 g, dim3 b, void **args, unsigned m, void *s) {
    (void)fn, (void)g, (void)b, (void)args, (void)m, (void)s;
    return last_error = 720;
}
int hipGetLastError(void) {
    const int e = last_error;
    last_error = 0;
    return e;
}
const char *hipGetErrorString(int e) { return e ? "failure" : "success"; }
int hipMalloc(void **p, size_t n) { return (*p = calloc(1, n ? n : 1)) ? 0 : 2; }
int hipHostMalloc(void **p, size_t n, unsigned f) { return (void)f, hipMalloc(p, n); }
int hipFree(void *p) { return free(p), 0; }
int hipHostFree(void *p) { return free(p), 0; }
int hipGetSymbolAddress(void **p, const void *s) { return (void)s, hipMalloc(p, (size_t)64 << 20); }
int hipMemcpyAsync(void *d, const void *s, size_t n, int k, void *st) { return (void)k, (void)st, memcpy(d, s, n), 0; }
int hipMemsetAsync(void *d, int v, size_t n, void *st) { return (void)st, memset(d, v, n), 0; }
/* (what is not the fake's own is ordinary host memory) */
int hipPointerGetAttributes(void *a, const void *p) { return (void)a, (void)p, last_error = 1; }
int hipSetDevice(int d) { return (void)d, 0; }
int hipDeviceSynchronize(void) { return 0; }
int hipStreamCreateWithFlags(void **s, unsigned f) { return (void)f, *s = &nfns, 0; }
int hipStreamDestroy(void *s) { return (void)s, 0; }
int hipStreamQuery(void *s) { return (void)s, note("query%.0s", "", 0, 0, 0), 0; }
int hipStreamSynchronize(void *s) { return (void)s, note("wait%.0s", "", 0, 0, 0), 0; }
int hipEventCreate(void **e) { return *e = &nfns, 0; }
int hipEventCreateWithFlags(void **e, unsigned f) { return (void)f, *e = &nfns, 0; }
int hipEventDestroy(void *e) { return (void)e, 0; }
int hipEventRecord(void *e, void *s) { return (void)e, (void)s, 0; }
int hipEventQuery(void *e) { return (void)e, 0; }
int hipEventSynchronize(void *e) { return (void)e, note("wait%.0s", "", 0, 0, 0), 0; }
int hipEventElapsedTime(float *ms, void *a, void *b) { return (void)a, (void)b, *ms = 0, 0; }
int hipStreamBeginCapture(void *s, int m) { return (void)s, (void)m, 0; }
int hipStreamEndCapture(void *s, void **g) { return (void)s, *g = &nfns, 0; }
int hipGraphInstantiate(void **e, void *g, void *n, char *b, size_t z) {
    return (void)g, (void)n, (void)b, (void)z, hipMalloc(e, 1);
}
int hipGraphDestroy(void *g) { return (void)g, 0; }
int hipGraphExecDestroy(void *g) { return note("destroy%.0s %p", "", g, 0, 0), 0; }
int hipGraphLaunch(void *g, void *s) { return (void)s, note("launch%.0s %p", "", g, 0, 0), 0; }
