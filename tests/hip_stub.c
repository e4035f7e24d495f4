/* A HIP runtime without a GPU, for CPU tests of the host code of libamps.so:
 * device memory is host memory, counted and limited; kernels are not run but
 * named in a log, with the copies, memsets and frees, in the order of the
 * calls; streams, events and graphs are empty shells.  Loaded before libamps.so it takes libamdhip64.so.7's place
 * (same SONAME and symbol versions). */
#include <stdint.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

typedef struct { unsigned x, y, z; } dim3_t;
enum { OK = 0, OUT_OF_MEMORY = 2 };

/* ---- what the tests read and set */
#define MAX_KERNELS 4096
static const void* fn_addr[MAX_KERNELS];
static const char* fn_name[MAX_KERNELS];
static int n_fn;
static char* log_text;
static size_t log_len, log_cap;
static size_t live, peak, limit = (size_t)-1;
static int capturing;

const char* stub_log(void) { return log_text ? log_text : ""; }
void stub_clear(void) { log_len = 0; if (log_text) log_text[0] = 0; peak = live; }
size_t stub_live(void) { return live; }
size_t stub_peak(void) { return peak; }
void stub_limit(size_t bytes) { limit = bytes; }

static void note(const char* what) {
    const size_t n = strlen(what);
    if (log_len + n + 3 > log_cap) log_text = realloc(log_text, log_cap = 2 * (log_cap + n + 3));
    if (capturing) log_text[log_len++] = '+';
    memcpy(log_text + log_len, what, n);
    log_len += n;
    log_text[log_len++] = '\n';
    log_text[log_len] = 0;
}

/* ---- memory */
typedef struct { size_t bytes; char pad[56]; } Head;
int hipMalloc(void** p, size_t bytes) {
    *p = NULL;
    if (bytes > limit || live > limit - bytes) return OUT_OF_MEMORY;
    Head* h = aligned_alloc(256, 256 + (bytes + 255) / 256 * 256);
    if (!h) return OUT_OF_MEMORY;
    memset(h, 0xA5, 256 + (bytes + 255) / 256 * 256);
    h->bytes = bytes;
    live += bytes;
    if (live > peak) peak = live;
    *p = (char*)h + 256;
    return OK;
}
int hipFree(void* p) {
    if (!p) return OK;
    note("free");
    Head* h = (Head*)((char*)p - 256);
    live -= h->bytes;
    free(h);
    return OK;
}
int hipHostMalloc(void** p, size_t bytes, unsigned flags) { (void)flags; *p = calloc(1, bytes); return OK; }
int hipHostFree(void* p) { free(p); return OK; }
int hipHostGetDevicePointer(void** d, void* h, unsigned flags) { (void)flags; *d = h; return OK; }
int hipMemcpy(void* d, const void* s, size_t n, int kind) { (void)kind; note("copy"); memcpy(d, s, n); return OK; }
int hipMemcpyAsync(void* d, const void* s, size_t n, int kind, void* st) { (void)st; return hipMemcpy(d, s, n, kind); }
int hipMemset(void* d, int v, size_t n) { note("memset"); memset(d, v, n); return OK; }
int hipMemsetAsync(void* d, int v, size_t n, void* st) { (void)st; return hipMemset(d, v, n); }

/* ---- kernels */
static struct { dim3_t g, b; size_t shmem; void* stream; } call;
void** __hipRegisterFatBinary(const void* data) { static void* h; (void)data; return &h; }
void __hipUnregisterFatBinary(void** h) { (void)h; }
void __hipRegisterFunction(void** h, const void* host, char* dev, const char* name, unsigned lim, void* tid, void* bid,
                           void* bd, void* gd, int* ws) {
    (void)h; (void)dev; (void)lim; (void)tid; (void)bid; (void)bd; (void)gd; (void)ws;
    if (n_fn < MAX_KERNELS) { fn_addr[n_fn] = host; fn_name[n_fn++] = name; }
}
int __hipPushCallConfiguration(dim3_t g, dim3_t b, size_t shmem, void* stream) {
    call.g = g; call.b = b; call.shmem = shmem; call.stream = stream;
    return OK;
}
int __hipPopCallConfiguration(dim3_t* g, dim3_t* b, size_t* shmem, void** stream) {
    *g = call.g; *b = call.b; *shmem = call.shmem; *stream = call.stream;
    return OK;
}
int hipLaunchKernel(const void* f, dim3_t g, dim3_t b, void** args, size_t shmem, void* stream) {
    (void)g; (void)b; (void)args; (void)shmem; (void)stream;
    for (int i = 0; i < n_fn; ++i)
        if (fn_addr[i] == f) { note(fn_name[i]); return OK; }
    note("unknown kernel");
    return OK;
}
int hipExtLaunchKernel(const void* f, dim3_t g, dim3_t b, void** args, size_t shmem, void* stream, void* e0, void* e1,
                       int flags) {
    (void)e0; (void)e1; (void)flags;
    return hipLaunchKernel(f, g, b, args, shmem, stream);
}
int hipOccupancyMaxActiveBlocksPerMultiprocessor(int* n, const void* f, int threads, size_t shmem) {
    (void)f; (void)threads; (void)shmem;
    *n = 2;
    return OK;
}

int hipLaunchHostFunc(void* s, void (*f)(void*), void* arg) { (void)s; note("host"); f(arg); return OK; }

/* ---- device, streams, events, graphs */
int hipGetDevice(int* d) { *d = 0; return OK; }
int hipDeviceGetAttribute(int* v, int attr, int dev) { (void)attr; (void)dev; *v = 256; return OK; }
const char* hipGetErrorString(int e) { return e == OUT_OF_MEMORY ? "out of memory" : "stub"; }
int hipGetLastError(void) { return OK; }
int hipStreamCreateWithFlags(void** s, unsigned flags) { (void)flags; *s = malloc(1); return OK; }
int hipStreamDestroy(void* s) { free(s); return OK; }
int hipStreamSynchronize(void* s) { (void)s; return OK; }
int hipEventCreate(void** e) { *e = malloc(1); return OK; }
int hipEventDestroy(void* e) { free(e); return OK; }
int hipEventRecord(void* e, void* s) { (void)e; (void)s; return OK; }
int hipEventElapsedTime(float* ms, void* a, void* b) { (void)a; (void)b; *ms = 1.0f; return OK; }
int hipStreamBeginCapture(void* s, int mode) { (void)s; (void)mode; capturing = 1; return OK; }
int hipStreamEndCapture(void* s, void** g) { (void)s; capturing = 0; *g = malloc(1); return OK; }
int hipGraphInstantiate(void** x, void* g, void** node, char* buf, size_t n) {
    (void)g; (void)node; (void)buf; (void)n;
    *x = malloc(1);
    return OK;
}
int hipGraphDestroy(void* g) { free(g); return OK; }
int hipGraphExecDestroy(void* x) { free(x); return OK; }
int hipGraphLaunch(void* x, void* s) { (void)x; (void)s; note("graph"); return OK; }
