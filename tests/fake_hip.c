/* A HIP runtime without a device, for tests of the library's host code: memory
 * is the host's, kernels are recorded and not run, time is the number of
 * kernels launched.  Loaded with RTLD_GLOBAL before libpennant_hip.so, whose
 * calls then come here. */
#include <stdint.h>
#include <stdlib.h>
#include <string.h>

typedef int hipError_t;
typedef void* hipStream_t;
typedef struct { uint32_t x, y, z; } dim3;
enum { OK = 0, OUT_OF_MEMORY = 2, INVALID_CONFIGURATION = 9, UNKNOWN = 999 };

/* failures: the n-th hipMalloc from now of at least fail_bytes, the n-th
 * hipMemcpyAsync or hipEventSynchronize from now; 0: none */
int64_t fake_fail_malloc, fake_fail_bytes, fake_fail_copy, fake_fail_wait;
int64_t fake_queued;                    /* kernels since the last wait for a stream */
int64_t fake_launches;                  /* kernels run so far */
int64_t fake_live;                      /* device bytes in use */
int64_t fake_copied;                    /* bytes of the last asynchronous copy */
int64_t fake_max_threads;               /* most threads of a launch along x */
char fake_slow[64];                     /* kernels with this in their name take 100 times as long */
static int64_t fake_time;
static char fake_log[1 << 20];          /* names of the kernels run */
static size_t fake_log_len;
int64_t fake_error;                     /* the error that hipGetLastError returns next */
static int capturing;
static int64_t captured, cap_time;
static char cap_log[1 << 16];
static size_t cap_len;

static hipError_t ret(hipError_t e) {
    if (e) fake_error = e;
    return e;
}

static struct { const void* f; const char* name; } kernels[4096];
static int nkernels;

const char* fake_names(void) {
    fake_log[fake_log_len] = 0;
    return fake_log;
}
void fake_clear(void) {
    fake_log_len = 0;
    fake_launches = 0;
    fake_max_threads = 0;
}
static int64_t cost(const char* name) { return fake_slow[0] && strstr(name, fake_slow) ? 100 : 1; }
static void put(char* log, size_t cap, size_t* len, const char* s, size_t n) {
    if (*len + n + 2 < cap) {
        memcpy(log + *len, s, n);
        *len += n;
    }
}

void** __hipRegisterFatBinary(const void* d) { static void* h; (void)d; return &h; }
void __hipUnregisterFatBinary(void** h) { (void)h; }
void __hipRegisterVar(void** m, void* v, char* a, const char* n, int e, size_t s, int c, int g) {
    (void)m; (void)v; (void)a; (void)n; (void)e; (void)s; (void)c; (void)g;
}
void __hipRegisterFunction(void** m, const void* f, char* dev, const char* name, unsigned lim, void* t, void* b,
                           void* bd, void* gd, int* w) {
    (void)m; (void)dev; (void)lim; (void)t; (void)b; (void)bd; (void)gd; (void)w;
    if (nkernels < 4096) {
        kernels[nkernels].f = f;
        kernels[nkernels++].name = name;
    }
}
static struct { dim3 g, b; size_t sh; hipStream_t s; } config;
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t sh, hipStream_t s) {
    config.g = g; config.b = b; config.sh = sh; config.s = s;
    return OK;
}
hipError_t __hipPopCallConfiguration(dim3* g, dim3* b, size_t* sh, hipStream_t* s) {
    *g = config.g; *b = config.b; *sh = config.sh; *s = config.s;
    return OK;
}
hipError_t hipLaunchKernel(const void* f, dim3 g, dim3 b, void** args, size_t sh, hipStream_t s) {
    (void)args; (void)sh; (void)s;
    const char* name = "?";
    for (int k = 0; k < nkernels; ++k)
        if (kernels[k].f == f) name = kernels[k].name;
    const uint64_t threads = (uint64_t)g.x * b.x;
    if (threads == 0 || threads > 0xffffffffu || !g.y || !g.z) return ret(INVALID_CONFIGURATION);
    if ((int64_t)threads > fake_max_threads) fake_max_threads = (int64_t)threads;
    if (capturing) {
        ++captured;
        cap_time += cost(name);
        put(cap_log, sizeof cap_log, &cap_len, name, strlen(name));
        put(cap_log, sizeof cap_log, &cap_len, "\n", 1);
        return OK;
    }
    ++fake_launches;
    ++fake_queued;
    fake_time += cost(name);
    put(fake_log, sizeof fake_log, &fake_log_len, name, strlen(name));
    put(fake_log, sizeof fake_log, &fake_log_len, "\n", 1);
    return OK;
}

hipError_t hipMalloc(void** p, size_t n) {
    if (fake_fail_malloc > 0 && (int64_t)n >= fake_fail_bytes && --fake_fail_malloc == 0) return ret(OUT_OF_MEMORY);
    int64_t* q = calloc(1, n + 64);
    if (!q) return ret(OUT_OF_MEMORY);
    q[0] = (int64_t)n;
    fake_live += (int64_t)n;
    *p = (char*)q + 64;
    return OK;
}
hipError_t hipFree(void* p) {
    if (p) {
        int64_t* q = (int64_t*)((char*)p - 64);
        fake_live -= q[0];
        free(q);
    }
    return OK;
}
hipError_t hipHostMalloc(void** p, size_t n, unsigned f) { (void)f; *p = calloc(1, n); return OK; }
hipError_t hipHostFree(void* p) { free(p); return OK; }
hipError_t hipMemset(void* p, int v, size_t n) { memset(p, v, n); return OK; }
hipError_t hipMemsetAsync(void* p, int v, size_t n, hipStream_t s) { (void)s; return hipMemset(p, v, n); }
hipError_t hipMemcpy(void* d, const void* s, size_t n, int k) { (void)k; memmove(d, s, n); return OK; }
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, int k, hipStream_t q) {
    (void)q;
    if (fake_fail_copy > 0 && --fake_fail_copy == 0) return ret(OUT_OF_MEMORY);
    fake_copied = (int64_t)n;
    return hipMemcpy(d, s, n, k);
}
hipError_t hipStreamCreate(hipStream_t* s) { *s = calloc(1, 8); return OK; }
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned f) { (void)f; return hipStreamCreate(s); }
hipError_t hipStreamDestroy(hipStream_t s) { free(s); return OK; }
hipError_t hipStreamSynchronize(hipStream_t s) { (void)s; fake_queued = 0; return OK; }
hipError_t hipDeviceSynchronize(void) { return OK; }
hipError_t hipStreamBeginCapture(hipStream_t s, int m) {
    (void)s; (void)m;
    capturing = 1;
    captured = cap_time = 0;
    cap_len = 0;
    return OK;
}
typedef struct { int64_t n, time; size_t len; char log[sizeof cap_log]; } graph;
hipError_t hipStreamEndCapture(hipStream_t s, void** g) {
    (void)s;
    graph* q = malloc(sizeof *q);
    capturing = 0;
    q->n = captured;
    q->time = cap_time;
    q->len = cap_len;
    memcpy(q->log, cap_log, cap_len);
    *g = q;
    return OK;
}
hipError_t hipGraphInstantiate(void** e, void* g, void* n, char* l, size_t z) {
    (void)n; (void)l; (void)z;
    *e = malloc(sizeof(graph));
    memcpy(*e, g, sizeof(graph));
    return OK;
}
hipError_t hipGraphDestroy(void* g) { free(g); return OK; }
hipError_t hipGraphExecDestroy(void* g) { free(g); return OK; }
hipError_t hipGraphLaunch(void* e, hipStream_t s) {
    (void)s;
    graph* q = e;
    fake_launches += q->n;
    fake_time += q->time;
    put(fake_log, sizeof fake_log, &fake_log_len, q->log, q->len);
    return OK;
}
hipError_t hipEventCreate(void** e) { *e = calloc(1, 8); return OK; }
hipError_t hipEventCreateWithFlags(void** e, unsigned f) { (void)f; return hipEventCreate(e); }
hipError_t hipEventDestroy(void* e) { free(e); return OK; }
hipError_t hipEventRecord(void* e, hipStream_t s) { (void)s; *(int64_t*)e = fake_time; return OK; }
hipError_t hipEventSynchronize(void* e) {
    (void)e;
    if (fake_fail_wait > 0 && --fake_fail_wait == 0) return ret(UNKNOWN);
    return OK;
}
hipError_t hipEventElapsedTime(float* ms, void* a, void* b) {
    *ms = (float)(*(int64_t*)b - *(int64_t*)a);
    return OK;
}
hipError_t hipGetDevice(int* d) { *d = 0; return OK; }
hipError_t hipGetDeviceCount(int* n) { *n = 1; return OK; }
hipError_t hipGetLastError(void) {
    const hipError_t e = (hipError_t)fake_error;
    fake_error = OK;
    return e;
}
const char* hipGetErrorString(hipError_t e) { return e ? "error" : "no error"; }
hipError_t hipGetSymbolAddress(void** p, const void* s) { *p = (void*)s; return OK; }
