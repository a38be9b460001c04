/* A CPU stand-in for the HIP runtime (the fake_hip fixture of tests/conftest.py).  Loaded with
 * RTLD_GLOBAL before libredukt_gpu.so, its definitions take the place of libamdhip64's for the
 * functions that library calls.  Device memory is host memory, kernels do nothing, and each
 * stream counts what was queued on it and how much of that is known to have ended: an event
 * that was queried successfully, or a synchronize, ends everything queued before it, on the
 * streams it waited for too.
 *   fake_hip_fail(name, k): call k (from 0) of that function from now on fails, once.
 *   fake_hip_failed(): whether that happened.
 *   fake_hip_pending(): streams with work that may still run. */
#define __HIP_PLATFORM_AMD__ 1
#include <hip/hip_runtime_api.h>
#include <pthread.h>
#include <stdlib.h>
#include <string.h>

enum { kMaxStreams = 64, kMaxNodes = 4096 };

typedef struct {
    int live, capturing;
    unsigned long queued, ended;
    unsigned long waits[kMaxStreams];   /* what of each stream this one's work waits for */
    struct graph* rec;
} Stream;
typedef struct {
    int stream;
    unsigned long at;
} Event;
struct node {
    const void* fn;
};
struct graph {
    size_t n;
    struct node node[kMaxNodes];
};

static Stream g_stream[kMaxStreams];   /* 0: the null stream */
static pthread_mutex_t g_mu = PTHREAD_MUTEX_INITIALIZER;
static char g_name[64];
static long g_left = -1;
static int g_failed;
static hipError_t g_last;

void fake_hip_fail(const char* name, long k) {
    strncpy(g_name, name, sizeof(g_name) - 1);
    g_left = k;
    g_failed = 0;
    g_last = hipSuccess;
}
int fake_hip_failed(void) { return g_failed; }
int fake_hip_pending(void) {
    int n = 0;
    for (int i = 0; i < kMaxStreams; i++) n += g_stream[i].ended < g_stream[i].queued;
    return n;
}

static int fails(const char* name) {
    pthread_mutex_lock(&g_mu);
    const int f = g_left >= 0 && strcmp(name, g_name) == 0 && g_left-- == 0;
    if (f) {
        g_failed = 1;
        g_last = hipErrorUnknown;
    }
    pthread_mutex_unlock(&g_mu);
    return f;
}
#define MAY_FAIL() \
    if (fails(__func__)) return hipErrorUnknown

static Stream* at(hipStream_t s) { return &g_stream[(size_t)s]; }

static void end(int s, unsigned long upto) {
    if (g_stream[s].ended >= upto) return;
    g_stream[s].ended = upto;
    for (int i = 0; i < kMaxStreams; i++) {
        const unsigned long w = g_stream[s].waits[i];
        g_stream[s].waits[i] = 0;
        end(i, w);
    }
}

static hipError_t launch(const void* fn, hipStream_t s) {
    Stream* st = at(s);
    if (st->capturing)
        st->rec->node[st->rec->n++].fn = fn;
    else
        st->queued++;
    return hipSuccess;
}

/* memory */
hipError_t hipMalloc(void** p, size_t n) {
    MAY_FAIL();
    *p = calloc(n ? n : 1, 1);
    return *p ? hipSuccess : hipErrorOutOfMemory;
}
hipError_t hipFree(void* p) {
    free(p);
    return hipSuccess;
}
hipError_t hipHostMalloc(void** p, size_t n, unsigned int flags) {
    (void)flags;
    return hipMalloc(p, n);
}
hipError_t hipHostFree(void* p) { return hipFree(p); }
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind k) {
    (void)k;
    MAY_FAIL();
    memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind k, hipStream_t st) {
    (void)k;
    MAY_FAIL();
    memcpy(d, s, n);
    at(st)->queued++;
    return hipSuccess;
}
hipError_t hipMemset(void* d, int v, size_t n) {
    memset(d, v, n);
    return hipSuccess;
}
hipError_t hipMemGetInfo(size_t* f, size_t* t) {
    *f = *t = (size_t)1 << 38;
    return hipSuccess;
}
hipError_t hipGetSymbolAddress(void** p, const void* sym) {
    (void)sym;
    return hipMalloc(p, (size_t)16 << 20);
}

/* streams and events */
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned int flags) {
    (void)flags;
    for (size_t i = 1; i < kMaxStreams; i++)
        if (!g_stream[i].live) {
            memset(&g_stream[i], 0, sizeof(Stream));
            g_stream[i].live = 1;
            *s = (hipStream_t)i;
            return hipSuccess;
        }
    return hipErrorOutOfMemory;
}
hipError_t hipStreamDestroy(hipStream_t s) {
    at(s)->live = 0;
    return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t s) {
    MAY_FAIL();
    pthread_mutex_lock(&g_mu);
    end((int)(size_t)s, at(s)->queued);
    pthread_mutex_unlock(&g_mu);
    return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned flags) {
    (void)flags;
    *e = (hipEvent_t)calloc(1, sizeof(Event));
    return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t e) {
    free(e);
    return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
    MAY_FAIL();
    Event* ev = (Event*)e;
    ev->stream = (int)(size_t)s;
    ev->at = at(s)->queued;
    return hipSuccess;
}
hipError_t hipEventQuery(hipEvent_t e) {
    MAY_FAIL();
    pthread_mutex_lock(&g_mu);
    end(((Event*)e)->stream, ((Event*)e)->at);
    pthread_mutex_unlock(&g_mu);
    return hipSuccess;
}
hipError_t hipStreamWaitEvent(hipStream_t s, hipEvent_t e, unsigned int flags) {
    (void)flags;
    MAY_FAIL();
    const Event* ev = (const Event*)e;
    if (at(s)->waits[ev->stream] < ev->at) at(s)->waits[ev->stream] = ev->at;
    at(s)->queued++;
    return hipSuccess;
}

/* launches */
typedef struct {
    dim3 g, b;
    size_t lds;
    hipStream_t s;
} Config;
static __thread Config t_config;
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t lds, hipStream_t s) {
    t_config = (Config){g, b, lds, s};
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* g, dim3* b, size_t* lds, hipStream_t* s) {
    *g = t_config.g, *b = t_config.b, *lds = t_config.lds, *s = t_config.s;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void* fn, dim3 g, dim3 b, void** args, size_t lds, hipStream_t s) {
    (void)g, (void)b, (void)args, (void)lds;
    MAY_FAIL();
    return launch(fn, s);
}
hipError_t hipLaunchCooperativeKernel(const void* fn, dim3 g, dim3 b, void** args, unsigned int lds, hipStream_t s) {
    return hipLaunchKernel(fn, g, b, args, lds, s);
}
hipError_t hipExtLaunchKernel(const void* fn, dim3 g, dim3 b, void** args, size_t lds, hipStream_t s, hipEvent_t e0,
                              hipEvent_t e1, int flags) {
    (void)e0, (void)e1, (void)flags;
    return hipLaunchKernel(fn, g, b, args, lds, s);
}
hipError_t hipGetLastError(void) {
    const hipError_t e = g_last;
    g_last = hipSuccess;
    return e;
}
const char* hipGetErrorString(hipError_t e) {
    (void)e;
    return "stand-in";
}

/* graphs: the kernels of a capture, in order */
hipError_t hipStreamBeginCapture(hipStream_t s, hipStreamCaptureMode mode) {
    (void)mode;
    MAY_FAIL();
    at(s)->rec = calloc(1, sizeof(struct graph));
    at(s)->capturing = 1;
    return hipSuccess;
}
hipError_t hipStreamEndCapture(hipStream_t s, hipGraph_t* g) {
    at(s)->capturing = 0;
    *g = (hipGraph_t)at(s)->rec;
    return hipSuccess;
}
hipError_t hipGraphGetNodes(hipGraph_t g, hipGraphNode_t* nodes, size_t* n) {
    struct graph* r = (struct graph*)g;
    for (size_t i = 0; nodes && i < r->n; i++) nodes[i] = (hipGraphNode_t)&r->node[i];
    *n = r->n;
    return hipSuccess;
}
hipError_t hipGraphKernelNodeGetParams(hipGraphNode_t node, hipKernelNodeParams* p) {
    p->func = (void*)((struct node*)node)->fn;
    return hipSuccess;
}
hipError_t hipGraphInstantiate(hipGraphExec_t* x, hipGraph_t g, hipGraphNode_t* en, char* log, size_t n) {
    (void)g, (void)en, (void)log, (void)n;
    MAY_FAIL();
    *x = (hipGraphExec_t)malloc(1);
    return hipSuccess;
}
hipError_t hipGraphExecKernelNodeSetParams(hipGraphExec_t x, hipGraphNode_t n, const hipKernelNodeParams* p) {
    (void)x, (void)n, (void)p;
    MAY_FAIL();
    return hipSuccess;
}
hipError_t hipGraphLaunch(hipGraphExec_t x, hipStream_t s) {
    (void)x;
    MAY_FAIL();
    at(s)->queued++;
    return hipSuccess;
}
hipError_t hipGraphExecDestroy(hipGraphExec_t x) {
    free(x);
    return hipSuccess;
}
hipError_t hipGraphDestroy(hipGraph_t g) {
    free(g);
    return hipSuccess;
}

/* the device and the code object */
hipError_t hipSetDevice(int d) {
    (void)d;
    return hipSuccess;
}
hipError_t hipGetDevice(int* d) {
    *d = 0;
    return hipSuccess;
}
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t a, int d) {
    (void)a, (void)d;
    *v = 256;
    return hipSuccess;
}
hipError_t hipFuncSetAttribute(const void* fn, hipFuncAttribute a, int v) {
    (void)fn, (void)a, (void)v;
    return hipSuccess;
}
hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int* n, const void* fn, int b, size_t lds) {
    (void)fn, (void)b, (void)lds;
    *n = 1;
    return hipSuccess;
}
void** __hipRegisterFatBinary(const void* data) {
    (void)data;
    static void* handle;
    return &handle;
}
void __hipRegisterFunction(void** m, const void* fn, char* a, const char* b, unsigned int c, void* d, void* e, dim3* f,
                           dim3* g, int* h) {
    (void)m, (void)fn, (void)a, (void)b, (void)c, (void)d, (void)e, (void)f, (void)g, (void)h;
}
void __hipRegisterVar(void** m, void* v, char* a, const char* b, int c, size_t d, int e, int f) {
    (void)m, (void)v, (void)a, (void)b, (void)c, (void)d, (void)e, (void)f;
}
void __hipUnregisterFatBinary(void** m) { (void)m; }
