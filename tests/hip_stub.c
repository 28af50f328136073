/* The HIP runtime calls of the package's libraries over ordinary memory, for tests of their host side without a GPU: streams
 * and graphs keep their order, a kernel does nothing, and an asynchronous copy happens when its stream is waited for - the last
 * moment at which the real one may.  Loaded RTLD_GLOBAL before the libraries, so that their calls come here. */
#include <stdbool.h>
#include <stdint.h>
#include <stdlib.h>
#include <string.h>

enum { kSuccess = 0, kInvalidValue = 1, kCaptureUnsupported = 900 };

typedef struct { /* one operation: a copy, or a kernel (n == 0) */
    void *dst;
    const void *src;
    size_t n;
} action;
typedef struct {
    action *a;
    size_t n, cap;
} list;
typedef struct stream {
    list queue, graph;
    bool capturing;
    struct stream *next;
} stream;

static stream g_null, *g_streams = &g_null;
static int g_error;
long stub_kernels, stub_captures, stub_graph_launches, stub_fail_instantiate;

static int set(int e)
{
    if (e)
        g_error = e;
    return e;
}
static stream *of(void *st) { return st ? st : &g_null; }
static void push(list *l, action a)
{
    if (l->n == l->cap)
        l->a = realloc(l->a, (l->cap = 2 * l->cap + 16) * sizeof(action));
    l->a[l->n++] = a;
}
static void drain(stream *s)
{
    for (size_t i = 0; i < s->queue.n; i++)
        if (s->queue.a[i].n)
            memcpy(s->queue.a[i].dst, s->queue.a[i].src, s->queue.a[i].n);
    s->queue.n = 0;
}
static void enqueue(void *st, action a) { push(of(st)->capturing ? &of(st)->graph : &of(st)->queue, a); }

/* what the tests ask */
long stub_pending(void *st) { return (long)of(st)->queue.n; }
int stub_error(void) { return g_error; }

int hipGetDeviceCount(int *n) { return *n = 1, kSuccess; }
int hipSetDevice(int d) { return d ? set(kInvalidValue) : kSuccess; }
const char *hipGetErrorString(int e) { return e == kCaptureUnsupported ? "operation not permitted when stream is capturing" : "error"; }
int hipGetLastError(void)
{
    const int e = g_error;
    g_error = 0;
    return e;
}
int hipDeviceSynchronize(void)
{
    for (stream *s = g_streams; s; s = s->next)
        drain(s);
    return kSuccess;
}
int hipMalloc(void **p, size_t n) /* whole pages, as the runtime gives */
{
    n = (n + 4096) / 4096 * 4096;
    *p = aligned_alloc(4096, n);
    memset(*p, 0, n);
    return kSuccess;
}
int hipFree(void *p) { return hipDeviceSynchronize(), free(p), kSuccess; }
int hipHostMalloc(void **p, size_t n, unsigned f) { return (void)f, hipMalloc(p, n); }
int hipHostFree(void *p) { return hipFree(p); }
int hipMemcpy(void *d, const void *s, size_t n, int k) { return (void)k, drain(&g_null), memcpy(d, s, n), kSuccess; }
int hipMemcpyAsync(void *d, const void *s, size_t n, int k, void *st) { return (void)k, enqueue(st, (action){d, s, n}), kSuccess; }
int hipStreamCreateWithFlags(void **st, unsigned f)
{
    stream *s = calloc(1, sizeof *s);
    (void)f;
    s->next = g_streams->next, g_streams->next = s;
    *st = s;
    return kSuccess;
}
int hipStreamDestroy(void *st)
{
    for (stream *s = g_streams; s; s = s->next)
        if (s->next == st)
            s->next = s->next->next;
    free(st);
    return kSuccess;
}
int hipStreamSynchronize(void *st) { return drain(of(st)), kSuccess; }
int hipStreamIsCapturing(void *st, int *state) { return *state = of(st)->capturing, kSuccess; }
int hipStreamBeginCapture(void *st, int mode)
{
    (void)mode;
    if (st == NULL)
        return set(kCaptureUnsupported); /* the null stream cannot be captured */
    of(st)->capturing = true, of(st)->graph.n = 0;
    stub_captures++;
    return kSuccess;
}
int hipStreamEndCapture(void *st, void **g)
{
    list *l = calloc(1, sizeof *l);
    for (size_t i = 0; i < of(st)->graph.n; i++)
        push(l, of(st)->graph.a[i]);
    of(st)->capturing = false;
    *g = l;
    return kSuccess;
}
int hipGraphGetNodes(void *g, void **nodes, size_t *n) { return (void)nodes, *n = ((list *)g)->n, kSuccess; }
int hipGraphInstantiate(void **e, void *g, void **node, char *log, size_t n)
{
    list *l = calloc(1, sizeof *l);
    (void)node, (void)log, (void)n;
    if (stub_fail_instantiate)
        return set(kInvalidValue);
    for (size_t i = 0; i < ((list *)g)->n; i++)
        push(l, ((list *)g)->a[i]);
    *e = l;
    return kSuccess;
}
static int drop(void *g) { return free(((list *)g)->a), free(g), kSuccess; }
int hipGraphDestroy(void *g) { return drop(g); }
int hipGraphExecDestroy(void *g) { return drop(g); }
int hipGraphLaunch(void *e, void *st)
{
    for (size_t i = 0; i < ((list *)e)->n; i++)
        push(&of(st)->queue, ((list *)e)->a[i]);
    stub_graph_launches++;
    return kSuccess;
}

/* the device functions' names, by the host stubs that launch them */
static struct { const void *f; const char *name; } g_kernels[4096];
static size_t g_nkernels;
const char *stub_last_kernel = "";

/* a launch is __hipPushCallConfiguration, the kernel's host stub, __hipPopCallConfiguration and hipLaunchKernel */
typedef struct { uint32_t x, y, z; } dim3;
static dim3 g_grid, g_block;
static size_t g_lds;
static void *g_stream;
int __hipPushCallConfiguration(dim3 g, dim3 b, size_t lds, void *st) { return g_grid = g, g_block = b, g_lds = lds, g_stream = st, kSuccess; }
int __hipPopCallConfiguration(dim3 *g, dim3 *b, size_t *lds, void **st) { return *g = g_grid, *b = g_block, *lds = g_lds, *st = g_stream, kSuccess; }
int hipLaunchKernel(const void *f, dim3 g, dim3 b, void **args, size_t lds, void *st)
{
    (void)g, (void)b, (void)args, (void)lds;
    for (size_t i = 0; i < g_nkernels; i++)
        if (g_kernels[i].f == f)
            stub_last_kernel = g_kernels[i].name;
    enqueue(st, (action){0});
    stub_kernels++;
    return kSuccess;
}
void **__hipRegisterFatBinary(const void *d)
{
    static void *handle;
    return (void)d, &handle;
}
void __hipUnregisterFatBinary(void **h) { (void)h; }
void __hipRegisterFunction(void **h, const void *f, char *d, const char *n, unsigned t, void *a, void *b, void *c, void *e, int *w)
{
    (void)h, (void)d, (void)t, (void)a, (void)b, (void)c, (void)e, (void)w;
    if (g_nkernels < sizeof g_kernels / sizeof *g_kernels)
        g_kernels[g_nkernels].f = f, g_kernels[g_nkernels++].name = n;
}
