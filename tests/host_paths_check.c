/* Host paths of the runtime on a HIP runtime of its own, without a GPU.
 *
 * The HIP entry points that libtl_int8.so calls are defined here, in the
 * executable, which the dynamic linker searches before libamdhip64.  Memory is
 * the host's, kernels are counted and not run, work on a stream is "queued"
 * until the next hipStreamSynchronize, and the operation number fail_at (a
 * launch or an asynchronous copy) returns an error.  A failing call must not
 * return with work still queued that reads or writes the caller's memory.  A
 * captured step may hold the address of any buffer that was there when it was
 * instantiated: none may be launched after such a buffer was freed.
 *
 * Built with -rdynamic and linked with the library; prints one line per
 * scenario and exits with the number of violations. */
#include <hip/hip_runtime_api.h>
#include <stdint.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#include "tl_int8.h"

static long ops, fail_at, queued;   /* operations since arm(); the one that fails (0: none); queued work */
static hipError_t last;
static int capturing;

static hipError_t op(void) {
    if (++ops == fail_at) return last = hipErrorLaunchFailure;
    if (!capturing) queued++;
    return hipSuccess;
}

/* device buffers and captured steps, by order of birth */
enum { MAXBUF = 1024, MAXEXEC = 64 };
static struct { void* p; long born; } bufs[MAXBUF];
static struct exec { long born; int stale; } *execs[MAXEXEC];
static long births;
static int stale_launches;

/* ---- the HIP entry points the library uses --------------------------------- */
hipError_t hipGetDeviceCount(int* n) { *n = 1; return hipSuccess; }
hipError_t hipGetDevice(int* d) { *d = 0; return hipSuccess; }
hipError_t hipGetDeviceProperties(hipDeviceProp_t* p, int d) {
    (void)d;
    memset(p, 0, sizeof *p);
    strcpy(p->gcnArchName, "gfx950");
    return hipSuccess;
}
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t a, int d) { (void)a; (void)d; *v = 256; return hipSuccess; }
const char* hipGetErrorString(hipError_t e) { return e == hipSuccess ? "ok" : "planted failure"; }
hipError_t hipGetLastError(void) { hipError_t e = last; last = hipSuccess; return e; }
hipError_t hipMalloc(void** p, size_t n) {
    *p = aligned_alloc(256, (n + 255) / 256 * 256);
    for (int i = 0; *p && i < MAXBUF; i++)
        if (!bufs[i].p) {
            bufs[i].p = *p;
            bufs[i].born = ++births;
            return hipSuccess;
        }
    return hipErrorOutOfMemory;
}
hipError_t hipFree(void* p) {
    for (int i = 0; p && i < MAXBUF; i++)
        if (bufs[i].p == p) {
            for (int j = 0; j < MAXEXEC; j++)
                if (execs[j] && execs[j]->born > bufs[i].born) execs[j]->stale = 1;
            bufs[i].p = NULL;
            break;
        }
    free(p);
    return hipSuccess;
}
hipError_t hipHostMalloc(void** p, size_t n, unsigned f) { (void)f; *p = calloc(1, n); return hipSuccess; }
hipError_t hipHostFree(void* p) { free(p); return hipSuccess; }
hipError_t hipHostGetDevicePointer(void** d, void* h, unsigned f) { (void)f; *d = h; return hipSuccess; }
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind k) { (void)k; memcpy(d, s, n); return hipSuccess; }
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind k, hipStream_t st) {
    (void)k; (void)st;
    hipError_t e = op();
    if (e == hipSuccess) memmove(d, s, n);
    return e;
}
hipError_t hipMemsetAsync(void* d, int v, size_t n, hipStream_t st) { (void)st; memset(d, v, n); return hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned f) { (void)f; *s = (hipStream_t)1; return hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t s) { (void)s; return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t s) { (void)s; queued = 0; return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t s, hipEvent_t e, unsigned f) { (void)s; (void)e; (void)f; return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t* e) { *e = (hipEvent_t)1; return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned f) { (void)f; return hipEventCreate(e); }
hipError_t hipEventDestroy(hipEvent_t e) { (void)e; return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) { (void)e; (void)s; return hipSuccess; }
hipError_t hipEventQuery(hipEvent_t e) { (void)e; return hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t a, hipEvent_t b) { (void)a; (void)b; *ms = 0.0f; return hipSuccess; }
hipError_t hipFuncSetAttribute(const void* f, hipFuncAttribute a, int v) { (void)f; (void)a; (void)v; return hipSuccess; }
hipError_t hipGetSymbolAddress(void** p, const void* s) { (void)s; static char scratch[256]; *p = scratch; return hipSuccess; }
hipError_t hipStreamBeginCapture(hipStream_t s, hipStreamCaptureMode m) { (void)s; (void)m; capturing = 1; return hipSuccess; }
hipError_t hipStreamEndCapture(hipStream_t s, hipGraph_t* g) { (void)s; capturing = 0; *g = (hipGraph_t)1; return hipSuccess; }
hipError_t hipGraphInstantiate(hipGraphExec_t* x, hipGraph_t g, hipGraphNode_t* n, char* b, size_t z) {
    (void)g; (void)n; (void)b; (void)z;
    for (int j = 0; j < MAXEXEC; j++)
        if (!execs[j]) {
            execs[j] = malloc(sizeof(struct exec));
            execs[j]->born = ++births;
            execs[j]->stale = 0;
            *x = (hipGraphExec_t)execs[j];
            return hipSuccess;
        }
    return hipErrorOutOfMemory;
}
hipError_t hipGraphDestroy(hipGraph_t g) { (void)g; return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t x) {
    for (int j = 0; j < MAXEXEC; j++)
        if ((void*)execs[j] == (void*)x) execs[j] = NULL;
    free(x);
    return hipSuccess;
}
hipError_t hipGraphLaunch(hipGraphExec_t x, hipStream_t s) {
    (void)s;
    stale_launches += ((struct exec*)x)->stale;
    return op();
}
static dim3 cfg_grid, cfg_block;
static size_t cfg_lds;
static hipStream_t cfg_stream;
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t l, hipStream_t s) {
    cfg_grid = g; cfg_block = b; cfg_lds = l; cfg_stream = s;
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* g, dim3* b, size_t* l, hipStream_t* s) {
    *g = cfg_grid; *b = cfg_block; *l = cfg_lds; *s = cfg_stream;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void* f, dim3 g, dim3 b, void** a, size_t l, hipStream_t s) {
    (void)f; (void)g; (void)b; (void)a; (void)l; (void)s;
    return op();
}

/* ---- a small model and the calls -------------------------------------------- */
enum { D = 512, HKV = 2, V = 256, MAXPOS = 256, LAYERS = 2 };

static tl_handle* make(int F, int max_seqs) {
    const tl_config c = {D, F, LAYERS, D / 64, HKV, 64, V, MAXPOS, 1e-5f, 10000.0f};
    tl_handle* h = NULL;
    if (tl_create(&c, max_seqs, &h) != TL_OK) {
        printf("tl_create: %s\n", tl_last_error(NULL));
        exit(100);
    }
    int8_t* w = calloc(1, (size_t)F * D);
    float* s = calloc(F, sizeof(float));
    const int8_t* ws[7] = {w, w, w, w, w, w, w};
    const float* ss[7] = {s, s, s, s, s, s, s};
    for (int l = 0; l < LAYERS; l++)
        if (tl_load_layer(h, l, ws, ss, s, s, TL_MEM_HOST) != TL_OK) exit(101);
    if (tl_load_lm_head(h, w, s, s, TL_MEM_HOST) != TL_OK || tl_load_embedding(h, w, s, TL_MEM_HOST) != TL_OK) exit(102);
    free(w);
    free(s);
    return h;
}

static float* rows;
static int32_t tokens[MAXPOS];
static float logits[(size_t)MAXPOS * V];

struct call {
    const char* name;
    int n, shift;
};

static int run(tl_handle* h, const struct call* c) {
    int32_t tok, n;
    float lg;
    if (!strcmp(c->name, "layer")) return tl_decode_layer(h, 0, 1, 7, rows + c->shift);
    if (!strcmp(c->name, "rows")) return tl_layer_rows(h, 0, 1, 7, c->n, rows + c->shift);
    if (!strcmp(c->name, "prefill")) return tl_prefill(h, 0, tokens, c->n, &tok, &lg);
    if (!strcmp(c->name, "logits")) return tl_prefill_logits(h, 0, tokens, c->n, logits);
    return tl_generate(h, 0, tokens, c->n, 1, -1, NULL, &tok, &n, NULL);
}

/* batches whose split-K scratch grows (1408 is no multiple of 512: no packed
 * form), back to the small ones, on one handle */
static int alternating_batches(void) {
    static const int sizes[] = {4, 40, 60, 0, 4, 40, 60};   /* 0: a scored prompt of 63 tokens */
    static int32_t start[60], out[60 * 4];
    tl_handle* h = make(1408, 60);
    int wrong = 0;
    for (size_t i = 0; i < sizeof sizes / sizeof sizes[0]; i++)
        wrong += (sizes[i] ? tl_decode_batch(h, sizes[i], tokens, start, 4, out)
                           : tl_prefill_logits(h, 0, tokens, 63, logits)) != TL_OK;
    printf("alternating batches: %d failed, %d launches of steps that hold a freed buffer\n", wrong, stale_launches);
    tl_destroy(h);
    return wrong + stale_launches;
}

int main(void) {
    static const struct call calls[] = {
        {"layer", 1, 0}, {"layer", 1, 1}, {"rows", 1, 0}, {"rows", 5, 0}, {"rows", 5, 3}, {"rows", 40, 0}, {"rows", 70, 0},
        {"rows", 70, 2}, {"prefill", 1, 0}, {"prefill", 20, 0}, {"prefill", 40, 0}, {"prefill", 70, 0}, {"logits", 20, 0},
        {"logits", 40, 0}, {"logits", 70, 0}, {"generate", 20, 0}};
    rows = aligned_alloc(256, sizeof(float) * (D * MAXPOS + 64));
    memset(rows, 0, sizeof(float) * (D * MAXPOS + 64));
    int bad = 0;
    for (size_t i = 0; i < sizeof calls / sizeof calls[0]; i++) {
        const struct call* c = &calls[i];
        tl_handle* h = make(1024, 4);
        ops = fail_at = 0;
        int wrong = run(h, c) != TL_OK || queued != 0;
        const long total = ops;
        for (long f = 1; f <= total; f++) {
            ops = 0;
            fail_at = f;
            const int r = run(h, c);
            fail_at = 0;
            if (r == TL_OK || queued != 0) wrong++;
            queued = 0;
            if (run(h, c) != TL_OK || queued != 0) wrong++;   /* and the handle works on */
        }
        printf("%s n=%d shift=%d: %ld operations, %d wrong\n", c->name, c->n, c->shift, total, wrong);
        bad += wrong;
        tl_destroy(h);
    }
    free(rows);
    bad += alternating_batches();
    return bad > 255 ? 255 : bad;
}
