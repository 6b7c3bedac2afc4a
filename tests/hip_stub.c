/* A HIP runtime of host memory, and kernels that do nothing, under fs_host.c:
 * lets a test without a GPU follow what the host code allocates, frees and
 * waits for. */
#include "../futspace_amd/csrc/fs_internal.h"

#include <stdlib.h>
#include <string.h>

int64_t stub_mallocs, stub_frees, stub_live, stub_limit = INT64_MAX;
int stub_capturing;
static hipError_t last;

static hipError_t take(void)
{
    hipError_t e = last;
    last = hipSuccess;
    return e;
}

/* Like the device's: a failed call stays the last error until it is asked for. */
hipError_t hipGetLastError(void) { return take(); }

hipError_t hipMalloc(void **p, size_t bytes)
{
    *p = NULL;
    if (stub_live + (int64_t)bytes > stub_limit)
        return last = hipErrorOutOfMemory;
    size_t *m = (size_t *)malloc(bytes + 64);
    m[0] = bytes;
    stub_live += (int64_t)bytes;
    stub_mallocs++;
    *p = (char *)m + 64;
    return hipSuccess;
}

hipError_t hipFree(void *p)
{
    if (!p)
        return hipSuccess;
    size_t *m = (size_t *)((char *)p - 64);
    stub_live -= (int64_t)m[0];
    stub_frees++;
    free(m);
    return hipSuccess;
}

hipError_t hipStreamIsCapturing(hipStream_t s, hipStreamCaptureStatus *st)
{
    (void)s;
    *st = stub_capturing ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone;
    return hipSuccess;
}

hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind k)
{
    (void)k;
    memcpy(d, s, n);
    return hipSuccess;
}

hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind k, hipStream_t st)
{
    (void)st;
    return hipMemcpy(d, s, n, k);
}

hipError_t hipMemsetAsync(void *d, int v, size_t n, hipStream_t s)
{
    (void)s;
    memset(d, v, n);
    return hipSuccess;
}

hipError_t hipGetDeviceCount(int *n) { *n = 1; return hipSuccess; }
hipError_t hipGetDevice(int *d) { *d = 0; return hipSuccess; }
hipError_t hipSetDevice(int d) { (void)d; return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t s) { (void)s; return hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t s) { (void)s; return hipSuccess; }
hipError_t hipStreamBeginCapture(hipStream_t s, hipStreamCaptureMode m) { (void)s; (void)m; return hipSuccess; }
hipError_t hipStreamEndCapture(hipStream_t s, hipGraph_t *g) { (void)s; *g = NULL; return hipSuccess; }
hipError_t hipGraphDestroy(hipGraph_t g) { (void)g; return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t g) { (void)g; return hipSuccess; }
hipError_t hipGraphLaunch(hipGraphExec_t g, hipStream_t s) { (void)g; (void)s; return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t *e) { *e = NULL; return hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t e) { (void)e; return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t e) { (void)e; return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) { (void)e; (void)s; return hipSuccess; }
const char *hipGetErrorString(hipError_t e) { return e == hipErrorOutOfMemory ? "out of memory" : "error"; }

hipError_t hipEventElapsedTime(float *ms, hipEvent_t a, hipEvent_t b)
{
    (void)a;
    (void)b;
    *ms = 0.0f;
    return hipSuccess;
}

hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned flags)
{
    static char streams[64];
    static int n;
    (void)flags;
    *s = (hipStream_t)&streams[n++ % 64];
    return hipSuccess;
}

hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600 *p, int d)
{
    (void)d;
    memset(p, 0, sizeof *p);
    return hipSuccess;
}

hipError_t hipGraphInstantiate(hipGraphExec_t *x, hipGraph_t g, hipGraphNode_t *n, char *log, size_t len)
{
    (void)g;
    (void)n;
    (void)log;
    (void)len;
    *x = NULL;
    return hipSuccess;
}

/* A launch returns the last error, as the real launchers do. */
#define LAUNCH(name, ...) int name(__VA_ARGS__) { return take(); }
#pragma GCC diagnostic ignored "-Wunused-parameter"

int fsk_device_init(void) { return 0; }
void fsk_default_tuning(fsk_tuning *t) { memset(t, 0, sizeof *t); }
int32_t fsk_render_max_rows(void) { return 1 << 22; }
int32_t fsk_batch_max_rows(void) { return 7680; }
int32_t fsk_limit_block_rows(int32_t w, int32_t h) { return 16; }
int32_t fsk_tile_columns(int32_t r, const fsk_tuning *t) { return 8; }
int32_t fsk_batch_grid(int32_t r, const fsk_tuning *t) { return 256; }
void fsk_batch_shape(int32_t r, int64_t a, int64_t b, fsk_tuning *t) {}
void fsk_batch_counters_init(uint32_t *c, int32_t g, int32_t n) {}
int32_t fsk_tame_level(const fsk_frame *f, int32_t s) { return 0; }
void fsk_map_recips(fsk_map *m) {}
double *fsk_scratch(int32_t d) { static double x[FSK_PARTIALS]; return x; }
LAUNCH(fsk_selftest, int w, unsigned long long *b, hipStream_t s)
LAUNCH(fsk_batch_run, const fsk_batch *b, hipStream_t s)
LAUNCH(fsk_render, const fsk_map *m, const fsk_frame *f, const fsk_tuning *t, uint32_t *o, int64_t p, hipStream_t s)
LAUNCH(fsk_render_nearest, const fsk_map *m, const fsk_frame *f, const fsk_tuning *t, uint32_t *o, int64_t p, hipStream_t s)
LAUNCH(fsk_render_slices, const fsk_map *m, const fsk_frame *f, const fsk_tuning *t, int32_t *o, int64_t p, hipStream_t s)
LAUNCH(fsk_render_slices_clear, const fsk_map *m, const fsk_frame *f, const fsk_tuning *t, int32_t *o, int64_t p, float *z, size_t n, int32_t *c, hipStream_t s)
LAUNCH(fsk_render2, const fsk_map *m, const fsk_frame *f, const float *c, const float *n, const uint32_t *d, int32_t k, uint32_t *o, int64_t p, hipStream_t s)
LAUNCH(fsk_height_quads, const int32_t *a, int32_t r, int32_t c, int32_t b, void *q, uint16_t *p, uint32_t *m, hipStream_t s)
LAUNCH(fsk_shade, const uint16_t *h, const uint32_t *m, int32_t r, int32_t c, const uint32_t *d, const float u[3], int32_t z, void *o, hipStream_t s)
LAUNCH(fsk_color_quads, const uint32_t *d, int32_t r, int32_t c, void *q, hipStream_t s)
LAUNCH(fsk_diff_color, const fsk_frame *f, const float *c, const float *sf, int32_t h, int32_t w, float k, const int32_t *r, float *i, hipStream_t s)
LAUNCH(fsk_diff_grad, const fsk_frame *f, const float *c, const float *sf, int32_t h, int32_t w, const int32_t *r, const float *g, float *p, float *k, int32_t a, double *d, int32_t n, hipStream_t s)
LAUNCH(fsk_diff_step_l2, const fsk_frame *f, const float *c, const float *sf, int32_t h, int32_t w, float k, const int32_t *r, const float *t, float *i, float *g, float *p, float *y, int32_t a, float *l, int32_t b, double *d, double *e, int32_t n, hipStream_t s)
LAUNCH(fsk_zero_f32, float *p, size_t n, hipStream_t s)
LAUNCH(fsk_fill_u32, uint32_t *p, size_t n, uint32_t v, hipStream_t s)
LAUNCH(fsk_l2_loss, const float *i, const float *t, size_t n, float *g, float *l, int32_t a, double *p, int32_t k, hipStream_t s)
LAUNCH(fsk_adam, float *p, const float *g, float *m, float *v, size_t n, double l, double b, double c, double e, int32_t t, int32_t f, float lo, float hi, hipStream_t s)
