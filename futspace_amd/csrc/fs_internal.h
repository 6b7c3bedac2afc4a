/*
 * fs_internal.h -- interface between the C host library (fs_host.c) and
 * the HIP kernel launchers (fs_kernels.hip).  Not installed; no torch or
 * HIP C++ types cross it.
 */
#ifndef FS_INTERNAL_H
#define FS_INTERNAL_H

#include <stdint.h>
#include <hip/hip_runtime_api.h>

#ifdef __cplusplus
extern "C" {
#endif

/* Device view of a resident map pair.
 *   hq: per texel (r,c) the bilinear quad of masked heights
 *       h(r,c), h(r,c+1), h(r+1,c), h(r+1,c+1) (indices wrap), packed as
 *       4 x u8 in a u32 (hbits 8) or 4 x u16 in a uint2 (hbits 16);
 *   cq: the same quad of shaded colours, one uint4 per shade texel. */
typedef struct {
    const void *hq;
    int32_t hrows, hcols, hbits;
    const void *cq;
    int32_t crows, ccols;
    float rhrows, rhcols, rcrows, rccols;   /* fsk_map_recips; set by the launchers */
} fsk_map;

/* Per-frame scalars, computed on the host exactly as `futhark c` does:
 *   lx = Lx*z, ly = Ly*z, rx = Rx*z, ry = Ry*z  (fut/voxel_renderer.fut:47-50)
 * with Lx = (-cos a) - sin a*fov, Ly = sin a - cos a*fov,
 *      Rx = cos a - sin a*fov,   Ry = (-sin a) - cos a*fov. */
typedef struct {
    float cam_x, cam_y, cam_h, horizon;
    float Lx, Ly, Rx, Ry;
    float d, z0, scale, fw;
    float rfw;           /* 1 / fw, correctly rounded (the host's f32 division) */
    int32_t n, rows, cols;
    uint32_t sky;
    int32_t tame;        /* fsk_tame_level; set by the launchers */
} fsk_frame;

/* FSK_TAME when every sample of the frame stays where the render kernel may
 * skip the out-of-range branches of the x86 casts: finite scalars, slice
 * depths increasing from z0 > 0, every sample coordinate below 2^22 and every
 * projected row below 2^30 in magnitude for any 16-bit height; else 0.
 * FSK_TAME_MOD when besides the coordinates are below 2^21 and max_side, the
 * longest side of the sampled maps, is at most 2^20, so that sides that are
 * no powers of two may be wrapped by reciprocals. */
#define FSK_TAME 1
#define FSK_TAME_MOD 2
int32_t fsk_tame_level(const fsk_frame *f, int32_t max_side);
/* The level of a frame over maps of any size: FSK_TAME or 0.  The line that
 * the tests evaluate by brute force is thereby the one that the launchers use. */
int32_t fsk_frame_tame(const fsk_frame *f);
/* A reciprocal of m a little below 1 / m, for such wraps; a map's four. */
float fsk_wrap_recip(int32_t m);
void fsk_map_recips(fsk_map *m);

/* Once per device, before its first render: uploads the kernels' constant
 * tables (the byte quantisation table of the colour path).  Thread-safe;
 * later calls on the same device return at once. */
int fsk_device_init(void);

/* The device address of `device`'s fixed scratch array of FSK_PARTIALS
 * doubles (set up by fsk_device_init; NULL before).  Shared by every caller
 * on that device. */
double *fsk_scratch(int32_t device);

/* render2 (ray march) of one frame into out[rows][pitch]: d_cs/d_sn[cols]
 * the host's cos / sin of angle + horz_ang per column, d_color the map's
 * unshaded colours [hrows][hcols], n = i32(distance / 4). */
int fsk_render2(const fsk_map *m, const fsk_frame *f, const float *d_cs, const float *d_sn,
                const uint32_t *d_color, int32_t n, uint32_t *d_out, int64_t pitch, hipStream_t s);

/* Tuning knobs of the render kernels (0 = automatic). */
typedef struct {
    int32_t tc;          /* frame columns per workgroup tile: 4 or 8 */
    int32_t wg_per_cu;   /* 1 or 2 workgroups per CU */
    int32_t chunk;       /* depth slices per chunk: 256..2048 */
} fsk_tuning;

/* The tuning a new context starts from: the FSX_RENDER_TC,
 * FSX_RENDER_WG_PER_CU and FSX_RENDER_CHUNK environment variables (unset:
 * 0, automatic). */
void fsk_default_tuning(fsk_tuning *t);

/* Plain render of one frame into out[rows][pitch] in the kernel shape
 * that t selects; the kernel builds its own slice table per depth chunk. */
int fsk_render(const fsk_map *m, const fsk_frame *f, const fsk_tuning *t, uint32_t *d_out,
               int64_t pitch, hipStream_t s);
/* Frame rows a render takes (frames taller than a tile's limit are rendered
 * in bands of rows), and the rows of a batched view. */
int32_t fsk_render_max_rows(void);
int32_t fsk_batch_max_rows(void);
/* The differentiable passes' limit on frames counts blocks of 64 columns by
 * this many rows (16, or 32 in frames of 2^22 pixels or more).  The adjoint's
 * own workgroups cover half as many rows each or more, and leave one partial
 * sum each: FSK_PARTIALS holds two for every block of the largest frame. */
int32_t fsk_limit_block_rows(int32_t w, int32_t h);
#define FSK_LIMIT_BLOCKS 32768
#define FSK_PARTIALS (2 * FSK_LIMIT_BLOCKS)

/* One view of a batched render, as the persistent kernel reads it. */
typedef struct {
    fsk_map m;
    fsk_frame f;
    int64_t offset;      /* first output element of the view */
    int32_t ntiles;
} fsk_batch_view;

/* A prepared batch: the device arrays stay valid while it is launched. */
typedef struct {
    const fsk_batch_view *views;   /* device */
    const uint32_t *items;         /* device: view << 16 | tile, grouped by queue */
    const uint32_t *qmeta;         /* device: qstart[nqueues], qlen[nqueues] */
    uint32_t *counters;            /* device: FSK_BATCH_COUNTERS(nqueues) claim counters */
    uint32_t *out;
    int32_t nqueues, max_rows, hbits, pow2;
    int32_t grid;                  /* persistent workgroups */
    fsk_tuning tune;
} fsk_batch;

/* Sets a tuning left automatic to the shape of a batch with views of up to
 * max_rows rows, of tiles4 tiles of 4 columns or tiles8 of 8 in all. */
void fsk_batch_shape(int32_t max_rows, int64_t tiles4, int64_t tiles8, fsk_tuning *t);
/* Columns per tile the kernels use for frames of max_rows rows. */
int32_t fsk_tile_columns(int32_t max_rows, const fsk_tuning *t);
/* Persistent workgroups for a batch (CUs x workgroups per CU). */
int32_t fsk_batch_grid(int32_t max_rows, const fsk_tuning *t);
/* The claim counters of a batch: one per queue and one of ended workgroups,
 * FSK_COUNTER_STRIDE words apart so that each has a cache line of its own.
 * fsk_batch_counters_init fills the host image that is uploaded with the
 * batch; every launch leaves them in that state again. */
#define FSK_COUNTER_STRIDE 64
#define FSK_BATCH_COUNTERS(nqueues) (((nqueues) + 1) * FSK_COUNTER_STRIDE)
void fsk_batch_counters_init(uint32_t *counters, int32_t grid, int32_t nqueues);
/* Run the persistent batched render. */
int fsk_batch_run(const fsk_batch *b, hipStream_t s);

/* Device self-test `which` (0-8) of the arithmetic shortcuts; adds the
 * number of mismatching inputs to *d_bad. */
int fsk_selftest(int which, unsigned long long *d_bad, hipStream_t s);

/* Map preparation.  fsk_height_quads also writes the map's largest masked
 * height to d_hmax, as FSK_HMAX_PARTS values whose maximum it is.  fsk_shade evaluates the sun-ray counts of the size^2
 * grid and writes the shaded colours of d_color (u32), or, with d_color
 * NULL, the shade factors sqrt(1 / (4*count + 1)) (f32). */
#define FSK_HMAX_PARTS 128
int fsk_height_quads(const int32_t *d_alt, int32_t rows, int32_t cols, int32_t hbits,
                     void *d_hq, uint16_t *d_hplain, uint32_t *d_hmax, hipStream_t s);
int fsk_shade(const uint16_t *d_hplain, const uint32_t *d_hmax, int32_t rows, int32_t cols,
              const uint32_t *d_color, const float sun[3], int32_t size, void *d_out,
              hipStream_t s);
int fsk_color_quads(const uint32_t *d_col, int32_t rows, int32_t cols, void *d_cq,
                    hipStream_t s);

/* Differentiable renderer (f32 colour planes, visibility held fixed).
 * fsk_render_slices writes, per pixel, the depth slice whose sample shows
 * there (-1: sky); fsk_diff_color turns it into img[3][rows][cols];
 * fsk_diff_grad adds dL/dcp into d_gcp[3][hc][wc] and dL/dsky_scale into
 * *d_gsky (both accumulate). */
int fsk_render_slices(const fsk_map *m, const fsk_frame *f, const fsk_tuning *t, int32_t *d_src,
                      int64_t pitch, hipStream_t s);
/* fsk_render_slices that also clears d_zero[zero_n] (float4-aligned) in
 * extra workgroups on the CUs its tiles leave idle, when enough are; sets
 * *cleared to 1 if it did (else the caller clears). */
int fsk_render_slices_clear(const fsk_map *m, const fsk_frame *f, const fsk_tuning *t,
                            int32_t *d_src, int64_t pitch, float *d_zero, size_t zero_n,
                            int32_t *cleared, hipStream_t s);
/* The stateless program of tests/futspace.fut: m.hq = i32 heights and
 * m.cq = i32 colours, both [hrows][hcols], nearest sampling; f.sky is the
 * program's sky (also its `empty` colour). */
int fsk_render_nearest(const fsk_map *m, const fsk_frame *f, const fsk_tuning *t,
                       uint32_t *d_out, int64_t pitch, hipStream_t s);
int fsk_diff_color(const fsk_frame *f, const float *d_cp, const float *d_sf, int32_t hc,
                   int32_t wc, float sky_scale, const int32_t *d_src, float *d_img, hipStream_t s);
int fsk_diff_grad(const fsk_frame *f, const float *d_cp, const float *d_sf, int32_t hc,
                  int32_t wc, const int32_t *d_src, const float *d_gimg, float *d_gcp,
                  float *d_gsky, int32_t sky_accumulate, double *d_partials, int32_t n_partials,
                  hipStream_t s);
/* The fused L2 step after the slice render: for each pixel the colour px
 * (written to d_img if not null), g = 2 (px - d_tgt) (written to d_g if not
 * null), the loss sum (px - tgt)^2 into *d_loss and dL/dcp into d_gcp (which
 * accumulates; the caller clears it first), dL/dsky_scale into *d_gsky.  The
 * loss and sky terms go through per-workgroup partials d_loss_part and
 * d_sky_part [n_partials each], summed in a fixed order. */
int fsk_diff_step_l2(const fsk_frame *f, const float *d_cp, const float *d_sf, int32_t hc,
                     int32_t wc, float sky_scale, const int32_t *d_src, const float *d_tgt,
                     float *d_img, float *d_g, float *d_gcp, float *d_gsky,
                     int32_t sky_accumulate, float *d_loss, int32_t loss_accumulate,
                     double *d_loss_part, double *d_sky_part, int32_t n_partials, hipStream_t s);
int fsk_zero_f32(float *d_p, size_t n, hipStream_t s);
/* One bias-corrected Adam step (step t >= 1) on d_p[n] with gradient d_g
 * and moments d_m, d_v, then d_p clamped to [lo, hi].  first: the moments
 * are zero and only written. */
int fsk_adam(float *d_p, const float *d_g, float *d_m, float *d_v, size_t n, double lr,
             double beta1, double beta2, double eps, int32_t step, int32_t first, float lo,
             float hi, hipStream_t s);
int fsk_fill_u32(uint32_t *d_p, size_t n, uint32_t v, hipStream_t s);
/* Reductions write one partial sum per workgroup into d_partials (at most
 * n_partials) and a one-workgroup pass adds their sum, in a fixed order,
 * to the scalar: no atomics on the scalar, reproducible results. */
int fsk_l2_loss(const float *d_img, const float *d_tgt, size_t n, float *d_g, float *d_loss,
                int32_t accumulate, double *d_partials, int32_t n_partials, hipStream_t s);

#ifdef __cplusplus
}
#endif
#endif
