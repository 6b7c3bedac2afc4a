/*
 * fs_kernels.hip -- gfx950 kernels of the futspace renderer.
 *
 * Compiled with -ffp-contract=off and correctly rounded f32 divide/sqrt:
 * every f32 expression below is evaluated in the reference's order
 * (fut/voxel_renderer.fut, fut/render_functions.fut, fut/effects.fut and
 * the matte argb operations they call), so frames are bit-exact with the
 * `futhark c` build of the reference on x86-64.
 *
 * Hot path (k_render): one workgroup owns a stripe of TC adjacent frame
 * columns for the whole depth range.  Lane (slice group g, column c) walks
 * KR consecutive slices per chunk; a prefix-min across slice groups gives
 * each lane the y-buffer value in front of its slices, so a lane knows
 * which of its samples rise strictly above everything nearer (the
 * reference's `scan occlude` + `scatter`, fut/voxel_renderer.fut:231,244).
 * Only those samples get the expensive bilinear argb colour.  The stripe
 * is assembled in LDS, filled top-down (`scan fill_vline` + sky,
 * :246-249) and written once, row-major.
 */
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <stdlib.h>

#include <algorithm>
#include <atomic>
#include <cmath>
#include <cstring>
#include <mutex>
#include <type_traits>

#include "fs_internal.h"

namespace {

/* ------------------------------------------------------------------ */
/* Scalar semantics                                                    */
/* ------------------------------------------------------------------ */

/* Texel index from a floor/ceil value.  gfx950's v_cvt_i32_f32 saturates
 * (NaN -> 0); indices only have to be exact where |v| < 2^24, because at
 * larger magnitudes every f32 is an integer and both bilinear weights are
 * zero, so the texel value is multiplied by 0. */
__device__ __forceinline__ int32_t idx_of(float v)
{
    return (int32_t)fminf(fmaxf(v, -1073741824.0f), 1073741824.0f);
}

/* i32.f32 as `futhark c` runs it on x86-64 (cvttss2si): NaN and values
 * outside [-2^31, 2^31) give INT_MIN. */
__device__ __forceinline__ int32_t i32_f32_x86(float v)
{
    bool ok = (v >= -2147483648.0f) && (v < 2147483648.0f);
    return ok ? (int32_t)fminf(fmaxf(v, -2147483648.0f), 2147483520.0f) : INT32_MIN;
}

/* i32.max 0 (i32.f32 rel), fut/voxel_renderer.fut:225, x86 semantics:
 * NaN, >= 2^31 and < -2^31 all give 0. */
__device__ __forceinline__ int32_t screen_row(float rel)
{
    return (rel < 2147483648.0f) ? max(0, (int32_t)fmaxf(rel, -1.0f)) : 0;
}

/* min(H, screen_row(rel)) with H = rows as float: truncating the median of
 * (rel, 0, H) equals clamping the truncation for every rel below 2^31;
 * rel >= 2^31 and NaN take the select's 0. */
__device__ __forceinline__ int32_t screen_row_clamped(float rel, float Hf)
{
    int32_t r = (int32_t)__builtin_amdgcn_fmed3f(rel, 0.0f, Hf);
    return (rel < 2147483648.0f) ? r : 0;
}

/* Futhark's signed `%` (floor-mod). */
__device__ __forceinline__ int32_t fmod_i32(int32_t a, int32_t m)
{
    int32_t r = a % m;
    return (r != 0 && ((r < 0) != (m < 0))) ? r + m : r;
}

template <bool POW2>
__device__ __forceinline__ int32_t wrap(int32_t v, int32_t m)
{
    return POW2 ? (v & (m - 1)) : fmod_i32(v, m);
}

/* Floor-mod of an integral f32 v, |v| < 2^21, by a side m <= 2^20 that is not
 * a power of two, with rm a little below 1 / m (fsk_wrap_recip).  v * rm is
 * then below the quotient, or at it, by less than 2^-21.4 of it, which is less
 * than 1 / m: its floor is the quotient's floor, or one less where m divides
 * v.  The remainder, exact in one FMA, is in [0, 2m), and the smaller of it
 * and it less m (as unsigned) is the result.  Six vector instructions where
 * the integer modulo takes some thirty; device self-test 8 compares the two. */
__device__ __forceinline__ int32_t wrap_tame(float v, int32_t m, float rm)
{
    const float q = floorf(v * rm);
    const uint32_t r = (uint32_t)(int32_t)__builtin_fmaf(-q, (float)m, v);
    return (int32_t)min(r, r - (uint32_t)m);
}

/* ------------------------------------------------------------------ */
/* matte argb, as restated for the reference (Gloss mixColors)         */
/* ------------------------------------------------------------------ */

/* f32.u32 b / 255 for a byte b, correctly rounded: one FMA correction
 * of the reciprocal product (exhaustively equal to the division for all
 * 256 bytes; checked on the device by the test suite). */
__device__ __forceinline__ float unit8(uint32_t b)
{
    const float inv = 1.0f / 255.0f;
    float fb = (float)b;
    float q0 = fb * inv;
    float r = __builtin_fmaf(-q0, 255.0f, fb);
    return __builtin_fmaf(r, inv, q0);
}

/* u32.f32 (clamp_channel v * 255); clamp passes NaN, u32 of NaN is 0. */
__device__ __forceinline__ uint32_t chan_u8(float v)
{
    /* the clamp is a median of three; a NaN v is caught by the final
     * select, so whatever the median does with it is discarded */
    float c = __builtin_amdgcn_fmed3f(v, 0.0f, 1.0f);
    uint32_t u = (uint32_t)(c * 255.0f);
    return (v == v) ? u : 0u;
}

/* Correctly rounded sqrt for t in [0, 1] or NaN: v_sqrt_f32 is within one
 * ulp, and the two FMA residuals pick the rounded root among its
 * neighbours.  Inputs are never negative or infinite here, which drops the
 * general sequence's special cases; inputs below 2^-96 (only reachable
 * within ~2^-90 of the map origin) take the general sqrt on a wave-uniform
 * branch, which skips it everywhere else.  The device self-test compares
 * this with the general sqrt on every f32 in [0, 1]. */
__device__ __forceinline__ float sqrt_unit(float t)
{
    float s = __builtin_amdgcn_sqrtf(t);
    float sm = __int_as_float(__float_as_int(s) - 1);
    float sp = __int_as_float(__float_as_int(s) + 1);
    float rm = __builtin_fmaf(-sm, s, t);
    float rp = __builtin_fmaf(-sp, s, t);
    s = (rm <= 0.0f) ? sm : s;
    s = (rp > 0.0f) ? sp : s;
    bool tiny = (t < 0x1p-96f) && (t > 0.0f);
    if (__ballot(tiny)) {
        /* the empty asm keeps the general sqrt inside the branch */
        float tt = t;
        asm volatile("" : "+v"(tt));
        if (tiny)
            s = __builtin_sqrtf(tt);
    }
    return s;
}

/* Correctly rounded sqrt of t >= 0 (or NaN): sqrt_unit's neighbour
 * correction holds for every non-negative f32; device self-test 7 checks
 * it against the correctly rounded sqrt on all of them. */
__device__ __forceinline__ float sqrt_rn(float t)
{
    return sqrt_unit(t);
}

__device__ __forceinline__ uint32_t from_rgba(float r, float g, float b, float a)
{
    return (chan_u8(a) << 24) | (chan_u8(r) << 16) | (chan_u8(g) << 8) | chan_u8(b);
}

/* argb.mix m1 c1 m2 c2.  When m1 + m2 rounds to exactly 1 the
 * normalisation divides by 1, which is exact, so the quotient is the
 * dividend; that skips three correctly rounded divisions on the common
 * bilinear path (weights (c - x) and (x - f) sum to 1 for |x| >= 1). */
__device__ __forceinline__ uint32_t argb_mix(float m1, uint32_t c1, float m2, uint32_t c2)
{
    float r1 = unit8((c1 >> 16) & 255u), g1 = unit8((c1 >> 8) & 255u);
    float b1 = unit8(c1 & 255u), a1 = unit8(c1 >> 24);
    float r2 = unit8((c2 >> 16) & 255u), g2 = unit8((c2 >> 8) & 255u);
    float b2 = unit8(c2 & 255u), a2 = unit8(c2 >> 24);
    float m12 = m1 + m2;
    float m1n = m1, m2n = m2;
    float al = (m1 * a1) + (m2 * a2);
    if (m12 != 1.0f) {
        m1n = m1 / m12;
        m2n = m2 / m12;
        al = al / m12;
    }
    float r = __builtin_sqrtf((m1n * (r1 * r1)) + (m2n * (r2 * r2)));
    float g = __builtin_sqrtf((m1n * (g1 * g1)) + (m2n * (g2 * g2)));
    float b = __builtin_sqrtf((m1n * (b1 * b1)) + (m2n * (b2 * b2)));
    return from_rgba(r, g, b, al);
}

/* ------------------------------------------------------------------ */
/* Samplers                                                            */
/* ------------------------------------------------------------------ */

/* png_height_filtered, fut/render_functions.fut:67-77, from the height
 * quad at (floor y, floor x). */
/* The maps are device memory.  Their gathers read through pointers of the
 * global address space: a map pointer the kernel read from memory (a
 * batch's view records) is generic, and loads through it would be flat
 * loads, which also count against the LDS wait counter, so every LDS wait
 * of the tile would wait for the gathers in flight too. */
#define FS_GLOBAL __attribute__((address_space(1)))
typedef uint32_t fs_u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t fs_u32x4 __attribute__((ext_vector_type(4)));

template <int HBITS, bool HP2, int TAME = 0>
__device__ __forceinline__ uint2 height_quad(const fsk_map &m, float x, float y)
{
    /* TAME: the frame's level (fsk_tame_level).  From FSK_TAME on |x| and |y|
     * are below 2^22, so that floor converts exactly without a clamp; at
     * FSK_TAME_MOD they are below 2^21 and wrap by reciprocals. */
    int32_t ix, iy;
    if (TAME == FSK_TAME_MOD && !HP2) {
        ix = wrap_tame(floorf(x), m.hcols, m.rhcols);
        iy = wrap_tame(floorf(y), m.hrows, m.rhrows);
    } else {
        ix = wrap<HP2>(TAME ? (int32_t)floorf(x) : idx_of(floorf(x)), m.hcols);
        iy = wrap<HP2>(TAME ? (int32_t)floorf(y) : idx_of(floorf(y)), m.hrows);
    }
    /* maps are at most 2^28 texels (host-checked), so 32-bit offsets; the
     * wrapped index is always inside the map, whatever x and y are */
    uint32_t t = HP2 ? ((uint32_t)iy << __builtin_ctz((uint32_t)m.hcols)) + (uint32_t)ix
                 : TAME == FSK_TAME_MOD ? __umul24((uint32_t)iy, (uint32_t)m.hcols) + (uint32_t)ix
                                        : (uint32_t)iy * (uint32_t)m.hcols + (uint32_t)ix;
    const FS_GLOBAL char *hq = (const FS_GLOBAL char *)m.hq;
    if (HBITS == 8)
        return make_uint2(*(const FS_GLOBAL uint32_t *)(hq + t * 4u), 0u);
    const fs_u32x2 v = *(const FS_GLOBAL fs_u32x2 *)(hq + t * 8u);
    return make_uint2(v.x, v.y);
}

template <int HBITS>
__device__ __forceinline__ float height_interp(uint2 q, float x, float y)
{
    float fx = floorf(x), cx = ceilf(x), fy = floorf(y), cy = ceilf(y);
    float h00, h01, h10, h11;
    if (HBITS == 8) {
        h00 = (float)(q.x & 255u);
        h01 = (float)((q.x >> 8) & 255u);
        h10 = (float)((q.x >> 16) & 255u);
        h11 = (float)(q.x >> 24);
    } else {
        h00 = (float)(q.x & 65535u);
        h01 = (float)(q.x >> 16);
        h10 = (float)(q.y & 65535u);
        h11 = (float)(q.y >> 16);
    }
    float wx0 = cx - x, wx1 = x - fx;
    float x_interpolated1 = (wx0 * h00) + (wx1 * h01);
    float x_interpolated2 = (wx0 * h10) + (wx1 * h11);
    return ((cy - y) * x_interpolated1) + ((y - fy) * x_interpolated2);
}

/* ------------------------------------------------------------------ */
/* Slice parameters: get_zs term (fut/voxel_renderer.fut:34), get_h_line */
/* (:43-60) and inv_z (:217) of slice k (0-based)                      */
/* ------------------------------------------------------------------ */

struct Slice {
    float sx, sy, dx, dy, iz;
};

__device__ __forceinline__ Slice slice_params(const fsk_frame &f, int32_t k)
{
    float i = (float)(k + 1);
    float z = (i / 2.0f) * ((2.0f * f.z0) + ((i - 1.0f) * f.d));
    float left_x = f.Lx * z, left_y = f.Ly * z;
    float right_x = f.Rx * z, right_y = f.Ry * z;
    Slice s;
    s.dx = (right_x - left_x) / f.fw;
    s.dy = (right_y - left_y) / f.fw;
    s.sx = left_x + f.cam_x;
    s.sy = left_y + f.cam_y;
    s.iz = (1.0f / z) * f.scale;
    return s;
}

/* RN(1 / z) for z > 0 whose reciprocal is a normal number: the hardware
 * reciprocal (within an ulp) and one Newton step with FMA.  Device self-test
 * 5 compares it with the correctly rounded division for every such z. */
__device__ __forceinline__ float rcp_rn(float z)
{
    float y = __builtin_amdgcn_rcpf(z);
    float e = __builtin_fmaf(-z, y, 1.0f);
    return __builtin_fmaf(e, y, y);
}

/* RN(a / b) from rb = RN(1 / b), for finite a and b >= 1 (Markstein's
 * correction: q = RN(a * rb) is within an ulp of a / b, the residual
 * a - q * b is exact in one FMA, and q + residual * rb rounds to the
 * nearest quotient).  The residual is not exact for quotients near the
 * subnormal range, and the signs of zero differ, so quotients below 2^-100
 * in magnitude take the division itself, on a wave-uniform branch (a plain
 * select would have every lane compute it).  Device self-test 6 compares it
 * with the correctly rounded division for every finite f32 a at a set of
 * frame widths b. */
__device__ __forceinline__ float div_rn(float a, float b, float rb)
{
    float q = a * rb;
    float r = __builtin_fmaf(-q, b, a);
    q = __builtin_fmaf(r, rb, q);
    const bool small = !(fabsf(q) >= 0x1p-100f);
    if (__ballot(small)) {
        /* the empty asm keeps the compiler from hoisting the division out
         * of the branch (it may otherwise evaluate it on every wave) */
        float aa = a;
        asm volatile("" : "+v"(aa));
        if (small)
            q = aa / b;
    }
    return q;
}

/* slice_params of a tame frame (z >= z0 > 0, finite scalars) with the two
 * divisions by the frame width and the reciprocal of z taken by rcp_rn and
 * div_rn (f.rfw = RN(1 / fw)).  Bit-identical to slice_params there. */
__device__ __forceinline__ Slice slice_params_tame(const fsk_frame &f, int32_t k)
{
    const float rfw = f.rfw;
    float i = (float)(k + 1);
    float z = (i / 2.0f) * ((2.0f * f.z0) + ((i - 1.0f) * f.d));
    float left_x = f.Lx * z, left_y = f.Ly * z;
    float right_x = f.Rx * z, right_y = f.Ry * z;
    Slice s;
    s.dx = div_rn(right_x - left_x, f.fw, rfw);
    s.dy = div_rn(right_y - left_y, f.fw, rfw);
    s.sx = left_x + f.cam_x;
    s.sy = left_y + f.cam_y;
    s.iz = rcp_rn(z) * f.scale;
    return s;
}

/* ------------------------------------------------------------------ */
/* The render kernel                                                   */
/* ------------------------------------------------------------------ */

/* Inclusive prefix sum over the 64 lanes of a wave, in registers: DPP
 * row shifts by 1, 2, 4 and 8 scan each row of 16 lanes (lanes shifted in
 * from outside the row read 0), then the last lane of row 0 is added to
 * rows 1 and 3 (row_bcast:15; rows 0 and 2 add the old value 0) and lane
 * 31 to rows 2 and 3 (row_bcast:31). */
__device__ __forceinline__ uint32_t wave_incl_sum(uint32_t x)
{
    x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x111, 0xf, 0xf, true);  /* row_shr:1 */
    x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x112, 0xf, 0xf, true);  /* row_shr:2 */
    x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x114, 0xf, 0xf, true);  /* row_shr:4 */
    x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x118, 0xf, 0xf, true);  /* row_shr:8 */
    x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x142, 0xa, 0xf, false); /* row_bcast:15 */
    x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x143, 0xc, 0xf, false); /* row_bcast:31 */
    return x;
}

/* Per-column minima over the slice groups of a wave of an 8-column tile
 * (lane = 8 * group + column, rows at most H): excl = the minimum over
 * the groups before the lane's (H for the first group), total = over all
 * eight.  In registers: DPP folds the two groups of each 16-lane row
 * (row_shr:8, then row_ror:8 to give the row's minimum to all its lanes),
 * and the permlane swaps hand every row the minima of all four rows with
 * the columns aligned (permlane32_swap exchanges rows 2-3 of its first
 * operand with rows 0-1 of its second; permlane16_swap the odd rows of the
 * first with the even rows of the second). */
__device__ __forceinline__ void wave_column_scan8(int32_t x, int32_t H, int32_t lane,
                                                  int32_t &excl, int32_t &total)
{
    /* the even group of the row in the odd group's lanes (row_shr:8; the
     * even group's lanes keep H) */
    const int32_t e = __builtin_amdgcn_update_dpp(H, x, 0x118, 0xf, 0xf, false);
    const int32_t i = min(x, e);
    const int32_t t = min(i, __builtin_amdgcn_update_dpp(H, i, 0x128, 0xf, 0xf, false));
    const auto y = __builtin_amdgcn_permlane32_swap(t, t, false, false);   /* T0 T1 T0 T1 | T2 T3 T2 T3 */
    const auto a = __builtin_amdgcn_permlane16_swap(y[0], y[0], false, false);   /* T0 | T1 */
    const auto b = __builtin_amdgcn_permlane16_swap(y[1], y[1], false, false);   /* T2 | T3 */
    const int32_t t0 = (int32_t)a[0], m01 = min(t0, (int32_t)a[1]);
    const int32_t m012 = min(m01, (int32_t)b[0]);
    total = min(m012, (int32_t)b[1]);
    const int32_t row = lane >> 4;
    const int32_t before = row == 0 ? H : row == 1 ? t0 : row == 2 ? m01 : m012;
    excl = (lane & 8) ? min(before, e) : before;
}

constexpr int kMaxWaves = 16;                    /* 1024-thread workgroups */
constexpr int kChunk = 2048;                     /* slices per chunk, at most */

/* Slice-table slots for chunks of up to `chunk` slices: the table is slot
 * major, slot j * SG + g holding slice g * kr + j of the chunk (slice group
 * g, its j-th slice), so that the slice groups of a wave read adjacent
 * records at an offset fixed per j.  Chunks are whole multiples of SG * 4
 * slots (the host rounds them), which covers the gather groups' reads past
 * kr. */
__host__ __device__ constexpr int tab_stride(int chunk)
{
    return chunk;
}
/* A queued visible sample: its slice group g, its slice j within the
 * group, its column c in the tile and its projected row, packed as
 * g << 22 | j << 17 | c << 13 | row (g < 256, j < 32, c < 16, row < 8192).
 * The long-span list packs c << 26 | first row << 13 | end row. */
constexpr uint32_t kQRowBits = 13;
constexpr uint32_t kQRowMask = (1u << kQRowBits) - 1u;
constexpr uint32_t kQColShift = 13, kQSliceShift = 17, kQGroupShift = 22;
constexpr uint32_t kQLaneMask = (0xFFu << kQGroupShift) | (15u << kQColShift);  /* g and c */
/* Frames up to kMaxRows rows are rendered whole columns at a time: the row
 * fields allow 8191, and a 4-column tile of that height still fits in LDS.
 * Taller ones, up to kMaxFrameRows, are rendered in bands of rows. */
constexpr int kMaxRows = 7680;
constexpr int kMaxFrameRows = 1 << 22;
constexpr int kChunkAlign = 4;                   /* chunks are multiples of SG * kChunkAlign */

/* blockIdx -> column tile.  Workgroups are dispatched round-robin over
 * the 8 XCDs (workgroup i runs on XCD i mod 8), so tile ranges are dealt
 * out per XCD: neighbouring stripes share one L2 for their height texels
 * and for merging their partial-line row writes. */
__device__ __forceinline__ int32_t xcd_tile(int32_t b, int32_t n)
{
    const int32_t X = 8;
    int32_t q = n / X, r = n % X, x = b % X, s = b / X;
    return (x < r) ? x * (q + 1) + s : r * (q + 1) + (x - r) * q + s;
}

struct RenderArgs {
    fsk_map m;
    fsk_frame f;
    uint32_t *out;
    int64_t pitch;
    int32_t ntiles;
    int32_t chunk_max;     /* slices per chunk, at most kChunk */
    int32_t band_rows;     /* banded renders: rows per workgroup */
    /* slice mode: workgroups ntiles .. ntiles + nzero - 1 clear zero[zero_n4]
     * (the fused step's gradient) on CUs the tiles leave idle */
    float4 *zero;
    size_t zero_n4;
    int32_t nzero;
};

/* Fewest idle workgroup slots worth a gradient clear inside the slice
 * render: with fewer, each would clear too much of the buffer and
 * outlast the tiles. */
constexpr int32_t kMinZeroBlocks = 64;

#ifndef FS_SQ_LUT
#define FS_SQ_LUT 1
#endif

/* RN(RN(b/255)^2) for every byte: the squared channel of to_rgba. */
__device__ __forceinline__ void fill_square_lut(float *lut, int32_t tid)
{
    if (tid < 256) {
        float u = unit8((uint32_t)tid);
        lut[tid] = u * u;
    }
}

__device__ __forceinline__ float sq8(const float *lut, uint32_t b)
{
#if FS_SQ_LUT
    return lut[b];
#else
    (void)lut;
    float u = unit8(b);
    return u * u;
#endif
}

/* One channel of argb.mix with the weights already normalised:
 * u32.f32(clamp(sqrt(m1' * c1^2 + m2' * c2^2)) * 255). */
__device__ __forceinline__ uint32_t mix_channel(float m1n, float s1, float m2n, float s2)
{
    return chan_u8(sqrt_unit((m1n * s1) + (m2n * s2)));
}

/* The common case of png_color_filtered: |x|, |y| >= 1 and four opaque
 * texels.  Then the weights (c - x), (x - f) are exact and sum to exactly
 * 1 (or are both 0 at an integer coordinate), so every normalisation is
 * the identity, every sqrt argument lies in {0} U [2^-39, 1] (weights are
 * multiples of 2^-23, squares at least 255^-2), the clamp never acts and
 * no NaN arises; alpha is 255 unless a weight sum is 0. */
__device__ __forceinline__ uint32_t mix_channel_exact(float m1, float s1, float m2, float s2)
{
    float t = (m1 * s1) + (m2 * s2);
    float s = __builtin_amdgcn_sqrtf(t);
    float sm = __int_as_float(__float_as_int(s) - 1);
    float sp = __int_as_float(__float_as_int(s) + 1);
    float rm = __builtin_fmaf(-sm, s, t);
    float rp = __builtin_fmaf(-sp, s, t);
    s = (rm <= 0.0f) ? sm : s;
    s = (rp > 0.0f) ? sp : s;
    return (uint32_t)(s * 255.0f);
}

/* The byte quantisation of a mixed channel, u32.f32(sqrt(t) * 255), by
 * table: the map t -> byte is non-decreasing on [0, 1], so the float bits
 * of t (clamped below at kQLo, where the byte is still 0) fall into one of
 * kQBuckets buckets of 2^16 consecutive bit patterns, and no bucket holds
 * more than one step of the byte.  Entry i of the table, with
 * u = max(bits(t) - kQLo, 0) in bucket i = u >> 16, is
 *     (base << 17) + 2^17 - step - (i << 16)   (mod 2^32)
 * (base: the byte at the bucket's first pattern; step: the offset of the
 * pattern where the byte becomes base + 1, or 2^16 if none), so that
 * (entry + u) >> 17 is the byte for every t of the bucket.  The table is
 * built on the host with the C library's correctly rounded sqrtf and is
 * checked against the sqrt sequence for every f32 in [0, 1] by the device
 * self-test. */
/* Scratch of the allocation-free fused step (fsx_render_f32_l2_step_noalloc):
 * per-workgroup partial sums, FSK_PARTIALS doubles per device, held until
 * the process ends.  Host code reaches it only through the address
 * hipGetSymbolAddress returns for the current device (fsk_scratch). */
static __device__ __align__(256) double scratch[FSK_PARTIALS];

constexpr uint32_t kQLo = 0x37810000u;           /* below sqrt(t) * 255 >= 1 */
constexpr int kQBuckets = 2048;                  /* (bits(1.0f) - kQLo) >> 16 = 2047 */
__device__ uint32_t g_qtab[kQBuckets];

/* (qt entry + u) for t = m1 * s1 + m2 * s2: the channel byte sits in bits
 * 17..24.  Needs t in [0, 1]. */
__device__ __forceinline__ uint32_t mix_q(const uint32_t *qt, float m1, float s1, float m2,
                                          float s2)
{
    float t = (m1 * s1) + (m2 * s2);
    uint32_t u = __builtin_elementwise_sub_sat(__float_as_uint(t), kQLo);
    return qt[u >> 16] + u;
}

/* color_fast with the table quantisation (qt: the bucket table in LDS). */
__device__ __forceinline__ uint32_t color_fast_q(uint4 q, const float *sq, const uint32_t *qt,
                                                 float wx0, float wx1, float wy0, float wy1)
{
    uint32_t out = 0;
#pragma unroll
    for (int sh = 16; sh >= 0; sh -= 8) {
        uint32_t X1 = mix_q(qt, wx0, sq8(sq, (q.x >> sh) & 255u), wx1,
                            sq8(sq, (q.y >> sh) & 255u)) >> 17;
        uint32_t X2 = mix_q(qt, wx0, sq8(sq, (q.z >> sh) & 255u), wx1,
                            sq8(sq, (q.w >> sh) & 255u)) >> 17;
        out |= (mix_q(qt, wy0, sq8(sq, X1), wy1, sq8(sq, X2)) >> 17) << sh;
    }
    bool opaque_sum = (wx0 + wx1 != 0.0f) && (wy0 + wy1 != 0.0f);
    return out | (opaque_sum ? 0xFF000000u : 0u);
}

__device__ __forceinline__ uint32_t color_fast(uint4 q, const float *sq, float wx0, float wx1,
                                               float wy0, float wy1)
{
    uint32_t out = 0;
#pragma unroll
    for (int sh = 16; sh >= 0; sh -= 8) {
        uint32_t X1 = mix_channel_exact(wx0, sq8(sq, (q.x >> sh) & 255u), wx1,
                                        sq8(sq, (q.y >> sh) & 255u));
        uint32_t X2 = mix_channel_exact(wx0, sq8(sq, (q.z >> sh) & 255u), wx1,
                                        sq8(sq, (q.w >> sh) & 255u));
        out |= mix_channel_exact(wy0, sq8(sq, X1), wy1, sq8(sq, X2)) << sh;
    }
    bool opaque_sum = (wx0 + wx1 != 0.0f) && (wy0 + wy1 != 0.0f);
    return out | (opaque_sum ? 0xFF000000u : 0u);
}

/* png_color_filtered (fut/render_functions.fut:95-105) evaluated channel
 * by channel: argb.mix is separable per channel once its weights are
 * normalised, so the two row mixes feed the column mix as bytes.
 *
 * argb.mix divides the weights by their sum m12.  A sum of exactly 1
 * makes the divisions exact no-ops; a sum of 0 (integer coordinate) makes
 * the reference's channels 0/0 = NaN, which quantise to byte 0 exactly as
 * the undivided zero weights do.  Bilinear weights sum to 0 or 1 whenever
 * |x|, |y| >= 1, so the divisions run only on waves where some lane has
 * another sum (a coordinate within 1 of the map origin); such waves, and
 * waves with translucent texels, take the general path below. */
template <bool CP2>
__device__ __forceinline__ uint4 color_quad(const fsk_map &m, float x, float y,
                                            int32_t tame = 0)
{
    int32_t ix, iy;
    if (!CP2 && tame >= FSK_TAME_MOD) {
        ix = wrap_tame(floorf(x), m.ccols, m.rccols);
        iy = wrap_tame(floorf(y), m.crows, m.rcrows);
    } else {
        ix = wrap<CP2>(idx_of(floorf(x)), m.ccols);
        iy = wrap<CP2>(idx_of(floorf(y)), m.crows);
    }
    /* colour maps have at most 65536^2 texels (host-checked), so the quad
     * index fits 32 bits; the byte offset is formed in 64 */
    uint32_t t = CP2 ? ((uint32_t)iy << __builtin_ctz((uint32_t)m.ccols)) + (uint32_t)ix
                     : (uint32_t)iy * (uint32_t)m.ccols + (uint32_t)ix;
    const fs_u32x4 v = ((const FS_GLOBAL fs_u32x4 *)m.cq)[t];
    return make_uint4(v.x, v.y, v.z, v.w);
}

/* The colour of a sample at (x, y) from its texel quad q; with qt (the
 * quantisation table in LDS) the fast path quantises by table. */
template <bool QT = false>
__device__ __forceinline__ uint32_t color_of_quad(uint4 q, const float *sq, float x, float y,
                                                  const uint32_t *qt = nullptr)
{
    float fx = floorf(x), cx = ceilf(x), fy = floorf(y), cy = ceilf(y);
    float wx0 = cx - x, wx1 = x - fx, wy0 = cy - y, wy1 = y - fy;
    bool easy = (fabsf(x) >= 1.0f) && (fabsf(y) >= 1.0f) &&
                (((q.x & q.y & q.z & q.w) >> 24) == 255u);
    if (__ballot(!easy) == 0)
        return QT ? color_fast_q(q, sq, qt, wx0, wx1, wy0, wy1)
                  : color_fast(q, sq, wx0, wx1, wy0, wy1);
    float mx = wx0 + wx1, my = wy0 + wy1;
    bool odd = !((mx == 1.0f || mx == 0.0f) && (my == 1.0f || my == 0.0f));
    float nx0 = wx0, nx1 = wx1, ny0 = wy0, ny1 = wy1;
    if (__ballot(odd)) {
        if (odd) {
            nx0 = wx0 / mx;
            nx1 = wx1 / mx;
            ny0 = wy0 / my;
            ny1 = wy1 / my;
        }
    }
    uint32_t out = 0;
#pragma unroll
    for (int sh = 16; sh >= 0; sh -= 8) {
        uint32_t X1 = mix_channel(nx0, sq8(sq, (q.x >> sh) & 255u), nx1, sq8(sq, (q.y >> sh) & 255u));
        uint32_t X2 = mix_channel(nx0, sq8(sq, (q.z >> sh) & 255u), nx1, sq8(sq, (q.w >> sh) & 255u));
        out |= mix_channel(ny0, sq8(sq, X1), ny1, sq8(sq, X2)) << sh;
    }
    /* alpha: (m1*a1 + m2*a2) / m12, mixed linearly */
    float ax1 = (wx0 * unit8(q.x >> 24)) + (wx1 * unit8(q.y >> 24));
    float ax2 = (wx0 * unit8(q.z >> 24)) + (wx1 * unit8(q.w >> 24));
    if (__ballot(odd)) {
        if (odd) {
            ax1 = ax1 / mx;
            ax2 = ax2 / mx;
        }
    }
    float ay = (wy0 * unit8(chan_u8(ax1))) + (wy1 * unit8(chan_u8(ax2)));
    if (__ballot(odd)) {
        if (odd)
            ay = ay / my;
    }
    return out | (chan_u8(ay) << 24);
}

constexpr int kShortSpan = 40;   /* span rows a lane paints itself */
constexpr int kGather = 4;       /* height gathers a lane keeps in flight */
constexpr int kColourBatch = 1;  /* visible samples a lane colours per pass */

/* Dynamic LDS of a tile render of tc columns by nt threads: slice table
 * (float4 + inv_z per slot), the tc x rows colour stripe, the
 * visible-sample queue (at most min(rows, chunk) samples per column and
 * chunk), the y-buffer in front of each lane's slices (u16 per thread) and
 * the long-span list. */
inline size_t render_lds_bytes(int tc, int nt, int32_t rows, int32_t chunk)
{
    size_t hp = (size_t)((rows + 3) & ~3);
    size_t q = (size_t)tc * (size_t)(rows < chunk ? rows : chunk);
    size_t longs = (size_t)tc * (size_t)(rows / kShortSpan + 1);
    return sizeof(float) * 5 * (size_t)tab_stride(chunk) +
           sizeof(uint32_t) * (hp * tc + q + (size_t)nt / 2 + 2 * longs);
}

/* One workgroup renders a stripe of TC adjacent columns over all slices,
 * chunk by chunk:
 *   0. the chunk's slice table (position, step, inv_z) into LDS;
 *   1. lane (slice group g, column c) projects its kr consecutive slices;
 *   2. prefix-min over slice groups (wave scan, then each lane takes the
 *      minimum of the earlier waves' totals and the chunk's carry-in)
 *      gives the y-buffer in front of each lane's slices;
 *   3. samples strictly above it are visible (scan occlude + scatter,
 *      fut/voxel_renderer.fut:231, :244): they are queued with the bottom
 *      of their span;
 *   4. each queued sample gets its bilinear argb colour and paints its span
 *      down to the next visible row below (the reference's top-down
 *      `scan fill_vline`, :246-249, seen from the sample's side).
 * Finally the stripe is written row by row with 0 replaced by the sky.  A
 * sample whose colour is 0 is transparent for fill_vline; if one occurs the
 * stripe is instead filled with a top-down scan over all rows. */
/* Workgroup-shared scalars of one tile render. */
template <int TC>
struct TileShared {
    float sq[256];                 /* squares table, filled once per workgroup */
    uint32_t qt[kQBuckets];        /* byte quantisation table (g_qtab) */
    int32_t wtot[kMaxWaves][TC];   /* wave totals of the prefix-min */
    int32_t wpre[kMaxWaves][TC];   /* wave prefixes of the transparent fill */
    int32_t carry[TC];
    uint32_t qn, nlong, transparent;
};

/* The colour tables of a tile workgroup: squares and the byte
 * quantisation table, copied from g_qtab in two halves -- load() issues
 * this thread's loads, store() writes them to LDS -- so that the loads'
 * latency passes under other work of the tile's first phase. */
template <int TC, int NT>
struct TileTables {
    static_assert(kQBuckets % NT == 0, "table split");
    uint32_t qv[kQBuckets / NT];
    __device__ __forceinline__ void load(int32_t tid)
    {
#pragma unroll
        for (int k = 0; k < kQBuckets / NT; k++)
            qv[k] = g_qtab[tid + k * NT];
    }
    __device__ __forceinline__ void store(TileShared<TC> &sh, int32_t tid) const
    {
        fill_square_lut(sh.sq, tid);
#pragma unroll
        for (int k = 0; k < kQBuckets / NT; k++)
            sh.qt[tid + k * NT] = qv[k];
    }
};

/* Nothing to do before a tile's rows are written. */
struct NoHook {
    __device__ __forceinline__ void operator()() const {}
};

/* No colour tables (tile modes without the argb colour path). */
struct NoTables {
    template <int TC>
    __device__ __forceinline__ void store(TileShared<TC> &, int32_t) const {}
};

/* What a tile writes per pixel: the u32 colour (the reference frame) or,
 * for the differentiable renderer, the index of the depth slice whose
 * sample shows there (-1 for sky).  The slice-index mode keeps the same
 * visibility and fill rules; a sample is transparent there iff its map
 * coordinate is integral in x or y, which is where argb.mix's weight sum
 * vanishes. */
enum { kOutColour = 0, kOutSlice = 1, kOutNearest = 2 };

/* kOutNearest is the stateless program of tests/futspace.fut:47-145: the
 * map is plain i32 colours (m.cq) and unmasked i32 heights (m.hq), sampled
 * at the truncated coordinate (floor-mod wrapped), and the column starts
 * as sky with sky as the `empty` colour of its fill (:110-121) -- colour 0
 * is an ordinary colour there.  The stripe holds colour ^ sky, so that its
 * 0 (unpainted) is the sky and a sky-coloured sample is the transparent
 * one. */
template <int MODE>
__device__ __forceinline__ uint32_t tile_value(uint32_t v, uint32_t sky)
{
    if (MODE == kOutColour)
        return v ? v : sky;
    if (MODE == kOutNearest)
        return v ^ sky;
    return v ? v - 1u : 0xFFFFFFFFu;
}

/* tile_value of a cell that is either painted with a non-zero value (v) or,
 * above its column's final y-buffer, unpainted (sky). */
template <int MODE>
__device__ __forceinline__ uint32_t painted_value(uint32_t v, bool sky_cell, uint32_t sky)
{
    if (MODE == kOutColour)
        return sky_cell ? sky : v;
    if (MODE == kOutNearest)
        return sky_cell ? sky : v ^ sky;
    return sky_cell ? 0xFFFFFFFFu : v - 1u;
}

/* Texel index of the stateless program's sample at (x, y): i32.f32 of
 * each coordinate (x86 truncation), floor-mod by the map size.  TAME as in
 * height_quad. */
template <bool P2, int TAME = 0>
__device__ __forceinline__ uint32_t nearest_index(const fsk_map &m, float x, float y)
{
    if (TAME && P2)
        return (uint32_t)wrap<P2>((int32_t)y, m.hrows) * (uint32_t)m.hcols +
               (uint32_t)wrap<P2>((int32_t)x, m.hcols);
    if (TAME == FSK_TAME_MOD)
        return __umul24((uint32_t)wrap_tame(truncf(y), m.hrows, m.rhrows), (uint32_t)m.hcols) +
               (uint32_t)wrap_tame(truncf(x), m.hcols, m.rhcols);
    int32_t ix = wrap<P2>(i32_f32_x86(x), m.hcols);
    int32_t iy = wrap<P2>(i32_f32_x86(y), m.hrows);
    return (uint32_t)iy * (uint32_t)m.hcols + (uint32_t)ix;
}

/* What the fill shows at row `row0` of a column whose nearest sample at or
 * above that row is transparent: the first opaque one beyond it, as a stripe
 * value (0: none, sky).  The visible samples are the strict running minima
 * of the projected rows over the whole depth range; a wave projects 64
 * slices at a time.  Every lane of the wave must call it. */
template <int HBITS, bool HP2, bool CP2, int MODE>
__device__ uint32_t column_above(const fsk_map &m, const fsk_frame &f, int32_t col, int32_t row0,
                                 const float *sq)
{
    const int32_t lane = threadIdx.x & 63;
    const float Hf = (float)f.rows, fcol = (float)col;
    int32_t run = f.rows;
    for (int32_t base = 0; base < f.n && run > 0; base += 64) {
        const int32_t k = base + lane;
        const Slice sl = slice_params(f, min(k, f.n - 1));
        const float x = sl.sx + (fcol * sl.dx);
        const float y = sl.sy + (fcol * sl.dy);
        float hgt;
        if (MODE == kOutNearest)
            hgt = (float)((const int32_t *)m.hq)[nearest_index<HP2>(m, x, y)];
        else
            hgt = height_interp<HBITS>(height_quad<HBITS, HP2>(m, x, y), x, y);
        const float rel = ((f.cam_h - hgt) * sl.iz) + f.horizon;
        const int32_t r = k < f.n ? screen_row_clamped(rel, Hf) : f.rows;
        int32_t v = r;
#pragma unroll
        for (int off = 1; off < 64; off <<= 1) {
            const int32_t o = __shfl_up(v, off);
            if (lane >= off)
                v = min(v, o);
        }
        const int32_t before = __shfl_up(v, 1);
        const bool visible = r < (lane == 0 ? run : min(run, before));
        uint32_t c = 0u;
        if (visible && r <= row0) {
            if (MODE == kOutColour)
                c = color_of_quad(color_quad<CP2>(m, x, y), sq, x, y);
            else if (MODE == kOutNearest)
                c = ((const uint32_t *)m.cq)[nearest_index<HP2>(m, x, y)] ^ f.sky;
            else
                c = (floorf(x) == ceilf(x) || floorf(y) == ceilf(y)) ? 0u : (uint32_t)(k + 1);
        }
        const uint64_t opaque = __ballot(c != 0u);
        if (opaque)
            return (uint32_t)__builtin_amdgcn_readlane((int)c, __builtin_ctzll(opaque));
        run = min(run, __builtin_amdgcn_readlane(v, 63));
    }
    return 0u;
}

/* chunk_max must be a multiple of NT/TC (the slice groups) and at most
 * CMAX; the LDS layout is sized for it.
 *
 * BAND: the tile covers rows row0 .. row0 + H - 1 of the frame only (out
 * points at row0), H = min(band_rows, f.rows - row0).  Rows are then counted
 * from row0 and clamped to [0, H]: a sample at or below the band is not
 * visible in it, and of those above it only the nearest is, at row 0, from
 * where it covers the band down to the next nearer one -- just what the
 * whole column shows there.  Should that sample be transparent, the rows it
 * covers show the next opaque one above, which column_above finds. */
template <int TC, int NT, int CMAX, int HBITS, bool HP2, bool CP2, int MODE = kOutColour,
          int GATHER = kGather, int CBATCH = kColourBatch, class Tables = NoTables,
          bool BAND = false, class Hook = NoHook>
__device__ __forceinline__ void render_tile(const fsk_map &m, const fsk_frame &f, uint32_t *out,
                                            int64_t pitch, int32_t tile, int32_t chunk_max,
                                            uint32_t *lds, TileShared<TC> &sh,
                                            const Tables &tables = Tables(), int32_t row0 = 0,
                                            int32_t band_rows = 0, Hook &&before_write = Hook())
{
    constexpr int NW = NT / 64;                  /* waves */
    constexpr int SG = NT / TC;                  /* slice groups */
    constexpr int KR = CMAX / SG;                /* slices per lane per chunk, at most */
    static_assert(NW <= kMaxWaves && KR % GATHER == 0 && GATHER % 2 == 0 && KR <= 32 &&
                      SG <= 256 && kChunkAlign % GATHER == 0,
                  "tile shape");
    const int32_t tabs = tab_stride(chunk_max);
    float4 *tl = (float4 *)lds;                                  /* [tabs] */
    float *tz = (float *)(lds + 4 * tabs);                       /* [tabs] */
    const int32_t H = BAND ? min(band_rows, f.rows - row0) : f.rows, n = f.n;
    const int32_t Hp = (H + 3) & ~3;
    uint32_t *stripe = lds + 5 * tabs;                           /* [TC][Hp] */
    const int32_t qcap = TC * min(H, chunk_max);                 /* visible rows differ */
    uint32_t *queue = stripe + (size_t)Hp * TC;                  /* [qcap] */
    uint16_t *lanein = (uint16_t *)(queue + qcap);               /* [NT] y-buffer per lane */
    uint32_t *longs = queue + qcap + NT / 2;                     /* [2][TC*(H/kShortSpan+1)] */

    const int32_t tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int32_t col0 = tile * TC;
    const int32_t c = tid % TC, g = tid / TC;
    const int32_t col = col0 + c;
    const bool colok = col < f.cols;
    const float fcol = (float)col;
    /* the rows' clamp; frame rows are below 2^24, so exact */
    const float topf = BAND ? (float)row0 : 0.0f;
    const float Hf = BAND ? (float)(row0 + H) : (float)H;

    /* The stripe is not cleared: the spans of a column's visible samples
     * tile the rows from its final y-buffer down to H (transparent samples
     * paint 0), and the rows above it are sky, which the write phase tells
     * apart by the y-buffer. */
    if (tid < TC)
        sh.carry[tid] = H;
    if (tid == 0) {
        sh.nlong = 0u;
        sh.transparent = 0u;
    }

    const int32_t nch = (n + chunk_max - 1) / chunk_max;
    const int32_t kr = nch > 0 ? (n + nch * SG - 1) / (nch * SG) : 0;
    const int32_t csz = kr * SG;

    for (int32_t base = 0; base < n; base += csz) {
        const int32_t cn = min(csz, n - base);
        /* phase 0: the chunk's slice records in slot order (slot j*SG + g
         * holds slice g*kr + j; slots past the chunk repeat its last
         * slice).  Each wave computes the slots of its own slice groups --
         * the only ones its projection reads -- so no workgroup barrier
         * separates this phase from the next: a wave starts projecting as
         * soon as its own records are in LDS.  Computing them per tile is
         * cheaper than copying a precomputed per-view table, even in
         * batches. */
        {
            constexpr int GPW = 64 / TC;             /* slice groups per wave */
            const int32_t nj = ((kr + GATHER - 1) / GATHER) * GATHER;
            auto table = [&](auto tame_tag) {
                constexpr bool TAMEP = decltype(tame_tag)::value;
                for (int32_t q = lane; q < nj * GPW; q += 64) {
                    const int32_t gq = wave * GPW + q % GPW, j = q / GPW;
                    const int32_t o = j * SG + gq;
                    const int32_t s = min(gq * kr + j, cn - 1);
                    Slice sl = TAMEP ? slice_params_tame(f, base + s) : slice_params(f, base + s);
                    tl[o] = make_float4(sl.sx, sl.sy, sl.dx, sl.dy);
                    tz[o] = sl.iz;
                }
            };
            if (f.tame)
                table(std::true_type{});
            else
                table(std::false_type{});
        }
        if (tid == 0)
            sh.qn = 0u;
        /* the wave reads back what its own lanes wrote: LDS operations of a
         * wave complete in order; the fence keeps the compiler from moving
         * the reads above the writes */
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");

        /* phase 1: rows are < 2^16, two per register.  Branch-free in
         * groups of GATHER samples: all of a group's height gathers are
         * issued before the first is used.  Samples past the chunk, the
         * slice group or the frame read a defined table slot and an in-map
         * texel; the fix-up below raises them to row H. */
        uint32_t ah[KR / 2];
        int32_t lmin = H;
        const float4 *tlg = tl + g;
        const float *tzg = tz + g;
        auto project = [&](auto tame_tag, auto full_tag) {
            constexpr int TAME = decltype(tame_tag)::value;
            constexpr bool FULL = decltype(full_tag)::value;
#pragma unroll
            for (int j0 = 0; j0 < KR; j0 += GATHER) {
                /* kr is uniform over the workgroup: whole groups past it
                 * are skipped, their rows stay H.  A full chunk (kr == KR)
                 * has no such group, and no branch between the groups, so
                 * the gathers of later groups may be issued early */
                if (!FULL && j0 >= kr) {
#pragma unroll
                    for (int u = 0; u < GATHER; u += 2)
                        ah[(j0 + u) / 2] = (uint32_t)H | ((uint32_t)H << 16);
                    continue;
                }
                float xs[GATHER], ys[GATHER], izs[GATHER];
                uint2 qs[GATHER];
#pragma unroll
                for (int u = 0; u < GATHER; u++) {
                    float4 L = tlg[(j0 + u) * SG];
                    xs[u] = L.x + (fcol * L.z);
                    ys[u] = L.y + (fcol * L.w);
                    izs[u] = tzg[(j0 + u) * SG];
                    if (MODE == kOutNearest)
                        qs[u] = make_uint2(
                            ((const uint32_t *)m.hq)[nearest_index<HP2, TAME>(m, xs[u], ys[u])],
                            0u);
                    else
                        qs[u] = height_quad<HBITS, HP2, TAME>(m, xs[u], ys[u]);
                }
#pragma unroll
                for (int u = 0; u < GATHER; u++) {
                    const int j = j0 + u;
                    float hgt = MODE == kOutNearest ? (float)(int32_t)qs[u].x
                                                    : height_interp<HBITS>(qs[u], xs[u], ys[u]);
                    float rel = ((f.cam_h - hgt) * izs[u]) + f.horizon;
                    /* a tame frame keeps |rel| < 2^30 (the stateless program's
                     * heights are unbounded): the cast of the clamped value
                     * is the whole x86 semantics */
                    constexpr bool ROWS = TAME && MODE != kOutNearest;
                    int32_t r = ROWS || BAND ? (int32_t)__builtin_amdgcn_fmed3f(rel, topf, Hf)
                                             : screen_row_clamped(rel, Hf);
                    if (BAND)
                        r = ROWS || rel < 2147483648.0f ? r - row0 : 0;
                    if (j & 1)
                        ah[j / 2] |= (uint32_t)r << 16;
                    else
                        ah[j / 2] = (uint32_t)r;
                    lmin = min(lmin, r);
                }
            }
        };
        /* middle: sides that are no powers of two at coordinates between 2^21
         * and 2^22 (or longer than 2^20) wrap by the integer modulo, still
         * without the x86 casts' clamps (1363 x 767, 1531 slices at x = 3e6:
         * 18.8 us, 19.5 through the casts; with reciprocals, nearer the
         * origin, 17.3) */
        constexpr std::integral_constant<int, HP2 ? FSK_TAME : FSK_TAME_MOD> best{};
        constexpr std::integral_constant<int, FSK_TAME> middle{};
        if (f.tame >= best && kr == KR)
            project(best, std::true_type{});
        else if (f.tame >= best)
            project(best, std::false_type{});
        else if (!HP2 && MODE != kOutNearest && f.tame >= FSK_TAME && kr == KR)
            project(middle, std::true_type{});
        else if (!HP2 && MODE != kOutNearest && f.tame >= FSK_TAME)
            project(middle, std::false_type{});
        else
            project(std::integral_constant<int, 0>{}, std::false_type{});
        /* lanes holding samples past the chunk, past kr (a last gather
         * group kr does not fill) or right of the frame: those samples
         * become row H */
        if (!colok || g * kr + kr > cn || (kr % GATHER) != 0) {
            lmin = H;
#pragma unroll
            for (int j = 0; j < KR; j++) {
                const bool ok = j < kr && g * kr + j < cn && colok;
                const uint32_t sh16 = (uint32_t)(j & 1) * 16u;
                uint32_t r = ok ? (ah[j / 2] >> sh16) & 0xFFFFu : (uint32_t)H;
                ah[j / 2] = (ah[j / 2] & ~(0xFFFFu << sh16)) | (r << sh16);
                lmin = min(lmin, (int32_t)r);
            }
        }

        /* phase 2 */
        int32_t excl;
        if constexpr (TC == 8) {
            int32_t total;
            wave_column_scan8(lmin, H, lane, excl, total);
            if (lane >= 64 - TC)
                sh.wtot[wave][c] = total;
        } else {
            int32_t v = lmin;
#pragma unroll
            for (int off = TC; off < 64; off <<= 1) {
                int32_t o = __shfl_up(v, off);
                if (lane >= off)
                    v = min(v, o);
            }
            excl = __shfl_up(v, TC);
            if (lane < TC)
                excl = H;
            if (lane >= 64 - TC)
                sh.wtot[wave][c] = v;
        }
        /* the chunk's carry-in is read before the barrier: the last slice
         * group overwrites it in phase 3 without a barrier in between (the
         * first chunk's is H) */
        const int32_t carry_in = base == 0 ? H : sh.carry[c];
        if (base == 0)
            tables.store(sh, tid);
        __syncthreads();
        /* exclusive prefix over the waves: each lane reads the totals of
         * the waves before its own (same address across the wave's lanes
         * of one column: broadcast reads) */
        int32_t run = min(carry_in, excl);
        for (int w = 0; w < wave; w++)
            run = min(run, sh.wtot[w][c]);

        /* phase 3: mark this lane's visible samples, reserve queue slots
         * with one wave-level prefix sum, then queue them in slice order.
         * A lane's samples take consecutive slots, so the bottom of a
         * sample's span (the y-buffer just before it: the next visible row
         * below in its column) is the row of the entry before it, or, for
         * the lane's first, the y-buffer in front of the lane (lanein) */
        const int32_t run_in = run;
        uint32_t vbits = 0u;
#pragma unroll
        for (int j = 0; j < KR; j++) {
            int32_t aj = (int32_t)((ah[j / 2] >> ((j & 1) * 16)) & 0xFFFFu);
            bool vis = aj < run;
            run = vis ? aj : run;
            vbits |= vis ? (1u << j) : 0u;
        }
        {
            uint32_t cnt = (uint32_t)__builtin_popcount(vbits);
            uint32_t incl = wave_incl_sum(cnt);
            uint32_t total = (uint32_t)__builtin_amdgcn_readlane((int)incl, 63);
            uint32_t b0 = 0;
            if (lane == 0 && total)
                b0 = atomicAdd(&sh.qn, total);
            b0 = __builtin_amdgcn_readfirstlane(b0);
            uint32_t slot = b0 + incl - cnt;
#pragma unroll
            for (int j = 0; j < KR; j++) {
                if (vbits & (1u << j)) {
                    int32_t aj = (int32_t)((ah[j / 2] >> ((j & 1) * 16)) & 0xFFFFu);
                    queue[slot] = ((uint32_t)g << kQGroupShift) | ((uint32_t)j << kQSliceShift) |
                                  ((uint32_t)c << kQColShift) | (uint32_t)aj;
                    slot++;
                }
            }
            lanein[tid] = (uint16_t)run_in;
        }
        /* the last slice group of each column holds the running minimum of
         * the whole chunk: the sh.carry into the next chunk */
        if (g == SG - 1)
            sh.carry[c] = run;
        __syncthreads();
        bool done = true;
#pragma unroll
        for (int j = 0; j < TC; j++)
            done = done && sh.carry[j] == 0;

        /* phase 4: colour and span, CBATCH queue entries per thread
         * at a time: their colour-quad gathers are all issued before the
         * first colour is computed */
        const uint32_t nq = sh.qn;
        for (uint32_t i0 = 0; i0 < nq; i0 += NT * CBATCH) {
            uint32_t es[CBATCH];
            float xs[CBATCH], ys[CBATCH];
            uint4 cqs[CBATCH];
#pragma unroll
            for (int u = 0; u < CBATCH; u++) {
                uint32_t e = queue[min(i0 + (uint32_t)(u * NT + tid), nq - 1u)];
                int32_t cc = (int32_t)((e >> kQColShift) & 15u);
                float4 L = tl[(int32_t)((e >> kQSliceShift) & 31u) * SG +
                              (int32_t)(e >> kQGroupShift)];
                float fc = (float)(col0 + cc);
                es[u] = e;
                xs[u] = L.x + (fc * L.z);
                ys[u] = L.y + (fc * L.w);
                if (MODE == kOutColour)
                    cqs[u] = color_quad<CP2>(m, xs[u], ys[u], f.tame);
            }
#pragma unroll
            for (int u = 0; u < CBATCH; u++) {
                const uint32_t i = i0 + (uint32_t)(u * NT + tid);
                if (i >= nq)
                    break;
                const uint32_t e = es[u];
                int32_t s = (int32_t)(e >> kQGroupShift) * kr + (int32_t)((e >> kQSliceShift) & 31u);
                int32_t cc = (int32_t)((e >> kQColShift) & 15u);
                int32_t row = (int32_t)(e & kQRowMask);
                const float x = xs[u], y = ys[u];
                uint32_t colour;
                if (MODE == kOutColour)
                    colour = color_of_quad<true>(cqs[u], sh.sq, x, y, sh.qt);
                else if (MODE == kOutNearest)
                    colour = ((const uint32_t *)m.cq)[nearest_index<HP2>(m, x, y)] ^ f.sky;
                else
                    colour = (floorf(x) == ceilf(x) || floorf(y) == ceilf(y))
                                 ? 0u : (uint32_t)(base + s + 1);
                /* a transparent sample paints 0 (fill_vline takes the
                 * colour above it) */
                if (colour == 0u)
                    sh.transparent = 1u;
                /* the entry before, if it is this lane's (same g and c),
                 * holds the row where this sample's span ends */
                const uint32_t ep = queue[i > 0 ? i - 1u : 0u];
                const bool first = i == 0 || ((e ^ ep) & kQLaneMask) != 0;
                int32_t bottom = first ? (int32_t)lanein[(int32_t)(e >> kQGroupShift) * TC + cc]
                                       : (int32_t)(ep & kQRowMask);
                uint32_t *dst = stripe + cc * Hp;
                int32_t stop = min(bottom, row + kShortSpan);
                for (int32_t r = row; r < stop; r++)
                    dst[r] = colour;
                if (bottom > stop) {
                    uint32_t li = atomicAdd(&sh.nlong, 1u);
                    longs[2 * li] = ((uint32_t)cc << 26) | ((uint32_t)stop << kQRowBits) |
                                    (uint32_t)bottom;
                    longs[2 * li + 1] = colour;
                }
            }
        }
        __syncthreads();
        if (done)
            break;
    }

    /* no chunk ran (no slices): publish the initial y-buffer (H, all sky) */
    if (n <= 0)
        __syncthreads();

    /* long spans: each wave paints every NW-th one with its 64 lanes */
    const uint32_t nl = sh.nlong;
    for (uint32_t li = (uint32_t)wave; li < nl; li += NW) {
        uint32_t d = longs[2 * li], colour = longs[2 * li + 1];
        int32_t cc = (int32_t)(d >> 26), r0 = (int32_t)((d >> kQRowBits) & kQRowMask);
        int32_t r1 = (int32_t)(d & kQRowMask);
        for (int32_t r = r0 + lane; r < r1; r += 64)
            stripe[cc * Hp + r] = colour;
    }
    if (nl)
        __syncthreads();

    before_write();
    const bool vec = (col0 + TC <= f.cols) && ((pitch & 3) == 0) &&
                     ((((uintptr_t)out) & 15u) == 0);
    /* a cell above its column's final y-buffer was never painted: 0 */
    auto cell = [&](int32_t cc, int32_t r, int32_t ybuf) -> uint32_t {
        return r < ybuf ? 0u : stripe[cc * Hp + r];
    };
    if (sh.transparent == 0u) {
        /* phase 5: every painted cell is final, the rest is sky.  TC/4
         * adjacent lanes share a row, so each store instruction writes
         * whole TC*4-byte row segments */
        constexpr int PARTS = TC / 4;
        const int32_t part = tid % PARTS;
        int32_t yb[4];
#pragma unroll
        for (int j = 0; j < 4; j++)
            yb[j] = sh.carry[part * 4 + j];
        /* the loop is written twice so that the whole-segment one keeps
         * its single 16-byte store: with the edge test inside one loop the
         * compiler shares the last element's store between the two forms
         * and splits the segment into a 12-byte and a 4-byte store */
        auto rows = [&](auto vec_tag) {
            constexpr bool VEC = decltype(vec_tag)::value;
            for (int32_t r = tid / PARTS; r < H; r += NT / PARTS) {
                uint32_t px[4];
#pragma unroll
                for (int j = 0; j < 4; j++)
                    px[j] = painted_value<MODE>(stripe[(part * 4 + j) * Hp + r], r < yb[j], f.sky);
                uint32_t *dst = out + (size_t)r * (size_t)pitch + col0 + part * 4;
                if (VEC) {
                    *(uint4 *)dst = make_uint4(px[0], px[1], px[2], px[3]);
                } else {
#pragma unroll
                    for (int j = 0; j < 4; j++)
                        if (col0 + part * 4 + j < f.cols)
                            dst[j] = px[j];
                }
            }
        };
        if (vec)
            rows(std::true_type{});
        else
            rows(std::false_type{});
        return;
    }

    /* phase 5 with sh.transparent samples: a zero cell takes the last
     * non-zero colour above it (fill_vline), else the sky; each thread
     * owns a block of consecutive rows */
    const int32_t per = (H + NT - 1) / NT;
    const int32_t r0 = min(tid * per, H), r1 = min(r0 + per, H);
    uint32_t pre[TC];
    int32_t yb[TC];
#pragma unroll
    for (int j = 0; j < TC; j++) {
        yb[j] = sh.carry[j];
        uint32_t p = 0u;
        for (int32_t r = r0; r < r1; r++) {
            uint32_t s = cell(j, r, yb[j]);
            p = s ? s : p;
        }
        pre[j] = p;
    }
    uint32_t *wfill = (uint32_t *)&sh.wtot[0][0];      /* [NW][TC] */
    uint32_t *wfpre = (uint32_t *)&sh.wpre[0][0];
    uint32_t *top = lds;                               /* [TC]; the slice table is done */
#pragma unroll
    for (int j = 0; j < TC; j++) {
        uint32_t v = pre[j];
#pragma unroll
        for (int off = 1; off < 64; off <<= 1) {
            uint32_t o = __shfl_up(v, off);
            if (lane >= off)
                v = v ? v : o;
        }
        uint32_t ex = __shfl_up(v, 1);
        pre[j] = lane == 0 ? 0u : ex;
        if (lane == 63)
            wfill[wave * TC + j] = v;
    }
    __syncthreads();
    if (wave == 0) {
#pragma unroll
        for (int half = 0; half < TC / 4; half++) {
            int32_t cc = (lane & 3) + 4 * half;
            uint32_t t = (lane >> 2) < NW ? wfill[(lane >> 2) * TC + cc] : 0u;
#pragma unroll
            for (int off = 4; off < 64; off <<= 1) {
                uint32_t o = __shfl_up(t, off);
                if (lane >= off)
                    t = t ? t : o;
            }
            uint32_t ex = __shfl_up(t, 4);
            if ((lane >> 2) < NW)
                wfpre[(lane >> 2) * TC + cc] = lane < 4 ? 0u : ex;
        }
    }
    if (BAND && row0 > 0) {
        /* a column that a transparent sample above the band covers from its
         * first row on: wave j finds what shows through in column j */
        static_assert(TC <= NW, "a wave per column");
        if (wave < TC && col0 + wave < f.cols && sh.carry[wave] == 0 && stripe[wave * Hp] == 0u) {
            const uint32_t above =
                column_above<HBITS, HP2, CP2, MODE>(m, f, col0 + wave, row0, sh.sq);
            if (lane == 0)
                top[wave] = above;
        } else if (wave < TC && lane == 0) {
            top[wave] = 0u;
        }
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < TC; j++) {
        uint32_t p = wfpre[wave * TC + j];
        if (BAND && row0 > 0)
            p = p ? p : top[j];
        pre[j] = pre[j] ? pre[j] : p;
    }
    /* written twice for the same reason as the loop above */
    auto rows = [&](auto vec_tag) {
        constexpr bool VEC = decltype(vec_tag)::value;
        for (int32_t r = r0; r < r1; r++) {
            uint32_t px[TC];
#pragma unroll
            for (int j = 0; j < TC; j++) {
                uint32_t s = cell(j, r, yb[j]);
                pre[j] = s ? s : pre[j];
                px[j] = tile_value<MODE>(pre[j], f.sky);
            }
            uint32_t *dst = out + (size_t)r * (size_t)pitch + col0;
            if (VEC) {
#pragma unroll
                for (int j = 0; j < TC; j += 4)
                    *(uint4 *)(dst + j) = make_uint4(px[j], px[j + 1], px[j + 2], px[j + 3]);
            } else {
#pragma unroll
                for (int j = 0; j < TC; j++)
                    if (col0 + j < f.cols)
                        dst[j] = px[j];
            }
        }
    };
    if (vec)
        rows(std::true_type{});
    else
        rows(std::false_type{});
}

template <int TC, int NT, int CMAX, int HBITS, bool HP2, bool CP2, int WPE, int MODE,
          bool BAND = false>
__global__ __launch_bounds__(NT, WPE) void k_render(RenderArgs a)
{
    extern __shared__ __align__(16) uint32_t lds[];  /* float4 slice table at its start */
    __shared__ TileShared<TC> sh;
    if constexpr (MODE == kOutSlice && !BAND) {
        if ((int32_t)blockIdx.x >= a.ntiles) {
            const size_t stride = (size_t)a.nzero * NT;
            for (size_t i = (size_t)(blockIdx.x - a.ntiles) * NT + threadIdx.x; i < a.zero_n4;
                 i += stride)
                a.zero[i] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
            return;
        }
    }
    const int32_t row0 = BAND ? (int32_t)blockIdx.y * a.band_rows : 0;
    uint32_t *out = BAND ? a.out + (size_t)row0 * (size_t)a.pitch : a.out;
    if constexpr (MODE == kOutColour) {
        /* the table loads go first: the tile's index arithmetic before them
         * had cost the 1080p frame 0.2 us */
        TileTables<TC, NT> tables;
        tables.load(threadIdx.x);
        render_tile<TC, NT, CMAX, HBITS, HP2, CP2, MODE, kGather, kColourBatch,
                    TileTables<TC, NT>, BAND>(a.m, a.f, out, a.pitch,
                                              xcd_tile(blockIdx.x, a.ntiles), a.chunk_max, lds,
                                              sh, tables, row0, a.band_rows);
    } else {
        render_tile<TC, NT, CMAX, HBITS, HP2, CP2, MODE, kGather, kColourBatch, NoTables, BAND>(
            a.m, a.f, out, a.pitch, xcd_tile(blockIdx.x, a.ntiles), a.chunk_max, lds, sh,
            NoTables(), row0, a.band_rows);
    }
}

/* render2 (fut/voxel_renderer.fut:257-305), the reference's ray-march
 * renderer.  The reference evaluates every dist = 0 ... n and keeps the hit
 * with the smallest dist (redstuff, :254-255); dists grow along the ray, so
 * that is the first hit (hits are the only elements that can win while the
 * miss distance i32(distance + 1) exceeds n, which the host checks).  The
 * colour is bilinear over the map's unshaded colours, evaluated for the
 * hit only.  cs/sn hold cos and sin of angle + horz_ang per column,
 * computed on the host with the C library as `futhark c` does.
 *
 * The terrain height under a ray point does not depend on the pixel's row:
 * a workgroup evaluates the heights of its 64 columns once for its ROWS rows,
 * a chunk of dists at a time, into LDS.  A pixel then searches them: along
 * dist the line of sight cam_h - dist * vert_ang is monotone, also in f32, so
 * if its lower end over a group of dists is not below the group's highest
 * terrain, none of them hits.  Wave w of the 16 evaluates group w of a chunk,
 * and so has the group's maximum in registers.  800 x 600 pixels, 200 steps:
 * 12 us, against 98 us with one thread per pixel marching through the map;
 * bound by the latency of its two phases on 247 workgroups.
 *
 * A camera on the ground, or one that looks steeply down from little above it,
 * has its hits within a few steps, and the full first chunk of 256 dists took
 * longer than the marching threads had (3840 x 2160: a call of 159 us, 79 by
 * the marching threads).  NEAR: where the line of sight of a workgroup's first
 * row comes below the ground under the camera within a chunk of 16 groups of
 * kR2Near dists, such a chunk goes first (93 us, with launch_render2's shapes;
 * 121 without).  Frames of one workgroup per CU go without it: 32 instead of
 * 34 us for such a camera at 800 x 600, but 40.2 instead of 39.6 for any other. */
struct Render2Args {
    fsk_map m;
    const uint32_t *color;     /* unshaded colours [hrows][hcols] */
    const float *cs, *sn;      /* [cols] */
    uint32_t *out;
    int64_t pitch;
    float cam_x, cam_y, cam_h, horizon;
    int32_t n, rows, cols;
};

template <bool P2>
__device__ __forceinline__ uint4 raw_color_quad(const uint32_t *col, int32_t rows, int32_t cols,
                                                float x, float y)
{
    const uint32_t fx = (uint32_t)wrap<P2>(idx_of(floorf(x)), cols);
    const uint32_t cx = (uint32_t)wrap<P2>(idx_of(ceilf(x)), cols);
    const uint32_t fy = (uint32_t)wrap<P2>(idx_of(floorf(y)), rows);
    const uint32_t cy = (uint32_t)wrap<P2>(idx_of(ceilf(y)), rows);
    const uint32_t w = (uint32_t)cols;
    return make_uint4(col[fy * w + fx], col[fy * w + cx], col[cy * w + fx], col[cy * w + cx]);
}

constexpr int kR2Group = 16;                      /* dists per group, a group per wave */
constexpr int kR2Near = 4;                        /* in the first chunk of a low camera */

template <int HBITS, bool HP2, int ROWS, int WPE, bool NEAR>
__global__ __launch_bounds__(1024, WPE) void k_render2(Render2Args a)
{
    __shared__ float sq[256];
    __shared__ float hs[16 * kR2Group][64], top[16][64];
    const int32_t lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int32_t x = blockIdx.x * 64 + lane;
    const float ca = a.cs[min(x, a.cols - 1)], sa = a.sn[min(x, a.cols - 1)];
    fill_square_lut(sq, threadIdx.x);
    constexpr int PX = ROWS / 16;
    float vert_ang[PX];
    int32_t hit[PX];
#pragma unroll
    for (int u = 0; u < PX; u++) {
        const int32_t y = blockIdx.y * ROWS + u * 16 + wave;
        vert_ang[u] = (a.horizon / 50.0f) + (((float)y / ((float)a.rows - 0.0f)) * (1.5f - 1.0f));
        hit[u] = -1;
    }
    /* a chunk of 16 groups of G dists; whether any pixel is left without a hit */
    auto march = [&](int32_t base, auto group) -> bool {
        constexpr int G = decltype(group)::value, B = G < 8 ? G : 8;
        const int32_t d0 = base + wave * G;
        float high = -INFINITY;
#pragma unroll
        for (int j0 = 0; j0 < G; j0 += B) {
            if (d0 + j0 > a.n) {
                /* past the march: nothing is below the lowest height */
#pragma unroll
                for (int j = j0; j < j0 + B; j++)
                    hs[wave * G + j][lane] = -INFINITY;
                continue;
            }
            float px[B], py[B];
            uint2 q[B];
#pragma unroll
            for (int j = 0; j < B; j++) {
                const float fd = (float)(d0 + j0 + j);
                px[j] = a.cam_x + (fd * ca);
                py[j] = a.cam_y + (fd * sa);
                q[j] = height_quad<HBITS, HP2>(a.m, px[j], py[j]);
            }
#pragma unroll
            for (int j = 0; j < B; j++) {
                float h = height_interp<HBITS>(q[j], px[j], py[j]);
                h = d0 + j0 + j <= a.n ? h : -INFINITY;
                hs[wave * G + j0 + j][lane] = h;
                high = fmaxf(high, h);
            }
        }
        top[wave][lane] = high;
        __syncthreads();
        const int32_t groups = min(16 * G, a.n + 1 - base + G - 1) / G;
        bool pending = false;
#pragma unroll
        for (int u = 0; u < PX; u++) {
            for (int32_t g = 0; g < groups && hit[u] < 0; g++) {
                const float f0 = (float)(base + g * G);
                const float t0 = a.cam_h - (f0 * vert_ang[u]);
                const float t1 = a.cam_h - ((f0 + (float)(G - 1)) * vert_ang[u]);
                if (!(fminf(t0, t1) < top[g][lane]))
                    continue;
                uint32_t below = 0u;
#pragma unroll
                for (int j = 0; j < G; j++)
                    below |= (a.cam_h - ((f0 + (float)j) * vert_ang[u])) < hs[g * G + j][lane]
                                 ? 1u << j : 0u;
                if (below)
                    hit[u] = base + g * G + __builtin_ctz(below);
            }
            pending = pending || hit[u] < 0;
        }
        /* also keeps the next chunk's heights from those still being read */
        return __syncthreads_or(pending);
    };
    int32_t base = 0;
    bool more = a.n >= 0;
    if constexpr (NEAR) {
        /* does the first row's line of sight come below the camera's ground
         * within the short chunk?  Only a guess of where the hits are, so that
         * one texel will do for the ground */
        const float vert_lo = (a.horizon / 50.0f) + (((float)(blockIdx.y * ROWS) /
                                                      ((float)a.rows - 0.0f)) * (1.5f - 1.0f));
        const uint32_t ground = height_quad<HBITS, HP2>(a.m, a.cam_x, a.cam_y).x &
                                (HBITS == 8 ? 0xFFu : 0xFFFFu);
        const bool low = (a.cam_h - ((float)(16 * kR2Near) * vert_lo)) < (float)ground;
        if (__builtin_amdgcn_readfirstlane(more && low)) {
            more = march(0, std::integral_constant<int, kR2Near>{});
            base = 16 * kR2Near;
        }
    }
    for (; more && base <= a.n; base += 16 * kR2Group)
        more = march(base, std::integral_constant<int, kR2Group>{});
    if (a.n < 0)
        __syncthreads();                          /* the squares */
#pragma unroll
    for (int u = 0; u < PX; u++) {
        const int32_t y = blockIdx.y * ROWS + u * 16 + wave;
        if (x >= a.cols || y >= a.rows)
            continue;
        uint32_t c = 0u;
        if (hit[u] >= 0) {
            const float fd = (float)hit[u];
            const float px = a.cam_x + (fd * ca), py = a.cam_y + (fd * sa);
            c = color_of_quad(raw_color_quad<HP2>(a.color, a.m.hrows, a.m.hcols, px, py), sq, px,
                              py);
        }
        a.out[(size_t)y * (size_t)a.pitch + (size_t)x] = c;
    }
}

/* ------------------------------------------------------------------ */
/* Map preparation kernels                                             */
/* ------------------------------------------------------------------ */

/* Ingest: `elem & mask` (fut/interactive.fut:189) and the bilinear quad
 * of each texel (right and lower neighbours wrap, as floor-mod does).  A
 * thread holds kQuadRows rows of one column, so that a row's heights are
 * read once and not again as the lower half of the row above, with all of
 * its reads in flight together. */
constexpr int kQuadRows = 4;

template <int HBITS>
__global__ __launch_bounds__(256) void k_height_quads(const int32_t *__restrict__ alt,
                                                      int32_t rows, int32_t cols,
                                                      void *__restrict__ hq,
                                                      uint16_t *__restrict__ hplain)
{
    const int32_t x = blockIdx.x * 256 + threadIdx.x;
    const int32_t y0 = blockIdx.y * kQuadRows;
    if (x >= cols)
        return;
    const uint32_t mk = HBITS == 8 ? 0xFFu : 0xFFFFu;
    const int32_t x1 = x + 1 == cols ? 0 : x + 1;
    uint32_t h0[kQuadRows + 1], h1[kQuadRows + 1];
#pragma unroll
    for (int j = 0; j <= kQuadRows; j++) {
        /* row `rows` is row 0; rows past it are not used */
        const int32_t y = y0 + j < rows ? y0 + j : 0;
        h0[j] = (uint32_t)alt[(size_t)y * cols + x] & mk;
        h1[j] = (uint32_t)alt[(size_t)y * cols + x1] & mk;
    }
#pragma unroll
    for (int j = 0; j < kQuadRows; j++) {
        if (y0 + j >= rows)
            break;
        const size_t t = (size_t)(y0 + j) * cols + x;
        if (HBITS == 8)
            ((uint32_t *)hq)[t] = h0[j] | (h1[j] << 8) | (h0[j + 1] << 16) | (h1[j + 1] << 24);
        else
            ((uint2 *)hq)[t] = make_uint2(h0[j] | (h1[j] << 16), h0[j + 1] | (h1[j + 1] << 16));
        hplain[t] = (uint16_t)h0[j];
    }
}

/* The largest of n heights (16-byte aligned) as one value per workgroup in
 * hmax[FSK_HMAX_PARTS]: a pass of its own, since one atomic maximum per
 * workgroup of k_height_quads took longer than reading the heights again
 * (2048^2: 12 against 4 us). */
__global__ __launch_bounds__(1024) void k_height_max(const uint16_t *__restrict__ hp, size_t n,
                                                     uint32_t *__restrict__ hmax)
{
    const size_t first = (size_t)blockIdx.x * 1024 + threadIdx.x;
    const size_t stride = (size_t)gridDim.x * 1024, n8 = n / 8;
    uint32_t top = 0u;
    for (size_t i = first; i < n8; i += stride) {
        const uint4 v = ((const uint4 *)hp)[i];
        const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
        for (int j = 0; j < 4; j++)
            top = max(top, max(w[j] & 0xFFFFu, w[j] >> 16));
    }
    for (size_t i = n8 * 8 + first; i < n; i += stride)
        top = max(top, (uint32_t)hp[i]);
    __shared__ uint32_t wtop[16];
#pragma unroll
    for (int off = 32; off > 0; off >>= 1)
        top = max(top, (uint32_t)__shfl_xor((int)top, off));
    if ((threadIdx.x & 63) == 0)
        wtop[threadIdx.x >> 6] = top;
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < 16; w++)
            top = max(top, wtop[w]);
        hmax[blockIdx.x] = top;
    }
}

__global__ void k_color_quads(const uint32_t *__restrict__ c, int32_t rows, int32_t cols,
                              uint4 *__restrict__ cq)
{
    int32_t x = blockIdx.x * blockDim.x + threadIdx.x;
    int32_t y = blockIdx.y;
    if (x >= cols)
        return;
    int32_t x1 = x + 1 == cols ? 0 : x + 1;
    int32_t y1 = y + 1 == rows ? 0 : y + 1;
    cq[(size_t)y * cols + x] = make_uint4(c[(size_t)y * cols + x], c[(size_t)y * cols + x1],
                                          c[(size_t)y1 * cols + x], c[(size_t)y1 * cols + x1]);
}

/* generate_shadowmap_accumulated, fut/effects.fut:108-125: for each
 * texel of the size^2 grid count the 255 sun-ray steps that pass below
 * the terrain by more than half a unit (nearest `png_height`,
 * fut/render_functions.fut:63-64), then darken with argb.mix -- or, for the
 * differentiable renderer, write the shade factor sqrt(1 / (4*count + 1)).
 *
 * The steps' offsets t * sun (t = 4 * dist) are the same for every texel:
 * the host forms them once (the same f32 products) and they arrive as
 * kernel arguments, i.e. in scalar registers.  A wave holds kShadeTexels
 * runs of 64 texels of one row, so a step's map row is one scalar too, and
 * a texel's step is nine vector instructions and a coalesced 2-byte load.
 * Under a sun above the horizon the ray climbs: (height + t * s1) - probe is
 * non-decreasing in t for a fixed probe, also in f32, so once it is at least
 * -0.5 against the map's largest height no later step can count, and the
 * wave leaves when that holds for its lowest texel (at sun height 0.1
 * after at most 65 of the 255 steps on an 8-bit map).  Measured, sun height
 * 0.1: 1024^2 grid 338 -> 25 us; 4096^2 grid, heights to 1024 (nearly every
 * step) 4.79 -> 0.64 ms, where the vector instructions bound it; before,
 * one texel per thread took every step with two general floor-mods. */
constexpr int kShadeSteps = 256;      /* dist = 1 .. 255 */
constexpr int kShadeTexels = 4;       /* texels per thread, 64 apart in x */
constexpr int kShadeGroup = 5;        /* steps between exit tests; 255 = 51 * 5 */

struct ShadeArgs {
    const uint16_t *hp;
    const uint32_t *hmax;             /* the map's largest height: k_height_max's parts */
    const uint32_t *col;              /* raw colours (not read for the shade factor) */
    void *out;
    int32_t hrows, hcols, size;
    float rrows, rcols;               /* 1 / hrows, 1 / hcols */
    /* t * s0, t * s1, t * s2 of step dist at [dist] */
    float dx[kShadeSteps], dh[kShadeSteps], dy[kShadeSteps];
};
static_assert(sizeof(ShadeArgs) <= 4096, "kernel argument size");

/* Floor-mod of a map coordinate.  kWrapPow2: a mask.  kWrapSmall: any side
 * m <= 2^16 and |v| < 2^22: v / m in f32 is within 2^-22 relative of the
 * quotient, which is below 2^22, so its floor is the integer quotient or
 * one off, and one correction either way gives the remainder.  kWrapX86:
 * every i32. */
enum { kWrapPow2 = 0, kWrapSmall = 1, kWrapX86 = 2 };

template <int WRAP>
__device__ __forceinline__ int32_t wrap_map(int32_t v, int32_t m, float rm)
{
    if (WRAP == kWrapPow2)
        return v & (m - 1);
    if (WRAP == kWrapX86)
        return fmod_i32(v, m);
    int32_t r = v - (int32_t)floorf((float)v * rm) * m;
    r = r < 0 ? r + m : r;
    return r >= m ? r - m : r;
}

/* WRAP kWrapX86 is for sun vectors that are not finite, whose probes take
 * the x86 cast's INT_MIN (a finite sun's offsets are at most 1020), and for
 * map sides or grids above 2^16. */
template <int WRAP, bool FACTOR>
__global__ __launch_bounds__(256) void k_shade(ShadeArgs a)
{
    const int32_t lane = threadIdx.x & 63;
    const int32_t y = __builtin_amdgcn_readfirstlane(blockIdx.y * 4 + (threadIdx.x >> 6));
    const int32_t x0 = blockIdx.x * (64 * kShadeTexels) + lane;
    if (y >= a.size)
        return;
    const size_t row = (size_t)wrap_map<WRAP>(y, a.hrows, a.rrows) * (size_t)a.hcols;
    static_assert(FSK_HMAX_PARTS == 128, "two parts per lane");
    float hmax = (float)max(a.hmax[lane], a.hmax[lane + 64]);
    const float fy = (float)y;
    float fx[kShadeTexels], height[kShadeTexels], low = 65536.0f;
    int32_t count[kShadeTexels];
#pragma unroll
    for (int u = 0; u < kShadeTexels; u++) {
        const int32_t x = x0 + 64 * u;
        fx[u] = (float)x;
        height[u] = (float)a.hp[row + (size_t)wrap_map<WRAP>(x, a.hcols, a.rcols)];
        low = fminf(low, x < a.size ? height[u] : low);
        count[u] = 0;
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        low = fminf(low, __shfl_xor(low, off));
        hmax = fmaxf(hmax, __shfl_xor(hmax, off));
    }
    const bool rises = a.dh[1] >= 0.0f;
    for (int32_t d0 = 1; d0 < kShadeSteps; d0 += kShadeGroup) {
        /* uniform over the wave: low and the step's values are */
        if (rises && ((low + a.dh[d0]) - hmax) >= -0.5f)
            break;
#pragma unroll
        for (int j = 0; j < kShadeGroup; j++) {
            const int32_t d = d0 + j;
            auto texel = [](float v) { return WRAP == kWrapX86 ? i32_f32_x86(v) : (int32_t)v; };
            const int32_t iy = __builtin_amdgcn_readfirstlane(
                wrap_map<WRAP>(texel(fy + a.dy[d]), a.hrows, a.rrows));
            const FS_GLOBAL char *hrow =
                (const FS_GLOBAL char *)(a.hp + (size_t)iy * (size_t)a.hcols);
#pragma unroll
            for (int u = 0; u < kShadeTexels; u++) {
                const uint32_t ix =
                    (uint32_t)wrap_map<WRAP>(texel(fx[u] + a.dx[d]), a.hcols, a.rcols);
                const float probe = (float)*(const FS_GLOBAL uint16_t *)(hrow + ix * 2u);
                count[u] += (((height[u] + a.dh[d]) - probe) < -0.5f) ? 1 : 0;
            }
        }
    }
    const float step_size = 4.0f;
#pragma unroll
    for (int u = 0; u < kShadeTexels; u++) {
        const int32_t x = x0 + 64 * u;
        if (x >= a.size)
            continue;
        const float amount = (float)count[u];
        const size_t t = (size_t)y * (size_t)a.size + (size_t)x;
        if (FACTOR)
            ((float *)a.out)[t] = __builtin_sqrtf(1.0f / ((step_size * amount) + 1.0f));
        else
            ((uint32_t *)a.out)[t] = argb_mix(step_size * amount, 0xFF000000u, 1.0f,
                                              a.col[row + (size_t)wrap_map<WRAP>(x, a.hcols, a.rcols)]);
    }
}

/* ------------------------------------------------------------------ */
/* Device self-tests of the arithmetic shortcuts                       */
/* ------------------------------------------------------------------ */

/* 0: unit8(b) == b / 255 (correctly rounded) for all bytes.
 * 1: sqrt_unit(t) == correctly rounded sqrt(t) for every f32 in [0, 1]
 *    and for NaNs.
 * 2: chan_u8(v) == u32.f32(clamp_channel(v) * 255) with the if-chain
 *    clamp, for every f32 bit pattern.
 * 3: screen_row_clamped(rel, H) == min(screen_row(rel), H) for every f32
 *    bit pattern at H = 1080.
 * 4: the quantisation table (g_qtab) gives u32.f32(sqrt(t) * 255), with
 *    the correctly rounded sqrt, for every f32 t in [0, 1].
 * 5: rcp_rn(z) == 1 / z (correctly rounded) for every f32 z in
 *    [2^-126, 2^126).
 * 6: div_rn(a, w, RN(1 / w)) == a / w for every finite f32 a and every
 *    frame width w of kSelftestWidths.
 * 7: sqrt_rn(t) == correctly rounded sqrt(t) for every f32 t >= 0
 *    (+inf included) and NaN stays NaN.
 * 8: wrap_tame(v, m) == the floor-mod of v by m for every integer |v| < 2^21
 *    and every side m of kSelftestSides. */
constexpr int32_t kSelftestWidths[] = {1920, 1280, 800, 640, 320, 3840, 128, 96, 1024,
                                       2048, 4096, 240, 1, 3, 7, 1000, 1366};
constexpr int kNSelftestWidths = sizeof kSelftestWidths / sizeof kSelftestWidths[0];
constexpr int32_t kSelftestSides[] = {1, 2, 3, 5, 7, 90, 100, 333, 777, 1000, 1363, 1500,
                                      4095, 65535, 1048575, 1048576};
constexpr int kNSelftestSides = sizeof kSelftestSides / sizeof kSelftestSides[0];

struct SelftestRecips {
    float rm[kNSelftestSides];
};

__global__ void k_selftest(int which, SelftestRecips recips, unsigned long long *bad)
{
    uint64_t n = which == 0 ? 256ull
                 : (which == 1 || which == 4) ? 0x3F800001ull
                 : which == 5 ? 0x7E000000ull
                 : which == 7 ? 0x7F800001ull
                 : which == 6 ? (uint64_t)kNSelftestWidths << 32
                 : which == 8 ? (uint64_t)kNSelftestSides << 22
                              : 0x100000000ull;
    uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    unsigned long long local = 0;
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) {
        uint32_t u = (uint32_t)i;
        bool ok = true;
        if (which == 7) {
            const float t = __uint_as_float(u);
            ok = __float_as_uint(sqrt_rn(t)) == __float_as_uint(__builtin_sqrtf(t));
            const float nan = __uint_as_float(0x7FC00000u | (u & 0x3FFFFFu));
            ok = ok && (sqrt_rn(nan) != sqrt_rn(nan));
        } else if (which == 8) {
            const int32_t v = (int32_t)(u & 0x3FFFFFu) - (1 << 21), s = (int32_t)(i >> 22);
            const int32_t m = kSelftestSides[s];
            ok = v == -(1 << 21) || wrap_tame((float)v, m, recips.rm[s]) == fmod_i32(v, m);
        } else if (which == 5) {
            u += 0x00800000u;
            const float z = __uint_as_float(u);
            ok = __float_as_uint(rcp_rn(z)) == __float_as_uint(1.0f / z);
        } else if (which == 6) {
            const float w = (float)kSelftestWidths[i >> 32];
            const float a = __uint_as_float(u);
            if ((u & 0x7F800000u) != 0x7F800000u)
                ok = __float_as_uint(div_rn(a, w, 1.0f / w)) == __float_as_uint(a / w);
        } else if (which == 0) {
            ok = __float_as_uint(unit8(u)) == __float_as_uint((float)u / 255.0f);
        } else if (which == 1) {
            float t = __uint_as_float(u);
            ok = __float_as_uint(sqrt_unit(t)) == __float_as_uint(__builtin_sqrtf(t));
            float nan = __uint_as_float(0x7FC00000u | (u & 0x3FFFFFu));
            ok = ok && (sqrt_unit(nan) != sqrt_unit(nan));
        } else if (which == 2) {
            float v = __uint_as_float(u);
            float c = (v < 0.0f) ? 0.0f : ((v > 1.0f) ? 1.0f : v);
            float sc = c * 255.0f;
            uint32_t want = (sc == sc) ? (uint32_t)sc : 0u;
            ok = chan_u8(v) == want;
        } else if (which == 3) {
            float rel = __uint_as_float(u);
            ok = screen_row_clamped(rel, 1080.0f) == min(screen_row(rel), 1080);
        } else {
            float t = __uint_as_float(u);
            const uint32_t want = (uint32_t)(__builtin_sqrtf(t) * 255.0f);
            ok = (mix_q(g_qtab, 1.0f, t, 0.0f, 0.0f) >> 17) == want;
        }
        if (!ok) {
            local += 1;
            atomicMin(bad + 1, (unsigned long long)u);
        }
    }
    if (local)
        atomicAdd(bad, local);
}

/* Per-device caches of device properties and kernel set-up (a process may
 * drive several devices; each has its own). */
constexpr int kMaxDevices = 64;

inline int current_device()
{
    int d = 0;
    if (hipGetDevice(&d) != hipSuccess || d < 0 || d >= kMaxDevices)
        d = 0;
    return d;
}

inline size_t lds_per_cu()
{
    static std::atomic<int> v[kMaxDevices];
    const int dev = current_device();
    int x = v[dev].load(std::memory_order_relaxed);
    if (x == 0) {
        if (hipDeviceGetAttribute(&x, hipDeviceAttributeMaxSharedMemoryPerMultiprocessor, dev) !=
                hipSuccess ||
            x <= 0)
            x = 65536;
        v[dev].store(x, std::memory_order_relaxed);
    }
    return (size_t)x;
}

inline int cu_count()
{
    static std::atomic<int> v[kMaxDevices];
    const int dev = current_device();
    int x = v[dev].load(std::memory_order_relaxed);
    if (x == 0) {
        if (hipDeviceGetAttribute(&x, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
            x <= 0)
            x = 256;
        v[dev].store(x, std::memory_order_relaxed);
    }
    return x;
}

/* Lets `kern` take all of a CU's LDS but its static shared memory, once per
 * device; returns that dynamic maximum (0 on failure, with *err set). */
inline int dyn_lds_max(const void *kern, std::atomic<int> *cache, hipError_t *err)
{
    const int dev = current_device();
    int x = cache[dev].load(std::memory_order_relaxed);
    if (x > 0)
        return x;
    hipFuncAttributes fa;
    hipError_t e = hipFuncGetAttributes(&fa, kern);
    if (e == hipSuccess) {
        x = (int)lds_per_cu() - (int)fa.sharedSizeBytes;
        e = hipFuncSetAttribute(kern, hipFuncAttributeMaxDynamicSharedMemorySize, x);
    }
    if (e != hipSuccess) {
        *err = e;
        return 0;
    }
    cache[dev].store(x, std::memory_order_relaxed);
    return x;
}

template <int TC, int NT, int CMAX, int HBITS, bool HP2, bool CP2, int WPE, int MODE>
hipError_t launch_render_cfg(const RenderArgs &a, hipStream_t s)
{
    auto kern = k_render<TC, NT, CMAX, HBITS, HP2, CP2, WPE, MODE>;
    static std::atomic<int> dyn_cache[kMaxDevices];
    hipError_t e = hipSuccess;
    const int dyn_max = dyn_lds_max((const void *)kern, dyn_cache, &e);
    if (!dyn_max)
        return e;
    size_t need = render_lds_bytes(TC, NT, a.f.rows, a.chunk_max);
    if (need > (size_t)dyn_max)
        return hipErrorInvalidValue;
    hipLaunchKernelGGL(kern, dim3(a.ntiles + a.nzero), dim3(NT), need, s, a);
    return hipGetLastError();
}

/* ------------------------------------------------------------------ */
/* Kernel shape and tuning                                             */
/* ------------------------------------------------------------------ */

/* Render kernel shape: columns per workgroup tile (8: 32-byte row
 * segments; 4: 16-byte segments), one 1024-thread or two 512-thread
 * workgroups per CU (two let one tile's barrier and gather stalls overlap
 * the other's work -- worth it when there are many more tiles than CUs, as
 * in batches; they need the LDS of two tiles, so their depth chunk is
 * shorter: at most 512 slices for 8 columns, 1024 for 4), and the
 * depth-chunk length.  Each context carries its own tuning (fsx_set_tuning,
 * the autotuner), which starts from the FSX_RENDER_TC /
 * FSX_RENDER_WG_PER_CU / FSX_RENDER_CHUNK environment variables; 0 means
 * automatic. */

struct Shape {
    int tc, nt, wg, chunk, cmax;
};

constexpr size_t kStaticLds = 12288;  /* headroom for the kernels' static shared memory */

/* Slices from which on a lane of a 1024-thread tile holds more than
 * kHalfChunk / (slice groups) of them: up to there the kernels of half the
 * chunk waste no registers and no passes on slices that are not there
 * (1100 x 400, 1024 slices). */
constexpr int kHalfChunk = 1024;

/* The automatic shape of one frame: what was measured best over widths of
 * 64 to 8192, 240 to 1240 rows and 64 to 4096 slices (us, 8x1 / 4x1 /
 * 8x2 = columns x workgroups per CU).
 *  - narrow: 4-column tiles still find a CU each, and a tile's time is its
 *    latency chain and its share of the work (640 x 480, 2048 slices: 12.9 /
 *    9.4 / 18.7);
 *  - one chunk of the 512-thread tile, whose barriers and phases are the
 *    shortest: up to 256 slices (64 x 240, 200: 7.2 / 7.4 / 6.4), or 512
 *    where there are more tiles than CUs (3840 x 1080, 500: 17.8 / 32.4 /
 *    13.5);
 *  - more tiles than CUs: two tiles on a CU instead of one after the other
 *    (2560 x 400, 1024: 16.8 / 19.2 / 13.8), unless the 1024-thread tile's
 *    last 2048-slice chunk is more than three quarters full, where it is as
 *    fast or faster (2560 x 1080, 2048: 26.2 / 27.4 / 27.1; 3000: 38.6 / 46.4
 *    / 35.6) but for frames of many rounds (8192 x 1080, 2048: 52.4 / 72.1 /
 *    49.8).
 * spare: the caller would use kMinZeroBlocks idle CUs, which 4-column tiles
 * may not leave. */
inline fsk_tuning frame_shape(int32_t rows, int32_t cols, int32_t n, bool spare)
{
    fsk_tuning t = {0, 0, 0};
    const int32_t cus = cu_count(), tiles4 = (cols + 3) / 4, tiles8 = (cols + 7) / 8;
    const bool two = 2 * (render_lds_bytes(8, 512, rows, 512) + kStaticLds) <= lds_per_cu();
    const bool narrow = tiles4 <= cus && !(spare && cus - tiles4 < kMinZeroBlocks);
    if (two && n <= (tiles8 > cus ? 512 : 256))
        t.wg_per_cu = 2;
    else if (narrow)
        t.tc = 4;
    else if (two && tiles8 > cus && (tiles8 > 3 * cus || (n - 1) % kChunk < 3 * kChunk / 4))
        t.wg_per_cu = 2;
    return t;
}

/* The shape of a frame of `rows` rows under tuning `tune`; with cols > 0 a
 * tuning left automatic follows frame_shape. */
inline Shape resolve_shape(int32_t rows, const fsk_tuning &tune, int32_t cols = 0, int32_t n = 0,
                           bool spare = false)
{
    const bool automatic = cols > 0 && !tune.tc && !tune.wg_per_cu && !tune.chunk;
    const fsk_tuning t = automatic ? frame_shape(rows, cols, n, spare) : tune;
    Shape s;
    s.cmax = kChunk;
    int chunk = (t.chunk >= 256 && t.chunk <= kChunk) ? t.chunk : 0;
    int c8 = chunk && chunk <= 512 ? chunk : 512;
    auto fits8 = [&](int c) {
        return render_lds_bytes(8, 1024, rows, c) + kStaticLds <= lds_per_cu();
    };
    if (t.tc != 4 && t.wg_per_cu == 2 &&
        2 * (render_lds_bytes(8, 512, rows, c8) + kStaticLds) <= lds_per_cu()) {
        s.tc = 8;
        s.nt = 512;
        s.wg = 2;
        s.chunk = c8;
        s.cmax = 512;
    } else if (t.tc != 4 && (chunk ? fits8(chunk) : fits8(kChunk) || fits8(kChunk / 2))) {
        /* left automatic, a frame too tall for 8-column tiles of the whole
         * chunk keeps them with half the chunk: measured faster than
         * 4-column tiles (2160 rows, 4096 slices: 49 against 55 us) */
        s.tc = 8;
        s.nt = 1024;
        s.wg = 1;
        s.chunk = chunk ? chunk : fits8(kChunk) ? kChunk : kChunk / 2;
    } else {
        s.tc = 4;
        int c2 = chunk ? chunk : 1024;
        c2 -= c2 % 128;
        if (t.wg_per_cu == 2 && 2 * (render_lds_bytes(4, 512, rows, c2) + kStaticLds) <=
                                    lds_per_cu()) {
            s.nt = 512;
            s.wg = 2;
            s.chunk = c2;
        } else {
            s.nt = 1024;
            s.wg = 1;
            s.chunk = chunk ? chunk : kChunk;
        }
    }
    /* a chunk holds whole groups of kChunkAlign slices per slice group;
     * tall frames take shorter chunks until the tile fits in LDS */
    auto need = [&](int c) {
        return render_lds_bytes(s.tc, s.nt, rows, c) + kStaticLds;
    };
    auto fit = [&]() {
        const int ga = (s.nt / s.tc) * kChunkAlign;
        s.chunk = s.chunk < ga ? ga : s.chunk - s.chunk % ga;
        while (s.chunk > ga && (size_t)s.wg * need(s.chunk) > lds_per_cu())
            s.chunk = (s.chunk / 2) - (s.chunk / 2) % ga;
        return (size_t)s.wg * need(s.chunk) <= lds_per_cu();
    };
    if (!fit() && s.tc == 4 && s.nt == 1024) {
        /* the tallest frames: 512-thread tiles, whose chunks go down to
         * 512 slices */
        s.nt = 512;
        s.wg = 1;
        fit();
    }
    if (s.nt == 1024) {
        if (automatic && n <= kHalfChunk && s.chunk > kHalfChunk)
            s.chunk = kHalfChunk;
        if (s.chunk <= kHalfChunk)
            s.cmax = kHalfChunk;
    }
    return s;
}

/* Frames of more than kMaxRows rows: 8-column tiles over bands of rows, each
 * as tall as its stripe fits in LDS beside chunks of at most kBandChunk
 * slices (half the whole-column tile's, for 1000 more rows a band).  A band
 * repeats its columns' projection, about 8 us per tile, and stores its rows
 * at the tile kernel's rate.  Measured on the stateless program's 800-column
 * frames: 10^4 rows 306 -> 23 us, 10^5 rows 3.04 -> 0.13 ms (2.4 TB/s of
 * stores), 10^6 rows 30.3 -> 1.39 ms, against one thread per column walking
 * the slices and storing its spans cell by cell. */
constexpr int kBandChunk = 1024;

template <int HBITS, bool HP2, bool CP2, int MODE>
hipError_t launch_bands(RenderArgs a, hipStream_t s)
{
    constexpr int TC = 8, NT = 1024, kGroups = NT / TC * kChunkAlign;
    if (a.f.rows > kMaxFrameRows)
        return hipErrorInvalidValue;
    auto kern = k_render<TC, NT, kBandChunk, HBITS, HP2, CP2, 4, MODE, true>;
    static std::atomic<int> dyn_cache[kMaxDevices];
    hipError_t e = hipSuccess;
    const int dyn_max = dyn_lds_max((const void *)kern, dyn_cache, &e);
    if (!dyn_max)
        return e;
    a.chunk_max = std::min(kBandChunk, std::max(1, (a.f.n + kGroups - 1) / kGroups) * kGroups);
    int32_t most = 64;
    while (most + 64 <= kMaxRows &&
           render_lds_bytes(TC, NT, most + 64, a.chunk_max) <= (size_t)dyn_max)
        most += 64;
    const int32_t bands = (a.f.rows + most - 1) / most;
    a.band_rows = ((a.f.rows + bands - 1) / bands + 63) & ~63;
    a.ntiles = (a.f.cols + TC - 1) / TC;
    const size_t need = render_lds_bytes(TC, NT, a.band_rows, a.chunk_max);
    if (need > (size_t)dyn_max)
        return hipErrorInvalidValue;
    hipLaunchKernelGGL(kern, dim3(a.ntiles, (a.f.rows + a.band_rows - 1) / a.band_rows), dim3(NT),
                       need, s, a);
    return hipGetLastError();
}

template <int HBITS, bool HP2, bool CP2, int MODE = kOutColour>
hipError_t launch_render(RenderArgs a, const fsk_tuning &tune, hipStream_t s,
                         int32_t *nzero = nullptr)
{
    if (a.f.rows > kMaxRows) {
        if (nzero)
            *nzero = 0;         /* no gradient clear */
        return launch_bands<HBITS, HP2, CP2, MODE>(a, s);
    }
    Shape sh = resolve_shape(a.f.rows, tune, a.f.cols, a.f.n,
                             MODE == kOutSlice && a.zero && a.zero_n4);
    a.chunk_max = sh.chunk;
    a.ntiles = (a.f.cols + sh.tc - 1) / sh.tc;
    /* slice mode: the workgroup slots the tiles leave free clear the
     * gradient, if there are enough of them */
    const int32_t spare = cu_count() * sh.wg - a.ntiles;
    a.nzero = (MODE == kOutSlice && a.zero && a.zero_n4 && spare >= kMinZeroBlocks) ? spare : 0;
    if (nzero)
        *nzero = a.nzero;
    const bool half = sh.cmax == kHalfChunk;
    if (sh.tc == 8) {
        if (sh.nt == 512)
            return launch_render_cfg<8, 512, 512, HBITS, HP2, CP2, 4, MODE>(a, s);
        return half ? launch_render_cfg<8, 1024, kHalfChunk, HBITS, HP2, CP2, 4, MODE>(a, s)
                    : launch_render_cfg<8, 1024, kChunk, HBITS, HP2, CP2, 4, MODE>(a, s);
    }
    if (sh.nt == 512)
        return launch_render_cfg<4, 512, kChunk, HBITS, HP2, CP2, 4, MODE>(a, s);
    return half ? launch_render_cfg<4, 1024, kHalfChunk, HBITS, HP2, CP2, 4, MODE>(a, s)
                : launch_render_cfg<4, 1024, kChunk, HBITS, HP2, CP2, 4, MODE>(a, s);
}

/* ------------------------------------------------------------------ */
/* Batched persistent render                                           */
/* ------------------------------------------------------------------ */

struct BatchArgs {
    const fsk_batch_view *views;
    const uint32_t *items;
    const uint32_t *qmeta;
    uint32_t *counters;
    uint32_t *out;
    int32_t nqueues, chunk_max;
};

/* Persistent workgroups take (view, tile) items from per-XCD queues: the
 * host deals each view's tiles out to the queues in contiguous blocks, so
 * neighbouring tiles of a view stay on one L2 (workgroup i runs on XCD
 * i mod 8).  Workgroup i takes item i / nqueues of queue i mod nqueues
 * first, and then what the queues' counters hand out, from the next queues
 * when its own is drained; it ends when all are.
 *
 * A claim is an atomic on memory all XCDs share, and those on one line go
 * one after the other: each counter has a line of its own, the first item
 * needs no claim, and a drained queue is told by reading its counter.  With
 * the eight counters in one line, and an atomic on each of them for every
 * workgroup that ran dry, the claims took longer than the tiles of a small
 * batch (4 views: 157 us).
 *
 * The counters are as fsk_batch_counters_init left them before the first
 * launch; the last workgroup to end leaves them so for the next one, so that
 * no launch has to reset them first.  Every claim of a workgroup has
 * returned before it counts itself as ended.
 *
 * Launches of one batch that overlap (two contexts, or an eager launch beside
 * a replay) share the counters: between them they hand out every item, some
 * of them twice, with the same pixels.  The ended workgroups are counted over
 * all of them by an atomic that wraps at a launch's worth, so that none is
 * lost; the last of all to end finds a whole number of launches and leaves the
 * counters reset.  A reset that reaches memory late, when its launch ends, over
 * the claims of another only has items handed out again, and that one's own end
 * resets the counters after it.  Resets by agent-scope stores, with the count
 * lowered by a second atomic, kept a launch's last workgroup and so the next
 * launch waiting: 0.3 to 1 us of a batch of 13 to 40 us. */
__host__ __device__ constexpr uint32_t batch_first_claim(uint32_t grid, uint32_t q, uint32_t nq)
{
    return (grid + nq - 1u - q) / nq;      /* workgroups that start on queue q */
}

template <int TC, int NT, int CMAX, int HBITS, bool HP2, bool CP2, int WPE>
__global__ __launch_bounds__(NT, WPE) void k_render_batch(BatchArgs b)
{
    extern __shared__ __align__(16) uint32_t lds[];  /* float4 slice table at its start */
    __shared__ TileShared<TC> sh;
    __shared__ uint32_t cur;
    {
        TileTables<TC, NT> tables;
        tables.load(threadIdx.x);
        tables.store(sh, threadIdx.x);    /* the claim loop's barrier publishes them */
    }
    const uint32_t nq = (uint32_t)b.nqueues;
    uint32_t q = blockIdx.x % nq, tried = 0u;
    uint32_t len = b.qmeta[nq + q], next = blockIdx.x / nq;
    bool claimed = true;                  /* next is this workgroup's */
    for (;;) {
        if (threadIdx.x == 0) {
            uint32_t v = 0xFFFFFFFFu;
            while (tried < nq) {
                uint32_t *count = b.counters + q * FSK_COUNTER_STRIDE;
                if (!claimed && __hip_atomic_load(count, __ATOMIC_RELAXED,
                                                  __HIP_MEMORY_SCOPE_AGENT) < len) {
                    next = atomicAdd(count, 1u);
                    claimed = true;
                }
                if (claimed && next < len) {
                    v = b.items[b.qmeta[q] + next];
                    break;
                }
                claimed = false;
                tried++;
                q = q + 1u == nq ? 0u : q + 1u;
                len = b.qmeta[nq + q];
            }
            cur = v;
        }
        __syncthreads();
        uint32_t it = cur;
        __syncthreads();
        if (it == 0xFFFFFFFFu)
            break;
        const fsk_batch_view &bv = b.views[it >> 16];
        /* while a queue is far from its end the next claim is made before
         * the tile's rows are written, and its round trip passes under
         * them; near the end an item claimed early would wait for this
         * workgroup while others run dry */
        auto claim = [&]() {
            if (threadIdx.x == 0) {
                claimed = next + gridDim.x / nq < len;
                if (claimed)
                    next = atomicAdd(b.counters + q * FSK_COUNTER_STRIDE, 1u);
            }
        };
        render_tile<TC, NT, CMAX, HBITS, HP2, CP2, kOutColour, kGather, kColourBatch, NoTables,
                    false, decltype(claim) &>(bv.m, bv.f, b.out + bv.offset, bv.f.cols,
                                              it & 0xFFFFu, b.chunk_max, lds, sh, NoTables(), 0,
                                              0, claim);
    }
    if (threadIdx.x == 0) {
        uint32_t *ended = b.counters + nq * FSK_COUNTER_STRIDE;
        if (atomicInc(ended, gridDim.x - 1u) == gridDim.x - 1u) {
            for (uint32_t i = 0; i < nq; i++)
                b.counters[i * FSK_COUNTER_STRIDE] = batch_first_claim(gridDim.x, i, nq);
        }
    }
}

template <int TC, int NT, int CMAX, int HBITS, bool HP2, bool CP2, int WPE>
hipError_t launch_batch_cfg(const fsk_batch *fb, int chunk, hipStream_t s)
{
    auto kern = k_render_batch<TC, NT, CMAX, HBITS, HP2, CP2, WPE>;
    static std::atomic<int> dyn_cache[kMaxDevices];
    hipError_t e = hipSuccess;
    const int dyn_max = dyn_lds_max((const void *)kern, dyn_cache, &e);
    if (!dyn_max)
        return e;
    size_t need = render_lds_bytes(TC, NT, fb->max_rows, chunk);
    if (need > (size_t)dyn_max)
        return hipErrorInvalidValue;
    BatchArgs b;
    b.views = fb->views;
    b.items = fb->items;
    b.qmeta = fb->qmeta;
    b.counters = fb->counters;
    b.out = fb->out;
    b.nqueues = fb->nqueues;
    b.chunk_max = chunk;
    hipLaunchKernelGGL(kern, dim3(fb->grid), dim3(NT), need, s, b);
    return hipGetLastError();
}

template <int HBITS, bool HP2, bool CP2>
hipError_t launch_batch(const fsk_batch *fb, hipStream_t s)
{
    Shape sh = resolve_shape(fb->max_rows, fb->tune);
    if (sh.tc == 8)
        return sh.nt == 512 ? launch_batch_cfg<8, 512, 512, HBITS, HP2, CP2, 4>(fb, sh.chunk, s)
                            : launch_batch_cfg<8, 1024, kChunk, HBITS, HP2, CP2, 4>(fb, sh.chunk, s);
    return sh.nt == 512 ? launch_batch_cfg<4, 512, kChunk, HBITS, HP2, CP2, 4>(fb, sh.chunk, s)
                        : launch_batch_cfg<4, 1024, kChunk, HBITS, HP2, CP2, 4>(fb, sh.chunk, s);
}

/* ------------------------------------------------------------------ */
/* Differentiable renderer: f32 colour planes                           */
/* ------------------------------------------------------------------ */

/* The f32 relaxation of the colour path: planes cp[3][hc][wc] in [0,1]
 * replace the u32 ARGB map, each texel scaled by its shade factor
 * sf = sqrt(1/(4*count + 1)) (argb.mix(4*count, black, 1, c) without
 * quantisation, fut/effects.fut:123), and argb.mix's channel rule
 * sqrt(m1'*a^2 + m2'*b^2) without u8 rounding (matte colour.fut, as
 * png_color_filtered calls it at fut/render_functions.fut:101-103).
 * Visibility is the integer renderer's, held fixed: src[r][c] is the
 * depth slice whose sample shows at the pixel, -1 for sky.  Sky pixels
 * are sky_base * sky_scale with sky_base = (0x90, 0x90, 0xE0) / 255
 * (argb.scale of 0xFF9090e0, fut/interactive.fut:163). */


/* Sum of n per-workgroup partials (f32 or f64) in f64 and in a fixed order
 * by one workgroup of NT threads, stored into *dst or added to it: thread t
 * adds part[t], part[t + NT], ... in that order (eight loads issued before
 * the first add), then the wave totals are added in wave order.  Every
 * thread of the workgroup must call it. */
template <int NT, typename T>
__device__ __forceinline__ void block_sum_partials(const T *__restrict__ part, int32_t n,
                                                   float *__restrict__ dst, int32_t accumulate)
{
    __shared__ double wsum[NT / 64];
    double acc = 0.0;
    for (int32_t base = 0; base < n; base += 8 * NT) {
        T v[8];
#pragma unroll
        for (int u = 0; u < 8; u++) {
            const int32_t i = base + u * NT + (int32_t)threadIdx.x;
            v[u] = i < n ? part[i] : (T)0;
        }
#pragma unroll
        for (int u = 0; u < 8; u++)
            acc += v[u];
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1)
        acc += __shfl_xor(acc, off);
    if ((threadIdx.x & 63) == 0)
        wsum[threadIdx.x >> 6] = acc;
    __syncthreads();
    if (threadIdx.x == 0) {
        double t = 0.0;
        for (int w = 0; w < NT / 64; w++)
            t += wsum[w];
        *dst = (float)(accumulate ? (double)*dst + t : t);
    }
}

struct DiffArgs {
    fsk_frame f;
    const float *cp;
    const float *sf;
    int32_t hc, wc;
    float rhc, rwc;        /* fsk_wrap_recip of them */
    float sky_scale;
    const int32_t *src;
    const float *gimg;     /* backward: dL/dimg [3][rows][cols] */
    float *img;            /* forward output [3][rows][cols] */
    float *gcp;            /* backward: dL/dcp accumulated [3][hc][wc] */
    float *gsky;           /* backward: dL/dsky_scale accumulated */
    double *partials;      /* per-workgroup partial sums (loss or sky) */
    const float *tgt;      /* fused step: the target frame [3][rows][cols] */
    float *gout;           /* fused step: dL/dimg written out (may be null) */
    double *sky_part;      /* fused step: per-workgroup sky terms */
};

/* The relaxed argb.mix channel: sqrt(m1' a^2 + m2' b^2) with weights
 * m1', m2' already normalised by norm_weights. */
__device__ __forceinline__ float mixn(float m1n, float a, float m2n, float b)
{
    return sqrt_rn((m1n * (a * a)) + (m2n * (b * b)));
}

/* One visible sample: texel offsets (fy,fx) (fy,cx) (cy,fx) (cy,cx) and
 * the bilinear weights, as png_color_filtered forms them
 * (fut/render_functions.fut:95-105) with floor-mod indices. */
struct Bilin {
    uint32_t t[4];
    float wx0, wx1, wy0, wy1;
    bool pair;               /* fx is not the map's last column */
};

/* The four texels of a bilinear quad from one plane.  When no lane of
 * the wave has its quad wrap round the map's last column, texels t1 and
 * t3 follow t0 and t2 in memory, and each pair is one 8-byte load (4-byte
 * aligned, which global loads allow).  At an integer x the quad's second
 * texel is its first (cx = fx) and the pair loads the next one instead;
 * the x weights are then 0 and their sum 0, so the colour is NaN whatever
 * the texel holds. */
typedef float float2_a4 __attribute__((ext_vector_type(2), aligned(4)));
__device__ __forceinline__ void quad_load(const float *P, const Bilin &b, bool pairs,
                                          float v[4])
{
    if (pairs) {
        const float2_a4 lo = *(const float2_a4 *)(P + b.t[0]);
        const float2_a4 hi = *(const float2_a4 *)(P + b.t[2]);
        v[0] = lo.x;
        v[1] = lo.y;
        v[2] = hi.x;
        v[3] = hi.y;
    } else {
#pragma unroll
        for (int t = 0; t < 4; t++)
            v[t] = P[b.t[t]];
    }
}

/* argb.mix's weights divided by their sum, for the x pair and the y pair
 * of a bilinear sample (w = wx0', wx1', wy0', wy1').  A pair sums to
 * exactly 1 unless its coordinate is an integer (sum 0) or within 1 of the
 * map origin, where the division is an exact no-op when skipped, so the
 * divisions run on a wave-uniform branch only when some lane of the wave
 * needs them (the empty asm keeps the compiler from evaluating them on
 * every wave). */
__device__ __forceinline__ void norm_weights(const Bilin &b, float w[4])
{
    w[0] = b.wx0;
    w[1] = b.wx1;
    w[2] = b.wy0;
    w[3] = b.wy1;
    const float sx = b.wx0 + b.wx1, sy = b.wy0 + b.wy1;
    const bool dx = sx != 1.0f, dy = sy != 1.0f;
    if (__ballot(dx || dy)) {
        float x0 = b.wx0, x1 = b.wx1, y0 = b.wy0, y1 = b.wy1;
        asm volatile("" : "+v"(x0), "+v"(x1), "+v"(y0), "+v"(y1));
        if (dx) {
            w[0] = x0 / sx;
            w[1] = x1 / sx;
        }
        if (dy) {
            w[2] = y0 / sy;
            w[3] = y1 / sy;
        }
    }
}

/* Texel offsets are 32-bit: a plane holds at most 2^31 texels (checked by
 * the host).  P2: both plane sides are powers of two, so the floor-mod is
 * a mask (also for the INT_MIN of an out-of-range cast). */
template <bool P2, bool TAME = false>
__device__ __forceinline__ Bilin bilin_of(const DiffArgs &a, int32_t k, int32_t col)
{
    const fsk_frame &f = a.f;
    const int32_t hc = a.hc, wc = a.wc;
    Slice sl = TAME ? slice_params_tame(f, k) : slice_params(f, k);
    float fcol = (float)col;
    float x = sl.sx + (fcol * sl.dx);
    float y = sl.sy + (fcol * sl.dy);
    float fx = floorf(x), cx = ceilf(x), fy = floorf(y), cy = ceilf(y);
    /* TAME: a tame frame keeps |x|, |y| < 2^22, where the x86 conversion
     * is the plain one */
    auto cvt = [](float v) { return TAME ? (int32_t)v : i32_f32_x86(v); };
    int32_t ify, icy, ifx, icx;
    if (TAME && !P2 && f.tame >= FSK_TAME_MOD) {
        ify = wrap_tame(fy, hc, a.rhc);
        icy = wrap_tame(cy, hc, a.rhc);
        ifx = wrap_tame(fx, wc, a.rwc);
        icx = wrap_tame(cx, wc, a.rwc);
    } else {
        ify = wrap<P2>(cvt(fy), hc);
        icy = wrap<P2>(cvt(cy), hc);
        ifx = wrap<P2>(cvt(fx), wc);
        icx = wrap<P2>(cvt(cx), wc);
    }
    const uint32_t ry = P2 ? (uint32_t)ify << __builtin_ctz((uint32_t)wc)
                           : (uint32_t)ify * (uint32_t)wc;
    const uint32_t rc = P2 ? (uint32_t)icy << __builtin_ctz((uint32_t)wc)
                           : (uint32_t)icy * (uint32_t)wc;
    Bilin b;
    b.t[0] = ry + (uint32_t)ifx;
    b.t[1] = ry + (uint32_t)icx;
    b.t[2] = rc + (uint32_t)ifx;
    b.t[3] = rc + (uint32_t)icx;
    b.wx0 = cx - x;
    b.wx1 = x - fx;
    b.wy0 = cy - y;
    b.wy1 = y - fy;
    b.pair = ifx < wc - 1;
    return b;
}

__device__ __forceinline__ float sky_base(int ch)
{
    return ch == 2 ? 224.0f / 255.0f : 144.0f / 255.0f;
}

/* The shaded texel values of a sample's quad: sf[t] and the three planes'
 * cv[ch][t].  All sixteen gathers are issued here, before any mix: the
 * mixes branch, and loads are not moved above a branch, so gathers
 * interleaved with them would wait for each other. */
__device__ __forceinline__ void sample_gather(const DiffArgs &a, const Bilin &b, size_t plane,
                                              float cv[3][4], float sf[4])
{
    /* one load per texel: the paired loads of quad_load measured slower
     * in the adjoint (its gathers sit under a per-lane branch) */
#pragma unroll
    for (int t = 0; t < 4; t++)
        sf[t] = a.sf[b.t[t]];
#pragma unroll
    for (int ch = 0; ch < 3; ch++) {
        const float *P = a.cp + ch * plane;
#pragma unroll
        for (int t = 0; t < 4; t++)
            cv[ch][t] = P[b.t[t]];
    }
}

/* The colour of a visible sample from its gathered quad, per channel (the
 * relaxed png_color_filtered); sv[ch][t] = cv[ch][t] * sf[t]. */
__device__ __forceinline__ void sample_mix(const Bilin &b, const float cv[3][4],
                                           const float sf[4], float w[4], float sv[3][4],
                                           float px[3])
{
    norm_weights(b, w);
#pragma unroll
    for (int ch = 0; ch < 3; ch++) {
#pragma unroll
        for (int t = 0; t < 4; t++)
            sv[ch][t] = cv[ch][t] * sf[t];
        float X1 = mixn(w[0], sv[ch][0], w[1], sv[ch][1]);
        float X2 = mixn(w[0], sv[ch][2], w[1], sv[ch][3]);
        px[ch] = mixn(w[2], X1, w[3], X2);
    }
}

/* Forward colour, one thread per pixel (2-D blocks of 64 columns x 4
 * rows: the gathers of neighbouring pixels share texels).  This kernel
 * gathers each channel's quad just before its mixes: with one pixel per
 * thread and many waves in flight that measured faster than issuing all
 * sixteen gathers first (which needs more registers per wave), and so did
 * one pixel per thread against two or four, and against listing each
 * column's runs to colour each visible sample once. */
template <bool P2, bool TAME>
__global__ __launch_bounds__(256) void k_diff_color(DiffArgs a)
{
    const int32_t col = blockIdx.x * 64 + (threadIdx.x & 63);
    const int32_t row = blockIdx.y * 4 + (threadIdx.x >> 6);
    const int32_t H = a.f.rows, W = a.f.cols;
    if (col >= W || row >= H)
        return;
    const size_t plane = (size_t)a.hc * a.wc, fplane = (size_t)H * W;
    const size_t p = (size_t)row * W + col;
    const int32_t k = a.src[p];
    float px[3];
    if (k < 0) {
#pragma unroll
        for (int ch = 0; ch < 3; ch++)
            px[ch] = sky_base(ch) * a.sky_scale;
    } else {
        const Bilin b = bilin_of<P2, TAME>(a, k, col);
        float sf[4], w[4];
        const bool pairs = __ballot(!b.pair) == 0;
        quad_load(a.sf, b, pairs, sf);
        norm_weights(b, w);
#pragma unroll
        for (int ch = 0; ch < 3; ch++) {
            float sv[4];
            quad_load(a.cp + ch * plane, b, pairs, sv);
#pragma unroll
            for (int t = 0; t < 4; t++)
                sv[t] *= sf[t];
            float X1 = mixn(w[0], sv[0], w[1], sv[1]);
            float X2 = mixn(w[0], sv[2], w[1], sv[3]);
            px[ch] = mixn(w[2], X1, w[3], X2);
        }
    }
#pragma unroll
    for (int ch = 0; ch < 3; ch++)
        a.img[ch * fplane + p] = px[ch];
}

constexpr uint32_t kNoKey = 0xFFFFFFFFu;     /* an empty texel slot, a lane with no sample */

/* One step of segment_sum_quad: each lane takes (v, f) of the lane CTRL
 * names (DPP) unless its accumulated range already holds its segment's
 * first lane (f).  Lanes with no source (shifted out of their row, or in
 * rows that ROWS leaves out) take (0, 0), which changes nothing. */
template <int CTRL, int ROWS, int N>
__device__ __forceinline__ void segment_step(float (&v)[N], int32_t &f)
{
    constexpr bool kShift = CTRL < 0x140;      /* row shifts read 0 outside the row */
    float d[N];
#pragma unroll
    for (int c = 0; c < N; c++)
        d[c] = __int_as_float(
            __builtin_amdgcn_update_dpp(0, __float_as_int(v[c]), CTRL, ROWS, 0xf, kShift));
    const int32_t fd = __builtin_amdgcn_update_dpp(0, f, CTRL, ROWS, 0xf, kShift);
    if (!f) {
#pragma unroll
        for (int c = 0; c < N; c++)
            v[c] += d[c];
        f = fd;
    }
}

/* Segmented inclusive prefix sum of a sample's four texel values over the
 * lanes of a wave, in registers: lanes holding the same texel quad (all
 * four keys equal, none of them kNoKey) in a contiguous run form a
 * segment, and each lane ends up with the sums of val from its segment's
 * first lane to itself, so the segment's last lane holds the segment's
 * totals.  Steps of 1, 2, 4 and 8 lanes scan each row of 16 lanes (DPP
 * row shifts); then the last lane of rows 0 and 2 is carried into rows 1
 * and 3 (row_bcast:15) and lane 31 into rows 2 and 3 (row_bcast:31).  A
 * wave in which no lane shares its quad with the lane before skips the
 * scan (every lane is a segment of its own).  Returns whether this lane
 * ends its segment. */
__device__ __forceinline__ bool segment_sum_quad(const uint32_t key[4], float (&val)[4][3])
{
    /* the keys of lane - 1 and lane + 1 (wave shifts; the first and the
     * last lane see a key that differs from their own).  Every lane reads
     * both neighbours: a DPP read from a lane that a branch has switched
     * off does not see that lane's key, so the comparisons are combined
     * without short-circuiting */
    uint32_t diff_prev = key[0] == kNoKey ? 1u : 0u, diff_next = diff_prev;
#pragma unroll
    for (int t = 0; t < 4; t++) {
        const int32_t k = (int32_t)key[t];
        diff_prev |= (uint32_t)(__builtin_amdgcn_update_dpp(~k, k, 0x138, 0xf, 0xf, false) ^ k);
        diff_next |= (uint32_t)(__builtin_amdgcn_update_dpp(~k, k, 0x130, 0xf, 0xf, false) ^ k);
    }
    const bool same_prev = diff_prev == 0u, same_next = diff_next == 0u;
    if (!__ballot(same_prev))
        return true;
    float v[12];
#pragma unroll
    for (int t = 0; t < 4; t++)
#pragma unroll
        for (int c = 0; c < 3; c++)
            v[t * 3 + c] = val[t][c];
    int32_t f = same_prev ? 0 : 1;
    /* once every lane's range holds its segment's first lane the later
     * steps change nothing: most segments are two or three lanes long */
    segment_step<0x111, 0xf>(v, f);            /* row_shr:1 */
    if (__ballot(!f)) {
        segment_step<0x112, 0xf>(v, f);        /* row_shr:2 */
        if (__ballot(!f)) {
            segment_step<0x114, 0xf>(v, f);    /* row_shr:4 */
            if (__ballot(!f)) {
                segment_step<0x118, 0xf>(v, f);    /* row_shr:8 */
                segment_step<0x142, 0xa>(v, f);    /* row_bcast:15 */
                segment_step<0x143, 0xc>(v, f);    /* row_bcast:31 */
            }
        }
    }
#pragma unroll
    for (int t = 0; t < 4; t++)
#pragma unroll
        for (int c = 0; c < 3; c++)
            val[t][c] = v[t * 3 + c];
    return !same_next;
}

/* Workgroups of the adjoint: 64 columns by 4 waves.  512 threads with a
 * table of 2048 texels: 1900 x 1000 98 against 89 us per fused step; 128 with
 * 512: 94 us. */
constexpr int kGradThreads = 256;
/* Rows per thread in the adjoint: 2, or 4 in frames of kGradTallPixels
 * pixels or more.  A run of equal src down a thread's rows is one evaluation
 * and one insertion, so more rows mean fewer of both per pixel, which pays
 * where a frame's runs are long and its workgroups many (2560 x 1440 over
 * 2048 slices: 72 against 83 us, 3840 x 2160 over 4096 slices: 119 against
 * 144 us), while smaller frames need the waves (1920 x 1080: 59 against 85
 * us).  8 rows: 88 against 92 us where heights of 10 bits make long runs,
 * 144 against 119 us where they do not. */
constexpr int64_t kGradTallPixels = (int64_t)3 << 20;
constexpr int kGradRowsLow = 2, kGradRowsTall = 4;
/* Texel slots of a workgroup's table (28 bytes each), and the workgroups of
 * a CU that they leave room for.  A texel that the table has no slot for
 * costs scattered global atomics.  With 2 rows, 512 pixels, distant ground
 * gives a workgroup up to some 1200 distinct texels: 1408 slots hold them
 * (1280 x 720: 45 us with 1408 slots and four workgroups, 52 with 1024 and
 * five, 59 with 816 and six).  With 4 rows, in frames whose runs are longer,
 * 944 slots and six workgroups: 92 us, 1024 and five 100 us, 512 and six 91
 * us there and 143 against 119 us over an 8-bit map.  With images to write
 * (out) a thread also holds its pixels until the run loop has ended, and six
 * or five workgroups would spill them (110 against 78 us for a 3840 x 2160
 * step that is nine tenths sky), so 4 rows take four workgroups too, and the
 * slots that these leave room for. */
constexpr int grad_cap(int rows, bool out)
{
    return rows == kGradRowsLow || out ? 1408 : 944;
}
constexpr int grad_waves(int rows, bool out)
{
    return rows == kGradRowsLow || out ? 4 : 6;
}
constexpr int kGradProbes = 4;
constexpr int kGradRunLog = 4;               /* texels of a row that hash to adjacent slots */

/* Add v[0..2] to texel `key` of the workgroup's LDS table (open addressing);
 * returns whether this call took a new slot.  A texel that finds no slot
 * within kGradProbes, or any new texel once kGradFill slots are taken, goes
 * straight to the global gradient.
 *
 * The sums are f64: an LDS f32 add takes 3 cycles per lane on this chip
 * (193 per wave, whatever the addresses), an f64 one 9 per wave.  With f32
 * sums the adds had bound the adjoint (72 of 98 us of a 1900 x 1000 step).
 *
 * The hash keeps runs of 2^kGradRunLog texels of a row together: adjacent
 * slots, which adjacent lanes flush, are then adjacent in memory, and a
 * wave's global atomics come as a few lines instead of one per lane
 * (1280 x 720: 94 -> 81 us per fused step; the flush no longer shows). */
template <int kGradCap>
__device__ __forceinline__ bool table_add(uint32_t *keys, double *vals, const uint32_t *fill,
                                          float *gcp, size_t plane, uint32_t key, const float v[3])
{
    constexpr uint32_t kRun = 1u << kGradRunLog;
    static_assert(kGradCap % kRun == 0 && kGradCap / kRun <= 256, "whole runs, 32-bit product");
    constexpr int kGradFill = kGradCap / 8 * 7;  /* slots taken before new texels go past it */
    uint32_t h = (__umul24(((key >> kGradRunLog) * 2654435761u) >> 8, kGradCap / kRun) >> 24) *
                     kRun + (key & (kRun - 1u));
    /* a relaxed atomic load, which becomes an LDS read: a volatile read
     * through this generic pointer was a flat load that waited for every
     * global atomic of the wave still in flight */
    const bool open = __hip_atomic_load(fill, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) <
                      (uint32_t)kGradFill;
#pragma unroll 1
    for (int p = 0; open && p < kGradProbes; p++) {
        uint32_t k = keys[h];
        bool mine = false;
        if (k == kNoKey) {
            k = atomicCAS(&keys[h], kNoKey, key);
            mine = k == kNoKey;
        }
        if (mine || k == key) {
#pragma unroll
            for (int ch = 0; ch < 3; ch++)
                __hip_atomic_fetch_add(&vals[ch * kGradCap + h], (double)v[ch],
                                       __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
            return mine;
        }
        h += kRun;
        h = h < (uint32_t)kGradCap ? h : h - kGradCap;
    }
#pragma unroll
    for (int ch = 0; ch < 3; ch++)
        if (v[ch] != 0.0f)
            unsafeAtomicAdd(&gcp[ch * plane + key], v[ch]);
    return false;
}

/* The texel terms of one visible sample k at column col whose pixels'
 * incoming gradients sum to run[3]: key[t] = texel t of the bilinear quad,
 * val[t][ch] = dL/d plane_ch at that texel.  For px = mix(wy0, X1, wy1, X2),
 * X1 = mix(wx0, s0, wx1, s1): d px / d s0 = wy0' * wx0' * s0 / px (X1
 * cancels), likewise for the other texels, 0 where px == 0. */
struct SampleEval {
    uint32_t t[4];           /* the quad's texels */
    float w[4];              /* norm_weights of the sample */
    float sf[4];             /* shade factors of the quad */
    float sv[3][4], px[3];   /* shaded texel values, pixel colour */
};

template <bool P2, bool TAME>
__device__ __forceinline__ void sample_eval(const DiffArgs &a, int32_t k, int32_t col,
                                            size_t plane, SampleEval &e)
{
    /* the caller's src may name slices past the frame's last, which the tame
     * bounds do not cover */
    Bilin b;
    if (TAME && !__ballot(k >= a.f.n))
        b = bilin_of<P2, TAME>(a, k, col);
    else
        b = bilin_of<P2, false>(a, k, col);
    float cv[3][4];
    sample_gather(a, b, plane, cv, e.sf);
    sample_mix(b, cv, e.sf, e.w, e.sv, e.px);
#pragma unroll
    for (int t = 0; t < 4; t++)
        e.t[t] = b.t[t];
}

__device__ __forceinline__ void sample_grad(const DiffArgs &a, const SampleEval &e,
                                            const float run[3], uint32_t key[4], float val[4][3])
{
    const float(&sv)[3][4] = e.sv;
    const float(&px)[3] = e.px;
    const float(&w)[4] = e.w;
    const float wt[4] = {w[2] * w[0], w[2] * w[1], w[3] * w[0], w[3] * w[1]};
    /* gradients are not bit-exact quantities: the hardware reciprocal
     * (within an ulp) stands in for the division, and the texel's weight
     * and shade factor are multiplied once */
    float q[3];
#pragma unroll
    for (int ch = 0; ch < 3; ch++)
        q[ch] = px[ch] > 0.0f ? run[ch] * __builtin_amdgcn_rcpf(px[ch]) : 0.0f;
#pragma unroll
    for (int t = 0; t < 4; t++) {
        const float ws = wt[t] * e.sf[t];
        key[t] = e.t[t];
#pragma unroll
        for (int ch = 0; ch < 3; ch++)
            val[t][ch] = (q[ch] * ws) * sv[ch][t];
    }
}

/* Adjoint.  A workgroup covers 64 adjacent columns x 4 kGradRows rows; each
 * thread holds kGradRows rows of one column.  A run of equal src down the column
 * is one visible sample: its incoming gradient is summed in registers and
 * pushed through the three mixes once.  For px = mix(wy0, X1, wy1, X2),
 * X1 = mix(wx0, s0, wx1, s1): d px / d s0 = wy0' * wx0' * s0 / px (X1
 * cancels), likewise for the other texels, 0 where px == 0.  A wave loops over
 * its lanes' runs, every lane at its next one wherever that starts: row by
 * row, a wave evaluated and inserted on each row where any lane began a run
 * (0.94 of a 4K view's rows; now 0.66 evaluations per row, 51 M instead of
 * 70 M vector instructions).  The texel terms are summed in two stages before
 * any global atomic: lanes of a wave whose runs hit the same texels (adjacent
 * columns magnifying one near texel) are merged by a segmented reduction
 * across the wave, so that the LDS table below sees distinct texels per
 * instruction; then an LDS hash table sums the terms per texel over the
 * whole block (neighbouring samples share texels: a block touches
 * several times fewer texels than it has sample-texel terms).  Few rows per
 * thread keep many waves in flight for the gathers.  Each table entry is then
 * added into the global f32 gradient with one atomic per channel.
 *
 * What bounds it: in large frames the vector instructions (3840 x 2160 fitting
 * view 127 -> 89 us); in small ones the inserts and the flush's atomics, with
 * the latency of a block's chain behind them (1280 x 720: 51 -> 46 us, 24
 * without inserts; 800 x 600 vjp 32 -> 26 us).
 *
 * FWD (the fused L2 step): the incoming gradient is not read but formed
 * here from the target, g = 2 (px - target), with the colour px of each
 * run's sample evaluated where the run starts (the same evaluation as
 * k_diff_color's, so img and g are bit-identical to the separate calls);
 * each workgroup leaves one partial of the loss, sum (px - target)^2, and one
 * of the sky term.  Otherwise each workgroup leaves one partial of the sky
 * term.
 *
 * OUT: img and g are written, where the caller asks for them, after the run
 * loop, a row of the wave at a time.  Written from within it, by the lanes
 * whose run was at hand and with six workgroups per CU, a 3840 x 2160 frame
 * that is all sky took 97 us and one that is two thirds sky 114; now 58 and
 * 94, of which the two images' 199 MB are 26 and 29. */
template <bool P2, bool TAME, bool FWD, bool OUT, int kGradRows>
__global__ __launch_bounds__(kGradThreads, grad_waves(kGradRows, OUT))
void k_diff_grad(DiffArgs a)
{
    constexpr int kGradCap = grad_cap(kGradRows, OUT);
    constexpr int kGradBlockRows = (kGradThreads / 64) * kGradRows;
    __shared__ uint32_t keys[kGradCap];
    __shared__ double vals[3 * kGradCap];
    __shared__ uint32_t fill;
    for (int32_t i = threadIdx.x; i < kGradCap; i += kGradThreads) {
        keys[i] = kNoKey;
        vals[i] = 0.0;
        vals[kGradCap + i] = 0.0;
        vals[2 * kGradCap + i] = 0.0;
    }
    if (threadIdx.x == 0)
        fill = 0u;
    const int32_t col = blockIdx.x * 64 + (threadIdx.x & 63);
    /* the row is the wave's: scalar, so that a pixel's address is a scalar
     * row pointer and the column */
    const int32_t wave = __builtin_amdgcn_readfirstlane((int32_t)threadIdx.x >> 6);
    const int32_t r0 = blockIdx.y * kGradBlockRows + wave * kGradRows;
    const int32_t H = a.f.rows, W = a.f.cols;
    const uint32_t lcol = (uint32_t)min(col, W - 1);
    const size_t plane = (size_t)a.hc * a.wc, fplane = (size_t)H * W;
    /* global-space views of the per-pixel inputs (loads through the
     * generic pointers came out as flat loads) */
    const FS_GLOBAL float *gin = (const FS_GLOBAL float *)(FWD ? a.tgt : a.gimg);
    const FS_GLOBAL int32_t *srcp = (const FS_GLOBAL int32_t *)a.src;
    int32_t src[kGradRows];
    float g[3][kGradRows];     /* FWD: the target; OUT: g, once that is known */
    float img[3][kGradRows];   /* OUT: the pixel */
#pragma unroll
    for (int j = 0; j < kGradRows; j++) {
        /* threads outside the frame load the pixel at its edge */
        const size_t row = (size_t)min(r0 + j, H - 1) * W;
        src[j] = (srcp + row)[lcol];
#pragma unroll
        for (int ch = 0; ch < 3; ch++)
            g[ch][j] = (gin + ch * fplane + row)[lcol];
    }
#pragma unroll
    for (int j = 0; j < kGradRows; j++)
        if (!(col < W && r0 + j < H))
            src[j] = INT32_MIN;
    __syncthreads();
    /* the sky term cancels where gradients of both signs meet: f64 keeps its
     * sum as exact as the gradients.  Its channels are weighted once per
     * thread: an all-sky 3840 x 2160 step without outputs 50 -> 32 us */
    double sky_acc = 0.0, loss_sum = 0.0, sky[3] = {0.0, 0.0, 0.0};
    /* one pixel of the fused step: its loss term and g = 2 (px - target) */
    auto pixel = [&](int j, const float px[3], float (&gd)[3]) {
#pragma unroll
        for (int ch = 0; ch < 3; ch++) {
            const float d = px[ch] - g[ch][j];
            gd[ch] = 2.0f * d;
            if constexpr (OUT) {
                img[ch][j] = px[ch];
                g[ch][j] = gd[ch];
            }
            /* the product is exact in f64 */
            loss_sum = __builtin_fma((double)d, (double)d, loss_sum);
        }
    };
    uint32_t starts = 0u;      /* rows where a run of a visible sample starts */
#pragma unroll
    for (int j = 0; j < kGradRows; j++) {
        const int32_t k = src[j];
        if (k >= 0 && (j == 0 || src[j - 1] != k))
            starts |= 1u << j;
        if (k < 0 && k != INT32_MIN) {
            float gd[3] = {g[0][j], g[1][j], g[2][j]};
            if constexpr (FWD) {
                const float px[3] = {sky_base(0) * a.sky_scale, sky_base(1) * a.sky_scale,
                                     sky_base(2) * a.sky_scale};
                pixel(j, px, gd);
            }
#pragma unroll
            for (int ch = 0; ch < 3; ch++)
                sky[ch] += (double)gd[ch];
        }
    }
#pragma unroll
    for (int ch = 0; ch < 3; ch++)
        sky_acc += sky[ch] * (double)sky_base(ch);
    while (__ballot(starts != 0u)) {
        float val[4][3];
        uint32_t key[4] = {kNoKey, kNoKey, kNoKey, kNoKey};
#pragma unroll
        for (int t = 0; t < 4; t++)
            val[t][0] = val[t][1] = val[t][2] = 0.0f;
        if (starts) {
            const int first = __builtin_ctz(starts);
            starts &= starts - 1u;
            int32_t k = src[0];
#pragma unroll
            for (int j = 1; j < kGradRows; j++)
                k = j == first ? src[j] : k;
            SampleEval e;
            sample_eval<P2, TAME>(a, k, col, plane, e);
            float run[3] = {0.0f, 0.0f, 0.0f};
            bool in = false;
#pragma unroll
            for (int j = 0; j < kGradRows; j++) {
                in = j == first || (in && src[j] == k);
                if (in) {
                    float gd[3] = {g[0][j], g[1][j], g[2][j]};
                    if constexpr (FWD)
                        pixel(j, e.px, gd);
#pragma unroll
                    for (int ch = 0; ch < 3; ch++)
                        run[ch] += gd[ch];
                }
            }
            sample_grad(a, e, run, key, val);
        }
        const bool last = segment_sum_quad(key, val);
#pragma unroll
        for (int t = 0; t < 4; t++) {
            bool inserted = false;
            if (last && key[t] != kNoKey)
                inserted = table_add<kGradCap>(keys, vals, &fill, a.gcp, plane, key[t], val[t]);
            /* the slot count is kept per wave, not per insertion: one
             * LDS atomic instead of one per inserting lane */
            const uint64_t ins = __ballot(inserted);
            if (ins && (threadIdx.x & 63) == 0)
                atomicAdd(&fill, (uint32_t)__popcll(ins));
        }
    }
    if constexpr (OUT) {
#pragma unroll
        for (int j = 0; j < kGradRows; j++) {
            const size_t row = (size_t)(r0 + j) * W;
            if (src[j] != INT32_MIN) {
#pragma unroll
                for (int ch = 0; ch < 3; ch++) {
                    if (a.img)
                        ((FS_GLOBAL float *)a.img + ch * fplane + row)[lcol] = img[ch][j];
                    if (a.gout)
                        ((FS_GLOBAL float *)a.gout + ch * fplane + row)[lcol] = g[ch][j];
                }
            }
        }
    }
    /* per-workgroup partials, summed in a fixed order by the next launch */
    __shared__ double wsky[kGradThreads / 64];
    __shared__ double wloss[kGradThreads / 64];
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        sky_acc += __shfl_xor(sky_acc, off);
        if (FWD)
            loss_sum += __shfl_xor(loss_sum, off);
    }
    if ((threadIdx.x & 63) == 0) {
        wsky[threadIdx.x >> 6] = sky_acc;
        if (FWD)
            wloss[threadIdx.x >> 6] = loss_sum;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        const int32_t blk = blockIdx.y * gridDim.x + blockIdx.x;
        double t = 0.0, tl = 0.0;
        for (int w = 0; w < kGradThreads / 64; w++) {
            t += wsky[w];
            if (FWD)
                tl += wloss[w];
        }
        if (FWD) {
            a.sky_part[blk] = t;
            a.partials[blk] = tl;
        } else {
            a.partials[blk] = t;
        }
    }
    for (int32_t i = threadIdx.x; i < kGradCap; i += kGradThreads) {
        const uint32_t key = keys[i];
        if (key == kNoKey)
            continue;
#pragma unroll
        for (int ch = 0; ch < 3; ch++) {
            const float v = (float)vals[ch * kGradCap + i];
            if (v != 0.0f)
                unsafeAtomicAdd(&a.gcp[ch * plane + key], v);
        }
    }
}

/* The fused step's two sums: its loss partials into *loss and its sky
 * partials into *gsky (= or +=), each in block_sum_partials' order (so
 * bit-identical to two calls of it), the two arrays' loads, shuffles and
 * final adds interleaved so that their latencies overlap. */
__global__ __launch_bounds__(1024) void k_sum_step(const double *__restrict__ loss_part,
                                                   const double *__restrict__ sky_part, int32_t n,
                                                   float *__restrict__ loss, int32_t loss_acc,
                                                   float *__restrict__ gsky, int32_t sky_acc)
{
    constexpr int NT = 1024;
    __shared__ double wsum[2][NT / 64];
    double a = 0.0, b = 0.0;
    for (int32_t base = 0; base < n; base += 8 * NT) {
        double va[8], vb[8];
#pragma unroll
        for (int u = 0; u < 8; u++) {
            const int32_t i = base + u * NT + (int32_t)threadIdx.x;
            va[u] = i < n ? loss_part[i] : 0.0;
            vb[u] = i < n ? sky_part[i] : 0.0;
        }
#pragma unroll
        for (int u = 0; u < 8; u++) {
            a += va[u];
            b += vb[u];
        }
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        a += __shfl_xor(a, off);
        b += __shfl_xor(b, off);
    }
    if ((threadIdx.x & 63) == 0) {
        wsum[0][threadIdx.x >> 6] = a;
        wsum[1][threadIdx.x >> 6] = b;
    }
    __syncthreads();
    if (threadIdx.x == 0 || threadIdx.x == 64) {
        const int k = threadIdx.x >> 6;
        double t = 0.0;
        for (int w = 0; w < NT / 64; w++)
            t += wsum[k][w];
        float *dst = k ? gsky : loss;
        *dst = (float)((k ? sky_acc : loss_acc) ? (double)*dst + t : t);
    }
}

/* L2 loss of the fitting harness: g = 2 * (img - target) and one partial
 * sum((img - target)^2) per workgroup. */
__global__ __launch_bounds__(256) void k_l2_loss(const float *__restrict__ img,
                                                 const float *__restrict__ tgt, size_t n,
                                                 float *__restrict__ g, float *__restrict__ part)
{
    __shared__ float wpart[4];
    float acc = 0.0f;
    const size_t stride = (size_t)gridDim.x * blockDim.x;
    const size_t n4 = n / 4;
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n4; i += stride) {
        float4 a = ((const float4 *)img)[i], b = ((const float4 *)tgt)[i];
        float4 d = make_float4(a.x - b.x, a.y - b.y, a.z - b.z, a.w - b.w);
        ((float4 *)g)[i] = make_float4(2.0f * d.x, 2.0f * d.y, 2.0f * d.z, 2.0f * d.w);
        acc += ((d.x * d.x) + (d.y * d.y)) + ((d.z * d.z) + (d.w * d.w));
    }
    for (size_t i = n4 * 4 + (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) {
        float d = img[i] - tgt[i];
        g[i] = 2.0f * d;
        acc += d * d;
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1)
        acc += __shfl_xor(acc, off);
    if ((threadIdx.x & 63) == 0)
        wpart[threadIdx.x >> 6] = acc;
    __syncthreads();
    if (threadIdx.x == 0)
        part[blockIdx.x] = (wpart[0] + wpart[1]) + (wpart[2] + wpart[3]);
}

/* One Adam step (no weight decay, bias-corrected moments) on n f32
 * parameters, then the parameters clamped to [lo, hi]: the fitting loop's
 * optimizer step and its projection back into the relaxation's domain in
 * one pass over parameter, gradient and moments (float4 where aligned).
 *   m = b1 m + (1 - b1) g,  v = b2 v + (1 - b2) g^2,
 *   p = clamp(p - (lr / (1 - b1^t)) m / (sqrt(v) / sqrt(1 - b2^t) + eps)) */
struct AdamArgs {
    float lr_t;          /* lr / (1 - b1^t) */
    float rbc2;          /* 1 / sqrt(1 - b2^t) */
    float b1, b2, omb1, omb2, eps, lo, hi;   /* omb = 1 - b, rounded once from double */
};

__device__ __forceinline__ float adam_one(float &p, float g, float &m, float &v,
                                          const AdamArgs &c)
{
    m = (c.b1 * m) + (c.omb1 * g);
    v = (c.b2 * v) + (c.omb2 * (g * g));
    /* the hardware sqrt and reciprocal (within an ulp or two): an
     * optimizer step has no bit-exact counterpart, and the correctly
     * rounded sequences would make this memory-bound pass VALU-bound */
    const float denom = (__builtin_amdgcn_sqrtf(v) * c.rbc2) + c.eps;
    p = fminf(fmaxf(p - (c.lr_t * (m * __builtin_amdgcn_rcpf(denom))), c.lo), c.hi);
    return p;
}

/* FIRST: the moments are zero and are not read (a fit's first step needs no
 * zeroed moments then; 12 of the pass's 28 bytes a parameter are its stores,
 * 8 the moments' loads: 4096^2 planes 237 -> 157 us, and two 33 us fills). */
template <bool FIRST>
__global__ __launch_bounds__(256) void k_adam(float *__restrict__ p, const float *__restrict__ g,
                                              float *__restrict__ m, float *__restrict__ v,
                                              size_t n, AdamArgs c)
{
    const float4 zero = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    const size_t stride = (size_t)gridDim.x * blockDim.x;
    const size_t n4 = n / 4;
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n4; i += stride) {
        float4 pp = ((float4 *)p)[i];
        float4 mm = FIRST ? zero : ((float4 *)m)[i], vv = FIRST ? zero : ((float4 *)v)[i];
        const float4 gg = ((const float4 *)g)[i];
        adam_one(pp.x, gg.x, mm.x, vv.x, c);
        adam_one(pp.y, gg.y, mm.y, vv.y, c);
        adam_one(pp.z, gg.z, mm.z, vv.z, c);
        adam_one(pp.w, gg.w, mm.w, vv.w, c);
        ((float4 *)p)[i] = pp;
        ((float4 *)m)[i] = mm;
        ((float4 *)v)[i] = vv;
    }
    for (size_t i = n4 * 4 + (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) {
        float pp = p[i], mm = FIRST ? 0.0f : m[i], vv = FIRST ? 0.0f : v[i];
        adam_one(pp, g[i], mm, vv, c);
        p[i] = pp;
        m[i] = mm;
        v[i] = vv;
    }
}

template <typename T>
__global__ __launch_bounds__(1024) void k_sum_partials(const T *__restrict__ part, int32_t n,
                                                       float *__restrict__ dst, int32_t accumulate)
{
    block_sum_partials<1024>(part, n, dst, accumulate);
}

/* A frame of one colour (the degenerate frames of the state's #math mode). */
__global__ void k_fill_u32(uint32_t *__restrict__ p, size_t n, uint32_t v)
{
    size_t stride = (size_t)gridDim.x * blockDim.x;
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride)
        p[i] = v;
}

/* Zero fill (a kernel, not a memset node, so that callers may capture it). */
__global__ void k_zero_f32(float *__restrict__ p, size_t n)
{
    size_t stride = (size_t)gridDim.x * blockDim.x;
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride)
        p[i] = 0.0f;
}

inline bool pow2(int32_t v)
{
    return v > 0 && (v & (v - 1)) == 0;
}

/* Host: u32.f32(sqrtf(t) * 255) for the f32 with bits tb (sqrtf is
 * correctly rounded, no contraction: this file is built with
 * -ffp-contract=off). */
uint32_t q_exact(uint32_t tb)
{
    float t;
    memcpy(&t, &tb, sizeof t);
    return (uint32_t)(sqrtf(t) * 255.0f);
}

/* The bucket table of mix_q (see kQLo): base byte per bucket and the offset
 * of its single step, found by bisection. */
void qtab_build(uint32_t *qt)
{
    for (int i = 0; i < kQBuckets; i++) {
        const uint32_t lo = kQLo + ((uint32_t)i << 16);
        const uint32_t hi = std::min(lo + 0xFFFFu, 0x3F800000u);
        const uint32_t base = q_exact(lo);
        uint32_t step = 0x10000u;
        if (q_exact(hi) != base) {
            uint32_t a = lo, b = hi;          /* q(a) == base < q(b) */
            while (b - a > 1) {
                const uint32_t m = a + (b - a) / 2;
                if (q_exact(m) > base)
                    b = m;
                else
                    a = m;
            }
            step = b - lo;
        }
        qt[i] = (base << 17) + 0x20000u - step - ((uint32_t)i << 16);
    }
}

std::mutex g_init_mu;
bool g_init_done[64];
double *g_scratch_ptr[64];   /* device address of `scratch` on each device */

}  // namespace

/* The adjoint's kernel for a's planes and frame, with `rows` rows per
 * thread; OUT where an image is to be written. */
template <bool FWD, bool OUT>
static void launch_diff_grad(const DiffArgs &a, int32_t rows, dim3 grid, hipStream_t s)
{
    constexpr int L = kGradRowsLow, T = kGradRowsTall;
    void (*const kern[2][2][2])(DiffArgs) = {
        {{k_diff_grad<false, false, FWD, OUT, L>, k_diff_grad<false, false, FWD, OUT, T>},
         {k_diff_grad<false, true, FWD, OUT, L>, k_diff_grad<false, true, FWD, OUT, T>}},
        {{k_diff_grad<true, false, FWD, OUT, L>, k_diff_grad<true, false, FWD, OUT, T>},
         {k_diff_grad<true, true, FWD, OUT, L>, k_diff_grad<true, true, FWD, OUT, T>}}};
    hipLaunchKernelGGL(kern[pow2(a.hc) && pow2(a.wc)][a.f.tame != 0][rows != kGradRowsLow], grid,
                       dim3(kGradThreads), 0, s, a);
}

/* render2 by the workgroups that a frame has: up to one per CU, 32 rows and
 * all the registers the kernel asks for; more than that, two on a CU (64
 * registers, which spill a little: 1920 x 1080 67 us instead of 75 per call,
 * but 160 x 120 41 instead of 39); and 128 rows, which share the heights,
 * where these still give each CU three and so fill a second round half
 * (3840 x 2160: 149 us instead of 164, with a camera on the ground 93 instead of
 * 107; 2900 x 1500, 2.2 per CU: 108 instead of 105). */
template <int HBITS, bool HP2>
static int launch_render2(const Render2Args &a, hipStream_t s)
{
    const uint32_t tiles = (uint32_t)(a.cols + 63) / 64;
    const int64_t low = (int64_t)tiles * ((a.rows + 31) / 32);
    const int64_t tall = (int64_t)tiles * ((a.rows + 127) / 128);
    const int rows = tall >= 3 * cu_count() ? 128 : 32;
    void (*kern)(Render2Args) = low <= cu_count() ? k_render2<HBITS, HP2, 32, 4, false>
                                : rows == 32 ? k_render2<HBITS, HP2, 32, 8, true>
                                             : k_render2<HBITS, HP2, 128, 8, true>;
    hipLaunchKernelGGL(kern, dim3(tiles, (a.rows + rows - 1) / rows), dim3(1024), 0, s, a);
    return hipGetLastError();
}

extern "C" {

int fsk_device_init(void)
{
    static uint32_t host_qt[kQBuckets];
    static bool built = false;
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess)
        return e;
    if (dev < 0 || dev >= 64)
        return hipErrorInvalidDevice;
    std::lock_guard<std::mutex> lock(g_init_mu);
    if (!built) {
        qtab_build(host_qt);
        built = true;
    }
    if (!g_init_done[dev]) {
        e = hipMemcpyToSymbol(HIP_SYMBOL(g_qtab), host_qt, sizeof host_qt, 0,
                              hipMemcpyHostToDevice);
        if (e != hipSuccess)
            return e;
        /* this device's copy of the scratch array: its address, not the
         * array's host-side name, is what kernels and copies may use */
        void *p = nullptr;
        e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess)
            return e;
        g_scratch_ptr[dev] = (double *)p;
        g_init_done[dev] = true;
    }
    return hipSuccess;
}

double *fsk_scratch(int32_t device)
{
    if (device < 0 || device >= 64)
        return nullptr;
    std::lock_guard<std::mutex> lock(g_init_mu);
    return g_init_done[device] ? g_scratch_ptr[device] : nullptr;
}

/* The automatic shape of a batch, by the tiles it would have (us per batch
 * of views of 320 x 240 to 1920 x 1080, 1024 to 4096 slices, as 8x1 / 4x1 /
 * 8x2): 4-column tiles while each finds a CU (2 views: 30 / 27 / 34), else
 * two 512-thread tiles per CU, whose stalls overlap (4 views: 76 / 93 / 70;
 * 40: 442 / 621 / 340; 256: 2690 / 3805 / 2180), where two fit in LDS. */
void fsk_batch_shape(int32_t max_rows, int64_t tiles4, int64_t tiles8, fsk_tuning *t)
{
    if (t->tc || t->wg_per_cu || t->chunk)
        return;
    if (tiles4 <= cu_count())
        t->tc = 4;
    else if (tiles8 > cu_count() &&
             2 * (render_lds_bytes(8, 512, max_rows, 512) + kStaticLds) <= lds_per_cu())
        t->wg_per_cu = 2;
}

int32_t fsk_tile_columns(int32_t max_rows, const fsk_tuning *t)
{
    return resolve_shape(max_rows, *t).tc;
}

int32_t fsk_batch_grid(int32_t max_rows, const fsk_tuning *t)
{
    Shape sh = resolve_shape(max_rows, *t);
    return cu_count() * sh.wg;
}

void fsk_default_tuning(fsk_tuning *t)
{
    const char *e = getenv("FSX_RENDER_TC");
    t->tc = e ? atoi(e) : 0;
    e = getenv("FSX_RENDER_WG_PER_CU");
    t->wg_per_cu = e ? atoi(e) : 0;
    e = getenv("FSX_RENDER_CHUNK");
    t->chunk = e ? atoi(e) : 0;
}

void fsk_batch_counters_init(uint32_t *counters, int32_t grid, int32_t nqueues)
{
    for (int32_t q = 0; q < nqueues; q++)
        counters[q * FSK_COUNTER_STRIDE] =
            batch_first_claim((uint32_t)grid, (uint32_t)q, (uint32_t)nqueues);
    counters[nqueues * FSK_COUNTER_STRIDE] = 0u;
}

int fsk_batch_run(const fsk_batch *b, hipStream_t s)
{
    if (b->max_rows > kMaxRows || b->nqueues < 1 || b->nqueues > 64)
        return hipErrorInvalidValue;
    if (b->hbits == 8)
        return b->pow2 ? launch_batch<8, true, true>(b, s) : launch_batch<8, false, false>(b, s);
    return b->pow2 ? launch_batch<16, true, true>(b, s) : launch_batch<16, false, false>(b, s);
}

static int32_t map_side(const fsk_map *m)
{
    return std::max(std::max(m->hrows, m->hcols), std::max(m->crows, m->ccols));
}

int fsk_render_slices_clear(const fsk_map *m, const fsk_frame *f, const fsk_tuning *t,
                            int32_t *d_src, int64_t pitch, float *d_zero, size_t zero_n,
                            int32_t *cleared, hipStream_t s)
{
    if (cleared)
        *cleared = 0;
    if (f->rows <= 0 || f->cols <= 0)
        return hipSuccess;
    RenderArgs a;
    a.m = *m;
    fsk_map_recips(&a.m);
    a.f = *f;
    a.f.tame = fsk_tame_level(f, map_side(m));
    if (a.f.n < 0)
        a.f.n = 0;
    a.out = (uint32_t *)d_src;
    a.pitch = pitch;
    a.ntiles = 0;
    a.chunk_max = kChunk;
    a.band_rows = 0;
    a.zero = nullptr;
    a.zero_n4 = 0;
    a.nzero = 0;
    /* float4 stores only */
    const bool z = d_zero && cleared && (((uintptr_t)d_zero) & 15u) == 0 && zero_n % 4 == 0;
    a.zero = z ? (float4 *)d_zero : nullptr;
    a.zero_n4 = z ? zero_n / 4 : 0;
    a.nzero = 0;
    int32_t nz = 0;
    bool hp2 = pow2(m->hrows) && pow2(m->hcols);
    hipError_t e;
    if (m->hbits == 8)
        e = hp2 ? launch_render<8, true, false, kOutSlice>(a, *t, s, &nz)
                : launch_render<8, false, false, kOutSlice>(a, *t, s, &nz);
    else
        e = hp2 ? launch_render<16, true, false, kOutSlice>(a, *t, s, &nz)
                : launch_render<16, false, false, kOutSlice>(a, *t, s, &nz);
    if (e == hipSuccess && cleared)
        *cleared = nz > 0;
    return e;
}

int fsk_render_slices(const fsk_map *m, const fsk_frame *f, const fsk_tuning *t, int32_t *d_src,
                      int64_t pitch, hipStream_t s)
{
    return fsk_render_slices_clear(m, f, t, d_src, pitch, nullptr, 0, nullptr, s);
}

/* Rows per thread of the adjoint on a w x h frame. */
static int32_t grad_rows(int32_t w, int32_t h)
{
    return (int64_t)w * (int64_t)h >= kGradTallPixels ? kGradRowsTall : kGradRowsLow;
}

static DiffArgs diff_args(const fsk_frame *f, const float *cp, const float *sf, int32_t hc,
                          int32_t wc, const int32_t *src)
{
    DiffArgs a;
    a.f = *f;
    a.f.tame = fsk_tame_level(f, std::max(hc, wc));
    a.rhc = fsk_wrap_recip(hc);
    a.rwc = fsk_wrap_recip(wc);
    a.cp = cp;
    a.sf = sf;
    a.hc = hc;
    a.wc = wc;
    a.sky_scale = 0.0f;
    a.src = src;
    a.gimg = nullptr;
    a.img = nullptr;
    a.gcp = nullptr;
    a.gsky = nullptr;
    a.partials = nullptr;
    a.tgt = nullptr;
    a.gout = nullptr;
    a.sky_part = nullptr;
    return a;
}

int fsk_render_nearest(const fsk_map *m, const fsk_frame *f, const fsk_tuning *t,
                       uint32_t *d_out, int64_t pitch, hipStream_t s)
{
    if (f->rows <= 0 || f->cols <= 0)
        return hipSuccess;
    RenderArgs a;
    a.m = *m;
    fsk_map_recips(&a.m);
    a.f = *f;
    a.f.tame = fsk_tame_level(f, map_side(m));
    if (a.f.n < 0)
        a.f.n = 0;
    a.out = d_out;
    a.pitch = pitch;
    a.ntiles = 0;
    a.chunk_max = kChunk;
    a.band_rows = 0;
    a.zero = nullptr;
    a.zero_n4 = 0;
    a.nzero = 0;
    return pow2(m->hrows) && pow2(m->hcols) ? launch_render<8, true, false, kOutNearest>(a, *t, s)
                                            : launch_render<8, false, false, kOutNearest>(a, *t, s);
}

int fsk_diff_color(const fsk_frame *f, const float *d_cp, const float *d_sf, int32_t hc,
                   int32_t wc, float sky_scale, const int32_t *d_src, float *d_img, hipStream_t s)
{
    if (f->rows <= 0 || f->cols <= 0)
        return hipSuccess;
    DiffArgs a = diff_args(f, d_cp, d_sf, hc, wc, d_src);
    a.sky_scale = sky_scale;
    a.img = d_img;
    dim3 grid((f->cols + 63) / 64, (f->rows + 3) / 4);
    const bool p2 = pow2(hc) && pow2(wc), tame = a.f.tame != 0;
    void (*kern)(DiffArgs) = p2 ? (tame ? k_diff_color<true, true> : k_diff_color<true, false>)
                                : (tame ? k_diff_color<false, true> : k_diff_color<false, false>);
    hipLaunchKernelGGL(kern, grid, dim3(256), 0, s, a);
    return hipGetLastError();
}

int fsk_l2_loss(const float *d_img, const float *d_tgt, size_t n, float *d_g, float *d_loss,
                int32_t accumulate, double *d_partials, int32_t n_partials, hipStream_t s)
{
    /* one f32 per workgroup */
    float *part = (float *)d_partials;
    size_t blocks = (n / 4 + 255) / 256;
    if (blocks > 4096)
        blocks = 4096;
    if (blocks == 0)
        blocks = 1;
    if ((int64_t)blocks > n_partials)
        return hipErrorInvalidValue;
    hipLaunchKernelGGL(k_l2_loss, dim3((unsigned)blocks), dim3(256), 0, s, d_img, d_tgt, n, d_g,
                       part);
    hipLaunchKernelGGL(k_sum_partials<float>, dim3(1), dim3(1024), 0, s, part, (int32_t)blocks,
                       d_loss, accumulate);
    return hipGetLastError();
}

int fsk_adam(float *d_p, const float *d_g, float *d_m, float *d_v, size_t n, double lr,
             double beta1, double beta2, double eps, int32_t step, int32_t first, float lo,
             float hi, hipStream_t s)
{
    if (n == 0)
        return hipSuccess;
    /* the hyper-parameters' derived constants in double, each rounded to
     * f32 once */
    AdamArgs c;
    c.lr_t = (float)(lr / (1.0 - pow(beta1, (double)step)));
    c.rbc2 = (float)(1.0 / sqrt(1.0 - pow(beta2, (double)step)));
    c.b1 = (float)beta1;
    c.b2 = (float)beta2;
    c.omb1 = (float)(1.0 - beta1);
    c.omb2 = (float)(1.0 - beta2);
    c.eps = (float)eps;
    c.lo = lo;
    c.hi = hi;
    size_t blocks = (n / 4 + 255) / 256;
    if (blocks > 16384)
        blocks = 16384;
    if (blocks == 0)
        blocks = 1;
    hipLaunchKernelGGL(first ? k_adam<true> : k_adam<false>, dim3((unsigned)blocks), dim3(256), 0, s,
                       d_p, d_g, d_m, d_v, n, c);
    return hipGetLastError();
}

int fsk_fill_u32(uint32_t *d_p, size_t n, uint32_t v, hipStream_t s)
{
    if (n == 0)
        return hipSuccess;
    size_t blocks = (n + 255) / 256;
    if (blocks > 8192)
        blocks = 8192;
    hipLaunchKernelGGL(k_fill_u32, dim3((unsigned)blocks), dim3(256), 0, s, d_p, n, v);
    return hipGetLastError();
}

int fsk_zero_f32(float *d_p, size_t n, hipStream_t s)
{
    if (n == 0)
        return hipSuccess;
    size_t blocks = (n + 255) / 256;
    if (blocks > 8192)
        blocks = 8192;
    hipLaunchKernelGGL(k_zero_f32, dim3((unsigned)blocks), dim3(256), 0, s, d_p, n);
    return hipGetLastError();
}

int fsk_diff_grad(const fsk_frame *f, const float *d_cp, const float *d_sf, int32_t hc,
                  int32_t wc, const int32_t *d_src, const float *d_gimg, float *d_gcp,
                  float *d_gsky, int32_t sky_accumulate, double *d_partials, int32_t n_partials,
                  hipStream_t s)
{
    if (f->rows <= 0 || f->cols <= 0)
        return hipSuccess;
    DiffArgs a = diff_args(f, d_cp, d_sf, hc, wc, d_src);
    a.gimg = d_gimg;
    a.gcp = d_gcp;
    a.gsky = d_gsky;
    a.partials = d_partials;
    const int32_t rows = grad_rows(f->cols, f->rows), br = kGradThreads / 64 * rows;
    dim3 grid((f->cols + 63) / 64, (f->rows + br - 1) / br);
    if ((int64_t)grid.x * grid.y > n_partials)
        return hipErrorInvalidValue;
    launch_diff_grad<false, false>(a, rows, grid, s);
    hipLaunchKernelGGL(k_sum_partials<double>, dim3(1), dim3(1024), 0, s, d_partials,
                       (int32_t)(grid.x * grid.y), d_gsky, sky_accumulate);
    return hipGetLastError();
}

int fsk_diff_step_l2(const fsk_frame *f, const float *d_cp, const float *d_sf, int32_t hc,
                     int32_t wc, float sky_scale, const int32_t *d_src, const float *d_tgt,
                     float *d_img, float *d_g, float *d_gcp, float *d_gsky,
                     int32_t sky_accumulate, float *d_loss, int32_t loss_accumulate,
                     double *d_loss_part, double *d_sky_part, int32_t n_partials, hipStream_t s)
{
    if (f->rows <= 0 || f->cols <= 0)
        return hipSuccess;
    DiffArgs a = diff_args(f, d_cp, d_sf, hc, wc, d_src);
    a.sky_scale = sky_scale;
    a.tgt = d_tgt;
    a.img = d_img;
    a.gout = d_g;
    a.gcp = d_gcp;
    a.gsky = d_gsky;
    a.partials = d_loss_part;
    a.sky_part = d_sky_part;
    const int32_t rows = grad_rows(f->cols, f->rows), br = kGradThreads / 64 * rows;
    dim3 grid((f->cols + 63) / 64, (f->rows + br - 1) / br);
    const int64_t nb = (int64_t)grid.x * grid.y;
    if (nb > n_partials)
        return hipErrorInvalidValue;
    if (d_img || d_g)
        launch_diff_grad<true, true>(a, rows, grid, s);
    else
        launch_diff_grad<true, false>(a, rows, grid, s);
    hipLaunchKernelGGL(k_sum_step, dim3(1), dim3(1024), 0, s, d_loss_part, d_sky_part,
                       (int32_t)nb, d_loss, loss_accumulate, d_gsky, sky_accumulate);
    return hipGetLastError();
}

int fsk_render2(const fsk_map *m, const fsk_frame *f, const float *d_cs, const float *d_sn,
                const uint32_t *d_color, int32_t n, uint32_t *d_out, int64_t pitch, hipStream_t s)
{
    if (f->rows <= 0 || f->cols <= 0)
        return hipSuccess;
    Render2Args a;
    a.m = *m;
    a.color = d_color;
    a.cs = d_cs;
    a.sn = d_sn;
    a.out = d_out;
    a.pitch = pitch;
    a.cam_x = f->cam_x;
    a.cam_y = f->cam_y;
    a.cam_h = f->cam_h;
    a.horizon = f->horizon;
    a.n = n;
    a.rows = f->rows;
    a.cols = f->cols;
    const bool p2 = pow2(m->hrows) && pow2(m->hcols);
    if (m->hbits == 8)
        return p2 ? launch_render2<8, true>(a, s) : launch_render2<8, false>(a, s);
    return p2 ? launch_render2<16, true>(a, s) : launch_render2<16, false>(a, s);
}

float fsk_wrap_recip(int32_t m)
{
    /* at most (1 - 2^-24) / m, so that its product with v, rounded, is not
     * above v / m, and at least (1 - 2^-21.6) / m (the least over the sides up
     * to 2^20 is (1 - 2^-21.68) / m, at 1047899) */
    const float r = 1.0f / (float)m;
    return nextafterf(nextafterf(r, 0.0f), 0.0f);
}

void fsk_map_recips(fsk_map *m)
{
    m->rhrows = fsk_wrap_recip(m->hrows);
    m->rhcols = fsk_wrap_recip(m->hcols);
    m->rcrows = m->crows > 0 ? fsk_wrap_recip(m->crows) : 0.0f;
    m->rccols = m->ccols > 0 ? fsk_wrap_recip(m->ccols) : 0.0f;
}

/* The frame's largest sample coordinate where its scalars and rows are
 * tame, else infinity. */
static double tame_extent(const fsk_frame *f)
{
    const float v[] = {f->cam_x, f->cam_y, f->cam_h, f->horizon, f->Lx, f->Ly,
                       f->Rx,    f->Ry,    f->d,     f->z0,      f->scale, f->fw};
    for (float x : v)
        if (!std::isfinite(x))
            return INFINITY;
    if (!(f->z0 > 0.0f) || !(f->d >= 0.0f) || !(f->scale > 0.0f) || !(f->fw >= 1.0f) ||
        f->n <= 0)
        return INFINITY;
    /* z_k = (k/2)(2 z0 + (k-1) d) is non-decreasing from z_1 = z0 (every
     * f32 step of get_zs' term is monotone for z0 > 0, d >= 0), so
     * inv_z <= scale / z0; a 1e-3 margin covers the roundings */
    const double n = (double)f->n, margin = 1.001;
    const double zmax = (n / 2.0) * (2.0 * (double)f->z0 + (n - 1.0) * (double)f->d) * margin;
    const double izmax = (double)f->scale / (double)f->z0 * margin;
    /* x = (lx + cam_x) + col * (rx - lx) / w over columns up to w + 7 (the
     * last tile's lanes past the frame) */
    const double span = ((double)f->fw + 8.0) / (double)f->fw;
    const double ax = std::fabs((double)f->Lx), bx = std::fabs((double)f->Rx);
    const double ay = std::fabs((double)f->Ly), by = std::fabs((double)f->Ry);
    const double xmax = (std::fabs((double)f->cam_x) + (ax + (ax + bx) * span) * zmax) * margin;
    const double ymax = (std::fabs((double)f->cam_y) + (ay + (ay + by) * span) * zmax) * margin;
    const double relmax =
        ((std::fabs((double)f->cam_h) + 65536.0) * izmax + std::fabs((double)f->horizon)) * margin;
    /* slice depths inside [2^-100, 2^100], where the table's reciprocal
     * (rcp_rn) is exact */
    const bool zok = (double)f->z0 >= 0x1p-100 && zmax <= 0x1p100;
    return zok && relmax < 1073741824.0 ? std::max(xmax, ymax) : INFINITY;
}

int32_t fsk_tame_level(const fsk_frame *f, int32_t max_side)
{
    const double extent = tame_extent(f);
    return extent < 2097152.0 && max_side <= 1 << 20 ? FSK_TAME_MOD
           : extent < 4194304.0 ? FSK_TAME : 0;
}

int32_t fsk_frame_tame(const fsk_frame *f)
{
    return fsk_tame_level(f, INT32_MAX);
}

int32_t fsk_render_max_rows(void)
{
    return kMaxFrameRows;
}

int32_t fsk_batch_max_rows(void)
{
    return kMaxRows;
}

int32_t fsk_limit_block_rows(int32_t w, int32_t h)
{
    return (int64_t)w * (int64_t)h >= (int64_t)1 << 22 ? 32 : 16;
}

int fsk_selftest(int which, unsigned long long *d_bad, hipStream_t s)
{
    if (which < 0 || which > 8)
        return hipErrorInvalidValue;
    SelftestRecips recips;
    for (int i = 0; i < kNSelftestSides; i++)
        recips.rm[i] = fsk_wrap_recip(kSelftestSides[i]);
    hipLaunchKernelGGL(k_selftest, dim3(4096), dim3(256), 0, s, which, recips, d_bad);
    return hipGetLastError();
}

int fsk_render(const fsk_map *m, const fsk_frame *f, const fsk_tuning *t, uint32_t *d_out,
               int64_t pitch, hipStream_t s)
{
    if (f->rows <= 0 || f->cols <= 0)
        return hipSuccess;
    RenderArgs a;
    a.m = *m;
    fsk_map_recips(&a.m);
    a.f = *f;
    a.f.tame = fsk_tame_level(f, map_side(m));
    if (a.f.n < 0)
        a.f.n = 0;
    a.out = d_out;
    a.pitch = pitch;
    a.ntiles = 0;
    a.chunk_max = kChunk;
    a.band_rows = 0;
    a.zero = nullptr;
    a.zero_n4 = 0;
    a.nzero = 0;
    bool hp2 = pow2(m->hrows) && pow2(m->hcols);
    bool cp2 = pow2(m->crows) && pow2(m->ccols);
    hipError_t e;
    if (m->hbits == 8) {
        if (hp2 && cp2) e = launch_render<8, true, true>(a, *t, s);
        else if (hp2) e = launch_render<8, true, false>(a, *t, s);
        else if (cp2) e = launch_render<8, false, true>(a, *t, s);
        else e = launch_render<8, false, false>(a, *t, s);
    } else {
        if (hp2 && cp2) e = launch_render<16, true, true>(a, *t, s);
        else if (hp2) e = launch_render<16, true, false>(a, *t, s);
        else if (cp2) e = launch_render<16, false, true>(a, *t, s);
        else e = launch_render<16, false, false>(a, *t, s);
    }
    return e;
}

int fsk_height_quads(const int32_t *d_alt, int32_t rows, int32_t cols, int32_t hbits,
                     void *d_hq, uint16_t *d_hplain, uint32_t *d_hmax, hipStream_t s)
{
    dim3 grid((cols + 255) / 256, (rows + kQuadRows - 1) / kQuadRows);
    void (*kern)(const int32_t *, int32_t, int32_t, void *, uint16_t *) =
        hbits == 8 ? k_height_quads<8> : k_height_quads<16>;
    hipLaunchKernelGGL(kern, grid, dim3(256), 0, s, d_alt, rows, cols, d_hq, d_hplain);
    hipLaunchKernelGGL(k_height_max, dim3(FSK_HMAX_PARTS), dim3(1024), 0, s, d_hplain,
                       (size_t)rows * (size_t)cols, d_hmax);
    return hipGetLastError();
}

int fsk_shade(const uint16_t *d_hplain, const uint32_t *d_hmax, int32_t rows, int32_t cols,
              const uint32_t *d_color, const float sun[3], int32_t size, void *d_out,
              hipStream_t s)
{
    ShadeArgs a;
    a.hp = d_hplain;
    a.hmax = d_hmax;
    a.col = d_color;
    a.out = d_out;
    a.hrows = rows;
    a.hcols = cols;
    a.size = size;
    a.rrows = 1.0f / (float)rows;
    a.rcols = 1.0f / (float)cols;
    const float step_size = 4.0f;
    for (int32_t d = 0; d < kShadeSteps; d++) {
        const float t = (float)d * step_size;
        a.dx[d] = t * sun[0];
        a.dh[d] = t * sun[1];
        a.dy[d] = t * sun[2];
    }
    /* kWrapSmall's range: sides and grid up to 2^16 and offsets up to 1020 */
    const bool finite = std::isfinite(sun[0]) && std::isfinite(sun[1]) && std::isfinite(sun[2]) &&
                        std::fabs(sun[0]) <= 1.5f && std::fabs(sun[2]) <= 1.5f;
    const bool small = rows <= 65536 && cols <= 65536 && size <= 65536;
    const int w = !(finite && small) ? kWrapX86
                  : pow2(rows) && pow2(cols) ? kWrapPow2 : kWrapSmall;
    void (*kern)(ShadeArgs);
    if (d_color)
        kern = w == kWrapPow2 ? k_shade<kWrapPow2, false>
               : w == kWrapSmall ? k_shade<kWrapSmall, false> : k_shade<kWrapX86, false>;
    else
        kern = w == kWrapPow2 ? k_shade<kWrapPow2, true>
               : w == kWrapSmall ? k_shade<kWrapSmall, true> : k_shade<kWrapX86, true>;
    dim3 grid((size + 64 * kShadeTexels - 1) / (64 * kShadeTexels), (size + 3) / 4);
    hipLaunchKernelGGL(kern, grid, dim3(256), 0, s, a);
    return hipGetLastError();
}

int fsk_color_quads(const uint32_t *d_col, int32_t rows, int32_t cols, void *d_cq, hipStream_t s)
{
    dim3 grid((cols + 255) / 256, rows);
    hipLaunchKernelGGL(k_color_quads, grid, dim3(256), 0, s, d_col, rows, cols, (uint4 *)d_cq);
    return hipGetLastError();
}

}  // extern "C"
