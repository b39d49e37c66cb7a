/*
 * ktm_device.hip -- gfx950 kernels and the device half of the C ABI of the
 * Kirchhoff prestack time-migration engine.
 *
 * Kernels (every one replaces a loop of Kirchhoff.c's kirchhoff()):
 *   k_geometry      per-trace rotation / CMP / offset class   Kirchhoff.c:1296-1310
 *                   (k_geometry_segy: from the raw trace headers)
 *   k_segy_decode   raw SEG-Y records -> FP32 traces + header words,
 *                   Kirchhoff.c:1281-1290 (the prep kernels below decode
 *                   records themselves when ingesting a raw block)
 *   k_prep_ref      FP32 double integral + trange=2 taps       Kirchhoff.c:1312-1328,1391-1392
 *   k_prep_closed   same operator as a 3-tap filter (FP32), from FP32 or
 *                   BF16/FP16-stored traces              (exact rewrite of 1312-1392)
 *   k_quantize      BF16/FP16 storage with per-trace scale and sixth-order
 *                   error feedback
 *   k_migrate       the image loop, Kirchhoff.c:1332-1404: one workgroup owns a
 *                   tile of image columns (one wave per column, all ns samples
 *                   in registers), streams the traces of a block through LDS in
 *                   trace order and accumulates F(floor(dsr/dt)) per sample
 *   k_postfft<PostKtm>  derivative/fold + low-pass, Kirchhoff.c:1457-1479, as
 *                   an FP64 FFT convolution (ktm_postfft.h; beyond 4096
 *                   samples the FP64 matrix product of ktm_postmx.h); its
 *                   transpose k_postfft<PostImg> + k_poststack_adjoint_tail
 *   k_image_records image<job>.su trace records (headers + big-endian
 *                   samples), Kirchhoff.c:1437-1598
 *   k_demigrate     exact transpose of k_migrate (CLOSED prep)
 *   k_synth_*       seeded synthetic surveys
 *
 * Build flags: -ffp-contract=off (no implicit FMA: every product and sum
 * that the reference rounds separately is rounded separately here; FMAs are
 * written explicitly where intended) and the default correctly-rounded FP32
 * divide/sqrt; packed-FP32 ops are disabled.
 */
#include <hip/hip_runtime.h>
#include <rocprim/device/device_radix_sort.hpp>

#include <mutex>

#include <math.h>

#include <stdint.h>
#include <stdlib.h>
#include <string.h>

#include "ktm_internal.h"
#include "ktm_devmath.h"
#include "ktm_postmx.h"
#include "ktm_postfft.h"

#define KTM_WAVE 64
#define KTM_CUS 256         /* compute units of the chip */

/* ------------------------------------------------------------------------ */
/* plan                                                                      */
/* ------------------------------------------------------------------------ */
struct ktm_plan {
    ktm_config cfg;
    ktm_tables tb;
    int device;
    int64_t row;            /* prepared trace row (elements), multiple of 8, >= ns+1 */
    float *d_t2;
    int32_t *d_t1;
    float *d_colx, *d_coly;
    int32_t *d_velx, *d_vely;
    float *d_slab_cx, *d_slab_cy;
    float *d_slab_x2thr;
    float *d_vel2;          /* [nvel_il][nvel_xl][nsm], squared like Kirchhoff.c:617 */
    float *d_w;             /* [ns+2] CLOSED weights */
    double *d_hconv2;       /* [2 ns] post-stack kernel, h2[m] = h[m mod ns] */
    double *d_pf_g;         /* [N] FFT form of the post-stack kernel */
    double2 *d_pf_tw;       /* [N] twiddles */
    int pf_n;                /* points of the FFT form, 0: the direct product */
    float *d_stage;         /* FP32 filtered traces of a BF16/FP16 block */
    size_t stage_cap;       /* elements of d_stage */
    float *d_pix_v2, *d_pix_rs; /* per-pixel v^2 and RN(1/(v^2 dt^2)), built for demigration */
    /* demigration trace order: sort keys and indices (in, out) and the
     * radix sort's temporary storage, grown on demand */
    uint64_t *d_dm_keys;
    int32_t *d_dm_idx;
    void *d_dm_tmp;
    size_t dm_cap, dm_tmp_bytes;
    uint32_t *d_dm_amax;    /* bits of max |km| of the last demigration */
    unsigned long long *d_dm_sum; /* sums of a demigration whose columns are in parts */
    size_t dm_sum_cap;      /* words of d_dm_sum */
    int64_t dm_sum_ntr;     /* most traces of a call that asked for them */
    float *d_scratch;       /* this device's copy of `scratch` (ktm_migrate_block_static) */
    /* compensated migration of small images: partial images of parts 1..
     * parts_max-1 of a trace block, [part][km, fold, comp][image or region] */
    float *d_parts;
    int parts_max;
};

static int scratch_address(int dev, float **out);
static int parts_workspace(ktm_plan *p);

#define HIP_TRY(expr)                                  \
    do {                                               \
        hipError_t e_ = (expr);                        \
        if (e_ != hipSuccess) return KTM_ERR_DEVICE;   \
    } while (0)

/* ------------------------------------------------------------------------ */
/* per-trace geometry, Kirchhoff.c:1296-1310 (and Kirchhoff_GHTest1.c:       */
/* 1302-1315 when scale_xy > 0)                                              */
/* ------------------------------------------------------------------------ */
struct GeoArgs {
    double ox, oy, scale, oh, dh;
    float sinA, cosA;
};

__device__ __forceinline__ void rotate_point(const GeoArgs &g, uint32_t hx, uint32_t hy,
                                             float &xt, float &yt)
{
    if (g.scale == 0.0) {
        /* htonl() gives uint32_t; minus the double origin; into an int */
        const int i = (int)((double)hx - g.ox);
        const int j = (int)((double)hy - g.oy);
        xt = g.cosA * (float)i + g.sinA * (float)j;
        yt = -g.sinA * (float)i + g.cosA * (float)j;
    } else {
        const int i = (int)((double)hx - g.ox / g.scale);
        const int j = (int)((double)hy - g.oy / g.scale);
        xt = (float)((double)(g.cosA * (float)i) * g.scale + (double)(g.sinA * (float)j) * g.scale);
        yt = (float)((double)(-g.sinA * (float)i) * g.scale + (double)(g.cosA * (float)j) * g.scale);
    }
}

__device__ __forceinline__ ktm_trace_geom trace_geometry(const GeoArgs &g, const int32_t *c)
{
    ktm_trace_geom r;
    rotate_point(g, (uint32_t)c[0], (uint32_t)c[1], r.sxt, r.syt);
    rotate_point(g, (uint32_t)c[2], (uint32_t)c[3], r.gxt, r.gyt);
    const float ex = r.sxt - r.gxt, ey = r.syt - r.gyt;
    const float h2 = (float)(0.25 * (double)(ex * ex + ey * ey));
    r.cmpx = (float)(0.5 * (double)(r.sxt + r.gxt));
    r.cmpy = (float)(0.5 * (double)(r.syt + r.gyt));
    r.off = (int)floor((2.0 * sqrt((double)h2) - g.oh) / g.dh);
    r.scale = 1.0f;
    return r;
}

__global__ void k_geometry(GeoArgs g, const int32_t *__restrict__ coords, int64_t ntr,
                           ktm_trace_geom *__restrict__ geom)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= ntr) return;
    geom[i] = trace_geometry(g, coords + 4 * i);
}

/* The same from raw SEG-Y trace records: header words 18-21 (sx, sy, gx,
 * gy; bytes 73-88, big-endian, Kirchhoff.c:1297,1302) of each record of
 * rec_words 4-byte words; the header words also go to coords if given. */
__global__ void k_geometry_segy(GeoArgs g, const uint32_t *__restrict__ raw, int64_t rec_words,
                                int64_t ntr, ktm_trace_geom *__restrict__ geom,
                                int32_t *__restrict__ coords)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= ntr) return;
    int32_t c[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) c[k] = (int32_t)__builtin_bswap32(raw[i * rec_words + 18 + k]);
    if (coords) {
#pragma unroll
        for (int k = 0; k < 4; ++k) coords[4 * i + k] = c[k];
    }
    geom[i] = trace_geometry(g, c);
}

/* ------------------------------------------------------------------------ */
/* trace preparation                                                         */
/* ------------------------------------------------------------------------ */

/* Where the prep kernels read trace samples: FP32 traces [ntr][ns], or raw
 * SEG-Y trace records as stored in the file (240-byte header + ns big-endian
 * words, Kirchhoff.c:1281-1290) with IBM (format 1) or IEEE (format 5)
 * samples.  Decoding inside the prep kernels makes the ingest of a block
 * one pass: the byte swap and IBM decode of Kirchhoff.c:1284-1290 happen
 * where the sample is consumed. */
enum { SRC_F32 = 0, SRC_SEGY_IBM = 1, SRC_SEGY_IEEE = 2, SRC_Q_BF16 = 3, SRC_Q_F16 = 4 };

struct TraceSrc {
    const void *p;
    int64_t rec_words;      /* 4-byte words per trace: ns, or 60 + ns for a record */
};

/* IBM hex float -> float as Kirchhoff.c:1287-1289 evaluates it:
 * (sign * fraction / 2^24) * (float)16^(exponent - 64), the power of 16
 * rounded to float on its own (inf above 2^127, 0 below 2^-149; a zero
 * fraction times inf is NaN).  The power is built from its bits: e4 is a
 * multiple of 4, so no value falls between two floats. */
__device__ __forceinline__ float ibm_word(uint32_t w)
{
    const float frac = (float)(w & 0x00ffffffu) * (1.0f / 16777216.0f);
    const int e4 = 4 * (int)((w >> 24) & 0x7fu) - 256;
    /* all three forms computed, then selected (no divergent branch) */
    const uint32_t norm = (uint32_t)(e4 + 127) << 23;                 /* -126 <= e4 <= 127 */
    const int sh = e4 + 149;                                          /* -149 <= e4 < -126 */
    const uint32_t sub = sh >= 0 ? (1u << (sh & 31)) : 0u;
    const uint32_t pb = e4 > 127 ? 0x7f800000u : (e4 >= -126 ? norm : sub);
    const float sf = (w >> 31) ? -frac : frac;
    return sf * __uint_as_float(pb);
}

/* Raw 32-bit word of sample t of trace i (no decode yet), and its decode:
 * split so that a tile's loads can all be in flight before any decode. */
template <int SRC>
__device__ __forceinline__ uint32_t load_word(const TraceSrc &s, int64_t i, int t)
{
    if (SRC == SRC_F32) return reinterpret_cast<const uint32_t *>(s.p)[i * s.rec_words + t];
    return reinterpret_cast<const uint32_t *>(s.p)[i * s.rec_words + 60 + t];
}

template <int SRC>
__device__ __forceinline__ float decode_word(uint32_t u)
{
    if (SRC == SRC_F32) return __uint_as_float(u);
    const uint32_t w = __builtin_bswap32(u);
    return SRC == SRC_SEGY_IBM ? ibm_word(w) : __uint_as_float(w);
}

/* the same for N words: where no exponent reaches 2^128 (one test for all)
 * the power of 16 is finite and the product of ibm_word is one exact scaling,
 * fraction x 2^(4 (exponent - 64) - 24), rounded once */
template <int SRC, int N>
__device__ __forceinline__ void decode_words(const uint32_t *u, float *x)
{
    if (SRC != SRC_SEGY_IBM) {
#pragma unroll
        for (int m = 0; m < N; ++m) x[m] = decode_word<SRC>(u[m]);
        return;
    }
    uint32_t big = 0u;
#pragma unroll
    for (int m = 0; m < N; ++m) big = max(big, u[m] & 0x7fu);   /* the exponent, as stored */
    if (__ballot(big >= 96u)) {
#pragma unroll
        for (int m = 0; m < N; ++m) x[m] = decode_word<SRC>(u[m]);
    } else {
#pragma unroll
        for (int m = 0; m < N; ++m) {
            const uint32_t w = __builtin_bswap32(u[m]);
            const float v = __builtin_amdgcn_ldexpf((float)(w & 0x00ffffffu), 4 * (int)(u[m] & 0x7fu) - 280);
            x[m] = __uint_as_float((__float_as_uint(v) & 0x7fffffffu) | (w & 0x80000000u));
        }
    }
}

template <int SRC>
__device__ __forceinline__ float load_sample(const TraceSrc &s, int64_t i, int t)
{
    return decode_word<SRC>(load_word<SRC>(s, i, t));
}

/* REFERENCE mode: the two FP32 running sums of Kirchhoff.c:1314-1324 per
 * trace, emitting
 *   F[T] = (float)(-2.0*p[T] + p[T-2] + p[T+2])         (Kirchhoff.c:1392)
 * as soon as p[T+2] exists (F[t-2] at step t), p[] the double integral of
 * which the last five values stay in registers.  p[-1] = p[1] and p[-2] =
 * p[2] are the mirror pad of Kirchhoff.c:1327-1328.
 *
 * A workgroup takes 64 traces.  Its first wave runs the recurrence, one lane
 * per trace, and nothing else: one step is a double add between two
 * conversions (the chain), the second sum and F.  Two helper waves feed it
 * through LDS, a tile of PREP_TS steps ahead: they load the samples
 * (PREP_AHEAD tiles ahead, two traces x 32 samples per instruction), decode
 * them, divide by 4 t2[t] (the increment of integral 1 does not depend on the
 * running sum), and store the F of the tile before.  Tile i's steps are
 * t = 32 (i - 1) + 2 ..., so its F start at a multiple of 32.  One barrier
 * per tile.
 * Bound by the recurrence's chain for few traces and by memory for a full
 * block: 50,000 IBM records of 1500 samples 319 -> 170 us (3.6 TB/s), 96
 * traces of 501 74 -> 32 us, against one wave that did all of it with a full
 * double division per sample.  Of the same block with 4 helper waves 180 us,
 * 8 200, tiles of 16 steps 250, and with the division in the recurrence wave
 * and tiles of 64 steps 350. */
#define PREP_TS 32
#define PREP_HELPERS 2
#define PREP_AHEAD 2        /* tiles in flight */
#define PREP_NT (KTM_WAVE * (1 + PREP_HELPERS))
template <int SRC>
__global__ void __launch_bounds__(PREP_NT)
k_prep_ref(const TraceSrc src, int64_t ntr, int ns, int64_t row, float dt,
           const float *__restrict__ t2, float *__restrict__ out)
{
    /* slot (b, j, k), b the tile's parity: the increment of integral 1 at the
     * tile's step k of trace j, (double)tr[t] / (4 t2[t]) (Kirchhoff.c:1314),
     * at t = 0 the sample itself; then, in its place, F of that step.  A
     * helper lane reads the F and writes the increment two tiles on of the
     * same slots, so one pair of buffers holds both. */
    union Slot { double inc; float f; };
    __shared__ Slot s[2][KTM_WAVE][PREP_TS + 1];
    constexpr int PER = PREP_TS / PREP_HELPERS;                 /* samples per helper lane */
    constexpr int STEP = KTM_WAVE * PREP_HELPERS / PREP_TS;     /* traces per helper pass */
    const int64_t tr0 = (int64_t)blockIdx.x * KTM_WAVE;
    const int ntl = (int)min((int64_t)KTM_WAVE, ntr - tr0);
    const int ntiles = (ns + PREP_TS - 1) / PREP_TS + 1;        /* steps up to ns + 1 */
    if (threadIdx.x < KTM_WAVE) {
        /* ---- the recurrence: tile i in phase i ---- */
        const int lane = threadIdx.x;
        const float last = load_sample<SRC>(src, tr0 + (lane < ntl ? lane : 0), ns - 1);
        float q = 0.0f, p = 0.0f;
        double dm1 = 0.0, dm2 = 0.0, dm3 = 0.0, dm4 = 0.0, d0 = 0.0;   /* p[t-1..t-4], p[t] */
        __syncthreads();
        for (int i = 0; i < ntiles; ++i) {
            const int t0 = (i - 1) * PREP_TS + 2;
            Slot *sl = s[i & 1][lane];
            if (t0 >= 4 && t0 + PREP_TS <= ns) {
                /* interior tile: every step is the t >= 4, t < ns case */
                double iv[PREP_TS];
#pragma unroll
                for (int k = 0; k < PREP_TS; ++k) iv[k] = sl[k].inc;
#pragma unroll
                for (int k = 0; k < PREP_TS; ++k) {
                    q = (float)((double)q + iv[k]);
                    dm4 = dm3; dm3 = dm2; dm2 = dm1; dm1 = d0;
                    p = p + q;
                    d0 = (double)p;
                    sl[k].f = (float)(-2.0 * dm2 + dm4 + d0);
                }
            } else {
                const int s_end = min(PREP_TS, ns + 2 - t0);
                for (int k = max(0, -t0); k < s_end; ++k) {
                    const int tk = t0 + k;
                    if (tk == 0) {
                        q = (float)sl[k].inc;   /* integral 1 at t */
                        p = q;                  /* integral 2 at t */
                        d0 = (double)p;
                        continue;
                    }
                    if (tk < ns)
                        q = (float)((double)q + sl[k].inc);
                    else
                        q = q + last / dt / dt / (float)tk / (float)tk;
                    dm4 = dm3; dm3 = dm2; dm2 = dm1; dm1 = d0;
                    p = p + q;
                    d0 = (double)p;
                    if (tk == 2)
                        sl[k].f = (float)(-2.0 * dm2 + d0 + d0);
                    else if (tk == 3)
                        sl[k].f = (float)(-2.0 * dm2 + dm2 + d0);
                    else if (tk >= 4)
                        sl[k].f = (float)(-2.0 * dm2 + dm4 + d0);
                }
            }
            __syncthreads();
        }
        return;
    }
    /* ---- helpers: lane (sub, tb) moves step sub of traces tb, tb + STEP .. */
    const int hid = threadIdx.x - KTM_WAVE;
    const int sub = hid & (PREP_TS - 1), tb = hid / PREP_TS;
    uint32_t wv[PREP_AHEAD][PER];       /* tile i in place i % PREP_AHEAD */
    float t2v[PREP_AHEAD];
    /* the workgroup's first record and output row; 32-bit offsets from there */
    const uint32_t *sp = reinterpret_cast<const uint32_t *>(src.p) + tr0 * src.rec_words +
                         (SRC == SRC_F32 ? 0 : 60);
    float *op = out + tr0 * row;
    const uint32_t rw = (uint32_t)src.rec_words, orow = (uint32_t)row;
    const bool full = ntl == KTM_WAVE;
    /* unconditional loads at clamped (in-bounds) positions, all in flight
     * together; out-of-range values are replaced after the decode */
    auto load = [&](int i, int a) __attribute__((always_inline)) {
        const int t = (i - 1) * PREP_TS + 2 + sub, tc = min(max(t, 0), ns - 1);
        if (full) {
            const uint32_t o = (uint32_t)tb * rw + (uint32_t)tc;
#pragma unroll
            for (int m = 0; m < PER; ++m) wv[a][m] = (sp + (uint32_t)(m * STEP) * rw)[o];
        } else {
#pragma unroll
            for (int m = 0; m < PER; ++m)
                wv[a][m] = sp[(uint32_t)min(tb + m * STEP, ntl - 1) * rw + (uint32_t)tc];
        }
        t2v[a] = t2[tc];
    };
    auto feed = [&](int i, int a) __attribute__((always_inline)) {
        const int t = (i - 1) * PREP_TS + 2 + sub;
        const double den = t > 0 && t < ns ? 4.0 * (double)t2v[a] : 1.0;
        const double rden = 1.0 / den;
        float x[PER];
        decode_words<SRC, PER>(wv[a], x);
        if (i < 2 || i * PREP_TS + 2 > ns) {
#pragma unroll
            for (int m = 0; m < PER; ++m) x[m] = t >= 0 && t < ns ? x[m] : 0.0f;
        }
#pragma unroll
        for (int m = 0; m < PER; ++m)
            /* x / den correctly rounded from RN(1/den), zeros, infinities,
             * NaN and a zero den as the division gives them */
            s[i & 1][tb + m * STEP][sub].inc = __builtin_amdgcn_div_fixup(
                div_cr((double)x[m], den, rden), den, (double)x[m]);
    };
    /* F of tile i, T = 32 (i - 1) + sub, and zeros from ns to the row's end */
    auto store = [&](int i) __attribute__((always_inline)) {
        const int T = (i - 1) * PREP_TS + sub;
        const uint32_t o = (uint32_t)tb * orow + (uint32_t)T;
        if (full && i > 0 && i * PREP_TS <= ns) {
#pragma unroll
            for (int m = 0; m < PER; ++m)
                (op + (uint32_t)(m * STEP) * orow)[o] = s[i & 1][tb + m * STEP][sub].f;
            return;
        }
        if (T < 0 || T >= row) return;
#pragma unroll
        for (int m = 0; m < PER; ++m) {
            const int j = tb + m * STEP;
            if (j < ntl) op[(uint32_t)(m * STEP) * orow + o] = T < ns ? s[i & 1][j][sub].f : 0.0f;
        }
    };
#pragma unroll
    for (int a = 0; a < PREP_AHEAD; ++a) load(a, a);
    feed(0, 0);
    __syncthreads();
    for (int i0 = 0; i0 < ntiles; i0 += PREP_AHEAD) {
#pragma unroll
        for (int a = 0; a < PREP_AHEAD; ++a) {
            const int i = i0 + a;
            if (i >= ntiles) break;
            /* phase i: tile i's registers are free, tile i + 1 is fed */
            load(i + PREP_AHEAD, a);
            store(i - 1);
            if (i + 1 < ntiles) feed(i + 1, (a + 1) % PREP_AHEAD);
            __syncthreads();
        }
    }
    store(ntiles - 1);
    store(ntiles);                          /* the row's end past the last tile */
}

/* CLOSED mode: F as the 3-tap filter of x[t] = trace[min(t,ns-1)] * w[t].
 * Derivation from Kirchhoff.c:1314-1328 (exact arithmetic): with
 * Q[k] = sum_{j<=k} x[j] and p[k] = sum_{j<=k} Q[j],
 *   T >= 2 : p[T+2] - 2p[T] + p[T-2] = x[T] + 2x[T+1] + x[T+2]
 *   T == 1 : p[3] - p[1]           = 2x[0] + 2x[1] + 2x[2] + x[3]
 *   T == 0 : 2(p[2] - p[0])        = 4x[0] + 4x[1] + 2x[2]
 * Shared by the F32 prep kernel and the BF16/FP16 staging in k_migrate so the
 * two storage modes differ only by quantisation. */
__device__ __forceinline__ float bf16_to_f32_(uint16_t h) { return __uint_as_float((uint32_t)h << 16); }
__device__ __forceinline__ float f16_to_f32_(uint16_t u)
{
    _Float16 h;
    __builtin_memcpy(&h, &u, 2);
    return (float)h;
}

__device__ __forceinline__ float closed_tap(int T, float x0, float x1, float x2, float x3)
{
    /* for T >= 2, x0..x2 are x[T], x[T+1], x[T+2]; for T < 2 they are x[0..3] */
    if (T >= 2) return (x0 + 2.0f * x1) + x2;
    if (T == 1) return ((2.0f * x0 + 2.0f * x1) + 2.0f * x2) + x3;
    return (4.0f * x0 + 4.0f * x1) + 2.0f * x2;
}

/* src: any 32-bit trace source of load_sample, or BF16/FP16 traces stored
 * by k_quantize (SRC_Q_*, [ntr][row] halves, rec_words = row) with the
 * per-trace scale in geom; the stored value times the scale stands for the
 * trace sample. */
template <int SRC>
__global__ void k_prep_closed(const TraceSrc src, const ktm_trace_geom *__restrict__ geom,
                              int64_t ntr, int ns, int64_t row, const float *__restrict__ w,
                              float *__restrict__ out)
{
    constexpr bool Q16 = SRC == SRC_Q_BF16 || SRC == SRC_Q_F16;
    const int64_t i = blockIdx.y;
    const int T = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= ntr || T >= row) return;
    float v = 0.0f;
    if (T < ns) {
        float x[4];
        const int b = T >= 2 ? T : 0;
        const float sc = Q16 ? geom[i].scale : 1.0f;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const int t = b + k;
            const int tt = t < ns ? t : ns - 1;
            float tr;
            if (Q16) {
                const uint16_t hq = reinterpret_cast<const uint16_t *>(src.p)[i * src.rec_words + tt];
                tr = sc * (SRC == SRC_Q_BF16 ? bf16_to_f32_(hq) : f16_to_f32_(hq));
            } else {
                tr = load_sample<SRC>(src, i, tt);
            }
            x[k] = t <= ns + 1 ? tr * w[t] : 0.0f;
        }
        v = closed_tap(T, x[0], x[1], x[2], x[3]);
    }
    out[i * row + T] = v;
}

/* BF16 (round to nearest even) and FP16 storage helpers */
__device__ __forceinline__ uint16_t f32_to_bf16(float f)
{
    uint32_t u = __float_as_uint(f);
    if ((u & 0x7fffffffu) > 0x7f800000u) return (uint16_t)((u >> 16) | 0x40u); /* NaN */
    u += 0x7fffu + ((u >> 16) & 1u);
    return (uint16_t)(u >> 16);
}
__device__ __forceinline__ float bf16_to_f32(uint16_t h) { return __uint_as_float((uint32_t)h << 16); }
__device__ __forceinline__ uint16_t f32_to_f16(float f)
{
    _Float16 h = (_Float16)f;
    uint16_t u;
    __builtin_memcpy(&u, &h, 2);
    return u;
}
__device__ __forceinline__ float f16_to_f32(uint16_t u)
{
    _Float16 h;
    __builtin_memcpy(&h, &u, 2);
    return (float)h;
}

/* scale = max |tr| (1 for an all-zero trace); the trace divided by scale is
 * rounded to BF16 or FP16 with sixth-order error feedback: sample t is
 * quantised as v = tr/scale + sum_k QA_k e[t-k] (e the rounding errors of
 * the previous samples), so the noise reaching the image is the rounding
 * noise shaped by N(z) = 1 - sum_k QA_k z^-k and then filtered by the [1,2,1]
 * anti-alias taps of the migration, H(z) = (1 + z^-1)^2.  QA minimise the
 * power of the shaped, filtered noise (|H|^2 has autocorrelation 6, 4, 1)
 * under N(1) = 0, which keeps the zero at DC of first-order feedback
 * (QA = 1): power 1.88 against 4 for first-order and 6 for none, the
 * low-frequency part 1.4 x first-order's where the unconstrained 4-tap
 * optimum has 4.4 x.  Measured on 74 random configurations: BF16 image
 * error (relative L2 against FP64) median 9.2e-4 -> 6.4e-4, max 1.6e-3 ->
 * 1.0e-3.  The coefficients are exact binary fractions and the feedback is
 * an FIR filter of bounded rounding errors, so it cannot run away.  A
 * workgroup is one wave of 64 traces: the max-abs sweep reads two traces x
 * 32 samples per load (max is exact in any order); the sequential
 * error-feedback sweep stages 32-sample tiles through LDS like k_prep_ref,
 * one lane per trace. */
#define QUANT_TS 32
#define QA1 1.625f
#define QA2 (-1.625f)
#define QA3 1.5f
#define QA4 (-1.0f)
#define QA5 0.625f
#define QA6 (-0.125f)
template <int DT, int SRC>
__global__ void __launch_bounds__(KTM_WAVE)
k_quantize(const TraceSrc src, int64_t ntr, int ns, int64_t row, uint16_t *__restrict__ q,
           ktm_trace_geom *__restrict__ geom)
{
    __shared__ float s_in[KTM_WAVE][QUANT_TS + 1];
    __shared__ uint16_t s_q[KTM_WAVE][QUANT_TS + 2];
    __shared__ float s_scale[KTM_WAVE];
    const int lane = threadIdx.x;
    const int sub = lane & (QUANT_TS - 1), half = lane / QUANT_TS;
    const int64_t tr0 = (int64_t)blockIdx.x * KTM_WAVE;
    const int ntl = (int)min((int64_t)KTM_WAVE, ntr - tr0);
    for (int m = 0; m < KTM_WAVE / 2; ++m) {
        const int j = min(2 * m + half, ntl - 1);
        float mx = 0.0f;
#pragma unroll 8
        for (int t = sub; t < ns; t += QUANT_TS) mx = fmaxf(mx, fabsf(load_sample<SRC>(src, tr0 + j, t)));
        for (int o = QUANT_TS / 2; o > 0; o >>= 1) mx = fmaxf(mx, __shfl_xor(mx, o));
        if (sub == 0) s_scale[2 * m + half] = mx;
    }
    __syncthreads();
    const float m_own = s_scale[lane];
    const float scale = m_own > 0.0f ? m_own : 1.0f;
    const float inv = 1.0f / scale;
    float e1 = 0.0f, e2 = 0.0f, e3 = 0.0f, e4 = 0.0f, e5 = 0.0f, e6 = 0.0f;   /* e[t-1] .. */
    for (int t0 = 0; t0 < ns; t0 += QUANT_TS) {
        const int t = t0 + sub;
        const int tc = t < ns ? t : ns - 1;
        uint32_t wv[KTM_WAVE / 2];
#pragma unroll
        for (int m = 0; m < KTM_WAVE / 2; ++m)
            wv[m] = load_word<SRC>(src, tr0 + min(2 * m + half, ntl - 1), tc);
#pragma unroll
        for (int m = 0; m < KTM_WAVE / 2; ++m) s_in[2 * m + half][sub] = decode_word<SRC>(wv[m]);
        __syncthreads();
        const int s_end = min(QUANT_TS, ns - t0);
        if (s_end == QUANT_TS) {
            float xk[QUANT_TS];
#pragma unroll
            for (int k = 0; k < QUANT_TS; ++k) xk[k] = s_in[lane][k];
#pragma unroll
            for (int k = 0; k < QUANT_TS; ++k) {
                const float fb = ((((QA1 * e1 + QA2 * e2) + QA3 * e3) + QA4 * e4) + QA5 * e5) + QA6 * e6;
                const float v = xk[k] * inv + fb;
                const uint16_t h = DT == KTM_TRACE_BF16 ? f32_to_bf16(v) : f32_to_f16(v);
                s_q[lane][k] = h;
                e6 = e5; e5 = e4; e4 = e3; e3 = e2; e2 = e1;
                e1 = v - (DT == KTM_TRACE_BF16 ? bf16_to_f32(h) : f16_to_f32(h));
            }
        } else for (int k = 0; k < s_end; ++k) {
            const float fb = ((((QA1 * e1 + QA2 * e2) + QA3 * e3) + QA4 * e4) + QA5 * e5) + QA6 * e6;
            const float v = s_in[lane][k] * inv + fb;
            const uint16_t h = DT == KTM_TRACE_BF16 ? f32_to_bf16(v) : f32_to_f16(v);
            s_q[lane][k] = h;
            e6 = e5; e5 = e4; e4 = e3; e3 = e2; e2 = e1;
            e1 = v - (DT == KTM_TRACE_BF16 ? bf16_to_f32(h) : f16_to_f32(h));
        }
        __syncthreads();
        if (sub < s_end) {
#pragma unroll 8
            for (int m = 0; m < KTM_WAVE / 2; ++m) {
                const int j = 2 * m + half;
                if (j < ntl) q[(tr0 + j) * row + t] = s_q[j][sub];
            }
        }
        __syncthreads();
    }
    for (int j = 0; j < ntl; ++j)
        for (int64_t T = ns + lane; T < row; T += KTM_WAVE) q[(tr0 + j) * row + T] = 0;
    if (lane < ntl) geom[tr0 + lane].scale = scale;
}

/* ------------------------------------------------------------------------ */
/* migration                                                                 */
/* ------------------------------------------------------------------------ */
struct MigArgs {
    const float *prep;               /* [ntr][row] filtered traces F(T) */
    const ktm_trace_geom *geom;
    int64_t ntr, row;
    float *km, *fold, *comp;
    const float *vel2;
    const int32_t *t1, *velx, *vely;
    const float *t2, *colx, *coly, *slab_cx, *slab_cy, *slab_x2thr;
    unsigned long long *counter;
    float ap_x2thr;                  /* aperture gate on the squared CMP distance */
    float aperture;                  /* for the conservative tile test only */
    float dt, rdt;                   /* dt and RN(1/dt) */
    int ns, nh, nxp, nyp, nx, ny, jobs_y, nvel_xl, nsm;
    int tiles_x, ntiles, tx_cols, ty_cols, run;
    int rx0, ry0, rx1, ry1;          /* migrated region [rx0,rx1) x [ry0,ry1) */
    int align16;                     /* prep (and so every row) 16-byte aligned */
    /* Kahan variants: the block's chunks of a workgroup's thread count of
     * traces dealt round-robin to nparts parts (chunk c to part c mod nparts), part = blockIdx.z, so that
     * every part spans the whole survey and its workgroups carry like loads;
     * part 0 adds into km/fold/comp, part p > 0 writes its sums into
     * parts + (p-1) * 3 * part_n, region layout [X-rx0][Y-ry0][h][t] */
    int64_t nparts, part_n;
    float *parts;
};

/* Reference semantics of one traveltime index (Kirchhoff.c:1381-1384):
 * FP32 true divisions and sums, the two square roots in double and summed in
 * double, rounded to float, FP32 division by dt, floor.  Returns ns when the
 * sample falls past the trace (the T<ns test of Kirchhoff.c:1387).  r and
 * rdt are RN(1/v2) and RN(1/dt). */
__device__ __forceinline__ int exact_T(float dIS2, float dIR2, float t2, float v2, float r,
                                       float dt, float rdt, int ns)
{
    const float s1 = t2 + div_cr(dIS2, v2, r);
    const float s2 = t2 + div_cr(dIR2, v2, r);
    const float dsr = (float)(sqrt_cr((double)s1) + sqrt_cr((double)s2));
    const float qq = div_cr(dsr, dt, rdt);
    return qq < (float)ns ? (int)qq : ns;
}

/* The fast form of the traveltime index, in samples from the start: with
 * rs = RN(1/(v2 dt^2)) (product and quotient in double, one rounding) and
 * tq = 0.25 t^2 (exact for t < 4096, else one rounding),
 *   q = RN( sqrt_hw(fma(dIS2, rs, tq)) + sqrt_hw(fma(dIR2, rs, tq)) ).
 * a1 = RN(fma(dIS2, rs, tq)) is within 2u of (t2e + dIS2/v2)/dt^2 (t2e =
 * t^2 dt^2 / 4), the reference's s1 = RN(t2 + RN(dIS2/v2)) within 2u of
 * t2e + dIS2/v2 (its t2 is t2e rounded once): 4u on the radicand, 2u after
 * the square root, plus 2u for v_sqrt_f32; the sum's rounding u; the
 * reference's RN(dsr) and RN(dsr/dt) 2u: |q - Q| <= 7u Q to first order;
 * its tolerance KTM_FAST_EPS_S = 8u leaves 1u for the second-order terms.
 * The 1 ulp figure of v_sqrt_f32 is checked exhaustively on [1, 4) by the GPU
 * tests, the whole bound on random and near-integer inputs.  The demigration and
 * the relaxed index take this form, the exact migration that of fast_p. */
#define KTM_FAST_EPS_S 4.8e-7f
__device__ __forceinline__ float fast_qs(float dIS2, float dIR2, float rs, float tq)
{
    return __builtin_amdgcn_sqrtf(__builtin_fmaf(dIS2, rs, tq)) +
           __builtin_amdgcn_sqrtf(__builtin_fmaf(dIR2, rs, tq));
}

/* per-sample constants of fast_qs */
__device__ __forceinline__ float fast_rs(float v2, float dt)
{
    return (float)(1.0 / ((double)v2 * (double)dt * (double)dt));
}
__device__ __forceinline__ float fast_tq(int t) { return (float)(0.25 * (double)t * (double)t); }

/* q >= 0 (a sum of square roots) clamped to lim, half a sample past an integer
 * T >= ns (demigration).  Beyond lim the reference's Q is > ns as well (|q - Q|
 * <= 1e-6 q), so the sample is discarded either way; the clamped value truncates
 * to T and is never ambiguous.  One clamp serves the index and the ambiguity
 * test. */
__device__ __forceinline__ float fast_clamp(float q, float lim) { return fminf(q, lim); }

/* floor of the clamped q */
__device__ __forceinline__ int fast_T(float qc) { return (int)qc; }

/* chunks of up to 4 staged rows (one of 8 counts twice) whose taps the Kahan
 * variants sum in plain FP32 before one compensated step: at most 32 terms */
#define KTM_KAHAN_CHUNKS 8

/* q clamped to [0, hi] in one instruction (v_med3_f32; q >= 0 is a sum of
 * square roots, so this is min(q, hi) without the canonicalisation of
 * fminf's operands, which the compiler otherwise repeats per sample) */
__device__ __forceinline__ float clamp_ns(float q, float hi)
{
    return __builtin_amdgcn_fmed3f(q, 0.0f, hi);
}

/* a non-negative float without infinity and NaN, the largest finite one in
 * their place */
__device__ __forceinline__ float finite(float x) { return fminf(x, 3.402823466e38f); }

/* The exact variants' form of q, in units of nsh = ns + 1/2: with
 * rsn = RN(1/(v2 dt^2 nsh^2)) and tqn = RN(t^2/(4 nsh^2)) (double, rounded
 * once)
 *   p = RN( sqrt_hw(fma(dIS2, rsn, tqn)) + sqrt_hw(fma(dIR2, rsn, tqn)) ),
 * q = p nsh without rounding.  The radicand's two constants carry one
 * rounding each, at most u of a sum of non-negative terms, and the FMA u: 2u,
 * as above (rs and the FMA), so |p nsh - Q| <= 7u Q holds unchanged.  p is
 * limited to 1 by the clamp modifier of its sum, at no cost (a v_med3 is a
 * quarter-rate instruction): a limited sample has Q > ns for certain, its
 * index is ns, and half a sample from an integer it is never ambiguous.
 * p is never NaN (which the limit would turn into 0, and floor_p into an index of
 * -1): v2 is at least KTM_V2_MIN, so rsn is finite, and the squared distances are
 * kept finite.  A trace without a position (NaN or infinite in the caller's
 * geometry), whose index is ns in the reference arithmetic, is so past the trace
 * by the limit. */
__device__ __forceinline__ float fast_rsn(float v2, float dt, float nsh)
{
    return (float)(1.0 / ((double)v2 * (double)dt * (double)dt * ((double)nsh * (double)nsh)));
}
__device__ __forceinline__ float fast_tqn(int t, float nsh)
{
    const double r = (double)t / (2.0 * (double)nsh);
    return (float)(r * r);
}
__device__ __forceinline__ float fast_p(float dIS2, float dIR2, float rsn, float tqn)
{
    return __builtin_amdgcn_fmed3f(__builtin_amdgcn_sqrtf(__builtin_fmaf(dIS2, rsn, tqn)) +
                                       __builtin_amdgcn_sqrtf(__builtin_fmaf(dIR2, rsn, tqn)),
                                   0.0f, 1.0f);
}

/* floor(q), q = p nsh, by one rounding: M = RN(q + (2^23 - 1/2)) holds
 * 2^23 + floor(q) in its mantissa when M >= 2^23, i.e. for q >= 1/4 (a tie,
 * q an integer, gives that integer or the one below; it is always
 * ambiguous); center = floor + 1/2 exactly; dev = q - center in
 * [-1/2, 1/2].  low: q may be below 1/4 (only t = 0 can be), where M is
 * raised to 2^23. */
#define KTM_FLOOR_MAGIC 8388607.5f
#define KTM_FLOOR_BITS 0x4B000000u     /* bits of 2^23 */
struct FloorP { float M, center, dev; };
__device__ __forceinline__ FloorP floor_p(float p, float nsh, bool low)
{
    FloorP r;
    r.M = __builtin_fmaf(p, nsh, KTM_FLOOR_MAGIC);
    if (low) r.M = fmaxf(r.M, 8388608.0f);
    r.center = r.M - KTM_FLOOR_MAGIC;
    r.dev = __builtin_fmaf(p, nsh, -r.center);
    return r;
}
__device__ __forceinline__ int floor_T(const FloorP &f)
{
    return (int)(__float_as_uint(f.M) - KTM_FLOOR_BITS);
}
/* An integer within eps (q + 1) of q: the distance to the nearest integer is
 * 1/2 - |dev|, so |dev| >= 1/2 - eps (q + 1) (the rounding of dev, 3e-8, is
 * inside the 8u against 7u of the bound).  The kernel takes the threshold at
 * the largest q that the trace can have in the wave's samples: one value per
 * trace instead of an FMA per sample, for a few more ambiguous samples. */
__device__ __forceinline__ float ambiguous_from(float q) { return 0.5f - KTM_FAST_EPS_S * (q + 1.0f); }

/* The reference traveltime index of a sample with every rule of the exact
 * path: the fast form, and where an integer lies within its error bound the
 * reference arithmetic.  low as in floor_p. */
__device__ __forceinline__ int reference_T(float dIS2, float dIR2, float rsn, float tqn, float t2,
                                           float v2, float dt, float rdt, int ns, bool low)
{
    const float nsh = (float)ns + 0.5f;
    const float p = fast_p(dIS2, dIR2, rsn, tqn);
    const FloorP f = floor_p(p, nsh, low);
    if (fabsf(f.dev) < ambiguous_from(p * nsh)) return floor_T(f);
    return exact_T(dIS2, dIR2, t2, v2, 1.0f / v2, dt, rdt, ns);
}

/* slots whose traveltime chains run side by side under one test */
constexpr int mig_group(int K) { return K % 3 == 0 ? 3 : K % 4 == 0 ? 4 : K % 5 == 0 ? 5 : 2; }

typedef __attribute__((address_space(3))) float lds_float;
typedef __attribute__((address_space(3))) void lds_void;
typedef __attribute__((address_space(3))) unsigned long long lds_u64;
typedef __attribute__((address_space(1))) const void global_void;

/* One workgroup = NW waves = NCOL image columns x W time segments.  Each lane
 * owns K samples t = seg*64K + 64k + lane of its column: the image values
 * (km, fold count, Kahan compensation) and the per-sample constants of the
 * traveltime stay in registers for the whole launch.
 *
 * Traces stream through LDS in trace order.  Blocks of NT traces are filtered
 * to those whose CMP can reach the tile (ordered compaction into a list);
 * the aperture and slab gates of the next 64 of the list are evaluated
 * lane-parallel (lane j = trace j), and the passing ones are walked in order.
 * Rows are staged C at a time into a ring of WN + 1 such chunks by loads that
 * write LDS directly: chunk q + 1 is in flight while chunk q is used, so the
 * loads' latency is hidden, no register holds a staged row, and one barrier
 * per chunk separates the two (the other slots keep the window's earlier
 * chunks for the re-summation below).
 *
 * Traveltime index, two variants:
 * - exact (the FP32 reference path, and the Kahan modes unless FASTIDX): the
 *   reference's index, resolved speculatively.  The fast form's floor is
 *   used at once; a sample whose p ns lies within the form's error bound of an
 *   integer (and is not past the trace for certain) is added with that index
 *   and remembered with the running sum before the add (one per lane and
 *   window of WN chunks; a lane's further ambiguous samples take the inline
 *   exact path).  At the end of the window one wave-wide pass computes the
 *   reference index of every lane's remembered sample together; where it
 *   differs from the fast one (a few percent of them) the sample's running sum
 *   is rebuilt from the saved value through the window's later traces in
 *   order, so every sample receives its additions in the reference's order
 *   and the result equals the inline exact path's bit for bit.
 * - FASTIDX: T = floor(min(q, ns)) of the fast form alone (CLOSED and 16-bit
 *   modes, whose contract is an error bound against FP64): no ambiguity
 *   test.
 * The source's square root of every slot is kept from one passing trace to the
 * next of the same source: traces in shot order, which most surveys come in,
 * cost one root per sample instead of two (12 offset classes x 2503 samples:
 * 6.3 -> 5.6 ms, the pair L, L^T of the 200-shot line 39.0 -> 36.5 ms), sources
 * at random 2 % more for the roots computed apart; with 12 slots and compensated
 * sums the roots do not fit the registers (33 of them in scratch).
 * A sample past the trace reads the zero F[ns] and does not count for fold.
 * With the gates each lane bounds, for its trace and every slot of the wave,
 * the largest q (the traveltime at the slot's largest constants): slots before
 * the first whose bound reaches the end of the trace need no count (and,
 * relaxed index, no clamp), and the bound over all slots sets the trace's
 * ambiguity threshold.
 * Bound by VALU issue.  In this mixed stream every VALU instruction takes a
 * SIMD about 4 cycles and a square root 8 (the doubled FMA and add rate of a
 * pure stream does not appear: 17.3 instructions per 64 contributions of
 * which 2.07 roots took 79 cycles), so what counts is their number: two FMA, two
 * roots, the clamped sum, three for floor and distance, the LDS address, the
 * add into the image, and 2/3 of an instruction for the test (14.5 in all with
 * the gates, the staging and the ambiguous samples).  Against rows staged
 * through registers between two barriers and every sample past the trace on
 * the rare path, the lane shapes and the kept root included: 16,000 traces x 1500
 * samples into 400 x 400 columns 298 -> 263 ms, 20,000 BF16-stored x 1251 into 150
 * x 150 222 -> 171 ms, the 40-shot line 3.91 -> 2.39 ms, 12 classes x 2503 samples
 * x 500 columns 11.5 -> 5.5 ms.  12 waves of K = 8 (six per SIMD) measured the same as 8 of K = 12
 * with 1500 samples, 16 waves in one workgroup 15 % slower (all of a CU's waves
 * at one barrier); slot groups of 2, 4 and 6 within 3 % of 3. */
template <int K, int W, int NW, int C, int WN, bool KAHAN, bool FASTIDX>
__global__ void __launch_bounds__(NW * KTM_WAVE) __attribute__((amdgpu_waves_per_eu(4, 4)))
k_migrate(const MigArgs a)
{
    constexpr int NT = NW * KTM_WAVE;
    constexpr int WPR = NW / C;             /* waves that stage one row of a chunk */
    constexpr bool SPEC = !FASTIDX;
    constexpr int G = mig_group(K);         /* slots side by side */
    constexpr int WT = WN * C;              /* traces of a window */
    constexpr int SB = KTM_WAVE / WT * WT;  /* traces whose gates are evaluated at once */
    constexpr int RING = WN + 1;            /* chunks in LDS: a window's and the next */
    static_assert(NW % C == 0 && WT <= 16 && K < 16 && K % G == 0 && (WN & (WN - 1)) == 0,
                  "remembered samples pack the slot and the trace in 4 bits each");
    extern __shared__ float4 lds4[];
    const int ldl = (int)a.row;             /* LDS row = prepared row (floats) */
    float *sF = reinterpret_cast<float *>(lds4);            /* [RING][C][ldl] */
    float2 *sMax = reinterpret_cast<float2 *>(sF + RING * C * ldl);   /* [NW][K] largest rs, tq */
    int *sSel = reinterpret_cast<int *>(sMax + NW * K);     /* [64 + C + NT], SB + C - 1 + NT used */
    int *sCnt = sSel + KTM_WAVE + C + NT;                   /* [NW]     */

    const int tid = threadIdx.x, lane = tid & (KTM_WAVE - 1);
    const int wv = __builtin_amdgcn_readfirstlane(tid / KTM_WAVE);
    /* XCD-aware tile order: consecutive workgroup ids go to different XCDs.
     * Each XCD takes runs of a.run consecutive tiles (a row of tiles in 3-D:
     * neighbouring columns share traces in its L2) and the runs are dealt
     * round-robin, so every XCD gets rows from the whole image; contiguous
     * bands per XCD left the edge bands (fewer traces within aperture) at
     * 0.73 of the mean work and the middle ones at 1.14. */
    const int wi = blockIdx.x >> 3;
    const int tile = (((wi / a.run) << 3) + (int)(blockIdx.x & 7)) * a.run + wi % a.run;
    if (tile >= a.ntiles) return;
    const int h = blockIdx.y;
    const int part = KAHAN ? (int)blockIdx.z : 0;
    const int tx = tile % a.tiles_x, ty = tile / a.tiles_x;
    const int cw = wv / W, seg = wv % W;    /* column within tile, time segment */
    const int X = a.rx0 + tx * a.tx_cols + cw % a.tx_cols;
    const int Y = a.ry0 + ty * a.ty_cols + cw / a.tx_cols;
    const bool col_ok = X < a.rx1 && Y < a.ry1;
    const int Xc = X < a.rx1 ? X : a.rx1 - 1, Yc = Y < a.ry1 ? Y : a.ry1 - 1;
    const float IX = a.colx[Xc], IY = a.coly[Yc];
    const int job = (Xc / a.nx) * a.jobs_y + (Yc / a.ny);
    const float scx = a.slab_cx[job], scy = a.slab_cy[job];
    const float sthr = a.slab_x2thr[job];
    const int ns = a.ns;
    const float nsf = (float)ns, nsh = nsf + 0.5f;
    /* M - past is 0 or less for an index below ns, 1 for ns */
    const float past = 8388608.0f + (nsf - 1.0f);

    /* conservative tile test: the CMP must be within aperture of some
     * column of the tile (exact per-column gates follow) */
    const int x0 = a.rx0 + tx * a.tx_cols, x1 = min(x0 + a.tx_cols, a.rx1) - 1;
    const int y0 = a.ry0 + ty * a.ty_cols, y1 = min(y0 + a.ty_cols, a.ry1) - 1;
    const float ccx = 0.5f * (a.colx[x0] + a.colx[x1]), ccy = 0.5f * (a.coly[y0] + a.coly[y1]);
    const float hx = 0.5f * fabsf(a.colx[x1] - a.colx[x0]);
    const float hy = 0.5f * fabsf(a.coly[y1] - a.coly[y0]);
    const float reach = a.aperture * 1.0001f + sqrtf(hx * hx + hy * hy) + 1.0f;
    const float reach2 = reach * reach;

    const int64_t pix = (((int64_t)Xc * a.nyp + Yc) * a.nh + h) * ns;
    const float *vel = a.vel2 + ((int64_t)a.velx[Xc] * a.nvel_xl + a.vely[Yc]) * a.nsm;
    float rs[K], tq[K], acc[K], cmp[K];
    float cnt[K];                           /* passing traces with T >= ns, per slot */
#pragma unroll
    for (int k = 0; k < K; ++k) {
        const int tl = seg * K * KTM_WAVE + k * KTM_WAVE + lane;
        cnt[k] = 0.0f;
        cmp[k] = 0.0f;
        if (tl < ns) {
            const float v2 = vel[a.t1[tl]];
            rs[k] = FASTIDX ? fast_rs(v2, a.dt) : fast_rsn(v2, a.dt, nsh);
            tq[k] = FASTIDX ? fast_tq(tl) : fast_tqn(tl, nsh);
            acc[k] = col_ok && part == 0 ? a.km[pix + tl] : 0.0f;
            if (KAHAN && col_ok && part == 0) cmp[k] = a.comp[pix + tl];
        } else {
            /* padding lane: q = 0.5, never flagged by the ambiguity test; it
             * reads F[0] into a value that is not stored */
            rs[k] = 0.0f;
            tq[k] = FASTIDX ? 0.0625f : 0.0625f / (nsh * nsh);
            acc[k] = 0.0f;
        }
        /* the slot's largest constants over the wave */
        float mr = rs[k], mt = tq[k];
        for (int d = KTM_WAVE / 2; d >= 1; d >>= 1) {
            mr = fmaxf(mr, __shfl_xor(mr, d));
            mt = fmaxf(mt, __shfl_xor(mt, d));
        }
        if (lane == 0) sMax[wv * K + k] = make_float2(mr, mt);
    }

    /* Kahan variants: the taps are summed onto y = -c in plain FP32 over
     * KTM_KAHAN_CHUNKS chunks (error <= (terms - 1) u times the terms'
     * magnitudes) and added to the image with one compensated step, which keeps
     * the compensated error bound of order u * sum |f| at a fraction of the
     * per-tap cost.  Plain variants add every tap into the image in trace order,
     * as the reference does. */
    float y[KAHAN ? K : 1];
#pragma unroll
    for (int k = 0; k < (KAHAN ? K : 1); ++k) y[k] = -cmp[k];
    int nfold = 0;
    auto fold_y = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int k = 0; k < (KAHAN ? K : 1); ++k) {
            const float yk = y[k];
            const float s = acc[k] + yk;
            y[k] = yk - (s - acc[k]);           /* -c, c = (s - acc) - y */
            acc[k] = s;
        }
    };

    uint32_t npass = 0, lastd = 0xffffffffu;    /* bits of the source distance of r1 (none: a NaN) */
    float r1[K];
#pragma unroll
    for (int k = 0; k < K; ++k) r1[k] = 0.0f;
    const int64_t cstep = KAHAN ? a.nparts * NT : NT;
    int64_t c0 = KAHAN ? (int64_t)part * NT : 0;
    /* the list of traces that can reach the tile, in order: sSel[head, n) */
    int head = 0, n = 0;
    auto refill = [&]() __attribute__((always_inline)) {
        while (n - head < SB + C && c0 < a.ntr) {
            if (head) {                          /* the rest to the front */
                const int left = n - head;       /* < SB + C <= NT */
                const int v = tid < left ? sSel[head + tid] : 0;
                __syncthreads();
                if (tid < left) sSel[tid] = v;
                head = 0;
                n = left;
            }
            const int64_t i = c0 + tid;
            bool pred = false;
            if (i < a.ntr) {
                const ktm_trace_geom g = a.geom[i];
                const float dx = g.cmpx - ccx, dy = g.cmpy - ccy;
                pred = g.off == h && dx * dx + dy * dy <= reach2;
            }
            const uint64_t m = __ballot(pred);
            const int pre = __popcll(m & ((1ull << lane) - 1ull));
            if (lane == 0) sCnt[wv] = __popcll(m);
            __syncthreads();
            int base = n, total = 0;
#pragma unroll
            for (int q = 0; q < NW; ++q) {
                const int v = sCnt[q];
                base += q < wv ? v : 0;
                total += v;
            }
            if (pred) sSel[base + pre] = (int)i;
            n += __builtin_amdgcn_readfirstlane(total);
            c0 += cstep;
            __syncthreads();
        }
    };
    /* start the loads of this wave's share of a chunk, part of the row of
     * trace ti, into ring slot s: WPR waves per row, 1 KiB pieces, lane l's 16
     * bytes to the piece's base + 16 l */
    const int rowbytes = ldl * (int)sizeof(float), jrow = wv / WPR;
    auto issue = [&](int ti, int s) __attribute__((always_inline)) {
        const char *src = reinterpret_cast<const char *>(a.prep + (int64_t)ti * a.row);
        char *dst = reinterpret_cast<char *>(sF + (s * C + jrow) * ldl);
        if (a.align16) {
            for (int o = (wv % WPR) * 1024; o < rowbytes; o += WPR * 1024) {
                const uint32_t lo = (uint32_t)lane * 16u;
                if (o + 1024 <= rowbytes || o + (int)lo < rowbytes)
                    __builtin_amdgcn_global_load_lds((global_void *)(src + o + lo),
                                                     (lds_void *)(dst + o), 16, 0, 0);
            }
        } else {                            /* rows that start at any float */
            for (int o = (wv % WPR) * 256; o < rowbytes; o += WPR * 256) {
                const uint32_t lo = (uint32_t)lane * 4u;
                if (o + (int)lo < rowbytes)
                    __builtin_amdgcn_global_load_lds((global_void *)(src + o + lo),
                                                     (lds_void *)(dst + o), 4, 0, 0);
            }
        }
    };

    refill();
    int slot = 0;                               /* ring slot of the current chunk */
    if (head + jrow < n) issue(__builtin_amdgcn_readfirstlane(sSel[head + jrow]), 0);
    while (n > head) {
        /* gates and distances of Kirchhoff.c:1334-1354 for the next 64 traces
         * at once (lane j = trace j), on squared distances with the exact
         * thresholds of ktm_gate_threshold */
        const int nb = min(SB, n - head);
        float g_is = 0.0f, g_ir = 0.0f;
        int g_ti = 0;
        bool gp = false;
        if (lane < nb) {
            g_ti = sSel[head + lane];
            const float4 *gg = reinterpret_cast<const float4 *>(a.geom + g_ti);
            const float4 g0 = gg[0], g1 = gg[1];
            const float ax = IX - g0.x, ay = IY - g0.y, bx = IX - g0.z, by = IY - g0.w;
            g_is = ax * ax + ay * ay;
            g_ir = bx * bx + by * by;
            const float cx = IX - g1.x, cy = IY - g1.y;
            const float ex = scx - g1.x, ey = scy - g1.y;
            gp = ex * ex + ey * ey < sthr && cx * cx + cy * cy < a.ap_x2thr;
        }
        const uint64_t pm = col_ok ? __ballot(gp) : 0ull;
        npass += __popcll(pm);
        if (SPEC) {
            g_is = finite(g_is);
            g_ir = finite(g_ir);
        }
        /* the slots that cannot reach the end of lane j's trace, the first
         * kend: their largest q (FMA and v_sqrt_f32 to 1 ulp each, so 1e-5
         * covers their rounding) is below ns - 1; and the trace's ambiguity
         * threshold, kend in its low 4 bits (which lower it by < 1e-6, taken
         * off first) */
        int kend = K;
        float qm = 0.0f;
#pragma unroll
        for (int k = K - 1; k >= 0; --k) {
            const float2 mx = sMax[wv * K + k];
            const float q = FASTIDX ? fast_qs(g_is, g_ir, mx.x, mx.y)
                                    : nsh * fast_p(g_is, g_ir, mx.x, mx.y);
            kend = q * 1.00001f < nsf - 1.0f ? kend : k;
            qm = fmaxf(qm, q);
        }
        const uint32_t g_lim =
            (__float_as_uint(ambiguous_from(qm * 1.00001f) - 1.0e-6f) & ~15u) | (uint32_t)kend;
        /* the lane's remembered sample of the window: slot | trace << 4 |
         * index << 8 (-1: none) and the sum before it */
        int qi = -1;
        float qs = 0.0f;
        for (int q = 0; q * C < nb; ++q) {
            /* chunk q's place in its window */
            const int wq = q & (WN - 1);
            /* chunk q has arrived and every wave is done with chunk q - 1,
             * so with the slot that chunk q + 1 goes to */
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            __syncthreads();
            const int nslot = slot == RING - 1 ? 0 : slot + 1;
            const int jn = (q + 1) * C + jrow;      /* this wave's row of chunk q + 1 */
            if (head + jn < n)
                issue(jn < SB ? __builtin_amdgcn_readlane(g_ti, jn)
                                    : __builtin_amdgcn_readfirstlane(sSel[head + jn]), nslot);

            uint32_t pmc = (uint32_t)(pm >> (q * C)) & ((1u << C) - 1u);
            const float *ring = sF + slot * C * ldl;
            while (pmc) {
                const int j = __builtin_ctz(pmc);    /* traces in order */
                pmc &= pmc - 1u;
                const float dIS2 = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(g_is), q * C + j));
                const float dIR2 = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(g_ir), q * C + j));
                const uint32_t lim = (uint32_t)__builtin_amdgcn_readlane((int)g_lim, q * C + j);
                const int kend = (int)(lim & 15u);
                const float *Fr = ring + j * ldl;
                /* the source term of every slot, kept while the source stays
                 * (traces of one shot follow each other) */
                if (__float_as_uint(dIS2) != lastd) {
                    lastd = __float_as_uint(dIS2);
#pragma unroll
                    for (int k = 0; k < K; ++k)
                        r1[k] = __builtin_amdgcn_sqrtf(__builtin_fmaf(dIS2, rs[k], tq[k]));
                }
                /* Hot loop, Kirchhoff.c:1374-1399: G slots at a time, their
                 * chains side by side */
                const uint32_t fr = (uint32_t)(uintptr_t)(lds_float *)Fr;
#pragma unroll
                for (int k = 0; k < K; k += G) {
                    uint32_t ad[G];
                    if (FASTIDX) {
                        float qg[G];
#pragma unroll
                        for (int i = 0; i < G; ++i)
                            qg[i] = r1[k + i] +
                                    __builtin_amdgcn_sqrtf(__builtin_fmaf(dIR2, rs[k + i], tq[k + i]));
                        if (k + G > kend) {
#pragma unroll
                            for (int i = 0; i < G; ++i) {
                                cnt[k + i] += qg[i] >= nsf ? 1.0f : 0.0f;
                                qg[i] = clamp_ns(qg[i], nsf);
                            }
                        }
#pragma unroll
                        for (int i = 0; i < G; ++i) ad[i] = ((uint32_t)fast_T(qg[i]) << 2) + fr;
                    } else {
                        float pg[G];
                        FloorP fg[G];
                        float far = 0.0f;       /* largest distance from the middle */
#pragma unroll
                        for (int i = 0; i < G; ++i) {
                            pg[i] = __builtin_amdgcn_fmed3f(
                                r1[k + i] + __builtin_amdgcn_sqrtf(__builtin_fmaf(dIR2, rs[k + i], tq[k + i])),
                                0.0f, 1.0f);
                            fg[i] = floor_p(pg[i], nsh, k + i == 0);
                            ad[i] = (__float_as_uint(fg[i].M) << 2) + (fr - 4u * KTM_FLOOR_BITS);
                            far = i ? fmaxf(far, fabsf(fg[i].dev)) : fabsf(fg[i].dev);
                        }
                        if (k + G > kend) {
                            /* past the trace, 0 or 1 */
#pragma unroll
                            for (int i = 0; i < G; ++i)
                                cnt[k + i] += __builtin_amdgcn_fmed3f(fg[i].M - past, 0.0f, 1.0f);
                        }
                        const float thr = __uint_as_float(lim);
                        if (far >= thr) {
                            const int jw = wq * C + j;
#pragma unroll
                            for (int i = 0; i < G; ++i) {
                                if (!(fabsf(fg[i].dev) >= thr)) continue;
                                const int kk = k + i;
                                const int T = floor_T(fg[i]);
                                if (qi < 0) {
                                    /* speculate: the fast index now, the
                                     * reference's at the end of the window */
                                    qi = kk | (jw << 4) | (T << 8);
                                    qs = KAHAN ? y[KAHAN ? kk : 0] : acc[kk];
                                    continue;
                                }
                                const int tl = seg * K * KTM_WAVE + kk * KTM_WAVE + lane;
                                const float v2 = vel[a.t1[tl]];
                                const int Te = exact_T(dIS2, dIR2, a.t2[tl], v2, 1.0f / v2, a.dt, a.rdt, ns);
                                cnt[kk] += (Te >= ns ? 1.0f : 0.0f) - (T >= ns ? 1.0f : 0.0f);
                                ad[i] = ((uint32_t)Te << 2) + fr;
                            }
                        }
                    }
#pragma unroll
                    for (int i = 0; i < G; ++i) {
                        const float f = *(lds_float *)(uintptr_t)ad[i];
                        if (KAHAN) y[KAHAN ? k + i : 0] = y[KAHAN ? k + i : 0] + f;
                        else acc[k + i] = acc[k + i] + f;
                    }
                }
            }
            const bool wend = wq == WN - 1 || (q + 1) * C >= nb;    /* end of the window */
            if (SPEC && wend && __ballot(qi >= 0)) {
                /* ---- the reference index of every lane's remembered sample ---- */
                const int w0 = (q - wq) * C;         /* the window's first trace */
                /* row of the window's trace jw: its chunk lies wq - jw / C
                 * slots before the current one */
                auto row_of = [&](int jw) __attribute__((always_inline)) {
                    const int s = slot - wq + jw / C;
                    return sF + ((s < 0 ? s + RING : s) * C + jw % C) * ldl;
                };
                const int jw = (qi >> 4) & 15, k = qi & 15;
                const float dIS2 = __shfl(g_is, w0 + (qi >= 0 ? jw : 0));
                const float dIR2 = __shfl(g_ir, w0 + (qi >= 0 ? jw : 0));
                const int tl = seg * K * KTM_WAVE + k * KTM_WAVE + lane;
                int Te = 0;
                float v2 = 1.0f, t2 = 0.0f;
                bool redo = false;
                if (qi >= 0) {
                    v2 = vel[a.t1[tl]];
                    t2 = a.t2[tl];
                    Te = exact_T(dIS2, dIR2, t2, v2, 1.0f / v2, a.dt, a.rdt, ns);
                    redo = Te != (qi >> 8);
                }
                if (__ballot(redo)) {
                    /* ---- rebuild the sums whose index was wrong: from the
                     * sum before it through the window's later passing
                     * traces in order (rare) ---- */
                    float s = 0.0f, rsk = 0.0f;
                    if (redo) s = qs + row_of(jw)[Te];
#pragma unroll
                    for (int kk = 0; kk < K; ++kk)
                        if (kk == k) rsk = rs[kk];
                    uint32_t later = (uint32_t)(pm >> w0) & ((1u << WT) - 1u);
                    while (later) {
                        const int jj = __builtin_ctz(later);
                        later &= later - 1u;
                        const float es = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(g_is), w0 + jj));
                        const float er = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(g_ir), w0 + jj));
                        const float *Fr = row_of(jj);
                        if (redo && jj > jw)
                            s = s + Fr[reference_T(es, er, rsk, fast_tqn(tl, nsh), t2, v2, a.dt,
                                                   a.rdt, ns, tl == 0)];
                    }
#pragma unroll
                    for (int kk = 0; kk < K; ++kk) {
                        if (!redo || kk != k) continue;
                        if (KAHAN) y[KAHAN ? kk : 0] = s;
                        else acc[kk] = s;
                        cnt[kk] +=
                            (Te >= ns ? 1.0f : 0.0f) - ((qi >> 8) >= ns ? 1.0f : 0.0f);
                    }
                }
                qi = -1;
            }
            if (KAHAN && wend && (nfold += C > 4 ? WN * (C / 4) : WN) >= KTM_KAHAN_CHUNKS) {
                nfold = 0;
                fold_y();
            }
            slot = nslot;
        }
        head += nb;
        refill();
    }
    if (KAHAN && nfold) fold_y();

    if (KAHAN && part > 0 && col_ok) {
        /* a later part of the block: its own sums, merged by k_merge_parts */
        float *pk = a.parts + (int64_t)(part - 1) * 3 * a.part_n;
        const int64_t rpix =
            (((int64_t)(X - a.rx0) * (a.ry1 - a.ry0) + (Y - a.ry0)) * a.nh + h) * ns;
#pragma unroll
        for (int k = 0; k < K; ++k) {
            const int t = seg * K * KTM_WAVE + k * KTM_WAVE + lane;
            if (t < ns) {
                pk[rpix + t] = acc[k];
                pk[a.part_n + rpix + t] = (float)npass - cnt[k];
                pk[2 * a.part_n + rpix + t] = -y[KAHAN ? k : 0];
            }
        }
        if (lane == 0 && seg == 0 && a.counter)
            atomicAdd(a.counter, (unsigned long long)npass * (unsigned long long)ns);
    } else if (col_ok) {
#pragma unroll
        for (int k = 0; k < K; ++k) {
            const int t = seg * K * KTM_WAVE + k * KTM_WAVE + lane;
            if (t < ns) {
                a.km[pix + t] = acc[k];
                /* fold adds the passing traces whose sample was inside the
                 * trace (Kirchhoff.c:1387-1396) */
                a.fold[pix + t] = a.fold[pix + t] + ((float)npass - cnt[k]);
                if (KAHAN) a.comp[pix + t] = -y[KAHAN ? k : 0];
            }
        }
        if (lane == 0 && seg == 0 && a.counter)
            atomicAdd(a.counter, (unsigned long long)npass * (unsigned long long)ns);
    }
}

/* The compensated sums of parts 1..nparts-1 of a trace block added to the
 * image (part 0 added into it directly): per sample, in FP64, the image's
 * km - comp and each part's km - comp in part order, rounded once to the new
 * km, with comp = km - the FP64 total (so km - comp keeps the total to
 * FP64); fold adds the parts' counts, which are exact.  One thread per
 * sample of the region. */
__global__ void k_merge_parts(const MigArgs a, int nparts)
{
    const int64_t ht = (int64_t)a.nh * a.ns;
    const int rny = a.ry1 - a.ry0;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < a.part_n;
         i += (int64_t)gridDim.x * blockDim.x) {
        const int64_t c = i / ht, r = i - c * ht;
        const int64_t pix = ((int64_t)(a.rx0 + c / rny) * a.nyp + (a.ry0 + c % rny)) * ht + r;
        double tot = (double)a.km[pix] - (double)a.comp[pix];
        float f = a.fold[pix];
        for (int p = 1; p < nparts; ++p) {
            const float *pk = a.parts + (int64_t)(p - 1) * 3 * a.part_n;
            tot += (double)pk[i] - (double)pk[2 * a.part_n + i];
            f += pk[a.part_n + i];
        }
        const float k = (float)tot;
        a.km[pix] = k;
        a.fold[pix] = f;
        a.comp[pix] = (float)((double)k - tot);
    }
}

/* Contributions of the traces outside the offset classes [0, nh): the
 * reference evaluates their loop body for every column in aperture and
 * drops the sum (the off test of Kirchhoff.c:1387); k_migrate never stages
 * them, so their (trace, column) pairs are counted here, with the gates of
 * k_migrate, for the contribution count.  One thread per trace. */
__global__ void k_count_outside(const MigArgs a)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= a.ntr) return;
    const ktm_trace_geom g = a.geom[i];
    if (g.off >= 0 && g.off < a.nh) return;
    uint64_t n = 0;
    for (int X = a.rx0; X < a.rx1; ++X) {
        const float cx = a.colx[X] - g.cmpx;
        if (!(cx * cx < a.ap_x2thr)) continue;   /* RN(cx^2 + cy^2) >= cx^2 */
        for (int Y = a.ry0; Y < a.ry1; ++Y) {
            const float cy = a.coly[Y] - g.cmpy;
            const int job = (X / a.nx) * a.jobs_y + (Y / a.ny);
            const float ex = a.slab_cx[job] - g.cmpx, ey = a.slab_cy[job] - g.cmpy;
            n += (ex * ex + ey * ey < a.slab_x2thr[job] && cx * cx + cy * cy < a.ap_x2thr) ? 1u : 0u;
        }
    }
    if (n) atomicAdd(a.counter, (unsigned long long)(n * (uint64_t)a.ns));
}

/* ------------------------------------------------------------------------ */
/* image reset and post-stack                                                */
/* ------------------------------------------------------------------------ */
__global__ void k_image_reset(float *km, float *fold, float *comp, int64_t n)
{
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
         i += (int64_t)gridDim.x * blockDim.x) {
        km[i] = 0.0f;
        fold[i] = 1.0f;
        if (comp) comp[i] = 0.0f;
    }
}

/* The post-stack low-pass of Kirchhoff.c:1457-1479 multiplies the DFT by the
 * even real spectrum anti_alias, i.e. it is the circular convolution
 * out[t] = sum_u h[(t-u) mod ns] d[u] with h the (real) inverse DFT of
 * anti_alias divided by ns, evaluated in FP64; h2[m] = h[m mod ns] for
 * m < 2 ns.  PS_NT: threads per workgroup of the transpose. */
#define PS_NT 256

/* x of the post-stack filter, Kirchhoff.c:1460: a float expression stored
 * into a double */
struct PostKtm {
    static __device__ __forceinline__ float3 load(const float *k, const float *f, int u)
    {
        return make_float3(k[u], k[u - 1], f[u]);
    }
    static __device__ __forceinline__ double value(float3 l, int u, float dt)
    {
        return (double)(-dt * (float)u * (l.x - l.y) * dt / l.z);
    }
};

/* ------------------------------------------------------------------------ */
/* seeded synthetic surveys                                                  */
/* ------------------------------------------------------------------------ */
/* One workgroup per trace: the DSR diffraction time of every scatterer,
 *   tau_j = sqrt((t0/2)^2 + |s-x_j|^2/v_j^2) + sqrt((t0/2)^2 + |g-x_j|^2/v_j^2),
 * v_j = v0 + vt*t0_j + vx*x_j, in LDS; then each sample sums the Ricker
 * wavelets (1 - 2 a) exp(-a), a = (pi f0 (t dt - tau_j))^2, of the scatterers
 * within 2/f0 (the wavelet is below 1e-13 there), in scatterer order. */
#define SYN_NT 256
#define SYN_MAXSCAT 1024
__global__ void __launch_bounds__(SYN_NT)
k_synth_traces(const ktm_trace_geom *__restrict__ geom, int64_t ntr, int ns, float dt,
               const float *__restrict__ scat, int nscat, float f0, float v0, float vt, float vx,
               float *__restrict__ traces)
{
    __shared__ float s_tau[SYN_MAXSCAT], s_amp[SYN_MAXSCAT];
    const int64_t i = blockIdx.x;
    if (i >= ntr) return;
    const ktm_trace_geom g = geom[i];
    for (int j = threadIdx.x; j < nscat; j += SYN_NT) {
        const double x = scat[4 * j], y = scat[4 * j + 1], t0 = scat[4 * j + 2];
        const double v = (double)v0 + (double)vt * t0 + (double)vx * x;
        const double h = 0.25 * t0 * t0, iv2 = 1.0 / (v * v);
        const double ds2 = (g.sxt - x) * (g.sxt - x) + (g.syt - y) * (g.syt - y);
        const double dg2 = (g.gxt - x) * (g.gxt - x) + (g.gyt - y) * (g.gyt - y);
        s_tau[j] = (float)(sqrt(h + ds2 * iv2) + sqrt(h + dg2 * iv2));
        s_amp[j] = scat[4 * j + 3];
    }
    __syncthreads();
    const float win = 2.0f / f0;
    const float pf = 3.14159265358979f * f0;
    float *o = traces + i * (int64_t)ns;
    for (int t = threadIdx.x; t < ns; t += SYN_NT) {
        const float tt = (float)t * dt;
        float acc = 0.0f;
        for (int j = 0; j < nscat; ++j) {
            const float d = tt - s_tau[j];
            if (fabsf(d) < win) {
                const float a = (pf * d) * (pf * d);
                acc += s_amp[j] * (1.0f - 2.0f * a) * expf(-a);
            }
        }
        o[t] = acc;
    }
}

/* counter-based Gaussian noise: SplitMix64 of (seed, index) -> two uniforms
 * -> Box-Muller; the value at an index does not depend on the launch shape */
__device__ __forceinline__ uint64_t splitmix64(uint64_t z)
{
    z += 0x9E3779B97F4A7C15ull;
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    return z ^ (z >> 31);
}

__global__ void k_synth_noise(float *traces, int64_t n, float sigma, uint64_t seed)
{
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
         i += (int64_t)gridDim.x * blockDim.x) {
        const uint64_t r = splitmix64(seed ^ splitmix64((uint64_t)i));
        const double u1 = ((double)(r >> 40) + 0.5) * (1.0 / 16777216.0);
        const double u2 = (double)((r >> 16) & 0xffffffull) * (1.0 / 16777216.0);
        const double z = sqrt(-2.0 * log(u1)) * cos(6.283185307179586 * u2);
        traces[i] += (float)(sigma * z);
    }
}

extern "C" int ktm_synth_traces(const ktm_plan *p, const ktm_trace_geom *geom, int64_t ntr,
                                const float *scat, int nscat, float f0, float v0, float vt,
                                float vx, float *traces, void *stream)
{
    if (!p || ntr < 0 || nscat < 0 || nscat > SYN_MAXSCAT || !(f0 > 0.0f)) return KTM_ERR_ARG;
    if (!ntr) return KTM_OK;
    if (!geom || !traces || (nscat && !scat)) return KTM_ERR_ARG;
    for (int64_t i0 = 0; i0 < ntr; i0 += 1 << 30) {
        const int64_t n = ntr - i0 < (1 << 30) ? ntr - i0 : (1 << 30);
        hipLaunchKernelGGL(k_synth_traces, dim3((unsigned)n), dim3(SYN_NT), 0, (hipStream_t)stream,
                           geom + i0, n, p->tb.s.ns, p->tb.s.dt, scat, nscat, f0, v0, vt, vx,
                           traces + i0 * p->tb.s.ns);
    }
    HIP_TRY(hipGetLastError());
    return KTM_OK;
}

extern "C" int ktm_synth_noise(float *traces, int64_t n, float sigma, uint64_t seed, void *stream)
{
    if (n < 0 || (n && !traces)) return KTM_ERR_ARG;
    if (!n) return KTM_OK;
    hipLaunchKernelGGL(k_synth_noise, dim3(4096), dim3(256), 0, (hipStream_t)stream, traces, n,
                       sigma, seed);
    HIP_TRY(hipGetLastError());
    return KTM_OK;
}

/* LDS read bandwidth probe: every workgroup fills 16 KB of LDS, then each
 * lane reads 16 bytes per step from a conflict-free rotating position,
 * folded with xor so the VALU work per byte stays well below the LDS rate;
 * one word per lane is written so the reads are not removed.  Reads
 * nblocks * 256 * iters * 4 * 16 bytes of LDS. */
__global__ void __launch_bounds__(256) k_probe_lds(uint32_t *__restrict__ out, int iters)
{
    __shared__ uint4 buf[4 * 256];
    const int tid = threadIdx.x;
    for (int k = 0; k < 4; ++k)
        buf[k * 256 + tid] = make_uint4(tid * 4u + k, tid ^ 0x55u, blockIdx.x, k * 7u + 1u);
    __syncthreads();
    uint32_t a = 0u, b = 0u;
    for (int i = 0; i < iters; ++i) {
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const uint4 v = buf[k * 256 + ((tid + i) & 255)];
            a ^= v.x ^ v.y;
            b ^= v.z ^ v.w;
        }
    }
    out[(int64_t)blockIdx.x * 256 + tid] = a ^ b;
}

extern "C" int ktm_probe_lds(uint32_t *out, int nblocks, int iters, void *stream)
{
    if (!out || nblocks < 1 || iters < 1) return KTM_ERR_ARG;
    hipLaunchKernelGGL(k_probe_lds, dim3((unsigned)nblocks), dim3(256), 0, (hipStream_t)stream,
                       out, iters);
    HIP_TRY(hipGetLastError());
    return KTM_OK;
}

/* ------------------------------------------------------------------------ */
/* self-tests of the numerical assumptions of the fast traveltime path       */
/* ------------------------------------------------------------------------ */
/* out_hw[i] = v_sqrt_f32(x[i]) */
__global__ void k_selftest_sqrt(const float *__restrict__ x, int64_t n, float *__restrict__ out_hw)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) out_hw[i] = __builtin_amdgcn_sqrtf(x[i]);
}

/* For in[i] = (dIS2, dIR2, t, v2) (t a sample index held as a float):
 * q_fast of the migration kernel, the reference Q = RN(dsr/dt) (float,
 * before the floor), and the T each selects; t2 is the table's value. */
__global__ void k_selftest_traveltime(const float4 *__restrict__ in, int64_t n, float dt, int ns,
                                      float *__restrict__ q_fast, float *__restrict__ q_ref,
                                      int *__restrict__ t_kernel, int *__restrict__ t_ref)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float4 in4 = in[i];
    const int t = (int)in4.z;
    const float4 v = make_float4(in4.x, in4.y, (float)(0.25 * t * t * dt * dt), in4.w);
    const float rdt = 1.0f / dt;
    const float q = fast_qs(v.x, v.y, fast_rs(v.w, dt), fast_tq(t));
    /* the decision procedure of k_migrate */
    const float nsf = (float)ns, nsh = nsf + 0.5f;
    const int T = reference_T(v.x, v.y, fast_rsn(v.w, dt, nsh), fast_tqn(t, nsh), v.z, v.w, dt, rdt,
                              ns, t == 0);
    /* the reference computed independently of exact_T: the compiler's
     * correctly rounded division and double square root */
    const float s1 = v.z + v.x / v.w, s2 = v.z + v.y / v.w;
    const float dsr = (float)(__builtin_sqrt((double)s1) + __builtin_sqrt((double)s2));
    const float qq = dsr / dt;
    q_fast[i] = q;
    q_ref[i] = qq;
    t_kernel[i] = T;
    t_ref[i] = qq < nsf ? (int)qq : ns;
}

/* the exact migration kernel's form of q, p nsh, without a further rounding */
__global__ void k_selftest_limited(const float4 *__restrict__ in, int64_t n, float dt, int ns,
                                   double *__restrict__ q)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float4 v = in[i];
    const float nsh = (float)ns + 0.5f;
    q[i] = (double)fast_p(v.x, v.y, fast_rsn(v.w, dt, nsh), fast_tqn((int)v.z, nsh)) * (double)nsh;
}

extern "C" int ktm_selftest_limited(const float *in4, int64_t n, float dt, int ns, double *q,
                                    void *stream)
{
    if (n < 0 || (n && (!in4 || !q))) return KTM_ERR_ARG;
    if (!n) return KTM_OK;
    hipLaunchKernelGGL(k_selftest_limited, dim3((unsigned)((n + 255) / 256)), dim3(256), 0,
                       (hipStream_t)stream, (const float4 *)in4, n, dt, ns, q);
    HIP_TRY(hipGetLastError());
    return KTM_OK;
}

extern "C" int ktm_selftest_sqrt(const float *x, int64_t n, float *out_hw, void *stream)
{
    if (n < 0 || (n && (!x || !out_hw))) return KTM_ERR_ARG;
    if (!n) return KTM_OK;
    hipLaunchKernelGGL(k_selftest_sqrt, dim3((unsigned)((n + 255) / 256)), dim3(256), 0,
                       (hipStream_t)stream, x, n, out_hw);
    HIP_TRY(hipGetLastError());
    return KTM_OK;
}

extern "C" int ktm_selftest_traveltime(const float *in4, int64_t n, float dt, int ns, float *q_fast,
                                       float *q_ref, int32_t *t_kernel, int32_t *t_ref, void *stream)
{
    if (n < 0 || (n && (!in4 || !q_fast || !q_ref || !t_kernel || !t_ref))) return KTM_ERR_ARG;
    if (!n) return KTM_OK;
    hipLaunchKernelGGL(k_selftest_traveltime, dim3((unsigned)((n + 255) / 256)), dim3(256), 0,
                       (hipStream_t)stream, (const float4 *)in4, n, dt, ns, q_fast, q_ref,
                       t_kernel, t_ref);
    HIP_TRY(hipGetLastError());
    return KTM_OK;
}


/* ------------------------------------------------------------------------ */
/* adjoint pair: demigration (L) and the post-stack transpose                */
/* ------------------------------------------------------------------------ */
/* Per-pixel velocity tables for trace-parallel kernels: v2 and rs =
 * RN(1/(v2 dt^2)) of every (column, sample), the values k_migrate derives
 * per lane. */
__global__ void k_pixel_velocity(const float *__restrict__ vel2, const int32_t *__restrict__ velx,
                                 const int32_t *__restrict__ vely, const int32_t *__restrict__ t1,
                                 int nxp, int nyp, int ns, int nvel_xl, int nsm, float dt,
                                 float *__restrict__ pv2, float *__restrict__ prs)
{
    const int64_t n = (int64_t)nxp * nyp * ns;
    for (int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; e < n;
         e += (int64_t)gridDim.x * blockDim.x) {
        const int t = (int)(e % ns);
        const int64_t c = e / ns;
        const int X = (int)(c / nyp), Y = (int)(c % nyp);
        const float v2 = vel2[((int64_t)velx[X] * nvel_xl + vely[Y]) * nsm + t1[t]];
        pv2[e] = v2;
        prs[e] = fast_rs(v2, dt);
    }
}

#define DM_TB 8                      /* traces per demigration workgroup, at most */
#define DM_PAD KTM_WAVE              /* words past g[ns - 1]: one per lane */

struct DemigArgs {
    const float *km;                 /* image [nxp][nyp][nh][ns] */
    const ktm_trace_geom *geom;
    const int32_t *order;            /* trace order (workgroup b takes order[b*tb ...]) */
    int64_t ntr;
    float *traces;                   /* out [ntr][ns] */
    unsigned long long *gsum;        /* columns in parts (gridDim.y > 1): [ntr][ns], zeroed */
    const float *pv2, *prs, *t2, *w, *colx, *coly, *slab_cx, *slab_cy, *slab_x2thr;
    const uint32_t *amax;            /* bits of max |km| (k_absmax) */
    float ap_x2thr, aperture, dt, rdt;
    int ns, nh, nxp, nyp, nx, ny, jobs_y, tb;
    int lg_terms;                    /* 2^lg_terms >= nxp * nyp * ns, terms per g[T] at most */
};

/* the fixed point of g: km is scaled by 2^E, max |km| < 2^emax, so that a sum
 * of 2^lg_terms terms stays below 2^59 */
__device__ __forceinline__ int demig_exponent(const DemigArgs &a)
{
    const float amax = __uint_as_float(*a.amax);
    int emax = 0;
    if (amax > 0.0f) (void)frexpf(amax, &emax);
    return 59 - emax - a.lg_terms;
}

/* trunc(m 2^E) as an integer.  NARROW (|m 2^E| < 2^51: a finite image of more
 * than 128 samples): the double sum with 1.5 * 2^52 holds it in its low bits;
 * the compiler's float to 64-bit conversion takes twice the instructions. */
template <bool NARROW> __device__ __forceinline__ unsigned long long to_fixed(float m, int E)
{
    if (!NARROW) return (unsigned long long)(long long)ldexpf(m, E);
    constexpr double MAGIC = 6755399441055744.0;
    const double s = __builtin_trunc(__builtin_amdgcn_ldexp((double)m, E)) + MAGIC;
    return (unsigned long long)__double_as_longlong(s) -
           (unsigned long long)__double_as_longlong(MAGIC);
}

/* sample t of L m from the trace's sums g[0..ns): the transpose of F =
 * closed_tap(x), x[t] = tr[min(t, ns-1)] * w[t], in double from the
 * fixed-point sums (q = 2^-E) */
__device__ __forceinline__ float demig_sample(const long long *gl, int t, int ns, const float *w,
                                              double q)
{
    double acc = 0.0;
    const int nt_ = t == ns - 1 ? 3 : 1;   /* tr[ns-1] also feeds x[ns], x[ns+1] */
    for (int u = 0; u < nt_; ++u) {
        const int tt = t + u;
        long long xb = 0;                  /* exact: |g| < 2^59, weights summing to <= 6 */
        if (tt >= 2 && tt < ns) xb += gl[tt];
        if (tt - 1 >= 2 && tt - 1 < ns) xb += 2 * gl[tt - 1];
        if (tt - 2 >= 2 && tt - 2 < ns) xb += gl[tt - 2];
        if (tt == 0) xb += 4 * gl[0] + 2 * gl[1];
        if (tt == 1) xb += 4 * gl[0] + 2 * gl[1];
        if (tt == 2) xb += 2 * gl[0] + 2 * gl[1];
        if (tt == 3) xb += gl[1];
        acc += (double)w[tt] * ((double)xb * q);
    }
    return (float)acc;
}

/* *out = bits of max |x| over n floats (out zeroed by k_zero_u32 first;
 * non-negative floats order like their bit patterns) */
__global__ void k_zero_u32(uint32_t *out) { *out = 0u; }
__global__ void k_absmax(const float *__restrict__ x, int64_t n, uint32_t *out)
{
    uint32_t m = 0u;
    for (int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; e < n;
         e += (int64_t)gridDim.x * blockDim.x)
        m = max(m, __float_as_uint(x[e]) & 0x7fffffffu);
    for (int d = KTM_WAVE / 2; d >= 1; d >>= 1) m = max(m, (uint32_t)__shfl_xor((int)m, d));
    if ((threadIdx.x & (KTM_WAVE - 1)) == 0) atomicMax(out, m);
}

/* Column index range whose centres can be within the aperture of a CMP at
 * coordinate c on an axis of n columns from col[0] to col[n-1]. */
__device__ __forceinline__ void aperture_span(const float *col, int n, float c, float aperture,
                                              int *lo, int *hi)
{
    *lo = 0;
    *hi = n - 1;
    if (n > 1) {
        const float step = (col[n - 1] - col[0]) / (float)(n - 1);
        if (step != 0.0f) {
            const float xc = (c - col[0]) / step, half = aperture / fabsf(step) + 2.0f;
            *lo = max(0, (int)floorf(xc - half));
            *hi = min(n - 1, (int)ceilf(xc + half));
        }
    }
}

/* Sort keys of the demigration trace order: offset class (out-of-class
 * traces last), then the CMP's image cell, row by row, so the traces one
 * workgroup takes lie close together and share their columns -- and within
 * eight cells of a row by source, so that traces of one shot come together
 * and share their source's roots.  The order is a matter of speed only, so
 * each field keeps just its low bits (12, 20, 18, 11 and 3). */
__global__ void k_demig_keys(const ktm_trace_geom *__restrict__ geom, int64_t ntr, int nh,
                             const float *__restrict__ colx, int nxp, const float *__restrict__ coly,
                             int nyp, uint64_t *__restrict__ keys, int32_t *__restrict__ idx)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= ntr) return;
    const ktm_trace_geom g = geom[i];
    const uint64_t cls = g.off >= 0 && g.off < nh ? (uint64_t)g.off : (uint64_t)nh;
    uint64_t cell[2] = {0, 0};
    const float *col[2] = {colx, coly};
    const int n[2] = {nxp, nyp};
    const float c[2] = {g.cmpx, g.cmpy};
    for (int d = 0; d < 2; ++d) {
        if (n[d] < 2) continue;
        const float step = (col[d][n[d] - 1] - col[d][0]) / (float)(n[d] - 1);
        if (step == 0.0f) continue;
        /* fminf/fmaxf return the number for a NaN operand */
        const float f = fminf(fmaxf(floorf((c[d] - col[d][0]) / step), -1.0f), (float)n[d]);
        cell[d] = (uint64_t)((int)f + 1);
    }
    uint32_t src = __float_as_uint(g.sxt) * 0x9E3779B1u ^ __float_as_uint(g.syt) * 0x85EBCA77u;
    src = (src ^ (src >> 15)) & 0x7ffu;
    keys[i] = (cls & 0xfffull) << 52 | (cell[1] & 0xfffffull) << 32 | (cell[0] >> 3 & 0x3ffffull) << 14 |
              (uint64_t)src << 3 | (cell[0] & 7ull);
    idx[i] = (int32_t)i;
}

/* add v to the LDS word at byte address ad */
__device__ __forceinline__ void lds_add(uint32_t ad, unsigned long long v)
{
    (void)__hip_atomic_fetch_add((lds_u64 *)(uintptr_t)ad, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

/* the largest of a wave's non-negative floats, in a scalar */
__device__ __forceinline__ float wave_max(float v)
{
    int m = __float_as_int(v);
#define KTM_DPP_MAX(ctrl, rows) m = max(m, __builtin_amdgcn_update_dpp(m, m, ctrl, rows, 0xf, false))
    KTM_DPP_MAX(0x111, 0xf);    /* row_shr 1, 2, 4, 8 */
    KTM_DPP_MAX(0x112, 0xf);
    KTM_DPP_MAX(0x114, 0xf);
    KTM_DPP_MAX(0x118, 0xf);
    KTM_DPP_MAX(0x142, 0xa);    /* row_bcast 15, 31 */
    KTM_DPP_MAX(0x143, 0xc);
#undef KTM_DPP_MAX
    return __int_as_float(__builtin_amdgcn_readlane(m, 63));
}

/* L, the exact transpose of migration with the CLOSED filter (km = L^T d).
 * A workgroup takes up to DM_TB traces, neighbours in the sort order of
 * k_demig_keys: the waves walk the image columns of the union of their
 * aperture boxes, gate every trace for the column exactly like k_migrate
 * (lane j = trace j), and for each passing trace and every sample t with
 * T(t) < ns add km[column][off][t] into that trace's g[T] (LDS atomics).
 * The column's image samples and rs are loaded once for all its traces.
 * g is 64-bit fixed point, km scaled by 2^E with max |km| < 2^(59 - E -
 * lg_terms), so no sum of at most 2^lg_terms terms passes 2^59 and the
 * filter's combinations of six stay below 2^62: integer LDS
 * atomics run at the rate of plain stores where float ones serialise over
 * the lanes (measured 22 vs 193 ms on the 48,000-trace line), and the
 * integer sums make L deterministic.  The quantum is 2^-E, at most
 * max |km| * 2^(lg_terms - 59).
 * Each trace is then the transpose of the 3-tap filter and of the sample
 * weights applied to its g.
 * Lane l owns samples l*K + ((k + l / P) mod K) of its wave's 64K-sample
 * segment, not k*64 + l: far from the CMP, T(t) grows slowly at early
 * times, and 64 consecutive samples land on a few T, whose atomics then
 * serialise; samples K apart land on distinct T, and with P = 32 / gcd(K, 32)
 * the 64 lanes' T spread over all banks where T(t) = t + const.  A sample past
 * the trace is clamped to ns + lane + 1/2 and adds into its lane's own unread
 * word (all lanes adding into one word serialised: with offsets up to 4 km
 * and 751 samples that was most of the time).
 * A sample whose fast-form q lies within the form's error bound of an
 * integer needs the reference arithmetic: each lane defers its first such
 * sample of a column and the wave resolves them after the column's traces,
 * every lane's together (the integer sums do not depend on the order of the
 * additions); a lane's further ones in the column take it inline.  The test is
 * k_migrate's: one threshold per trace, at the largest q of its samples in
 * the column, for G slots at a time.
 * FASTIDX: the index floor(min(q, ns + lane + 1/2)) of the fast form alone,
 * the transpose of k_migrate's FASTIDX variant (floor(min(q, ns)) there: both
 * are >= ns for q >= ns, so they index the same samples).
 * Few traces leave the chip idle (demig_parts): gridDim.y parts then take every
 * gridDim.y-th column of a group's box each, add their sums into gsum
 * (integers: in any order) and k_demig_finish forms the traces.
 * Bound by VALU issue like k_migrate, the image samples' conversion to fixed
 * point and the gates shared by the traces of a column.  48,000 traces x 1501
 * samples, 1600 columns: 23.0 -> 18.9 ms against a test, a branch and a
 * quarter-rate floor per slot and addresses formed anew for every column;
 * 3001 traces x 751 of a wide-azimuth patch of 61 x 61 columns, relaxed
 * index: 25.7 -> 3.0 ms, by the words past the trace and the column parts. */
template <int K, int W, bool FASTIDX>
__global__ void __launch_bounds__(8 * KTM_WAVE) __attribute__((amdgpu_waves_per_eu(4, 4)))
k_demigrate(const DemigArgs a)
{
    constexpr int NCOL = 8 / W;
    constexpr int G = mig_group(K);                /* slots side by side */
    extern __shared__ unsigned long long sg[];     /* [tb][ns + DM_PAD] fixed point */
    __shared__ int32_t sIdx[DM_TB];
    const int tid = threadIdx.x, lane = tid & (KTM_WAVE - 1);
    const int wv = __builtin_amdgcn_readfirstlane(tid / KTM_WAVE);
    const int cw = wv / W, seg = wv % W;
    const int ns = a.ns, ldg = ns + DM_PAD;
    const int64_t b0 = (int64_t)blockIdx.x * a.tb;
    const int nb = (int)min((int64_t)a.tb, a.ntr - b0);
    for (int e = tid; e < a.tb * ldg; e += 8 * KTM_WAVE) sg[e] = 0ull;
    const int E = demig_exponent(a);
    const bool narrow = a.lg_terms >= 8 && __builtin_amdgcn_readfirstlane((int)*a.amax) < 0x7f800000;
    /* lane j < nb of every wave holds trace j of the workgroup */
    ktm_trace_geom g;
    memset(&g, 0, sizeof g);
    bool valid = false;
    int gi = 0;
    int xlo = a.nxp, xhi = -1, ylo = a.nyp, yhi = -1;
    if (lane < nb) {
        gi = a.order[b0 + lane];
        g = a.geom[gi];
        valid = g.off >= 0 && g.off < a.nh;
        if (valid) {
            aperture_span(a.colx, a.nxp, g.cmpx, a.aperture, &xlo, &xhi);
            aperture_span(a.coly, a.nyp, g.cmpy, a.aperture, &ylo, &yhi);
        }
    }
    if (tid < nb) sIdx[tid] = gi;
    for (int m = KTM_WAVE / 2; m >= 1; m >>= 1) {
        xlo = min(xlo, __shfl_xor(xlo, m));
        xhi = max(xhi, __shfl_xor(xhi, m));
        ylo = min(ylo, __shfl_xor(ylo, m));
        yhi = max(yhi, __shfl_xor(yhi, m));
    }
    xlo = __builtin_amdgcn_readfirstlane(xlo); xhi = __builtin_amdgcn_readfirstlane(xhi);
    ylo = __builtin_amdgcn_readfirstlane(ylo); yhi = __builtin_amdgcn_readfirstlane(yhi);
    __syncthreads();
    const float qlim = (float)(ns + lane) + 0.5f;  /* clamp of q */
    constexpr int P = K % 8 == 0 ? 4 : K % 4 == 0 ? 8 : 16;
    static_assert(K % 2 == 0 && K <= 12, "P = 32 / gcd(K, 32)");
    const int rot = lane / P % K, tbase = seg * K * KTM_WAVE + lane * K;
    auto slot_t = [&](int k) __attribute__((always_inline)) {   /* sample of slot k */
        return tbase + (k + rot < K ? k + rot : k + rot - K);
    };
    /* past the end, tq puts q beyond every clamp */
    const float tq_past = 0.25f * (float)(ns + 2 * KTM_WAVE) * (float)(ns + 2 * KTM_WAVE);
    float tq[K];
    uint32_t to[K];                                /* the slot's sample, at most ns - 1 */
#pragma unroll
    for (int k = 0; k < K; ++k) {
        const int t = slot_t(k);
        tq[k] = t < ns ? fast_tq(t) : tq_past;
        to[k] = (uint32_t)min(t, ns - 1);
    }
    const float tq_max = fast_tq(min(ns, (seg + 1) * K * KTM_WAVE) - 1);
    const int nbx = xhi - xlo + 1, nby = yhi - ylo + 1;
    const int ncols = nbx > 0 && nby > 0 ? nbx * nby : 0;
    const int cstep = NCOL * (int)gridDim.y;
    for (int cidx = cw + NCOL * (int)blockIdx.y; cidx < ncols; cidx += cstep) {
        const int X = xlo + cidx / nby, Y = ylo + cidx % nby;
        const float IX = a.colx[X], IY = a.coly[Y];
        const int job = (X / a.nx) * a.jobs_y + (Y / a.ny);
        float g_is = 0.0f, g_ir = 0.0f;
        bool gp = false;
        if (valid) {
            const float ex = a.slab_cx[job] - g.cmpx, ey = a.slab_cy[job] - g.cmpy;
            const float cx = IX - g.cmpx, cy = IY - g.cmpy;
            gp = ex * ex + ey * ey < a.slab_x2thr[job] && cx * cx + cy * cy < a.ap_x2thr;
            const float ax = IX - g.sxt, ay = IY - g.syt, bx = IX - g.gxt, by = IY - g.gyt;
            g_is = ax * ax + ay * ay;
            g_ir = bx * bx + by * by;
        }
        uint64_t pm = __ballot(gp);
        if (!pm) continue;
        const int64_t pixc = ((int64_t)X * a.nyp + Y) * ns;
        const float *rc = a.prs + pixc;
        float rs[K];
        unsigned long long mq[K];          /* km samples, fixed point */
#pragma unroll
        for (int k = 0; k < K; ++k) {
            rs[k] = rc[to[k]];
            mq[k] = 0ull;
        }
        float g_thr = 0.0f;                /* lane j: trace j's ambiguity threshold */
        if (!FASTIDX) {
            float m = rs[0];
#pragma unroll
            for (int k = 1; k < K; ++k) m = fmaxf(m, rs[k]);
            g_thr = ambiguous_from(fminf(fast_qs(g_is, g_ir, wave_max(m), tq_max) * 1.00001f,
                                         (float)ns + 1.0f));
        }
        uint32_t lastd = 0xffffffffu;      /* bits of the source distance of r1 (none: a NaN) */
        float r1[K];
#pragma unroll
        for (int k = 0; k < K; ++k) r1[k] = 0.0f;
        int cur = -1;                      /* offset class whose samples mq holds */
        /* one ambiguous sample per lane deferred to the end of the column:
         * its slot | trace << 8 (-1: none) and its fixed-point value */
        int qkj = -1;
        unsigned long long qv = 0;
        while (pm) {
            const int j = __builtin_ctzll(pm);
            pm &= pm - 1ull;
            const float dIS2 = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(g_is), j));
            const float dIR2 = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(g_ir), j));
            const int offj = __builtin_amdgcn_readlane(g.off, j);
            if (offj != cur) {
                cur = offj;
                const float *mk = a.km + (((int64_t)X * a.nyp + Y) * a.nh + offj) * ns;
                float m[K];
#pragma unroll
                for (int k = 0; k < K; ++k) m[k] = mk[to[k]];
                if (narrow) {
#pragma unroll
                    for (int k = 0; k < K; ++k) mq[k] = to_fixed<true>(m[k], E);
                } else {
#pragma unroll
                    for (int k = 0; k < K; ++k) mq[k] = to_fixed<false>(m[k], E);
                }
            }
            /* the source's roots, kept for the column's traces of one source */
            if (__float_as_uint(dIS2) != lastd) {
                lastd = __float_as_uint(dIS2);
#pragma unroll
                for (int k = 0; k < K; ++k)
                    r1[k] = __builtin_amdgcn_sqrtf(__builtin_fmaf(dIS2, rs[k], tq[k]));
            }
            const uint32_t gl = (uint32_t)(uintptr_t)(lds_u64 *)(sg + j * ldg);
            if (FASTIDX) {
#pragma unroll
                for (int k = 0; k < K; ++k) {
                    const float qc = fast_clamp(
                        r1[k] + __builtin_amdgcn_sqrtf(__builtin_fmaf(dIR2, rs[k], tq[k])), qlim);
                    lds_add(((uint32_t)fast_T(qc) << 3) + gl, mq[k]);
                }
                continue;
            }
            const float thr = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(g_thr), j));
#pragma unroll
            for (int k = 0; k < K; k += G) {
                uint32_t ad[G];
                float dev[G], far = 0.0f;
#pragma unroll
                for (int i = 0; i < G; ++i) {
                    const float qc = fast_clamp(
                        r1[k + i] + __builtin_amdgcn_sqrtf(__builtin_fmaf(dIR2, rs[k + i], tq[k + i])), qlim);
                    /* floor_p's rounding, on q itself; t = 0 is in slot 0 */
                    float M = qc + KTM_FLOOR_MAGIC;
                    if (k + i == 0) M = fmaxf(M, 8388608.0f);
                    dev[i] = qc - (M - KTM_FLOOR_MAGIC);
                    ad[i] = (__float_as_uint(M) << 3) + (gl - 8u * KTM_FLOOR_BITS);
                    far = i ? fmaxf(far, fabsf(dev[i])) : fabsf(dev[i]);
                }
                if (far >= thr) {
#pragma unroll
                    for (int i = 0; i < G; ++i) {
                        if (!(fabsf(dev[i]) >= thr)) continue;
                        int T = ns + lane;
                        if (qkj < 0) {
                            /* deferred: the integer sums do not depend on the
                             * order of their additions */
                            qkj = (k + i) | (j << 8);
                            qv = mq[k + i];
                        } else {
                            /* (hidden, so that the compiler does not hold
                             * every slot's addresses in registers) */
                            uint32_t t = to[k + i];
                            asm volatile("" : "+v"(t));
                            const float v2 = a.pv2[pixc + t];
                            const int Te = exact_T(dIS2, dIR2, a.t2[t], v2, 1.0f / v2, a.dt, a.rdt, ns);
                            if (Te < ns && tq[k + i] != tq_past) T = Te;
                        }
                        ad[i] = ((uint32_t)T << 3) + gl;
                    }
                }
#pragma unroll
                for (int i = 0; i < G; ++i) lds_add(ad[i], mq[k + i]);
            }
        }
        if (!FASTIDX && __ballot(qkj >= 0)) {
            /* the deferred samples of the column, every lane's together:
             * one reference-arithmetic pass instead of one per ambiguous
             * lane and slot (the trace's distances from its lane, all lanes
             * active for the shuffle) */
            const int jq = qkj >= 0 ? qkj >> 8 : 0;
            const float dIS2 = __shfl(g_is, jq), dIR2 = __shfl(g_ir, jq);
            if (qkj >= 0) {
                const int t = slot_t(qkj & 0xff);
                if (t < ns) {
                    const float v2 = a.pv2[pixc + t];
                    const int T = exact_T(dIS2, dIR2, a.t2[t], v2, 1.0f / v2, a.dt, a.rdt, ns);
                    if (T < ns) atomicAdd(&sg[jq * ldg + T], qv);
                }
            }
        }
    }
    __syncthreads();
    if (gridDim.y > 1) {
        for (int e = tid; e < nb * ns; e += 8 * KTM_WAVE) {
            const int j = e / ns, t = e - j * ns;
            const unsigned long long v = sg[j * ldg + t];
            if (v) atomicAdd(a.gsum + (int64_t)sIdx[j] * ns + t, v);
        }
        return;
    }
    const double q = ldexp(1.0, -E);
    for (int e = tid; e < nb * ns; e += 8 * KTM_WAVE) {
        const int j = e / ns, t = e - j * ns;
        a.traces[(int64_t)sIdx[j] * ns + t] =
            demig_sample(reinterpret_cast<const long long *>(sg + j * ldg), t, ns, a.w, q);
    }
}

/* the traces of a demigration whose columns were taken in parts: one
 * workgroup per trace */
__global__ void __launch_bounds__(256) k_demig_finish(const DemigArgs a)
{
    const double q = ldexp(1.0, -demig_exponent(a));
    const int64_t o = (int64_t)blockIdx.x * a.ns;
    for (int t = threadIdx.x; t < a.ns; t += 256)
        a.traces[o + t] = demig_sample(reinterpret_cast<const long long *>(a.gsum + o), t, a.ns, a.w, q);
}

__global__ void k_zero_u64(unsigned long long *p, int64_t n)
{
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
         i += (int64_t)gridDim.x * blockDim.x)
        p[i] = 0ull;
}

/* Transpose of the post-stack chain image = P0 H C D km of Kirchhoff.c:
 * 1457-1479 (D: first difference with d[0] = 0, C: -dt^2 t / fold[t],
 * H: the even circular low-pass, P0: out[0] = 0):  km_bar = D^T C H P0 img.
 * H is symmetric (h even), so w = H P0 img is the post-stack convolution of
 * img itself (k_postfft<PostImg> or k_postmx<PostImg>, written into out);
 * this kernel finishes a
 * trace per workgroup in place: uu[t] = C[t] w[t] (FP64, uu[0] = uu[ns] = 0),
 * out[t] = uu[t] - uu[t + 1]. */
struct PostImg {
    static __device__ __forceinline__ float3 load(const float *im, const float *, int u)
    {
        return make_float3(im[u], 0.0f, 0.0f);
    }
    static __device__ __forceinline__ double value(float3 l, int, float) { return (double)l.x; }
};

__global__ void __launch_bounds__(PS_NT) k_poststack_adjoint_tail(const float *__restrict__ fold,
                                                                  int ns, float dt, float *out)
{
    extern __shared__ double uu[];                     /* [ns + 1] */
    const int64_t tr = blockIdx.x;
    float *o = out + tr * ns;
    const float *f = fold + tr * ns;
    for (int t = threadIdx.x; t <= ns; t += PS_NT) {
        double v = 0.0;
        if (t >= 1 && t < ns) v = -(double)dt * (double)dt * (double)t / (double)f[t] * (double)o[t];
        uu[t] = v;
    }
    __syncthreads();
    for (int t = threadIdx.x; t < ns; t += PS_NT) o[t] = (float)(uu[t] - uu[t + 1]);
}

/* ------------------------------------------------------------------------ */
/* host glue                                                                 */
/* The velocity check of ktm_plan_create on the device: every sample an image
 * column reads (column x, y at grid node velx[x], vely[y], time index t1[t])
 * must be > 0 and < 3e19, whose square stays finite (a velocity <= 0 or NaN
 * would divide by zero at Kirchhoff.c:1381); a failing sample sets *bad. */
__global__ void k_velocity_check(const float *__restrict__ vel, const int32_t *__restrict__ velx,
                                 const int32_t *__restrict__ vely, const int32_t *__restrict__ t1,
                                 int nxp, int nyp, int ns, int nvel_xl, int nsm, uint32_t *bad)
{
    const int64_t n = (int64_t)nxp * nyp * ns;
    for (int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; e < n;
         e += (int64_t)gridDim.x * blockDim.x) {
        const int t = (int)(e % ns);
        const int64_t c = e / ns;
        const int x = (int)(c / nyp), y = (int)(c % nyp);
        const float v = vel[((int64_t)velx[x] * nvel_xl + vely[y]) * nsm + t1[t]];
        if (!(v > 0.0f) || !(v < 3.0e19f)) *bad = 1u;
    }
}

/* v -> v^2 in place (Kirchhoff.c:617), one FP32 product each, at least
 * KTM_V2_MIN: below it (v < 3e-13 m/s) every sample away from the source and the
 * receiver is past the trace either way, and 1/(v dt)^2 would overflow */
#define KTM_V2_MIN 1.0e-25f
__global__ void k_square(float *__restrict__ v, int64_t n)
{
    for (int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; e < n;
         e += (int64_t)gridDim.x * blockDim.x)
        v[e] = fmaxf(v[e] * v[e], KTM_V2_MIN);
}

/* ------------------------------------------------------------------------ */
template <typename T>
static int upload(T **dst, const T *src, size_t n)
{
    *dst = nullptr;
    if (hipMalloc((void **)dst, sizeof(T) * (n ? n : 1)) != hipSuccess) return KTM_ERR_NOMEM;
    if (n && hipMemcpy(*dst, src, sizeof(T) * n, hipMemcpyHostToDevice) != hipSuccess)
        return KTM_ERR_DEVICE;
    return KTM_OK;
}

extern "C" void ktm_plan_destroy(ktm_plan *p)
{
    if (!p) return;
    void *bufs[] = {p->d_t2, p->d_t1, p->d_colx, p->d_coly, p->d_velx, p->d_vely,
                    p->d_slab_cx, p->d_slab_cy, p->d_slab_x2thr, p->d_vel2, p->d_w, p->d_hconv2,
                    p->d_stage, p->d_pix_v2, p->d_pix_rs, p->d_dm_keys, p->d_dm_idx,
                    p->d_dm_tmp, p->d_dm_amax, p->d_dm_sum, p->d_parts, p->d_pf_g, p->d_pf_tw};
    for (void *b : bufs)
        if (b) (void)hipFree(b);
    ktm_tables_free(&p->tb);
    free(p);
}

extern "C" int ktm_plan_create(ktm_plan **out, const ktm_config *cfg, int ns, float dt, int nsm,
                               float dtm, const float *vel)
{
    if (!out || !cfg || !vel) return KTM_ERR_ARG;
    *out = nullptr;
    if (ns < 4 || ns > KTM_MAX_NS) return KTM_ERR_UNSUPPORTED;
    ktm_plan *p = (ktm_plan *)calloc(1, sizeof(ktm_plan));
    if (!p) return KTM_ERR_NOMEM;
    p->cfg = *cfg;
    int st = ktm_tables_build(cfg, ns, dt, nsm, dtm, &p->tb);
    if (st != KTM_OK) { free(p); return st; }
    if (hipGetDevice(&p->device) != hipSuccess) { ktm_plan_destroy(p); return KTM_ERR_DEVICE; }
    if ((st = scratch_address(p->device, &p->d_scratch)) != KTM_OK) {
        ktm_plan_destroy(p);
        return st;
    }
    p->row = ((int64_t)ns + 1 + 7) / 8 * 8;
    const ktm_tables *tb = &p->tb;
    st = upload(&p->d_t2, tb->t2, (size_t)ns);
    if (st == KTM_OK) st = upload(&p->d_t1, tb->t1, (size_t)ns);
    if (st == KTM_OK) st = upload(&p->d_colx, tb->colx, (size_t)tb->s.nxp);
    if (st == KTM_OK) st = upload(&p->d_coly, tb->coly, (size_t)tb->s.nyp);
    if (st == KTM_OK) st = upload(&p->d_velx, tb->velx, (size_t)tb->s.nxp);
    if (st == KTM_OK) st = upload(&p->d_vely, tb->vely, (size_t)tb->s.nyp);
    if (st == KTM_OK) st = upload(&p->d_slab_cx, tb->slab_cx, (size_t)tb->s.no_job);
    if (st == KTM_OK) st = upload(&p->d_slab_cy, tb->slab_cy, (size_t)tb->s.no_job);
    if (st == KTM_OK) st = upload(&p->d_slab_x2thr, tb->slab_x2thr, (size_t)tb->s.no_job);
    /* the velocity model: checked where the image reads it, then squared
     * (Kirchhoff.c:617), on the device */
    const size_t nv = (size_t)cfg->nvel_ilines * cfg->nvel_xlines * nsm;
    if (st == KTM_OK) st = upload(&p->d_vel2, vel, nv);
    if (st == KTM_OK) {
        uint32_t *d_bad = nullptr, bad = 0;
        if (hipMalloc((void **)&d_bad, sizeof(uint32_t)) != hipSuccess) {
            st = KTM_ERR_NOMEM;
        } else {
            const int64_t nchk = (int64_t)tb->s.nxp * tb->s.nyp * ns;
            const unsigned g = (unsigned)(nchk / 256 < 8192 ? (nchk + 255) / 256 : 8192);
            hipLaunchKernelGGL(k_zero_u32, dim3(1), dim3(1), 0, 0, d_bad);
            hipLaunchKernelGGL(k_velocity_check, dim3(g), dim3(256), 0, 0, p->d_vel2, p->d_velx,
                               p->d_vely, p->d_t1, tb->s.nxp, tb->s.nyp, ns, cfg->nvel_xlines, nsm,
                               d_bad);
            hipLaunchKernelGGL(k_square, dim3(8192), dim3(256), 0, 0, p->d_vel2, (int64_t)nv);
            if (hipGetLastError() != hipSuccess ||
                hipMemcpy(&bad, d_bad, sizeof(uint32_t), hipMemcpyDeviceToHost) != hipSuccess)
                st = KTM_ERR_DEVICE;
            (void)hipFree(d_bad);
            if (st == KTM_OK && bad) st = KTM_ERR_VELOCITY;
        }
    }
    if (st == KTM_OK) st = upload(&p->d_w, tb->w, (size_t)ns + 2);
    if (st == KTM_OK) {
        double *h2 = (double *)malloc(sizeof(double) * 2 * (size_t)ns);
        if (!h2) st = KTM_ERR_NOMEM;
        for (int m = 0; st == KTM_OK && m < 2 * ns; ++m) h2[m] = tb->hconv[m < ns ? m : m - ns];
        if (st == KTM_OK) st = upload(&p->d_hconv2, h2, 2 * (size_t)ns);
        free(h2);
    }
    if (st == KTM_OK && (p->pf_n = postfft_size(ns)) != 0) {
        const size_t n = (size_t)p->pf_n;
        double *g = (double *)malloc(sizeof(double) * 5 * n);
        if (!g) st = KTM_ERR_NOMEM;
        if (st == KTM_OK) {
            postfft_host_tables(tb->hconv, ns, p->pf_n, g, g + n, g + 3 * n);
            st = upload(&p->d_pf_g, g, n);
            if (st == KTM_OK) st = upload(&p->d_pf_tw, reinterpret_cast<const double2 *>(g + n), n);
        }
        free(g);
    }
    if (st == KTM_OK) st = parts_workspace(p);
    if (st != KTM_OK) { ktm_plan_destroy(p); return st; }
    *out = p;
    return KTM_OK;
}

extern "C" int ktm_plan_setup(const ktm_plan *p, ktm_setup *out)
{
    if (!p || !out) return KTM_ERR_ARG;
    *out = p->tb.s;
    return KTM_OK;
}

extern "C" int64_t ktm_plan_trace_row(const ktm_plan *p) { return p ? p->row : 0; }


extern "C" int64_t ktm_plan_image_size(const ktm_plan *p)
{
    if (!p) return 0;
    return (int64_t)p->tb.s.nxp * p->tb.s.nyp * p->tb.s.nh * p->tb.s.ns;
}

static GeoArgs geo_args(const ktm_plan *p)
{
    GeoArgs g;
    g.ox = p->cfg.ox; g.oy = p->cfg.oy; g.scale = p->cfg.scale_xy;
    g.oh = p->cfg.oh; g.dh = p->cfg.dh;
    g.sinA = p->tb.s.sinA; g.cosA = p->tb.s.cosA;
    return g;
}

extern "C" int ktm_geometry(const ktm_plan *p, const int32_t *coords, int64_t ntr,
                            ktm_trace_geom *geom, void *stream)
{
    if (!p || ntr < 0 || (ntr && (!coords || !geom))) return KTM_ERR_ARG;
    if (!ntr) return KTM_OK;
    hipStream_t s = (hipStream_t)stream;
    const int nt = 256;
    hipLaunchKernelGGL(k_geometry, dim3((unsigned)((ntr + nt - 1) / nt)), dim3(nt), 0, s,
                       geo_args(p), coords, ntr, geom);
    HIP_TRY(hipGetLastError());
    return KTM_OK;
}

/* prep kernels of one trace source (geometry already written) */
template <int SRC>
static int prep_launch(const ktm_plan *p, const TraceSrc src, int64_t ntr, int prep_mode,
                       int dtype, void *prepared, ktm_trace_geom *geom, hipStream_t s)
{
    const int ns = p->tb.s.ns;
    if (dtype == KTM_TRACE_F32) {
        if (prep_mode == KTM_PREP_REFERENCE) {
            hipLaunchKernelGGL(k_prep_ref<SRC>, dim3((unsigned)((ntr + KTM_WAVE - 1) / KTM_WAVE)),
                               dim3(PREP_NT), 0, s, src, ntr, ns, p->row, p->tb.s.dt, p->d_t2,
                               (float *)prepared);
        } else {
            if (ntr > 65535 * 1024LL) return KTM_ERR_UNSUPPORTED;
            const int nt = 256;
            for (int64_t i0 = 0; i0 < ntr; i0 += 65535) {
                const int64_t n = ntr - i0 < 65535 ? ntr - i0 : 65535;
                const TraceSrc si = {reinterpret_cast<const uint32_t *>(src.p) + i0 * src.rec_words,
                                     src.rec_words};
                hipLaunchKernelGGL(k_prep_closed<SRC>,
                                   dim3((unsigned)((p->row + nt - 1) / nt), (unsigned)n), dim3(nt),
                                   0, s, si, geom + i0, n, ns, p->row, p->d_w,
                                   (float *)prepared + i0 * p->row);
            }
        }
    } else {
        const int nt = KTM_WAVE;
        const dim3 grid((unsigned)((ntr + nt - 1) / nt));
        if (dtype == KTM_TRACE_BF16)
            hipLaunchKernelGGL((k_quantize<KTM_TRACE_BF16, SRC>), grid, dim3(nt), 0, s, src, ntr, ns,
                               p->row, (uint16_t *)prepared, geom);
        else
            hipLaunchKernelGGL((k_quantize<KTM_TRACE_F16, SRC>), grid, dim3(nt), 0, s, src, ntr, ns,
                               p->row, (uint16_t *)prepared, geom);
    }
    HIP_TRY(hipGetLastError());
    return KTM_OK;
}

static int prep_check(const ktm_plan *p, int prep_mode, int dtype)
{
    if (prep_mode != KTM_PREP_REFERENCE && prep_mode != KTM_PREP_CLOSED) return KTM_ERR_ARG;
    if (dtype != KTM_TRACE_F32 && dtype != KTM_TRACE_BF16 && dtype != KTM_TRACE_F16)
        return KTM_ERR_ARG;
    /* reduced-precision storage keeps the raw trace; its filter (the closed
     * form) is applied when a block is migrated */
    if (dtype != KTM_TRACE_F32 && prep_mode != KTM_PREP_CLOSED) return KTM_ERR_UNSUPPORTED;
    (void)p;
    return KTM_OK;
}

extern "C" int ktm_prep(const ktm_plan *p, const float *traces, const int32_t *coords,
                        int64_t ntr, int prep_mode, int dtype, void *prepared,
                        ktm_trace_geom *geom, void *stream)
{
    if (!p || ntr < 0) return KTM_ERR_ARG;
    if (!ntr) return KTM_OK;
    if (!traces || !coords || !prepared || !geom) return KTM_ERR_ARG;
    int st = prep_check(p, prep_mode, dtype);
    if (st != KTM_OK) return st;
    st = ktm_geometry(p, coords, ntr, geom, stream);
    if (st != KTM_OK) return st;
    const TraceSrc src = {traces, p->tb.s.ns};
    return prep_launch<SRC_F32>(p, src, ntr, prep_mode, dtype, prepared, geom, (hipStream_t)stream);
}

extern "C" int ktm_ingest(const ktm_plan *p, const void *raw, int64_t ntr, int format,
                          int prep_mode, int dtype, void *prepared, ktm_trace_geom *geom,
                          int32_t *coords, void *stream)
{
    if (!p || ntr < 0) return KTM_ERR_ARG;
    if (!ntr) return KTM_OK;
    if (!raw || !prepared || !geom || ((uintptr_t)raw & 3u)) return KTM_ERR_ARG;
    if (format != KTM_SEGY_IBM && format != KTM_SEGY_IEEE) return KTM_ERR_ARG;
    int st = prep_check(p, prep_mode, dtype);
    if (st != KTM_OK) return st;
    hipStream_t s = (hipStream_t)stream;
    const TraceSrc src = {raw, 60 + (int64_t)p->tb.s.ns};
    const int nt = 256;
    hipLaunchKernelGGL(k_geometry_segy, dim3((unsigned)((ntr + nt - 1) / nt)), dim3(nt), 0, s,
                       geo_args(p), (const uint32_t *)raw, src.rec_words, ntr, geom, coords);
    HIP_TRY(hipGetLastError());
    if (format == KTM_SEGY_IBM)
        return prep_launch<SRC_SEGY_IBM>(p, src, ntr, prep_mode, dtype, prepared, geom, s);
    return prep_launch<SRC_SEGY_IEEE>(p, src, ntr, prep_mode, dtype, prepared, geom, s);
}

/* raw SEG-Y records -> FP32 traces and header words: one workgroup per
 * record (the sample loop is contiguous, no index division) */
template <int SRC>
__global__ void k_segy_decode(const TraceSrc src, int64_t ntr, int ns, float *__restrict__ traces,
                              int32_t *__restrict__ coords)
{
    const int64_t i = blockIdx.x;
    if (i >= ntr) return;
    if (traces)
        for (int t = threadIdx.x; t < ns; t += blockDim.x)
            traces[i * ns + t] = load_sample<SRC>(src, i, t);
    if (coords && threadIdx.x < 4)
        coords[4 * i + threadIdx.x] = (int32_t)__builtin_bswap32(
            reinterpret_cast<const uint32_t *>(src.p)[i * src.rec_words + 18 + threadIdx.x]);
}

extern "C" int ktm_segy_decode(const void *raw, int64_t ntr, int ns, int format, float *traces,
                               int32_t *coords, void *stream)
{
    if (ntr < 0 || ns < 4) return KTM_ERR_ARG;
    if (!ntr) return KTM_OK;
    if (!raw || ((uintptr_t)raw & 3u)) return KTM_ERR_ARG;
    if (format != KTM_SEGY_IBM && format != KTM_SEGY_IEEE) return KTM_ERR_ARG;
    const TraceSrc src = {raw, 60 + (int64_t)ns};
    const int nt = 256;
    if (ntr > 0x7fffffffLL) return KTM_ERR_UNSUPPORTED;
    const dim3 grid((unsigned)ntr);
    hipStream_t s = (hipStream_t)stream;
    if (format == KTM_SEGY_IBM)
        hipLaunchKernelGGL(k_segy_decode<SRC_SEGY_IBM>, grid, dim3(nt), 0, s, src, ntr, ns, traces,
                           coords);
    else
        hipLaunchKernelGGL(k_segy_decode<SRC_SEGY_IEEE>, grid, dim3(nt), 0, s, src, ntr, ns, traces,
                           coords);
    HIP_TRY(hipGetLastError());
    return KTM_OK;
}

/* ------------------------------------------------------------------------ */
/* SEG-Y output on the device                                                */
/* ------------------------------------------------------------------------ */

/* IEEE -> IBM hex float, truncating (the encoder of the host's SEG-Y
 * writer): v = M 2^s with a 24-bit M (top bit 23), e2 = s + 24 (frexp's
 * exponent), e16 = ceil(e2 / 4), mantissa M >> (4 e16 - e2).  Zero, NaN and
 * inf encode as 0. */
__device__ __forceinline__ uint32_t float_to_ibm(float v)
{
    const uint32_t b = __float_as_uint(v);
    const uint32_t E = (b >> 23) & 0xffu, F = b & 0x7fffffu;
    if (E == 0xffu || (E == 0u && F == 0u)) return 0u;
    uint32_t M;
    int e2;
    if (E) {
        M = F | 0x800000u;
        e2 = (int)E - 126;
    } else {                                /* subnormal: normalise */
        const int sh = __builtin_clz(F) - 8;
        M = F << sh;
        e2 = -125 - sh;
    }
    const int e16 = (e2 + 3) >> 2;
    const uint32_t mant = M >> (4 * e16 - e2);
    return (b & 0x80000000u) | ((uint32_t)(e16 + 64) << 24) | mant;
}

/* samples of ntr records: records[r][60 + t] = big-endian word of
 * traces[r][t]; one workgroup per record */
template <int FMT>
__global__ void k_encode_samples(const float *__restrict__ traces, int64_t ntr, int ns,
                                 uint32_t *__restrict__ rec)
{
    const int64_t r = blockIdx.x;
    if (r >= ntr) return;
    for (int t = threadIdx.x; t < ns; t += blockDim.x) {
        const float v = traces[r * ns + t];
        const uint32_t w = FMT == KTM_SEGY_IBM ? float_to_ibm(v) : __float_as_uint(v);
        rec[r * (60 + (int64_t)ns) + 60 + t] = __builtin_bswap32(w);
    }
}

/* headers [ntr][60 words] into the records (or zeros) */
__global__ void k_copy_headers(const uint32_t *__restrict__ hdr, int64_t ntr, int ns,
                               uint32_t *__restrict__ rec)
{
    const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= ntr * 60) return;
    const int64_t r = e / 60;
    rec[r * (60 + (int64_t)ns) + (e - r * 60)] = hdr ? hdr[e] : 0u;
}

struct ImgHdrArgs {
    double start_il, start_xl, inc_il, inc_xl, il_dist, xl_dist, oh, dh;
    int ox_i, oy_i;                 /* (int)ox, (int)oy of Kirchhoff.c:1492-1493 */
    float cosA, sinA;
    int nx, ny, nyp, Nx, nh, ns, job, jobs_y;
    uint32_t dt_us;                 /* (unsigned short)(dt * 1e6), Kirchhoff.c:1447 */
};

/* word w of the 240-byte header of image<job>.su's record r = (xc ny + yc) nh +
 * ih of the job's slab, Kirchhoff.c:1437-1598: the fields the reference sets,
 * big-endian, the rest zero */
__device__ __forceinline__ uint32_t image_header_word(const ImgHdrArgs &a, int64_t r, int w)
{
    const int ih = (int)(r % a.nh);
    const int64_t c = r / a.nh;
    const int xc = (int)(c / a.ny), yc = (int)(c % a.ny);
    const int X = xc + (a.job / a.jobs_y) * a.nx;
    const int Y = yc + (a.job % a.jobs_y) * a.ny;
    const double il = a.start_il + X * a.inc_il;                 /* Kirchhoff.c:1482 */
    const double xl = a.start_xl + Y * a.inc_xl;                 /* Kirchhoff.c:1483 */
    const int xm = (int)(il * a.il_dist);                        /* Kirchhoff.c:1485 */
    const int ym = (int)(xl * a.xl_dist);                        /* Kirchhoff.c:1486 */
    const float cx = (float)a.ox_i + a.cosA * (float)xm - a.sinA * (float)ym;
    const float cy = (float)a.oy_i + a.sinA * (float)xm + a.cosA * (float)ym;
    const int tracl = a.nx * a.ny * a.nh * a.job + 1 + (xc * a.ny + yc) * a.nh + ih;
    switch (w) {
    case 0: return __builtin_bswap32((uint32_t)tracl);                      /* tracl */
    case 5: return __builtin_bswap32((uint32_t)(X + a.Nx * Y + 1));         /* cdp */
    case 9: return __builtin_bswap32((uint32_t)(int)ceil(a.oh + ih * a.dh));    /* offset */
    case 18: case 19: case 20: case 21: return __builtin_bswap32(1u);       /* sx..gy */
    case 28: return __builtin_bswap32((uint32_t)(a.ns & 0xffff));           /* ns, 114 */
    case 29: return __builtin_bswap32(a.dt_us << 16);                       /* dt, 116 */
    case 45: return __builtin_bswap32((uint32_t)(int)cx);                   /* cdpx */
    case 46: return __builtin_bswap32((uint32_t)(int)cy);                   /* cdpy */
    case 47: return __builtin_bswap32((uint32_t)(int)il);                   /* iline */
    case 48: return __builtin_bswap32((uint32_t)(int)xl);                   /* xline */
    case 51: case 55: case 56: case 58:         /* mess: 0 in the first record, */
        return r > 0 ? __builtin_bswap32(9999u) : 0u;       /* then 9999 (:1224, 1589) */
    case 59: return __builtin_bswap32(9999u);                               /* :1589-1590 */
    default: return 0u;
    }
}

/* image<job>.su: one workgroup per record r, its header by the first 60 lanes
 * (a kernel of its own with one lane per record took 53 us of 160,000 records'
 * 410) and its image row [X][Y][ih][t] byte-swapped into place; 16-byte
 * vectors when ns % 4 == 0 (image rows and records then start 16-byte aligned:
 * 240-byte header, 4 (60 + ns)-byte records) */
template <bool V4>
__global__ void __launch_bounds__(128) k_image_records(const float *__restrict__ image,
                                                        const ImgHdrArgs a,
                                                        uint32_t *__restrict__ rec)
{
    const int64_t r = blockIdx.x;
    const int ih = (int)(r % a.nh);
    const int64_t c = r / a.nh;
    const int64_t X = c / a.ny + (int64_t)(a.job / a.jobs_y) * a.nx;
    const int64_t Y = c % a.ny + (int64_t)(a.job % a.jobs_y) * a.ny;
    const float *src = image + ((X * a.nyp + Y) * a.nh + ih) * a.ns;
    uint32_t *dst = rec + r * (60 + (int64_t)a.ns) + 60;
    if (threadIdx.x < 60) dst[(int)threadIdx.x - 60] = image_header_word(a, r, (int)threadIdx.x);
    if (V4) {
        const int n4 = a.ns / 4;
        for (int i = threadIdx.x; i < n4; i += blockDim.x) {
            uint4 w = reinterpret_cast<const uint4 *>(src)[i];
            w.x = __builtin_bswap32(w.x);
            w.y = __builtin_bswap32(w.y);
            w.z = __builtin_bswap32(w.z);
            w.w = __builtin_bswap32(w.w);
            reinterpret_cast<uint4 *>(dst)[i] = w;
        }
    } else {
        for (int t = threadIdx.x; t < a.ns; t += blockDim.x)
            dst[t] = __builtin_bswap32(__float_as_uint(src[t]));
    }
}

extern "C" int ktm_segy_encode(const float *traces, int64_t ntr, int ns, int format,
                               const void *headers, void *records, void *stream)
{
    if (ntr < 0 || ns < 1) return KTM_ERR_ARG;
    if (!ntr) return KTM_OK;
    if (!traces || !records || ((uintptr_t)records & 3u) || ((uintptr_t)headers & 3u))
        return KTM_ERR_ARG;
    if (format != KTM_SEGY_IBM && format != KTM_SEGY_IEEE) return KTM_ERR_ARG;
    hipStream_t s = (hipStream_t)stream;
    const int nt = 256;
    if (ntr > 0x7fffffffLL || (ntr * 60 + nt - 1) / nt > 0x7fffffffLL) return KTM_ERR_UNSUPPORTED;
    hipLaunchKernelGGL(k_copy_headers, dim3((unsigned)((ntr * 60 + nt - 1) / nt)), dim3(nt), 0, s,
                       (const uint32_t *)headers, ntr, ns, (uint32_t *)records);
    if (format == KTM_SEGY_IBM)
        hipLaunchKernelGGL(k_encode_samples<KTM_SEGY_IBM>, dim3((unsigned)ntr), dim3(nt), 0, s,
                           traces, ntr, ns, (uint32_t *)records);
    else
        hipLaunchKernelGGL(k_encode_samples<KTM_SEGY_IEEE>, dim3((unsigned)ntr), dim3(nt), 0, s,
                           traces, ntr, ns, (uint32_t *)records);
    HIP_TRY(hipGetLastError());
    return KTM_OK;
}

extern "C" int ktm_image_records(const ktm_plan *p, const float *image, int job, void *records,
                                 void *stream)
{
    if (!p || !image || !records || ((uintptr_t)records & 3u)) return KTM_ERR_ARG;
    const ktm_setup *st = &p->tb.s;
    if (job < 0 || job >= st->no_job) return KTM_ERR_ARG;
    const ktm_config *c = &p->cfg;
    ImgHdrArgs a;
    a.start_il = c->start_iline; a.start_xl = c->start_xline;
    a.inc_il = c->inc_iline; a.inc_xl = c->inc_xline;
    a.il_dist = c->iline_distance; a.xl_dist = c->xline_distance;
    a.oh = c->oh; a.dh = c->dh;
    a.ox_i = (int)c->ox; a.oy_i = (int)c->oy;
    a.cosA = st->cosA; a.sinA = st->sinA;
    a.nx = st->nx; a.ny = st->ny; a.nyp = st->nyp; a.Nx = st->Nx; a.nh = st->nh; a.ns = st->ns;
    a.job = job; a.jobs_y = c->jobs_y;
    a.dt_us = (uint32_t)(uint16_t)(st->dt * 1000000);
    const int64_t nrec = (int64_t)a.nx * a.ny * a.nh;
    if (nrec > 0x7fffffffLL) return KTM_ERR_UNSUPPORTED;
    hipStream_t s = (hipStream_t)stream;
    const bool v4 = a.ns % 4 == 0 && ((uintptr_t)records & 15u) == 0 && ((uintptr_t)image & 15u) == 0;
    if (v4)
        hipLaunchKernelGGL(k_image_records<true>, dim3((unsigned)nrec), dim3(128), 0, s, image, a,
                           (uint32_t *)records);
    else
        hipLaunchKernelGGL(k_image_records<false>, dim3((unsigned)nrec), dim3(128), 0, s, image, a,
                           (uint32_t *)records);
    HIP_TRY(hipGetLastError());
    return KTM_OK;
}

extern "C" int ktm_image_reset(const ktm_plan *p, float *km, float *fold, float *comp, void *stream)
{
    if (!p || !km || !fold) return KTM_ERR_ARG;
    const int64_t n = ktm_plan_image_size(p);
    hipLaunchKernelGGL(k_image_reset, dim3(2048), dim3(256), 0, (hipStream_t)stream, km, fold, comp, n);
    HIP_TRY(hipGetLastError());
    return KTM_OK;
}

/* kernel choice */
typedef void (*mig_fn)(const MigArgs);
struct MigShape {
    mig_fn fn;
    int K, W, NW, C, RING;   /* samples per lane, waves per column, waves, rows per chunk, chunks */
};

/* accum is KTM_ACCUM_PLAIN or KTM_ACCUM_KAHAN, optionally with KTM_INDEX_FAST */
template <int K, int W, int NW, int C, int WN>
static MigShape mig_shape(int accum)
{
    const bool kahan = (accum & ~KTM_INDEX_FAST) == KTM_ACCUM_KAHAN;
    if (accum & KTM_INDEX_FAST)         /* no window to keep */
        return {kahan ? k_migrate<K, W, NW, C, 1, true, true> : k_migrate<K, W, NW, C, 1, false, true>,
                K, W, NW, C, 2};
    return {kahan ? k_migrate<K, W, NW, C, WN, true, false> : k_migrate<K, W, NW, C, WN, false, false>,
            K, W, NW, C, WN + 1};
}

/* every shape, by samples per column; the ring of rows within half of a
 * CU's LDS (two workgroups of 8 waves) or all of it (one of 16, or one of 8 for
 * few columns).  Chunks of 8 rows wherever that ring holds two of them, with
 * windows of up to 16 traces as it allows: half the barriers of chunks of 4 and
 * twice the rows in flight.  The 800-column, 1001-sample line (4 x 4) 2.80 ->
 * 2.41 ms, 12,000 traces into 1600 columns x 4 classes of 640 samples (10 x 1)
 * 3.31 -> 3.13 and of 2001 (8 x 4) 8.90 -> 8.21, 500 samples into 60 columns (2 x
 * 4) 0.78 -> 0.70; compensated sums and the relaxed index 2 to 13 % as well.
 * 1280 and 1536 samples and beyond 2048 keep 4 (two chunks of 8 do not fit). */
static const struct MigRow { int cap; MigShape (*make)(int); } mig_rows[] = {
    {256, mig_shape<2, 2, 8, 8, 2>},    {384, mig_shape<6, 1, 8, 8, 2>},
    {512, mig_shape<2, 4, 8, 8, 2>},    {512, mig_shape<4, 2, 8, 8, 2>},
    {512, mig_shape<8, 1, 8, 8, 2>},    {640, mig_shape<10, 1, 8, 8, 2>},
    {768, mig_shape<6, 2, 8, 8, 2>},    {768, mig_shape<12, 1, 8, 8, 2>},
    {1024, mig_shape<2, 8, 8, 8, 1>},   {1024, mig_shape<4, 4, 8, 8, 1>},
    {1024, mig_shape<8, 2, 8, 8, 1>},   {1280, mig_shape<10, 2, 8, 4, 2>},
    {1536, mig_shape<6, 4, 8, 4, 2>},   {1536, mig_shape<12, 2, 8, 4, 2>},
    {2048, mig_shape<8, 4, 16, 8, 1>},  {2048, mig_shape<8, 4, 8, 4, 1>},
    {2560, mig_shape<10, 4, 16, 4, 2>}, {3072, mig_shape<12, 4, 16, 4, 2>},
    {4096, mig_shape<8, 8, 16, 2, 2>},  {4096, mig_shape<8, 8, 8, 4, 1>},
    {5120, mig_shape<10, 8, 16, 2, 2>}, {6144, mig_shape<12, 8, 16, 2, 2>},
    {6144, mig_shape<12, 8, 8, 2, 2>}};

/* dynamic LDS: the ring of rows, the slots' largest constants, the trace list,
 * counts */
static size_t mig_lds(const MigShape &m, int64_t row)
{
    return sizeof(float) * (size_t)(m.RING * m.C * row + 2 * m.NW * m.K) +
           sizeof(int) * (size_t)(KTM_WAVE + m.C + m.NW * KTM_WAVE + m.NW);
}

/* instructions of a trace, per wave of K slots (k_migrate) */
static double mig_trace(int K, int accum)
{
    return accum & KTM_INDEX_FAST ? 8.0 * K + 25.0 : 10.7 * K + 40.0;
}

/* Relative time of a shape with wgs workgroups (columns x offset classes x
 * parts of the traces, as if every trace reached all of them) that take `share`
 * of the traces each: a SIMD runs its waves' sum over the chip's CUs (whole
 * workgroups while there are few), at full rate from four resident waves.  Two
 * waves run at 0.65 of that rate (3500 samples into 200 columns: 2.39 ms at four
 * waves on 100 CUs, 1.74 at two on 200); one and three lie beside it.
 * Against 8 or 12 slots with 2 or 4 waves by length alone: 751 samples take 12 x 1
 * instead of 8 x 2 (a 61 x 61 patch with the relaxed index 5.0 -> 3.3 ms), 1251
 * 10 x 2 instead of 12 x 2 (150 x 150 columns 187 -> 171), 2503 10 x 4 instead of
 * 12 x 4 (12 classes of 500 columns 6.75 -> 5.9), and 32 columns of 501 samples
 * 2 x 4 instead of 4 x 2 (60 -> 45 us).  The 800-column, 1001-sample line, chunks
 * of 4 rows: 4 x 4 2.96 ms, 8 x 2 3.92, 2 x 8 3.22.  Eight waves of long rows
 * against sixteen: 200 columns of 1700 samples 1.46 ms, 1.75; of 3500 1.74, 2.39; of
 * 6144 2.50, 2.96; 60 x 60 columns of 3500 5.65, 4.42. */
static double mig_cost(const MigShape &m, size_t lds, double wgs, double share, int accum)
{
    static const double rate[5] = {0.0, 0.40, 0.65, 0.85, 1.0};
    const double per_cu = wgs / KTM_CUS;
    const double waves = (per_cu < 8.0 ? ceil(per_cu) : per_cu) * m.NW / 4.0;
    const double fit = (double)(160 * 1024 / lds) * m.NW / 4.0;    /* resident, by LDS */
    const double at_once = waves < 4.0 && waves < fit ? waves : fit < 4.0 ? fit : 4.0;
    const int i = at_once < 4.0 ? (int)at_once : 3;
    return waves * share * mig_trace(m.K, accum) / (rate[i] + (at_once - i) * (rate[i + 1] - rate[i]));
}

/* Tiles of the region [rx0,rx1) x [ry0,ry1): ncol columns, a row on a 2-D
 * line, as square as possible in 3-D. */
static void tile_layout(const ktm_setup *s, int ncol, MigArgs *a)
{
    a->tx_cols = s->nyp == 1 ? ncol : (ncol == 8 ? 4 : ncol == 4 ? 2 : ncol);
    a->ty_cols = ncol / a->tx_cols;
    a->tiles_x = (a->rx1 - a->rx0 + a->tx_cols - 1) / a->tx_cols;
    const int tiles_y = (a->ry1 - a->ry0 + a->ty_cols - 1) / a->ty_cols;
    a->ntiles = a->tiles_x * tiles_y;
}

/* Compensated sums do not need the reference's order of additions, so a
 * block whose image region gives fewer than 10240 workgroups (20 per
 * workgroup slot, 256 CUs x 2) is split along its traces into parts, each
 * part a workgroup per tile with its own sums, merged afterwards.  On the
 * 1600-column, 1501-sample line (400 tiles) L^T took 33.7 ms unsplit, 27.6
 * with 7 parts, 25.2 with 12 and 24.2 with 24. */
#define KTM_PART_TARGET_WGS 10240
#define KTM_MAX_PARTS 32
#define KTM_PARTS_MAX_BYTES (1ull << 30)

static int parts_for(int64_t wgs)
{
    if (wgs >= KTM_PART_TARGET_WGS) return 1;
    const int64_t n = (KTM_PART_TARGET_WGS + wgs - 1) / wgs;
    return n > KTM_MAX_PARTS ? KTM_MAX_PARTS : (int)n;
}

/* The shape, tiles and parts of a block of ntr traces into the region of a. */
static MigShape pick_migrate(const ktm_setup *s, int64_t row, int accum, int64_t ntr, int parts_max,
                             MigArgs *a)
{
    const int64_t ncol = (int64_t)(a->rx1 - a->rx0) * (a->ry1 - a->ry0) * s->nh;
    MigShape best = {};
    MigArgs with = *a;
    double tbest = 0.0;
    for (const MigRow &r : mig_rows) {
        if (r.cap < s->ns) continue;
        const MigShape m = r.make(accum);
        MigArgs b = *a;
        tile_layout(s, m.NW / m.W, &b);
        /* compensated sums of a small region: the traces in parts */
        double share = 1.0;
        b.nparts = 1;
        if ((accum & ~KTM_INDEX_FAST) == KTM_ACCUM_KAHAN) {
            const int64_t chunk = m.NW * KTM_WAVE, nchunks = (ntr + chunk - 1) / chunk;
            b.nparts = parts_for((int64_t)b.ntiles * s->nh);
            if (b.nparts > parts_max) b.nparts = parts_max;
            if (b.nparts > nchunks) b.nparts = nchunks;      /* no part without a chunk */
            const double most = (double)((nchunks + b.nparts - 1) / b.nparts * chunk) / (double)ntr;
            if (b.nparts > 1 && most < 1.0) share = most;
        }
        const double wgs = (double)((ncol * m.W + m.NW - 1) / m.NW) * (double)b.nparts;
        const double t = mig_cost(m, mig_lds(m, row), wgs, share, accum);
        if (!best.fn || t < tbest) {
            best = m;
            with = b;
            tbest = t;
        }
    }
    *a = with;
    return best;
}

/* the partial images of the compensated split, sized for the whole image
 * (a job region needs at most that) at the shape of least instructions a trace
 * (the fewest tiles of those that a block takes, so the most parts), allocated
 * once with the plan so that neither migration entry point allocates them; none
 * for a large image */
static int parts_workspace(ktm_plan *p)
{
    const ktm_setup *s = &p->tb.s;
    MigArgs a;
    memset(&a, 0, sizeof a);
    a.rx1 = s->nxp; a.ry1 = s->nyp;
    MigShape m = {};
    for (const MigRow &r : mig_rows) {
        if (r.cap < s->ns) continue;
        const MigShape c = r.make(KTM_ACCUM_KAHAN);
        if (!m.fn || c.W * mig_trace(c.K, 0) < m.W * mig_trace(m.K, 0)) m = c;
    }
    tile_layout(s, m.NW / m.W, &a);
    int n = parts_for((int64_t)a.ntiles * s->nh);
    const uint64_t per = 3ull * sizeof(float) * (uint64_t)s->nxp * s->nyp * s->nh * s->ns;
    if (n > 1 && (uint64_t)(n - 1) * per > KTM_PARTS_MAX_BYTES)
        n = 1 + (int)(KTM_PARTS_MAX_BYTES / per);
    p->parts_max = n > 1 ? n : 1;
    if (p->parts_max > 1 &&
        hipMalloc((void **)&p->d_parts, (size_t)(p->parts_max - 1) * per) != hipSuccess) {
        p->d_parts = nullptr;
        return KTM_ERR_NOMEM;
    }
    return KTM_OK;
}

/* n elements that a call cannot do without.  The sums of column parts, which a
 * demigration can do without, are given back for them (hipFree waits for the
 * kernels that use them). */
template <class T> static int plan_alloc(ktm_plan *p, T **dst, size_t n)
{
    for (;;) {
        const hipError_t e = hipMalloc((void **)dst, n * sizeof(T));
        if (e == hipSuccess) return KTM_OK;
        *dst = nullptr;
        (void)hipGetLastError();
        if (e != hipErrorOutOfMemory || !p->d_dm_sum) return KTM_ERR_NOMEM;
        (void)hipFree(p->d_dm_sum);
        p->d_dm_sum = nullptr;
        p->dm_sum_cap = 0;
    }
}

/* FP32 filtered traces of a BF16/FP16 block, into stage (ntr * row floats)
 * or, when stage is NULL, into a workspace the plan owns and grows on demand
 * (the only allocation on the migration path) */
static int decode_block(const ktm_plan *cp, const void *prepared, int dtype,
                        const ktm_trace_geom *geom, int64_t ntr, hipStream_t s, float *stage,
                        const float **out)
{
    ktm_plan *p = const_cast<ktm_plan *>(cp);
    float *dst = stage;
    if (!dst) {
        const size_t need = (size_t)ntr * (size_t)p->row;
        if (need > p->stage_cap) {
            if (p->d_stage) HIP_TRY(hipFree(p->d_stage));
            p->d_stage = nullptr;
            p->stage_cap = 0;
            if (plan_alloc(p, &p->d_stage, need) != KTM_OK) return KTM_ERR_NOMEM;
            p->stage_cap = need;
        }
        dst = p->d_stage;
    }
    const int nt = 256;
    for (int64_t i0 = 0; i0 < ntr; i0 += 65535) {
        const int64_t n = ntr - i0 < 65535 ? ntr - i0 : 65535;
        const dim3 grid((unsigned)((p->row + nt - 1) / nt), (unsigned)n);
        const TraceSrc src = {reinterpret_cast<const uint16_t *>(prepared) + i0 * p->row, p->row};
        if (dtype == KTM_TRACE_BF16)
            hipLaunchKernelGGL(k_prep_closed<SRC_Q_BF16>, grid, dim3(nt), 0, s, src, geom + i0, n,
                               p->tb.s.ns, p->row, p->d_w, dst + i0 * p->row);
        else
            hipLaunchKernelGGL(k_prep_closed<SRC_Q_F16>, grid, dim3(nt), 0, s, src, geom + i0, n,
                               p->tb.s.ns, p->row, p->d_w, dst + i0 * p->row);
    }
    HIP_TRY(hipGetLastError());
    *out = dst;
    return KTM_OK;
}

static int migrate_block(const ktm_plan *p, const void *prepared, int dtype, int prep_mode,
                         const ktm_trace_geom *geom, int64_t ntr, int accum, int job, float *km,
                         float *fold, float *comp, uint64_t *counter, void *stream, float *stage);

extern "C" int ktm_migrate_block(const ktm_plan *p, const void *prepared, int dtype, int prep_mode,
                                 const ktm_trace_geom *geom, int64_t ntr, int accum, int job,
                                 float *km, float *fold, float *comp, uint64_t *counter,
                                 void *stream)
{
    return migrate_block(p, prepared, dtype, prep_mode, geom, ntr, accum, job, km, fold, comp,
                         counter, stream, nullptr);
}

/* ---- the allocation-free entry point ----
 * The BF16/FP16 decode workspace of ktm_migrate_block_static is this array:
 * every GPU the library runs on holds its own copy (KTM_STATIC_STAGE_FLOATS
 * floats, 64 MiB) until the process ends.  Host code never passes the name
 * `scratch` to a kernel (on the host it is only a stand-in for the symbol):
 * each plan keeps the device address hipGetSymbolAddress gave for its device
 * at ktm_plan_create, looked up once per device. */
static __device__ __align__(256) float scratch[KTM_STATIC_STAGE_FLOATS];

#define KTM_MAX_DEVICES 64
static float *g_scratch_ptr[KTM_MAX_DEVICES];
static std::mutex g_scratch_mu;

/* the device address of `scratch` on device dev, which must be current */
static int scratch_address(int dev, float **out)
{
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (dev < 0 || dev >= KTM_MAX_DEVICES) return KTM_ERR_UNSUPPORTED;
    if (!g_scratch_ptr[dev]) {
        void *ptr = nullptr;
        if (hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)) != hipSuccess || !ptr)
            return KTM_ERR_DEVICE;
        g_scratch_ptr[dev] = reinterpret_cast<float *>(ptr);
    }
    *out = g_scratch_ptr[dev];
    return KTM_OK;
}

extern "C" int ktm_migrate_block_static(const ktm_plan *p, const void *prepared, int dtype,
                                        int prep_mode, const ktm_trace_geom *geom, int64_t ntr,
                                        int accum, int job, float *km, float *fold, float *comp,
                                        uint64_t *counter, void *stream)
{
    if (!p || ntr < 0) return KTM_ERR_ARG;
    if (!p->d_scratch) return KTM_ERR_DEVICE;
    if (dtype != KTM_TRACE_F32 &&
        (uint64_t)ntr * (uint64_t)p->row > (uint64_t)KTM_STATIC_STAGE_FLOATS)
        return KTM_ERR_UNSUPPORTED;
    return migrate_block(p, prepared, dtype, prep_mode, geom, ntr, accum, job, km, fold, comp,
                         counter, stream, p->d_scratch);
}

static int migrate_block(const ktm_plan *p, const void *prepared, int dtype, int prep_mode,
                         const ktm_trace_geom *geom, int64_t ntr, int accum, int job, float *km,
                         float *fold, float *comp, uint64_t *counter, void *stream, float *stage)
{
    if (!p || !km || !fold || ntr < 0) return KTM_ERR_ARG;
    if (!ntr) return KTM_OK;
    if (!prepared || !geom) return KTM_ERR_ARG;
    const int acc_mode = accum & ~KTM_INDEX_FAST;
    if (acc_mode != KTM_ACCUM_PLAIN && acc_mode != KTM_ACCUM_KAHAN) return KTM_ERR_ARG;
    if (acc_mode == KTM_ACCUM_KAHAN && !comp) return KTM_ERR_ARG;
    if (dtype != KTM_TRACE_F32 && dtype != KTM_TRACE_BF16 && dtype != KTM_TRACE_F16) return KTM_ERR_ARG;
    if (dtype != KTM_TRACE_F32 && prep_mode != KTM_PREP_CLOSED) return KTM_ERR_UNSUPPORTED;
    /* the relaxed index is an option of the CLOSED operator only: the FP32
     * reference prep needs the reference's index (its taps cancel) */
    if ((accum & KTM_INDEX_FAST) && prep_mode != KTM_PREP_CLOSED) return KTM_ERR_UNSUPPORTED;
    const ktm_setup *s = &p->tb.s;
    if (job >= s->no_job) return KTM_ERR_ARG;
    hipStream_t hs = (hipStream_t)stream;
    const float *F = reinterpret_cast<const float *>(prepared);
    if (dtype != KTM_TRACE_F32) {
        const int st = decode_block(p, prepared, dtype, geom, ntr, hs, stage, &F);
        if (st != KTM_OK) return st;
    }
    MigArgs a;
    memset(&a, 0, sizeof a);
    a.prep = F; a.align16 = ((uintptr_t)F & 15u) == 0; a.geom = geom; a.ntr = ntr; a.row = p->row;
    a.km = km; a.fold = fold; a.comp = comp;
    a.vel2 = p->d_vel2; a.t1 = p->d_t1; a.velx = p->d_velx; a.vely = p->d_vely;
    a.t2 = p->d_t2; a.colx = p->d_colx; a.coly = p->d_coly;
    a.slab_cx = p->d_slab_cx; a.slab_cy = p->d_slab_cy; a.slab_x2thr = p->d_slab_x2thr;
    a.counter = (unsigned long long *)counter;
    a.ap_x2thr = p->tb.ap_x2thr;
    a.aperture = (float)p->cfg.aperture;
    a.dt = s->dt;
    a.rdt = 1.0f / s->dt;
    a.ns = s->ns; a.nh = s->nh; a.nxp = s->nxp; a.nyp = s->nyp; a.nx = s->nx; a.ny = s->ny;
    a.jobs_y = p->cfg.jobs_y; a.nvel_xl = p->cfg.nvel_xlines; a.nsm = s->nsm;
    if (job < 0) {
        a.rx0 = 0; a.ry0 = 0; a.rx1 = s->nxp; a.ry1 = s->nyp;
    } else { /* slab of Kirchhoff.c:1341-1347, job -> slice as in 287-295 */
        a.rx0 = (job / p->cfg.jobs_y) * s->nx; a.rx1 = a.rx0 + s->nx;
        a.ry0 = (job % p->cfg.jobs_y) * s->ny; a.ry1 = a.ry0 + s->ny;
    }
    a.part_n = (int64_t)(a.rx1 - a.rx0) * (a.ry1 - a.ry0) * s->nh * s->ns;
    a.parts = p->d_parts;
    const MigShape m = pick_migrate(s, p->row, accum, ntr, p->parts_max, &a);
    const mig_fn fn = m.fn;
    const int nthreads = m.NW * KTM_WAVE, nparts = (int)a.nparts;
    const size_t lds = mig_lds(m, p->row);
    if (lds > 160 * 1024) return KTM_ERR_UNSUPPORTED;
    /* runs of a row of tiles, but at least 8 runs per XCD */
    a.run = a.ntiles / 64 < a.tiles_x ? a.ntiles / 64 : a.tiles_x;
    if (a.run < 1) a.run = 1;
    const int64_t span = 8 * (int64_t)a.run;
    const int64_t nblk = ((int64_t)a.ntiles + span - 1) / span * span;
    if (nblk > 0x7fffffffLL) return KTM_ERR_UNSUPPORTED;
    const dim3 grid((unsigned)nblk, (unsigned)s->nh, (unsigned)nparts);
    HIP_TRY(hipFuncSetAttribute((const void *)fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    /* at most 2^24 traces a launch: the kernels count a sample's passing
     * traces in floats */
    for (int64_t i0 = 0; i0 < ntr; i0 += 1 << 24) {
        MigArgs b = a;
        b.ntr = ntr - i0 < (1 << 24) ? ntr - i0 : (1 << 24);
        b.prep = a.prep + i0 * a.row;
        b.geom = a.geom + i0;
        hipLaunchKernelGGL(fn, grid, dim3(nthreads), lds, hs, b);
        if (nparts > 1) {
            const int64_t nb = (a.part_n + 255) / 256;
            hipLaunchKernelGGL(k_merge_parts, dim3((unsigned)(nb < 8192 ? nb : 8192)), dim3(256), 0,
                               hs, b, nparts);
        }
        if (counter)
            hipLaunchKernelGGL(k_count_outside, dim3((unsigned)((b.ntr + 255) / 256)), dim3(256), 0,
                               hs, b);
    }
    HIP_TRY(hipGetLastError());
    return KTM_OK;
}

extern "C" int ktm_poststack(const ktm_plan *p, const float *km, const float *fold, float *out,
                             void *stream)
{
    if (!p || !km || !fold || !out) return KTM_ERR_ARG;
    const ktm_setup *s = &p->tb.s;
    const int64_t ntraces = (int64_t)s->nxp * s->nyp * s->nh;
    const hipError_t e =
        p->pf_n ? postfft_launch<PostKtm>(km, fold, ntraces, s->ns, s->dt, p->d_pf_g, p->d_pf_tw,
                                             out, (hipStream_t)stream)
                   : postmx_launch<PostKtm>(km, fold, ntraces, s->ns, s->dt, p->d_hconv2, out,
                                            (hipStream_t)stream);
    return e == hipSuccess ? KTM_OK : e == hipErrorInvalidValue ? KTM_ERR_UNSUPPORTED : KTM_ERR_DEVICE;
}

extern "C" int ktm_device_alloc(void **ptr, size_t bytes)
{
    if (!ptr) return KTM_ERR_ARG;
    *ptr = nullptr;
    return hipMalloc(ptr, bytes ? bytes : 1) == hipSuccess ? KTM_OK : KTM_ERR_NOMEM;
}

extern "C" int ktm_device_free(void *ptr)
{
    return hipFree(ptr) == hipSuccess ? KTM_OK : KTM_ERR_DEVICE;
}

extern "C" int ktm_copy_to_device(void *dst, const void *src, size_t bytes)
{
    return hipMemcpy(dst, src, bytes, hipMemcpyHostToDevice) == hipSuccess ? KTM_OK : KTM_ERR_DEVICE;
}

extern "C" int ktm_copy_to_host(void *dst, const void *src, size_t bytes)
{
    return hipMemcpy(dst, src, bytes, hipMemcpyDeviceToHost) == hipSuccess ? KTM_OK : KTM_ERR_DEVICE;
}

extern "C" int ktm_device_sync(void)
{
    return hipDeviceSynchronize() == hipSuccess ? KTM_OK : KTM_ERR_DEVICE;
}

/* ---- host pipeline runtime (ktm_internal.h) ---- */
extern "C" int ktm_rt_pinned_alloc(void **p, size_t bytes)
{
    if (!p) return KTM_ERR_ARG;
    *p = nullptr;
    return hipHostMalloc(p, bytes ? bytes : 1, hipHostMallocDefault) == hipSuccess ? KTM_OK
                                                                                  : KTM_ERR_NOMEM;
}
extern "C" void ktm_rt_pinned_free(void *p)
{
    if (p) (void)hipHostFree(p);
}
extern "C" int ktm_rt_stream_create(void **s)
{
    if (!s) return KTM_ERR_ARG;
    *s = nullptr;
    hipStream_t h = nullptr;
    if (hipStreamCreate(&h) != hipSuccess) return KTM_ERR_DEVICE;
    *s = h;
    return KTM_OK;
}
extern "C" void ktm_rt_stream_destroy(void *s)
{
    if (s) (void)hipStreamDestroy((hipStream_t)s);
}
extern "C" int ktm_rt_stream_sync(void *s)
{
    return hipStreamSynchronize((hipStream_t)s) == hipSuccess ? KTM_OK : KTM_ERR_DEVICE;
}
extern "C" int ktm_rt_stream_wait(void *s, void *e)
{
    return hipStreamWaitEvent((hipStream_t)s, (hipEvent_t)e, 0) == hipSuccess ? KTM_OK
                                                                            : KTM_ERR_DEVICE;
}
extern "C" int ktm_rt_event_create(void **e)
{
    if (!e) return KTM_ERR_ARG;
    *e = nullptr;
    hipEvent_t h = nullptr;
    if (hipEventCreate(&h) != hipSuccess) return KTM_ERR_DEVICE;
    *e = h;
    return KTM_OK;
}
extern "C" void ktm_rt_event_destroy(void *e)
{
    if (e) (void)hipEventDestroy((hipEvent_t)e);
}
extern "C" int ktm_rt_event_record(void *e, void *s)
{
    return hipEventRecord((hipEvent_t)e, (hipStream_t)s) == hipSuccess ? KTM_OK : KTM_ERR_DEVICE;
}
extern "C" int ktm_rt_event_sync(void *e)
{
    return hipEventSynchronize((hipEvent_t)e) == hipSuccess ? KTM_OK : KTM_ERR_DEVICE;
}
extern "C" int ktm_rt_event_elapsed_ms(void *e0, void *e1, float *ms)
{
    return hipEventElapsedTime(ms, (hipEvent_t)e0, (hipEvent_t)e1) == hipSuccess ? KTM_OK
                                                                               : KTM_ERR_DEVICE;
}
extern "C" int ktm_rt_copy_h2d_async(void *dst, const void *src, size_t bytes, void *s)
{
    return hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, (hipStream_t)s) == hipSuccess
               ? KTM_OK : KTM_ERR_DEVICE;
}
extern "C" int ktm_rt_copy_d2h_async(void *dst, const void *src, size_t bytes, void *s)
{
    return hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, (hipStream_t)s) == hipSuccess
               ? KTM_OK : KTM_ERR_DEVICE;
}

static int pixel_tables(const ktm_plan *cp, hipStream_t hs)
{
    ktm_plan *p = const_cast<ktm_plan *>(cp);
    if (p->d_pix_v2) return KTM_OK;
    const ktm_setup *s = &p->tb.s;
    const size_t n = (size_t)s->nxp * s->nyp * s->ns;
    if (plan_alloc(p, &p->d_pix_v2, n) != KTM_OK) return KTM_ERR_NOMEM;
    if (plan_alloc(p, &p->d_pix_rs, n) != KTM_OK) {
        (void)hipFree(p->d_pix_v2);
        p->d_pix_v2 = nullptr;
        return KTM_ERR_NOMEM;
    }
    hipLaunchKernelGGL(k_pixel_velocity, dim3(4096), dim3(256), 0, hs, p->d_vel2, p->d_velx,
                       p->d_vely, p->d_t1, s->nxp, s->nyp, s->ns, p->cfg.nvel_xlines, s->nsm,
                       s->dt, p->d_pix_v2, p->d_pix_rs);
    HIP_TRY(hipGetLastError());
    return KTM_OK;
}

/* The sums of column parts take at most 256 MiB */
#define DM_MAX_PARTS 16
#define DM_SUM_MAX_WORDS (32ll << 20)

/* lane shapes by length: K samples per lane, W waves per column */
typedef void (*demig_fn)(const DemigArgs);
struct DemigShape { int cap, K, W; demig_fn fn[2]; };   /* fn: reference index, relaxed index */
template <int K, int W> constexpr DemigShape demig_shape()
{
    return {K * W * KTM_WAVE, K, W, {k_demigrate<K, W, false>, k_demigrate<K, W, true>}};
}
static const DemigShape demig_shapes[] = {
    demig_shape<6, 1>(),  demig_shape<8, 1>(),  demig_shape<10, 1>(), demig_shape<12, 1>(),
    demig_shape<8, 2>(),  demig_shape<10, 2>(), demig_shape<12, 2>(), demig_shape<8, 4>(),
    demig_shape<10, 4>(), demig_shape<12, 4>(), demig_shape<8, 8>(),  demig_shape<10, 8>(),
    demig_shape<12, 8>()};                  /* KTM_MAX_NS */

/* columns of an axis within the aperture of a point, at most */
static int64_t columns_in_reach(const float *col, int n, double aperture)
{
    const double step = n > 1 ? fabs((double)col[n - 1] - col[0]) / (n - 1) : 0.0;
    const double c = step > 0.0 ? 2.0 * aperture / step + 1.0 : (double)n;
    return c < n ? (int64_t)c : n;
}

/* how a demigration is laid out: its lanes, traces per workgroup, the columns
 * that one trace reaches at most, workgroups that run at once */
struct DemigLayout { const DemigShape *sh; size_t lds; int tb, slots; int64_t cols; };

/* Parts in which n traces take their columns: the cheapest of 1 to
 * DM_MAX_PARTS if it is 10 % cheaper than 1.  Microseconds: a workgroup costs
 * its waves 0.27 per slot, trace and column and 3.5 per column (reference index,
 * four waves per SIMD) and 0.6 per pass over its sums; the chip takes 0.83 of
 * that time per round of workgroups (some reach fewer columns) and the whole of it
 * for the last ones; parts cost 34 for two more launches, 1.5e-5 per part and
 * sample for the 64-bit atomic adds and 3e-5 per sample for clearing and finishing.
 * Fitted to 1 to 16 parts of 8 to 12,000 traces of 63 to 5000 samples on 4 to 800
 * columns of a line and 30 x 30 to 120 x 120 of a patch: of the parts tried the
 * choice is within 0.8 % of the best on average, and at worst 4 % slower than
 * undivided.
 * 96 traces x 1001 on 800 columns: 1 part 1096 us, 16 150; 3000: 1 part 1165, 8
 * 975; 6000 on 4 columns: 1 part 128, 16 254; 3001 x 751 on 61 x 61: 1 part 5.75
 * ms, 6 3.99, 16 3.86. */
static int demig_parts(const DemigLayout &l, int64_t n, int ns)
{
    const int64_t nblk = (n + l.tb - 1) / l.tb;
    if (nblk >= 4 * l.slots) return 1;      /* four rounds are even enough */
    const int64_t per = (l.cols * l.sh->W + 7) / 8;
    const double col = 0.27 * l.sh->K * (double)(n < l.tb ? n : l.tb) + 3.5;
    const double sums = 0.6 * l.tb * ns / 512.0, size = (double)n * ns;
    int best = 1;
    double tbest = 0.0;
    for (int p = 1; p <= DM_MAX_PARTS; ++p) {
        const double rounds = 1.0 + 0.83 * (double)(nblk * p) / l.slots;
        const double t = rounds * ((double)((per + p - 1) / p) * col + sums) +
                         (p > 1 ? 34.0 + (1.5e-5 * p + 3e-5) * size : 0.0);
        if (p == 1) tbest = 0.9 * t;
        else if (t < tbest) {
            best = p;
            tbest = t;
        }
    }
    return best;
}

/* the demigration trace order of n traces (sorted by k_demig_keys) into
 * plan-owned buffers that grow with n; *order points at the sorted indices */
static int demig_order(const ktm_plan *cp, const ktm_trace_geom *geom, int64_t n,
                       hipStream_t hs, const int32_t **order)
{
    ktm_plan *p = const_cast<ktm_plan *>(cp);
    const ktm_setup *s = &p->tb.s;
    if (n > 0x7fffffffLL || s->nh >= (1 << 21)) return KTM_ERR_UNSUPPORTED;
    if ((size_t)n > p->dm_cap) {
        if (p->d_dm_keys) HIP_TRY(hipFree(p->d_dm_keys));
        if (p->d_dm_idx) HIP_TRY(hipFree(p->d_dm_idx));
        p->d_dm_keys = nullptr;
        p->d_dm_idx = nullptr;
        p->dm_cap = 0;
        if (plan_alloc(p, &p->d_dm_keys, 2 * (size_t)n) != KTM_OK) return KTM_ERR_NOMEM;
        if (plan_alloc(p, &p->d_dm_idx, 2 * (size_t)n) != KTM_OK) return KTM_ERR_NOMEM;
        p->dm_cap = (size_t)n;
    }
    uint64_t *k_in = p->d_dm_keys, *k_out = p->d_dm_keys + n;
    int32_t *i_in = p->d_dm_idx, *i_out = p->d_dm_idx + n;
    size_t need = 0;
    HIP_TRY(rocprim::radix_sort_pairs(nullptr, need, k_in, k_out, i_in, i_out, (size_t)n, 0u, 64u,
                                      hs));
    if (need > p->dm_tmp_bytes) {
        if (p->d_dm_tmp) HIP_TRY(hipFree(p->d_dm_tmp));
        p->d_dm_tmp = nullptr;
        p->dm_tmp_bytes = 0;
        char *tmp = nullptr;
        if (plan_alloc(p, &tmp, need) != KTM_OK) return KTM_ERR_NOMEM;
        p->d_dm_tmp = tmp;
        p->dm_tmp_bytes = need;
    }
    hipLaunchKernelGGL(k_demig_keys, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, hs, geom, n,
                       s->nh, p->d_colx, s->nxp, p->d_coly, s->nyp, k_in, i_in);
    HIP_TRY(hipGetLastError());
    size_t have = p->dm_tmp_bytes;
    HIP_TRY(rocprim::radix_sort_pairs(p->d_dm_tmp, have, k_in, k_out, i_in, i_out, (size_t)n, 0u,
                                      64u, hs));
    *order = i_out;
    return KTM_OK;
}

/* The sums of column parts for calls of up to n traces, after everything that
 * a call cannot do without.  They grow with n up to the most traces that take
 * parts, whether or not this call does: a call of no more traces than an earlier
 * one allocates and frees nothing.  Without memory for them calls are not
 * divided until one of more traces asks again. */
static void demig_sums(ktm_plan *p, const DemigLayout &l, int64_t n)
{
    if (n <= p->dm_sum_ntr) return;
    p->dm_sum_ntr = n;
    const int ns = p->tb.s.ns;
    int64_t nblk = (n + l.tb - 1) / l.tb;
    if (nblk > 4 * l.slots) nblk = 4 * l.slots;
    while (nblk && demig_parts(l, nblk * l.tb, ns) == 1) --nblk;
    const int64_t most = nblk * l.tb;
    int64_t words = (n < most ? n : most) * ns;
    if (words > DM_SUM_MAX_WORDS) words = DM_SUM_MAX_WORDS;
    if ((size_t)words <= p->dm_sum_cap) return;
    if (p->d_dm_sum) (void)hipFree(p->d_dm_sum);
    p->d_dm_sum = nullptr;
    p->dm_sum_cap = 0;
    if (hipMalloc((void **)&p->d_dm_sum, (size_t)words * sizeof(unsigned long long)) == hipSuccess) {
        p->dm_sum_cap = (size_t)words;
    } else {
        p->d_dm_sum = nullptr;
        (void)hipGetLastError();
    }
}

static int demigrate(const ktm_plan *p, const float *km, const ktm_trace_geom *geom, int64_t ntr,
                     float *traces, bool fast, void *stream);

extern "C" int ktm_demigrate(const ktm_plan *p, const float *km, const ktm_trace_geom *geom,
                             int64_t ntr, float *traces, void *stream)
{
    return demigrate(p, km, geom, ntr, traces, false, stream);
}

extern "C" int ktm_demigrate_index(const ktm_plan *p, const float *km, const ktm_trace_geom *geom,
                                   int64_t ntr, float *traces, int index, void *stream)
{
    if (index != 0 && index != KTM_INDEX_FAST) return KTM_ERR_ARG;
    return demigrate(p, km, geom, ntr, traces, index == KTM_INDEX_FAST, stream);
}

static int demigrate(const ktm_plan *p, const float *km, const ktm_trace_geom *geom, int64_t ntr,
                     float *traces, bool fast, void *stream)
{
    if (!p || ntr < 0) return KTM_ERR_ARG;
    if (!ntr) return KTM_OK;
    if (!km || !geom || !traces) return KTM_ERR_ARG;
    hipStream_t hs = (hipStream_t)stream;
    int st = pixel_tables(p, hs);
    if (st != KTM_OK) return st;
    const ktm_setup *s = &p->tb.s;
    /* cell indices of the sort key take 21 bits per axis */
    if (s->nxp >= (1 << 21) - 2 || s->nyp >= (1 << 21) - 2) return KTM_ERR_UNSUPPORTED;
    DemigArgs a;
    memset(&a, 0, sizeof a);
    a.km = km; a.geom = geom; a.ntr = ntr; a.traces = traces;
    a.pv2 = p->d_pix_v2; a.prs = p->d_pix_rs; a.t2 = p->d_t2; a.w = p->d_w;
    a.colx = p->d_colx; a.coly = p->d_coly;
    a.slab_cx = p->d_slab_cx; a.slab_cy = p->d_slab_cy; a.slab_x2thr = p->d_slab_x2thr;
    a.ap_x2thr = p->tb.ap_x2thr; a.aperture = (float)p->cfg.aperture;
    a.dt = s->dt; a.rdt = 1.0f / s->dt;
    a.ns = s->ns; a.nh = s->nh; a.nxp = s->nxp; a.nyp = s->nyp; a.nx = s->nx; a.ny = s->ny;
    a.jobs_y = p->cfg.jobs_y;
    /* fixed-point scale of g: max |km| and a bound on the terms per g[T] */
    a.lg_terms = 0;
    while ((1ull << a.lg_terms) < (unsigned long long)s->nxp * s->nyp * s->ns) ++a.lg_terms;
    if (!p->d_dm_amax) {
        ktm_plan *pm = const_cast<ktm_plan *>(p);
        if (plan_alloc(pm, &pm->d_dm_amax, 1) != KTM_OK) return KTM_ERR_NOMEM;
    }
    a.amax = p->d_dm_amax;
    const int64_t nimg = (int64_t)s->nxp * s->nyp * s->nh * s->ns;
    hipLaunchKernelGGL(k_zero_u32, dim3(1), dim3(1), 0, hs, p->d_dm_amax);
    hipLaunchKernelGGL(k_absmax, dim3(1024), dim3(256), 0, hs, km, nimg, p->d_dm_amax);
    /* traces per workgroup: DM_TB, fewer so that two workgroups share a CU
     * (g rows of 8 bytes per sample within 76 KB), or one beyond that */
    DemigLayout l;
    const size_t row = sizeof(unsigned long long) * (size_t)(s->ns + DM_PAD);
    l.tb = (int)((76 * 1024) / row);
    l.slots = l.tb < 2 ? KTM_CUS : 2 * KTM_CUS;
    if (l.tb < 2) l.tb = (int)((152 * 1024) / row);
    if (l.tb > DM_TB) l.tb = DM_TB;
    if (l.tb < 1) return KTM_ERR_UNSUPPORTED;
    a.tb = l.tb;
    l.lds = row * (size_t)l.tb;
    l.sh = demig_shapes;
    while (l.sh->cap < s->ns) ++l.sh;       /* ns <= KTM_MAX_NS by ktm_plan_create */
    l.cols = columns_in_reach(p->tb.colx, s->nxp, p->cfg.aperture) *
             columns_in_reach(p->tb.coly, s->nyp, p->cfg.aperture);
    const demig_fn fn = l.sh->fn[fast ? 1 : 0];
    HIP_TRY(hipFuncSetAttribute((const void *)fn, hipFuncAttributeMaxDynamicSharedMemorySize,
                                (int)l.lds));
    for (int64_t i0 = 0; i0 < ntr; i0 += 1 << 30) {
        const int64_t n = ntr - i0 < (1 << 30) ? ntr - i0 : (1 << 30);
        DemigArgs b = a;
        b.geom = geom + i0;
        b.traces = traces + i0 * s->ns;
        b.ntr = n;
        if ((st = demig_order(p, b.geom, n, hs, &b.order)) != KTM_OK) return st;
        demig_sums(const_cast<ktm_plan *>(p), l, n);
        const int64_t nblk = (n + l.tb - 1) / l.tb;
        /* few traces: their columns in parts, where the sums have their place */
        int parts = demig_parts(l, n, s->ns);
        if ((size_t)(n * s->ns) > p->dm_sum_cap) parts = 1;
        if (parts > 1) {
            b.gsum = p->d_dm_sum;
            hipLaunchKernelGGL(k_zero_u64, dim3(2048), dim3(256), 0, hs, b.gsum, n * s->ns);
        }
        hipLaunchKernelGGL(fn, dim3((unsigned)nblk, (unsigned)parts), dim3(8 * KTM_WAVE), l.lds, hs, b);
        if (parts > 1)
            hipLaunchKernelGGL(k_demig_finish, dim3((unsigned)n), dim3(256), 0, hs, b);
    }
    HIP_TRY(hipGetLastError());
    return KTM_OK;
}

extern "C" int ktm_poststack_adjoint(const ktm_plan *p, const float *img, const float *fold,
                                     float *km_bar, void *stream)
{
    if (!p || !img || !fold || !km_bar) return KTM_ERR_ARG;
    const ktm_setup *s = &p->tb.s;
    const int64_t ntraces = (int64_t)s->nxp * s->nyp * s->nh;
    if (ntraces > 0x7fffffffLL) return KTM_ERR_UNSUPPORTED;
    hipStream_t hs = (hipStream_t)stream;
    const hipError_t e =
        p->pf_n ? postfft_launch<PostImg>(img, fold, ntraces, s->ns, s->dt, p->d_pf_g,
                                             p->d_pf_tw, km_bar, hs)
                   : postmx_launch<PostImg>(img, fold, ntraces, s->ns, s->dt, p->d_hconv2, km_bar,
                                            hs);
    if (e != hipSuccess) return e == hipErrorInvalidValue ? KTM_ERR_UNSUPPORTED : KTM_ERR_DEVICE;
    hipLaunchKernelGGL(k_poststack_adjoint_tail, dim3((unsigned)ntraces), dim3(PS_NT),
                       sizeof(double) * (size_t)(s->ns + 1), hs, fold, s->ns, s->dt, km_bar);
    HIP_TRY(hipGetLastError());
    return KTM_OK;
}
