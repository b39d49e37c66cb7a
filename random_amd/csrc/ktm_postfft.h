/*
 * ktm_postfft.h -- the real circular convolution of ktm_postmx.h,
 *   out[j][t] = sum_u h[(t - u) mod ns] x[j][u]   (t = 0 stored as 0),
 * by FFT in FP64: with N the smallest of 256, 512, ..., 8192 and 3072 that is
 * >= 2 ns - 1, the kernel
 * wrapped into N points, g[d] = h[d] (0 <= d < ns) and g[N - d] = h[ns - d]
 * (0 < d < ns), zero between, makes the length-N circular convolution of the
 * zero-padded trace equal the length-ns one on t < ns:
 *   out = IDFT_N(G . DFT_N(x)) / N,   G = DFT_N(g)  (h is even, so is g, and
 * G is real),
 * the O(ns log ns) form of Kirchhoff.c:1465-1478 (FFTW forward, filter,
 * backward, / ns: here the 1/ns is in h) and EOM.c:1386-1413.  g is real,
 * so two traces go through one complex transform, x_a + i x_b, and come
 * out as its real and imaginary parts.
 *
 * k_postfft, in place in LDS without any reordering: the forward transform
 * leaves X[k] where its decimation does and the inverse takes it from there,
 * so the filter table lies in that order.  A pass over blocks of L points
 * combines, in registers, the R points L / R apart that a lane holds (at most
 * 16) and multiplies them by powers of a twiddle; the next works on blocks of
 * L / R:
 *   N -> N / 16 -> 16 -> done, the middle step of radix N / 256 = 2, 4, 8 or
 *   12 (512 to 3072 points), 16 (4096) or 2 and 16 (8192), none for 256.
 * N / 16 blocks of 16 are transformed, filtered and transformed back without
 * leaving the registers.  Between the first and the last pass a wave works on
 * 1024 points of its own (768 of 3072): whole blocks of N / 16, so these
 * passes need no barrier, and a workgroup has two in all (none up to 1024
 * points, where a wave holds 1024 / N transforms).  The first pass reads the
 * traces (the prologue Pro of ktm_postmx.h), whose second half is padding, the
 * last one writes t < ns <= N / 2; both with consecutive lanes on consecutive
 * samples.  LDS rows are padded by one double2 per 16 so that lanes 16 points
 * apart spread over the banks.
 * 160,000 traces of 1500 samples: 1.3 to 1.7 ms, 1.39 on average (2.1 before,
 * with a Stockham reordering and two barriers in every pass), 2.1 TB/s of traces
 * and fold in and image out.  It is bound by FP64 instructions (about 1500 per lane, 0.9
 * ms at one per four cycles) and by LDS latency at the three waves per SIMD
 * that 52 KB per workgroup leave: without its input loads it takes 1.2 ms.
 */
#ifndef KTM_POSTFFT_H
#define KTM_POSTFFT_H

#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>
#include <stdlib.h>


__device__ __forceinline__ double2 pf_add(double2 a, double2 b) { return make_double2(a.x + b.x, a.y + b.y); }
__device__ __forceinline__ double2 pf_sub(double2 a, double2 b) { return make_double2(a.x - b.x, a.y - b.y); }
__device__ __forceinline__ double2 pf_mul(double2 a, double2 w)
{
    return make_double2(__builtin_fma(a.x, w.x, -(a.y * w.y)), __builtin_fma(a.x, w.y, a.y * w.x));
}
/* a * (-i) forward, a * (+i) inverse */
template <bool INV> __device__ __forceinline__ double2 pf_rot(double2 a)
{
    return INV ? make_double2(-a.y, a.x) : make_double2(a.y, -a.x);
}
template <bool INV> __device__ __forceinline__ double2 pf_conj(double2 w)
{
    return INV ? make_double2(w.x, -w.y) : w;
}

template <bool INV> __device__ __forceinline__ void pf_dft2(double2 &a0, double2 &a1)
{
    const double2 t = a0;
    a0 = pf_add(t, a1);
    a1 = pf_sub(t, a1);
}

template <bool INV>
__device__ __forceinline__ void pf_dft4(double2 &a0, double2 &a1, double2 &a2, double2 &a3)
{
    const double2 t0 = pf_add(a0, a2), t1 = pf_sub(a0, a2);
    const double2 t2 = pf_add(a1, a3), t3 = pf_rot<INV>(pf_sub(a1, a3));
    a0 = pf_add(t0, t2);
    a2 = pf_sub(t0, t2);
    a1 = pf_add(t1, t3);
    a3 = pf_sub(t1, t3);
}

template <bool INV>
__device__ __forceinline__ void pf_dft3(double2 &a0, double2 &a1, double2 &a2)
{
    /* X0 = a0 + a1 + a2, X1,2 = a0 - (a1 + a2)/2 -+ i sqrt(3)/2 (a1 - a2) (forward) */
    constexpr double S3 = 0.86602540378443864676;
    const double2 t1 = pf_add(a1, a2);
    const double2 t2 = make_double2(a0.x - 0.5 * t1.x, a0.y - 0.5 * t1.y);
    const double2 d = pf_sub(a1, a2);
    const double2 t3 = INV ? make_double2(-S3 * d.y, S3 * d.x) : make_double2(S3 * d.y, -S3 * d.x);
    a0 = pf_add(a0, t1);
    a1 = pf_add(t2, t3);
    a2 = pf_sub(t2, t3);
}

/* exp(-2 pi i m / 12), m = 1, 2, 3, 4, 6 */
__device__ __forceinline__ double2 pf_w12(int m)
{
    constexpr double S3 = 0.86602540378443864676;
    switch (m) {
    case 1: return make_double2(S3, -0.5);
    case 2: return make_double2(0.5, -S3);
    case 3: return make_double2(0.0, -1.0);
    case 4: return make_double2(-0.5, -S3);
    default: return make_double2(-1.0, 0.0);   /* 6 */
    }
}

/* exp(-2 pi i m / 16), m = 0..9 */
__device__ __forceinline__ double2 pf_w16(int m)
{
    const double c1 = 0.92387953251128673848, s1 = 0.38268343236508978178;
    const double c2 = 0.70710678118654752440;
    switch (m) {
    case 0: return make_double2(1.0, 0.0);
    case 1: return make_double2(c1, -s1);
    case 2: return make_double2(c2, -c2);
    case 3: return make_double2(s1, -c1);
    case 4: return make_double2(0.0, -1.0);
    case 6: return make_double2(-c2, -c2);
    default: return make_double2(-c1, s1);   /* 9 */
    }
}

/* In-place DFT of R = 16, 12, 8, 4 or 2 points v[o], v[o + 1], ...; the
 * result X[k] ends in v[o + pf_slot<R>(k)]. */
template <int R> __device__ __forceinline__ constexpr int pf_slot(int k)
{
    return R == 16 ? 4 * (k & 3) + (k >> 2)
           : R == 12 ? 4 * (k % 3) + k / 3
           : R == 8 ? 4 * (k & 1) + (k >> 1) : k;
}

/* HALF: the inputs of the second half are zero (R = 16) */
template <int R, bool INV, bool HALF = false> __device__ __forceinline__ void pf_dft(double2 *v)
{
    if (R == 2) {
        pf_dft2<INV>(v[0], v[1]);
    } else if (R == 4) {
        pf_dft4<INV>(v[0], v[1], v[2], v[3]);
    } else if (R == 12) {
        /* n = 4 n1 + n2: 3-point DFTs over n1, twiddle W12^(n2 k1), 4-point over n2 */
#pragma unroll
        for (int n2 = 0; n2 < 4; ++n2) pf_dft3<INV>(v[n2], v[4 + n2], v[8 + n2]);
#pragma unroll
        for (int k1 = 1; k1 < 3; ++k1)
#pragma unroll
            for (int n2 = 1; n2 < 4; ++n2)
                v[4 * k1 + n2] = pf_mul(v[4 * k1 + n2], pf_conj<INV>(pf_w12(n2 * k1)));
#pragma unroll
        for (int k1 = 0; k1 < 3; ++k1) pf_dft4<INV>(v[4 * k1], v[4 * k1 + 1], v[4 * k1 + 2], v[4 * k1 + 3]);
    } else if (R == 8) {
        /* n = 4 n1 + n2: 2-point DFTs over n1, twiddle W8^(n2 k1), 4-point over n2 */
#pragma unroll
        for (int n2 = 0; n2 < 4; ++n2) pf_dft2<INV>(v[n2], v[4 + n2]);
#pragma unroll
        for (int n2 = 1; n2 < 4; ++n2) v[4 + n2] = pf_mul(v[4 + n2], pf_conj<INV>(pf_w16(2 * n2)));
#pragma unroll
        for (int k1 = 0; k1 < 2; ++k1) pf_dft4<INV>(v[4 * k1], v[4 * k1 + 1], v[4 * k1 + 2], v[4 * k1 + 3]);
    } else {
        /* n = 4 n1 + n2: 4-point DFTs over n1, twiddle W16^(n2 k1), 4-point over n2 */
#pragma unroll
        for (int n2 = 0; n2 < 4; ++n2) {
            if (HALF) {
                const double2 a = v[n2], b = v[4 + n2], ib = pf_rot<INV>(b);
                v[n2] = pf_add(a, b);
                v[4 + n2] = pf_add(a, ib);
                v[8 + n2] = pf_sub(a, b);
                v[12 + n2] = pf_sub(a, ib);
            } else {
                pf_dft4<INV>(v[n2], v[4 + n2], v[8 + n2], v[12 + n2]);
            }
        }
#pragma unroll
        for (int k1 = 1; k1 < 4; ++k1)
#pragma unroll
            for (int n2 = 1; n2 < 4; ++n2)
                v[4 * k1 + n2] = pf_mul(v[4 * k1 + n2], pf_conj<INV>(pf_w16(n2 * k1)));
#pragma unroll
        for (int k1 = 0; k1 < 4; ++k1) pf_dft4<INV>(v[4 * k1], v[4 * k1 + 1], v[4 * k1 + 2], v[4 * k1 + 3]);
    }
}

__device__ __forceinline__ int pf_pad(int i) { return i + (i >> 4); }

/* points per wave, threads per transform and per workgroup, transforms per
 * workgroup for an N-point transform */
template <int N> struct PfShape {
    static constexpr int E = N == 3072 ? 768 : 1024;
    static constexpr int TPF = N == 3072 ? 256 : N / 16;
    static constexpr int NT = TPF < 64 ? 64 : TPF;
    static constexpr int FPW = NT / TPF;
    static constexpr int ROW = N + N / 16; /* padded LDS row (double2) */
    static constexpr int WAVES_PER_EU = N == 3072 ? 3 : 2;
};

struct PfArgs {
    const float *in, *fold;
    int64_t ntraces;
    int ns;
    float dt;
    const double *G;
    const double2 *tw;
    float *out;
};

/* powers 1, 2, 4, 8 (as far as R needs them) of W_L^q, L points of N */
template <int N, int L, int R>
__device__ __forceinline__ void pf_twiddle(double2 *w, const double2 *__restrict__ tw, int q)
{
    w[1] = tw[q * (N / L)];
    if (R > 2) w[2] = tw[2 * q * (N / L)];
    if (R > 4) w[4] = tw[4 * q * (N / L)];
    if (R > 8) w[8] = tw[8 * q * (N / L)];
}

/* element r of v times the power r of the twiddle, those not in w being
 * products of them; SLOT: element r lies where pf_dft left it */
template <int R, bool INV, bool SLOT> __device__ __forceinline__ void pf_turn(double2 *v, double2 *w)
{
#pragma unroll
    for (int r = 3; r < R; ++r) {
        const int hi = r & (r - 1) ? (r & 8 ? 8 : r & 4 ? 4 : 2) : 0;
        if (hi) w[r] = pf_mul(w[hi], w[r - hi]);
    }
#pragma unroll
    for (int r = 1; r < R; ++r) {
        const int o = SLOT ? pf_slot<R>(r) : r;
        v[o] = pf_mul(v[o], pf_conj<INV>(w[r]));
    }
}

/* LDS accesses of a wave are done in order: the compiler has to keep it */
__device__ __forceinline__ void pf_wave_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

/* The passes over blocks of L < N points, forward, filter and inverse, of the
 * E points of one wave from buf on; e0: the wave's first point in its
 * transform. */
template <int N, int L>
__device__ __forceinline__ void pf_inner(double2 *buf, int lane, int e0, const PfArgs &a)
{
    constexpr int E = PfShape<N>::E;
    if constexpr (L == 16) {
        constexpr int NBF = E / 16;
        static_assert(NBF <= 64, "one block of 16 per lane");
        if (NBF == 64 || lane < NBF) {
            double g[16];
#pragma unroll
            for (int r = 0; r < 16; ++r) g[r] = a.G[r * (N / 16) + ((e0 / 16 + lane) & (N >= 1024 ? -1 : N / 16 - 1))];
            double2 v[16], x[16], *b = buf + 17 * lane;
#pragma unroll
            for (int r = 0; r < 16; ++r) v[r] = b[r];
            pf_dft<16, false>(v);
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const double2 y = v[pf_slot<16>(r)];
                x[r] = make_double2(y.x * g[r], y.y * g[r]);
            }
            pf_dft<16, true>(x);
#pragma unroll
            for (int r = 0; r < 16; ++r) b[r] = x[pf_slot<16>(r)];
        }
    } else {
        constexpr int R = L / 16 <= 16 ? L / 16 : L / 256;
        constexpr int S = L / R, SP = S + S / 16, NB = E / R / 64;
        static_assert(NB * R <= 16 && NB * R * 64 == E, "16 points per lane, all lanes busy");
#pragma unroll
        for (int b = 0; b < NB; ++b) {
            const int j = lane + 64 * b, q = j % S;
            double2 v[R], w[16], *p = buf + pf_pad(j / S * L + q);
            pf_twiddle<N, L, R>(w, a.tw, q);
#pragma unroll
            for (int r = 0; r < R; ++r) v[r] = p[r * SP];
            pf_dft<R, false>(v);
            pf_turn<R, false, true>(v, w);
#pragma unroll
            for (int r = 0; r < R; ++r) p[r * SP] = v[pf_slot<R>(r)];
        }
        pf_wave_sync();
        pf_inner<N, S>(buf, lane, e0, a);
        pf_wave_sync();
#pragma unroll
        for (int b = 0; b < NB; ++b) {
            const int j = lane + 64 * b, q = j % S;
            double2 v[R], w[16], *p = buf + pf_pad(j / S * L + q);
            pf_twiddle<N, L, R>(w, a.tw, q);
#pragma unroll
            for (int r = 0; r < R; ++r) v[r] = p[r * SP];
            pf_turn<R, true, false>(v, w);
            pf_dft<R, true>(v);
#pragma unroll
            for (int r = 0; r < R; ++r) p[r * SP] = v[pf_slot<R>(r)];
        }
    }
}

template <class Pro, int N>
__global__ void __launch_bounds__(PfShape<N>::NT)
    __attribute__((amdgpu_waves_per_eu(PfShape<N>::WAVES_PER_EU)))
k_postfft(const PfArgs a)
{
    typedef PfShape<N> S;
    constexpr int M = N / 16, MP = M + M / 16;
    extern __shared__ double2 pf_lds[];
    const int tid = threadIdx.x;
    /* 3072 points: 192 of the 256 threads work in the first and the last pass;
     * which wave idles differs from workgroup to workgroup, since a wave's
     * index in its workgroup fixes the SIMD it runs on */
    const int rot = N == 3072 ? 64 * ((blockIdx.x >> 3) + (blockIdx.x >> 8)) : 0;
    const int f = tid / S::TPF, tj = (tid + rot) % S::TPF;
    const bool busy = S::TPF == M || tj < M;
    double2 *p = pf_lds + f * S::ROW + pf_pad(tj);
    const int64_t tra = ((int64_t)blockIdx.x * S::FPW + f) * 2;
    double2 v[16], w[16];
    if (busy) {
        /* Inputs u >= N / 2 >= ns are zeros.  All samples are asked for at once,
         * where there is none at an index that has one: behind a branch each,
         * their 16 latencies in a row took 0.4 ms of 160,000 traces' 1.9. */
        const int64_t last = a.ntraces - 1;
        const int64_t ta = (tra < last ? tra : last) * a.ns, tb = (tra + 1 < last ? tra + 1 : last) * a.ns;
        float3 ka[8] = {}, kb[8] = {};
        if (a.ns > 1) {
#pragma unroll
            for (int r = 0; r < 8; ++r) {
                const int u = min(max(tj + r * M, 1), a.ns - 1);
                ka[r] = Pro::load(a.in + ta, a.fold + ta, u);
                kb[r] = Pro::load(a.in + tb, a.fold + tb, u);
            }
        }
        __builtin_amdgcn_sched_barrier(0);
        pf_twiddle<N, N, 16>(w, a.tw, tj);
#pragma unroll
        for (int r = 0; r < 8; ++r) {
            const int u = tj + r * M;
            const bool in = u >= 1 && u < a.ns;
            v[r] = make_double2(in && tra <= last ? Pro::value(ka[r], u, a.dt) : 0.0,
                                in && tra < last ? Pro::value(kb[r], u, a.dt) : 0.0);
        }
        pf_dft<16, false, true>(v);
        pf_turn<16, false, true>(v, w);
#pragma unroll
        for (int r = 0; r < 16; ++r) p[r * MP] = v[pf_slot<16>(r)];
    }
    if (N > S::E) __syncthreads(); else pf_wave_sync();
    const int wave = tid / 64, e0 = wave * S::E;
    pf_inner<N, M>(pf_lds + pf_pad(e0), tid % 64, N > S::E ? e0 : 0, a);
    if (N > S::E) __syncthreads(); else pf_wave_sync();
    if (!busy) return;
    pf_twiddle<N, N, 16>(w, a.tw, tj);
#pragma unroll
    for (int r = 0; r < 16; ++r) v[r] = p[r * MP];
    pf_turn<16, true, false>(v, w);
    pf_dft<16, true>(v);
    constexpr double inv_n = 1.0 / (double)N;
    float *o = a.out + tra * a.ns;
#pragma unroll
    for (int r = 0; r < 8; ++r) {           /* t >= N / 2 >= ns is not stored */
        const int t = tj + r * M;
        if (t < a.ns) {
            const double2 y = v[pf_slot<16>(r)];
            if (tra < a.ntraces) o[t] = t == 0 ? 0.0f : (float)(y.x * inv_n);
            if (tra + 1 < a.ntraces) o[a.ns + t] = t == 0 ? 0.0f : (float)(y.y * inv_n);
        }
    }
}

/* The transform length for ns samples: the smallest of 256, 512, 1024, 2048,
 * 3072, 4096, 8192 that is >= 2 ns - 1, or 0 beyond (the caller then takes
 * the direct product of ktm_postmx.h). */
static inline int postfft_size(int ns)
{
    static const int sizes[] = {256, 512, 1024, 2048, 3072, 4096, 8192};
    for (int n : sizes)
        if (n >= 2 * ns - 1) return n;
    return 0;
}

/* in-place DFT of n (a power of two) complex doubles, twiddles
 * exp(-2 pi i q / n) = tw[q step]: bit reversal, then log2 n butterfly stages */
static inline void postfft_host_fft(double *G, int n, const double *tw, int step)
{
    for (int i = 1, j = 0; i < n; ++i) {
        int bit = n >> 1;
        for (; j & bit; bit >>= 1) j ^= bit;
        j ^= bit;
        if (i < j) {
            const double tr = G[2 * i], ti = G[2 * i + 1];
            G[2 * i] = G[2 * j]; G[2 * i + 1] = G[2 * j + 1];
            G[2 * j] = tr; G[2 * j + 1] = ti;
        }
    }
    for (int len = 2; len <= n; len <<= 1) {
        const int half = len >> 1, stride = n / len * step;
        for (int s = 0; s < n; s += len)
            for (int k = 0; k < half; ++k) {
                const double wr = tw[2 * k * stride], wi = tw[2 * k * stride + 1];
                double *a = G + 2 * (s + k), *b = G + 2 * (s + k + half);
                const double br = b[0] * wr - b[1] * wi, bi = b[0] * wi + b[1] * wr;
                b[0] = a[0] - br; b[1] = a[1] - bi;
                a[0] += br; a[1] += bi;
            }
    }
}

/* Host tables of the FFT form for the even kernel h[0..ns): G = DFT_N(g), N
 * doubles in the order in which k_postfft reads it, and the twiddles exp(-2 pi i m / N), m < N, N double2 ({re, im}),
 * into caller arrays; work: 2 N doubles.  G in double, by radix-2 transforms
 * (of the three decimated sequences for 3072 points); twiddles from cos/sin
 * of the exact angle. */
static inline void postfft_host_tables(const double *h, int ns, int n, double *Gr, double *tw,
                                       double *G)
{
    const double two_pi = 6.283185307179586476925286766559;
    for (int m = 0; m < n; ++m) {
        tw[2 * m] = cos(two_pi * m / n);
        tw[2 * m + 1] = -sin(two_pi * m / n);
    }
    const int r = n & (n - 1) ? 3 : 1, l = n / r;
    /* the transforms F_q of the r sequences g[r j + q] in G's r parts, then
     * G[k] = sum_q W^(q k) F_q[k mod l] */
    for (int j = 0; j < n; ++j) {
        const int d = j < ns ? j : j > n - ns ? ns - (n - j) : -1;   /* g[n - e] = h[ns - e] */
        double *f = G + 2 * (j % r * l + j / r);
        f[0] = d >= 0 ? h[d] : 0.0;
        f[1] = 0.0;
    }
    for (int q = 0; q < r; ++q) postfft_host_fft(G + 2 * q * l, l, tw, r);
    /* position m = 16 b + t of block b: digits of radix 16, then n / 256 (of 512
     * for 8192: 2, then 16), then 16, the first digit of k the lowest */
    for (int m = 0; m < n; ++m) {
        int k = 0, one = 1;
        for (int len = n, p = m; len > 1;) {
            const int rad = len == n || len <= 16 ? 16 : len / 16 <= 16 ? len / 16 : len / 256;
            len /= rad;
            k += one * (p / len);
            one *= rad;
            p %= len;
        }
        double re = 0.0;
        for (int q = 0; q < r; ++q) {
            const double *f = G + 2 * (q * l + k % l), *w = tw + 2 * ((long long)q * k % n);
            re += f[0] * w[0] - f[1] * w[1];
        }
        Gr[m % 16 * (n / 16) + m / 16] = re;
    }
}

/* Launch k_postfft<Pro> over ntraces traces of ns samples; G and tw are the
 * device copies of postfft_host_tables for n = postfft_size(ns). */
template <class Pro>
static hipError_t postfft_launch(const float *in, const float *fold, int64_t ntraces, int ns,
                                 float dt, const double *G, const double2 *tw, float *out,
                                 hipStream_t stream)
{
    void (*fn)(const PfArgs) = nullptr;
    const int n = postfft_size(ns);
    int nt = 0, fpw = 0;
#define PF_CASE(n) case n: fn = k_postfft<Pro, n>; nt = PfShape<n>::NT; fpw = PfShape<n>::FPW; break
    switch (n) {
    PF_CASE(256);
    PF_CASE(512);
    PF_CASE(1024);
    PF_CASE(2048);
    PF_CASE(3072);
    PF_CASE(4096);
    PF_CASE(8192);
    default: return hipErrorInvalidValue;
    }
#undef PF_CASE
    const PfArgs a = {in, fold, ntraces, ns, dt, G, tw, out};
    const size_t lds = sizeof(double2) * (size_t)fpw * (size_t)(n + n / 16);
    const int64_t nblk = (ntraces + 2 * fpw - 1) / (2 * fpw);
    if (nblk > 0x7fffffffLL) return hipErrorInvalidValue;
    hipError_t e = hipFuncSetAttribute((const void *)fn, hipFuncAttributeMaxDynamicSharedMemorySize,
                                       (int)lds);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(fn, dim3((unsigned)nblk), dim3(nt), lds, stream, a);
    return hipGetLastError();
}

#endif
