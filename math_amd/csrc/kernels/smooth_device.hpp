// Lines of smooth length (factors 2, 3, 5 and 7, up to 4096 points) that are
// neither 2^k nor 3 * 2^k: a direct mixed-radix FFT of the line's own length
// in place of Bluestein's two padded ones (a line of 1920 points: one FFT of
// 15 x 8 x 16 instead of two of 4096).
//
// Radices, strides and threads per line are run-time values (a table of a few
// words per length, read as scalars), the butterflies are compiled per radix:
// hundreds of lengths share eleven radices, and a shape compiled per length
// would not fit the batch kernels.  A tile is T / tpl whole lines; a thread
// takes up to 16 points in every pass (gen_nb butterflies of the pass's
// radix), gathers them from LDS at j + r * n/R, and scatters to the Stockham
// positions.  The planner puts an odd radix first, so the scatter with stride
// R of the first pass meets no bank conflict without padding.  The first pass
// reads HBM, the last writes it.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "fft_device.hpp"

namespace mdft {

// ---------------------------------------------------------------------------
// odd radices
// ---------------------------------------------------------------------------
// forward 5-point DFT in place: sums and differences of the mirrored inputs,
// X1,4 = a1 -+ i*b1, X2,3 = a2 -+ i*b2
__device__ __forceinline__ void dft5(float2& x0, float2& x1, float2& x2, float2& x3, float2& x4)
{
    const float c1 = 0.30901699437494742410f, c2 = -0.80901699437494742410f;
    const float s1 = 0.95105651629515357212f, s2 = 0.58778525229247312917f;
    const float2 p1 = cadd(x1, x4), p2 = cadd(x2, x3), d1 = csub(x1, x4), d2 = csub(x2, x3);
    const float2 a1 = make_float2(__builtin_fmaf(c2, p2.x, __builtin_fmaf(c1, p1.x, x0.x)),
                                  __builtin_fmaf(c2, p2.y, __builtin_fmaf(c1, p1.y, x0.y)));
    const float2 a2 = make_float2(__builtin_fmaf(c1, p2.x, __builtin_fmaf(c2, p1.x, x0.x)),
                                  __builtin_fmaf(c1, p2.y, __builtin_fmaf(c2, p1.y, x0.y)));
    const float2 b1 = make_float2(__builtin_fmaf(s2, d2.x, s1 * d1.x), __builtin_fmaf(s2, d2.y, s1 * d1.y));
    const float2 b2 = make_float2(__builtin_fmaf(-s1, d2.x, s2 * d1.x), __builtin_fmaf(-s1, d2.y, s2 * d1.y));
    x0 = cadd(x0, cadd(p1, p2));
    x1 = make_float2(a1.x + b1.y, a1.y - b1.x);
    x4 = make_float2(a1.x - b1.y, a1.y + b1.x);
    x2 = make_float2(a2.x + b2.y, a2.y - b2.x);
    x3 = make_float2(a2.x - b2.y, a2.y + b2.x);
}

// forward 7-point DFT in place, the same way
__device__ __forceinline__ void dft7(float2 (&u)[7])
{
    const float c[3] = {0.62348980185873353053f, -0.22252093395631440429f, -0.90096886790241912624f};
    const float s[3] = {0.78183148246802980871f, 0.97492791218182360702f, 0.43388373911755812048f};
    float2 p[3], d[3];
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        p[k] = cadd(u[k + 1], u[6 - k]);
        d[k] = csub(u[k + 1], u[6 - k]);
    }
    const float2 x0 = u[0];
    u[0] = cadd(x0, cadd(p[0], cadd(p[1], p[2])));
#pragma unroll
    for (int k = 1; k <= 3; ++k) {
        float2 a = x0, b = make_float2(0.0f, 0.0f);
#pragma unroll
        for (int m = 1; m <= 3; ++m) {
            const int e = (k * m) % 7, f = e <= 3 ? e : 7 - e;  // cos is even, sin odd
            const float cc = c[f - 1], ss = e <= 3 ? s[f - 1] : -s[f - 1];
            a = make_float2(__builtin_fmaf(cc, p[m - 1].x, a.x), __builtin_fmaf(cc, p[m - 1].y, a.y));
            b = m == 1 ? make_float2(ss * d[0].x, ss * d[0].y)
                       : make_float2(__builtin_fmaf(ss, d[m - 1].x, b.x), __builtin_fmaf(ss, d[m - 1].y, b.y));
        }
        u[k] = make_float2(a.x + b.y, a.y - b.x);
        u[7 - k] = make_float2(a.x - b.y, a.y + b.x);
    }
}

// 9 = 3 x 3: input n = 3*n1 + n2, output k = k1 + 3*k2, twiddles W9^(n2*k1)
__device__ __forceinline__ void dft9(float2 (&u)[9])
{
    dft3(u[0], u[3], u[6]);
    dft3(u[1], u[4], u[7]);
    dft3(u[2], u[5], u[8]);
    const float2 w1 = make_float2(0.76604444311897803520f, -0.64278760968653932632f);
    const float2 w2 = make_float2(0.17364817766693034885f, -0.98480775301220805937f);
    const float2 w4 = make_float2(-0.93969262078590838405f, -0.34202014332566873304f);
    u[4] = cmul(u[4], w1);
    u[5] = cmul(u[5], w2);
    u[7] = cmul(u[7], w2);
    u[8] = cmul(u[8], w4);
    dft3(u[0], u[1], u[2]);
    dft3(u[3], u[4], u[5]);
    dft3(u[6], u[7], u[8]);
    // u[3*k1 + k2] holds output k1 + 3*k2
    const float2 t[9] = {u[0], u[3], u[6], u[1], u[4], u[7], u[2], u[5], u[8]};
#pragma unroll
    for (int i = 0; i < 9; ++i) u[i] = t[i];
}

// prime-factor (Good-Thomas) Q x 5, Q = 2 or 3: input n = (5*n1 + Q*n2) mod R,
// output k = (E1*k1 + E5*k2) mod R (E1 = 1 mod Q and 0 mod 5, E5 the other way)
template <int Q>
__device__ __forceinline__ void dft_pfa5(float2 (&u)[5 * Q])
{
    constexpr int R = 5 * Q, E1 = Q == 2 ? 5 : 10, E5 = 6;
    float2 a[Q][5];
#pragma unroll
    for (int n1 = 0; n1 < Q; ++n1) {
#pragma unroll
        for (int n2 = 0; n2 < 5; ++n2) a[n1][n2] = u[(5 * n1 + Q * n2) % R];
        dft5(a[n1][0], a[n1][1], a[n1][2], a[n1][3], a[n1][4]);
    }
#pragma unroll
    for (int k2 = 0; k2 < 5; ++k2) {
        if constexpr (Q == 2) {
            const float2 x = a[0][k2], y = a[1][k2];
            a[0][k2] = cadd(x, y);
            a[1][k2] = csub(x, y);
        } else {
            dft3(a[0][k2], a[1][k2], a[Q - 1][k2]);
        }
#pragma unroll
        for (int k1 = 0; k1 < Q; ++k1) u[(E1 * k1 + E5 * k2) % R] = a[k1][k2];
    }
}

template <int R>
__device__ __forceinline__ void dft_smooth(float2 (&u)[R])
{
    if constexpr (R == 3)
        dft3(u[0], u[1], u[2]);
    else if constexpr (R == 5)
        dft5(u[0], u[1], u[2], u[3], u[4]);
    else if constexpr (R == 7)
        dft7(u);
    else if constexpr (R == 9)
        dft9(u);
    else if constexpr (R == 10)
        dft_pfa5<2>(u);
    else if constexpr (R == 15)
        dft_pfa5<3>(u);
    else
        dft_fwd<R>(u);
}

// ---------------------------------------------------------------------------
// one tile
// ---------------------------------------------------------------------------
// butterflies of radix R a thread takes in a pass (16 points at most)
__host__ __device__ constexpr int gen_nb(int radix) { return radix >= 9 ? 1 : 16 / radix; }

// words of LDS a tile of `threads` threads needs: two planes of T * 16 points
// and the line strides' padding (gen_line_stride)
__host__ __device__ constexpr int gen_lds_floats(int threads) { return 2 * 17 * threads; }

// Line stride in words.  Columns (lines fastest): a wave's 32 lanes of a cycle
// cover 32/q' positions of q' lines, so a stride of q = 32/q' times an odd
// number keeps them apart; a stride past n costs at most 64 words a tile where
// q > 1 and two a line where q = 1.
template <bool COLS>
__device__ __forceinline__ int gen_line_stride(int n, int lines)
{
    if (!COLS) return n;
    const int q = lines >= 32 ? 1 : lines > 16 ? 1 : lines > 8 ? 2 : lines > 4 ? 4 : lines > 2 ? 8 : lines > 1 ? 16 : 0;
    return q == 0 ? n : ((n + q - 1) & ~(2 * q - 1)) + q;
}

template <int R, bool FIRST, bool LAST, bool COLS, int IO>
struct GenPassRun {
    static constexpr int NB = gen_nb(R);
    struct Tile {
        const AxisJob* job;
        const ImageIO* io;
        int t, tpl;
        bool valid;
        int64_t base;   // columns: the thread's line; rows: the tile's first line (uniform)
        uint32_t off;   // rows: the thread's line inside the tile
        int64_t iline;  // image input and output: the line's index
        float *re, *im;
        uint32_t sgn;
    };

    __device__ __forceinline__ static void run(const Tile& x, const GenPass& pass, const float2* rows)
    {
        const AxisJob& job = *x.job;
        const int nbf = pass.nbf, ns = pass.ns;
        constexpr int Q = tw_quads<R>();
        float4 w[NB][Q];
        int jj[NB], kk[NB];
#pragma unroll
        for (int b = 0; b < NB; ++b) {
            // a thread past the last butterfly repeats it and writes nothing
            const int j = x.t + b * x.tpl;
            jj[b] = j < nbf ? j : nbf - 1;
            if constexpr (FIRST) {
                kk[b] = 0;
            } else {
                kk[b] = LAST ? jj[b] : jj[b] - ns * (int)__umulhi((uint32_t)jj[b], pass.magic);
#pragma unroll
                for (int r2 = 0; r2 < Q; ++r2) w[b][r2] = load4_at(rows, uint32_t(kk[b]) * 32u + 16u * r2);
            }
        }
        float2 u[NB][R];
        if constexpr (FIRST && (IO & IO_LUM) != 0) {
            float lum[NB * R];
            load_luminance<NB * R>(
                *x.io,
                [&](int i) { return x.iline * x.io->ils + int64_t(jj[i / R] + (i % R) * nbf) * x.io->iel; }, lum);
#pragma unroll
            for (int i = 0; i < NB * R; ++i) u[i / R][i % R] = make_float2(lum[i], 0.0f);
        } else if constexpr (FIRST) {
#pragma unroll
            for (int b = 0; b < NB; ++b) {
#pragma unroll
                for (int r = 0; r < R; ++r) {
                    if constexpr (COLS)
                        u[b][r] = load_global(job.src + x.base + int64_t(jj[b]) * job.es + int64_t(r * nbf) * job.es);
                    else
                        u[b][r] = load_at(job.src + x.base + r * nbf, x.off + uint32_t(jj[b]));
                }
            }
#pragma unroll
            for (int b = 0; b < NB; ++b)
#pragma unroll
                for (int r = 0; r < R; ++r) u[b][r] = cxor(u[b][r], x.sgn);
        } else {
            __syncthreads();  // the previous pass is written
#pragma unroll
            for (int b = 0; b < NB; ++b)
#pragma unroll
                for (int r = 0; r < R; ++r) {
                    const int q = jj[b] + r * nbf;
                    u[b][r] = make_float2(x.re[q], x.im[q]);
                }
            if constexpr (!LAST) __syncthreads();  // and read
        }
#pragma unroll
        for (int b = 0; b < NB; ++b) {
            if constexpr (!FIRST) {
                if constexpr (R == 16) {
                    dft_twiddled<16>(u[b], w[b]);
                } else {
                    float2 wt[R];
                    expand_twiddles<R>(wt, w[b]);
#pragma unroll
                    for (int r = 1; r < R; ++r) u[b][r] = cmul(u[b][r], wt[r]);
                    dft_smooth<R>(u[b]);
                }
            } else {
                dft_smooth<R>(u[b]);
            }
            if (x.t + b * x.tpl >= nbf) continue;
            if constexpr (!LAST) {
                const int q0 = (jj[b] - kk[b]) * R + kk[b];
#pragma unroll
                for (int r = 0; r < R; ++r) {
                    x.re[q0 + r * ns] = u[b][r].x;
                    x.im[q0 + r * ns] = u[b][r].y;
                }
            } else if (x.valid) {
#pragma unroll
                for (int r = 0; r < R; ++r) {
                    const float2 y = cscale(cxor(u[b][r], x.sgn), job.scale);
                    if constexpr ((IO & IO_MAG) != 0)
                        x.io->mag[x.iline * x.io->mls + int64_t(jj[b] + r * nbf) * x.io->mel] =
                            cabs_scaled(y, x.io->mscale);
                    else if constexpr (COLS)
                        store_global(job.dst + x.base + int64_t(jj[b]) * job.es + int64_t(r * nbf) * job.es, y);
                    else
                        store_at(job.dst + x.base + r * nbf, x.off + uint32_t(jj[b]), y);
                }
            }
        }
    }
};

template <bool FIRST, bool LAST, bool COLS, int IO, class TileT>
__device__ __forceinline__ void gen_pass(const TileT& x, const GenPass& pass, const float2* rows)
{
    // uniform: the pass table is read as scalars.  Every radix has its own copy of
    // the tile's fields (one struct for all of them: 300 x 200 9.9 us instead of 9.6)
    switch (pass.radix) {
#define MDFT_GEN_CASE(R)                                                                                           \
    case R: {                                                                                                      \
        using P = GenPassRun<R, FIRST, LAST, COLS, IO>;                                                            \
        const typename P::Tile y{x.job, x.io, x.t, x.tpl, x.valid, x.base, x.off, x.iline, x.re, x.im, x.sgn};       \
        P::run(y, pass, rows);                                                                                     \
        break;                                                                                                     \
    }
        MDFT_GEN_CASE(2)
        MDFT_GEN_CASE(3)
        MDFT_GEN_CASE(4)
        MDFT_GEN_CASE(5)
        MDFT_GEN_CASE(7)
        MDFT_GEN_CASE(8)
        MDFT_GEN_CASE(9)
        MDFT_GEN_CASE(10)
        MDFT_GEN_CASE(12)
        MDFT_GEN_CASE(15)
        MDFT_GEN_CASE(16)
#undef MDFT_GEN_CASE
    default: break;
    }
}

// the pass table at the head of a length's twiddle block, read as scalars
__device__ __forceinline__ GenPass gen_read_pass(const float2* tw, int p)
{
    auto w = (const __attribute__((address_space(4))) uint32_t*)(uintptr_t)tw + p * 4;
    GenPass g;
    g.radix = __builtin_amdgcn_readfirstlane(w[0]);
    g.ns = __builtin_amdgcn_readfirstlane(w[1]);
    g.nbf = __builtin_amdgcn_readfirstlane(w[2]);
    g.magic = (uint32_t)__builtin_amdgcn_readfirstlane(w[3]);
    return g;
}

template <int THREADS, bool COLS, int IO = 0>
__device__ __forceinline__ void smooth_tile(const AxisJob& job, int tile, float* lds, int tid, ImageIO io = ImageIO{})
{
    struct {
        const AxisJob* job;
        const ImageIO* io;
        int t, tpl;
        bool valid;
        int64_t base;
        uint32_t off;
        int64_t iline;
        float *re, *im;
        uint32_t sgn;
    } x;
    const int n = job.n, tpl = job.tpl, lines = THREADS / tpl;
    const int ll = COLS ? tid % lines : tid / tpl;
    x.job = &job;
    x.io = &io;
    x.tpl = tpl;
    // threads past the last whole line (rows: the line index; columns: the position) take no part
    const bool extra = COLS ? tid / lines >= tpl : ll >= lines;
    x.t = extra ? 0x3fffffff - 8 * tpl : COLS ? tid / lines : tid % tpl;
    const int lane = extra ? 0 : ll;
    const int line = tile * lines + lane;
    x.valid = line < job.count && !extra;
    // a line past the last one reads the tile's first and stores nothing
    const int from = line < job.count ? lane : 0;
    x.base = COLS ? int64_t(tile * lines + from) * job.ls : int64_t(tile) * lines * job.ls;
    x.off = COLS ? 0u : uint32_t(from) * uint32_t(job.ls);
    x.iline = tile * lines + from;
    const int lst = gen_line_stride<COLS>(n, lines);
    x.re = lds + lane * lst;
    x.im = lds + 17 * THREADS + lane * lst;
    x.sgn = job.inverse ? 0x80000000u : 0u;
    const float2* rows = job.tw + GEN_TABLE;
    GenPass pass = gen_read_pass(job.tw, 0);
    gen_pass<true, false, COLS, IO>(x, pass, rows);
    for (int p = 1; p + 1 < job.npass; ++p) {
        pass = gen_read_pass(job.tw, p);
        gen_pass<false, false, COLS, IO>(x, pass, rows);
        rows += pass.ns * 4;
    }
    pass = gen_read_pass(job.tw, job.npass - 1);
    gen_pass<false, true, COLS, IO>(x, pass, rows);
}

}  // namespace mdft
