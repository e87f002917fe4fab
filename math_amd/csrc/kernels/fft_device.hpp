// Device-side building blocks of the 2-D DFT line passes (gfx950 / CDNA4).
//
// One "axis pass" transforms `count` lines of logical length n, laid out with
// element stride es and line stride ls inside a row-major complex<float>
// image (rows: es = 1, ls = w; columns: es = w, ls = 1).  A line of length n
// is transformed through an FFT of length M: directly when n is a power of
// two or 3 * 2^k in [192, 6144] (M = n; other smooth lengths run in
// smooth_device.hpp), otherwise by Bluestein's chirp-z
// method with M >= 2n - 1: the reference's padded length bit_ceil(2n - 2)
// (src/gpu/dft/function.cpp:32-45), or 3 * 2^k when that is shorter, and the
// chirp tables of function.cpp:49-92 generated in FP64 on the device.
//
// A workgroup owns LPW whole lines (a "tile").  Each thread holds EPT points
// (16, 32, 12 or 24, see the shapes below) of one line or of two in VGPRs, at
// positions t + i*TPL (TPL = M/EPT threads per line).  The FFT is a Stockham
// autosort in passes of up to radix 32, DIT form: pass p gathers its operands
// from LDS at the thread's fixed positions, runs a radix-R butterfly with the
// pass's twiddle row fused into it in registers and scatters to the Stockham
// positions.  The first pass needs no twiddles and reads straight from HBM; the
// last pass leaves its results at the thread's own positions, so it writes
// straight to HBM and Bluestein's two FFTs chain without an LDS exchange.  LDS
// holds one exchange buffer of real and imaginary planes (one plane, used twice,
// for 24 and 32 points per thread) in the layouts of lds_maps.inc, conflict-free
// for every exchange.
//
// Only the forward FFT exists: an inverse transform is conj(FFT(conj(x))),
// folded into the load, the D multiply and the store.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace mdft {

// ---------------------------------------------------------------------------
// complex helpers
// ---------------------------------------------------------------------------
__device__ __forceinline__ float2 cadd(float2 a, float2 b) { return make_float2(a.x + b.x, a.y + b.y); }
__device__ __forceinline__ float2 csub(float2 a, float2 b) { return make_float2(a.x - b.x, a.y - b.y); }
// Products are written with explicit fused multiply-adds and the library is
// built with -ffp-contract=off, so every rounding is fixed by the source and a
// line gives bitwise the same result in every kernel that runs it.
__device__ __forceinline__ float2 cmul(float2 a, float2 b)
{
    return make_float2(__builtin_fmaf(a.x, b.x, -(a.y * b.y)), __builtin_fmaf(a.x, b.y, a.y * b.x));
}
// a * conj(b)
__device__ __forceinline__ float2 cmulc(float2 a, float2 b)
{
    return make_float2(__builtin_fmaf(a.x, b.x, a.y * b.y), __builtin_fmaf(a.y, b.x, -(a.x * b.y)));
}
__device__ __forceinline__ float2 cconj(float2 a) { return make_float2(a.x, -a.y); }
// conj(a * b)
__device__ __forceinline__ float2 cmul_conj(float2 a, float2 b)
{
    return make_float2(__builtin_fmaf(a.x, b.x, -(a.y * b.y)), __builtin_fmaf(-a.x, b.y, -(a.y * b.x)));
}
// flip the sign of the imaginary part when sgn is 0x80000000 (conjugate), keep it when 0
__device__ __forceinline__ float2 cxor(float2 a, uint32_t sgn)
{
    return make_float2(a.x, __uint_as_float(__float_as_uint(a.y) ^ sgn));
}
__device__ __forceinline__ float2 cscale(float2 a, float s) { return make_float2(a.x * s, a.y * s); }

// ---------------------------------------------------------------------------
// compile-time line geometry
// ---------------------------------------------------------------------------
// A line's FFT has a "shape" S:
//  * S in [1, 12]: M = 2^S, radix-16 passes (16 points per thread) and one
//    remainder pass;
//  * S = 13, 14: 32 points per thread, passes 32 x 16 x 16 and 32 x 32 x 16, and
//    the LDS exchange one component at a time, so a line takes half the threads
//    and half the LDS of 16 points per thread (8192 points: 256 threads and
//    33 KB, 16384: 512 threads and 66 KB), a CU holds twice the lines, and
//    there is one exchange less than with radix 16;
//  * S = F3_BASE + k: M = 3 * 2^k (Bluestein convolutions, and lines of
//    exactly 3 * 2^k points transformed directly), 12 points per
//    thread: radix-4 passes, one radix-2 pass when k is odd, and a final
//    radix-12 pass (a 3 x 4 prime-factor butterfly).  6144 points: 24 per thread
//    in passes 8 x 8 x 8 x 12 (six passes of radix 4 and 2 took up to 15 % longer).
// The shape is a function of the line length and axis, so a line runs the
// same schedule in every kernel.
// S + X2: the same with two lines per thread (column tiles).  The lines of a tile share the
// chirp, the diagonal and the twiddles at a position, which one line per thread
// loads anew for every line (42 of the 60 loads of a Bluestein line's thread);
// a thread with two lines loads them once for both, reads two adjacent columns
// with one 16-byte load, and a tile has twice the columns (runs of a row twice
// as long) on the same LDS, the lines exchanging one after the other.
constexpr int MAX_LOGM = 14;
constexpr int X2 = 64;
__host__ __device__ constexpr int base_of(int s) { return s & 63; }
__host__ __device__ constexpr int lines_per_thread(int s) { return (s & X2) ? 2 : 1; }
// waves per SIMD the tile kernels are compiled for (at most 128 VGPRs)
constexpr int TILE_WAVES = 4;
constexpr int F3_BASE = 32;
constexpr int F3_MIN_K = 6;   // M = 192: the radix-12 pass follows at least two radix-4 passes
constexpr int F3_MAX_K = 11;  // M = 6144: 24 points per thread, 256 threads per line
__host__ __device__ constexpr bool is_f3(int s) { return base_of(s) >= F3_BASE && base_of(s) < 60; }
__host__ __device__ constexpr int f3_k(int s) { return base_of(s) - F3_BASE; }
// 8192 and 16384 points: 32 per thread
__host__ __device__ constexpr bool is_wide(int s) { return base_of(s) == 13 || base_of(s) == 14; }
// shapes with an X2 form: from 1024 points a 256-thread tile holds at most four lines
__host__ __device__ constexpr bool has_x2(int s)
{
    return (base_of(s) >= 10 && base_of(s) <= 12) || (is_f3(s) && (f3_k(s) == 9 || f3_k(s) == 10));
}
__host__ __device__ constexpr int m_of(int s) { return is_f3(s) ? (3 << f3_k(s)) : (1 << base_of(s)); }
// points of a line per thread
__host__ __device__ constexpr int ept_of(int s)
{
    return is_f3(s) ? (f3_k(s) == 11 ? 24 : 12) : is_wide(s) ? 32 : base_of(s) < 4 ? (1 << base_of(s)) : 16;
}
// threads per line
__host__ __device__ constexpr int tpl_of(int s) { return m_of(s) / ept_of(s); }
__host__ __device__ constexpr int npass_of(int s)
{
    return is_f3(s)     ? (f3_k(s) == 11 ? 4 : (f3_k(s) - 2) / 2 + (f3_k(s) - 2) % 2 + 1)
           : is_wide(s) ? 3
                        : (base_of(s) + 3) / 4;
}
// radix of pass p (1 when p is past the last pass)
__host__ __device__ constexpr int radix_of(int s, int p)
{
    if (p >= npass_of(s)) return 1;
    if (is_f3(s)) {
        const int a = f3_k(s) - 2;
        if (a == 9) return p < 3 ? 8 : 12;
        return p < a / 2 ? 4 : (p == npass_of(s) - 1 ? 12 : 2);
    }
    if (is_wide(s)) return p == 0 || (base_of(s) == 14 && p == 1) ? 32 : 16;
    return 1 << ((base_of(s) - 4 * p) >= 4 ? 4 : (base_of(s) - 4 * p));
}
// Stockham stride before pass p: the product of the earlier radices
__host__ __device__ constexpr int ns_of(int s, int p)
{
    int ns = 1;
    for (int q = 0; q < p; ++q) ns *= radix_of(s, q);
    return ns;
}

// Twiddle rows of pass p >= 1 (stride Ns = ns_of(s, p), radix R): row k
// (k < Ns) holds powers of w = exp(-2*pi*i*k/(Ns*R)):
//  * radix 16: w, w^2, w^4, w^8, the base twiddles of dft_twiddled (32 bytes,
//    four rows per cache line; the other stage twiddles are rotations);
//  * radix 32 (a pass of few rows): all 16 stage twiddles of dft_twiddled,
//    w^16, w^8, w^4 * {1, W8}, w^2 * {1, W16, W16^2, W16^3}, w * {1, W32, .. W32^7};
//  * other radices: w^1, w^2, w^3, w^4; the other powers are products of these
//    (expand_twiddles).
//  * 6144 points (full_rows): w^1 .. w^7 for radix 8, w^1 .. w^6, w^8, w^10 for
//    radix 12, so a product of two stands for three of them at most: with rows
//    of four the error against FP64 was 5 % above that of radix-4 passes.
__host__ __device__ constexpr bool full_rows(int s) { return is_f3(s) && f3_k(s) == 11; }
__host__ __device__ constexpr int tw_row(int radix, bool full = false) { return full ? 8 : radix == 32 ? 16 : 4; }
// entry e of row k: exp(-2*pi*i*q/(Ns*R)) with q = power * k + rotation * Ns*R/32
__host__ __device__ constexpr int tw_power(int radix, int e, bool full = false)
{
    if (full) return radix == 8 ? (e < 7 ? e + 1 : 0) : e < 6 ? e + 1 : 2 * e - 4;
    return radix == 16 ? (1 << e) : radix == 32 ? (e == 0 ? 16 : e == 1 ? 8 : e < 4 ? 4 : e < 8 ? 2 : 1) : e + 1;
}
__host__ __device__ constexpr int tw_rotation(int radix, int e)
{
    return radix != 32 || e < 2 ? 0 : e < 4 ? (e - 2) * 4 : e < 8 ? (e - 4) * 2 : e - 8;
}
__host__ __device__ constexpr int64_t tw_pass_len(int s, int p)
{
    return p >= 1 && p < npass_of(s) ? int64_t(ns_of(s, p)) * tw_row(radix_of(s, p), full_rows(s)) : 0;
}
__host__ __device__ constexpr int64_t tw_pass_off(int s, int p)
{
    int64_t off = 0;
    for (int q = 1; q < p; ++q) off += tw_pass_len(s, q);
    return off;
}
__host__ __device__ constexpr int64_t tw_len(int s)
{
    int64_t t = 0;
    for (int p = 1; p < npass_of(s); ++p) t += tw_pass_len(s, p);
    return t;
}
// Every shape has a block of one table: powers of two 1..MAX_LOGM, then
// 3 * 2^k for k in [F3_MIN_K, F3_MAX_K].
__host__ __device__ constexpr int64_t tw_off(int s)
{
    int64_t t = 0;
    const int plast = is_f3(s) ? MAX_LOGM + 1 : base_of(s);
    for (int l = 1; l < plast; ++l) t += tw_len(l);
    if (is_f3(s))
        for (int k = F3_MIN_K; k < f3_k(s); ++k) t += tw_len(F3_BASE + k);
    return t;
}
__host__ __device__ constexpr int64_t tw_total() { return tw_off(F3_BASE + F3_MAX_K + 1); }

// LDS layout of the exchange written by pass P: line position p is stored at
// word p + c * (p >> sh) of the line's slice, with (c, sh) chosen per FFT
// shape, workgroup size, axis and pass by gen_lds_maps.py (lds_maps.inc) so
// that (a) offsets stay linear, f(t + i*TPL) = f(t) + f(i*TPL) for the next
// pass's reads and f(base + r*NS) = f(base) + f(r*NS) for this pass's writes,
// making every LDS access a base register plus an immediate, and (b) no
// write or read instruction has a bank conflict (32 banks, 32 lanes per cycle).
struct LdsMap {
    int shape, threads, cols, pass, c, sh;
};
constexpr LdsMap kLdsMaps[] = {
#include "lds_maps.inc"
};
__host__ __device__ constexpr LdsMap lds_map(int shape, int threads, bool cols, int pass)
{
    for (const LdsMap& e : kLdsMaps)
        if (e.shape == base_of(shape) && e.threads == threads && e.cols == (cols ? 1 : 0) && e.pass == pass) return e;
    return LdsMap{shape, threads, cols ? 1 : 0, pass, -1, 0};  // missing: rejected by a static_assert
}
template <int S, int THREADS, bool COLS, int P>
__host__ __device__ constexpr int lds_pos(int p)
{
    constexpr LdsMap m = lds_map(S, THREADS, COLS, P);
    static_assert(m.c >= 0, "no LDS layout generated for this shape, workgroup size and pass");
    return p + m.c * (p >> m.sh);
}

template <int S, int THREADS>
struct LineCfg {
    static constexpr int M = m_of(S);
    static constexpr int EPT = ept_of(S);
    static constexpr int TPL = tpl_of(S);        // threads per line
    static constexpr int L = lines_per_thread(S);
    static constexpr int SLOTS = THREADS / TPL;  // lines side by side in the workgroup
    static constexpr int LPW = SLOTS * L;        // lines per tile
    static constexpr int NPASS = npass_of(S);
    // exchange the real parts, then the imaginary parts, through one plane
    static constexpr bool SPLIT = EPT > 16;
    static_assert(!SPLIT || L == 1, "32 points per thread: one line");
    static_assert(TPL <= THREADS, "line does not fit the workgroup");
    static_assert(SLOTS * TPL == THREADS, "workgroup must hold whole lines");
    // words of one line's slice: the largest padded position over the exchanges
    template <bool COLS, int P = 0>
    static constexpr int padm()
    {
        if constexpr (P + 1 >= NPASS) {
            return M;
        } else {
            const int a = lds_pos<S, THREADS, COLS, P>(M - 1) + 1;
            const int b = padm<COLS, P + 1>();
            return a > b ? a : b;
        }
    }
    // Line stride in LDS words.  Lanes of one wave cover q consecutive
    // positions of 32/q lines (rows: q = TPL; columns, lines fastest:
    // q = 32/SLOTS); a stride of q times an odd number puts them on distinct
    // banks (the same rule gen_lds_maps.py assumes).
    template <bool COLS>
    static constexpr int lstride()
    {
        const int q = COLS ? (SLOTS >= 32 ? 1 : 32 / SLOTS) : (TPL >= 32 ? 0 : TPL);
        const int pm = padm<COLS>();
        if (q == 0) return pm;
        int s = pm;
        while (s % (2 * q) != q) ++s;
        return s;
    }
    template <bool COLS>
    static constexpr int lds_floats()
    {
        return NPASS > 1 ? (SPLIT ? 1 : 2) * SLOTS * lstride<COLS>() : 0;
    }
};

// ---------------------------------------------------------------------------
// radix-R forward DFT in registers (R <= 32), natural order in and out
// ---------------------------------------------------------------------------
// cos(2*pi*m/32), sin(2*pi*m/32), m < 16
__device__ constexpr float kC32[16] = {
    1.0f, 0.98078528040323043f, 0.92387953251128674f, 0.83146961230254524f,
    0.70710678118654757f, 0.55557023301960229f, 0.38268343236508984f, 0.19509032201612833f,
    0.0f, -0.19509032201612819f, -0.38268343236508973f, -0.55557023301960196f,
    -0.70710678118654746f, -0.83146961230254535f, -0.92387953251128674f, -0.98078528040323043f
};
__device__ constexpr float kS32[16] = {
    0.0f, 0.19509032201612825f, 0.38268343236508978f, 0.55557023301960218f,
    0.70710678118654746f, 0.83146961230254524f, 0.92387953251128674f, 0.98078528040323043f,
    1.0f, 0.98078528040323043f, 0.92387953251128674f, 0.83146961230254546f,
    0.70710678118654757f, 0.55557023301960218f, 0.38268343236508989f, 0.19509032201612861f
};

// d * exp(-2*pi*i*m/32) for a compile-time m < 16
template <int m>
__device__ __forceinline__ float2 twc(float2 d)
{
    if constexpr (m == 0) {
        return d;
    } else if constexpr (m == 8) {
        return make_float2(d.y, -d.x);
    } else if constexpr (m == 4) {
        const float r = 0.70710678118654752440f;
        return make_float2(r * (d.x + d.y), r * (d.y - d.x));
    } else if constexpr (m == 12) {
        const float r = 0.70710678118654752440f;
        return make_float2(r * (d.y - d.x), -r * (d.x + d.y));
    } else {
        const float c = kC32[m], s = kS32[m];
        return make_float2(__builtin_fmaf(d.x, c, d.y * s), __builtin_fmaf(d.y, c, -(d.x * s)));
    }
}

__host__ __device__ constexpr int bitrev_small(int v, int bits)
{
    int r = 0;
    for (int i = 0; i < bits; ++i) {
        r = (r << 1) | (v & 1);
        v >>= 1;
    }
    return r;
}

// ---------------------------------------------------------------------------
// Radix 16 and 32: decimation in time with the pass's twiddles fused in.
//
// A pass multiplies input r by w^r and takes the R-point DFT.  Split even and
// odd r: stage h (h = 1, 2, 4, .. R/2) combines a and b into a +- t*b with
// t = w^(R/2h) * exp(-2*pi*i*k/2h), k < h.  The products never stand alone:
// a + t*b is four fused multiply-adds, a - t*b = 2a - (a + t*b) two more, so a
// twiddled radix-2 butterfly costs 6 instructions (8 for a product and two
// sums, or where a - t*b is formed by itself), and only w^(R/2), .., w^2, w
// and their constant rotations (t at k >= h/2 is -i times the one at k - h/2,
// a swap of operands) are needed: 8 twiddles for radix 16 instead of 15.  A
// radix-16 pass issues 224 VALU instructions, against 274 for 15 products, 11
// derived twiddles and a DIF butterfly.  Radices 2, 4 and 8 keep separate
// products: there the fused form saves nothing.
// ---------------------------------------------------------------------------
// a, b <- a + t*b, a - t*b with t rotated by -i when NEGI.  FULL: a - t*b by
// four fused multiply-adds of its own (8 instructions), which leaves out the
// rounding of a + t*b that 2a - (a + t*b) carries along.
template <bool NEGI, bool FULL>
__device__ __forceinline__ void bfly_tw(float2& a, float2& b, float2 t)
{
    // (-i*t)*b = (t.x*b.y + t.y*b.x) - i*(t.x*b.x - t.y*b.y)
    float2 y;
    if constexpr (NEGI) {
        y.x = __builtin_fmaf(t.y, b.x, __builtin_fmaf(t.x, b.y, a.x));
        y.y = __builtin_fmaf(t.y, b.y, __builtin_fmaf(-t.x, b.x, a.y));
    } else {
        y.x = __builtin_fmaf(-t.y, b.y, __builtin_fmaf(t.x, b.x, a.x));
        y.y = __builtin_fmaf(t.y, b.x, __builtin_fmaf(t.x, b.y, a.y));
    }
    if constexpr (!FULL) {
        b = make_float2(__builtin_fmaf(2.0f, a.x, -y.x), __builtin_fmaf(2.0f, a.y, -y.y));
    } else if constexpr (NEGI) {
        b = make_float2(__builtin_fmaf(-t.y, b.x, __builtin_fmaf(-t.x, b.y, a.x)),
                        __builtin_fmaf(-t.y, b.y, __builtin_fmaf(t.x, b.x, a.y)));
    } else {
        b = make_float2(__builtin_fmaf(t.y, b.y, __builtin_fmaf(-t.x, b.x, a.x)),
                        __builtin_fmaf(-t.y, b.x, __builtin_fmaf(-t.x, b.y, a.y)));
    }
    a = y;
}

// a, b <- a + t*b, a - t*b with t = exp(-2*pi*i*m/32), m < 16
template <int m>
__device__ __forceinline__ void bfly_const(float2& a, float2& b)
{
    if constexpr (m == 0) {
        const float2 t = b;
        b = csub(a, t);
        a = cadd(a, t);
    } else if constexpr (m == 8) {
        const float2 t = make_float2(b.y, -b.x);
        b = csub(a, t);
        a = cadd(a, t);
    } else if constexpr (m == 4 || m == 12) {
        const float r = 0.70710678118654752440f;
        // m = 4: r*(x + y) + i*r*(y - x); m = 12: r*(y - x) - i*r*(x + y)
        const float p = b.x + b.y, q = b.y - b.x;
        const float2 t = m == 4 ? make_float2(p, q) : make_float2(q, -p);
        b = make_float2(__builtin_fmaf(-r, t.x, a.x), __builtin_fmaf(-r, t.y, a.y));
        a = make_float2(__builtin_fmaf(r, t.x, a.x), __builtin_fmaf(r, t.y, a.y));
    } else {
        bfly_tw<false, false>(a, b, make_float2(kC32[m], -kS32[m]));
    }
}

// stage H of the untwiddled DFT over bit-reversed u.  ZHI: inputs R/2 + 1 ..
// are zero (bit-reversed: every odd slot but the first), so the pairs of stage
// 1 after the first are copies.
template <int R, int H, int BASE, int K, bool ZHI>
__device__ __forceinline__ void dit_bfly(float2* u)
{
    if constexpr (BASE < R) {
        if constexpr (K < H) {
            if constexpr (ZHI && H == 1 && BASE > 0)
                u[BASE + 1] = u[BASE];
            else
                bfly_const<K*(32 / (2 * H))>(u[BASE + K], u[BASE + K + H]);
            dit_bfly<R, H, BASE, K + 1, ZHI>(u);
        } else {
            dit_bfly<R, H, BASE + 2 * H, 0, ZHI>(u);
        }
    }
}

template <int R, int H, bool ZHI>
__device__ __forceinline__ void dit_stages(float2* u)
{
    if constexpr (H < R) {
        dit_bfly<R, H, 0, 0, ZHI>(u);
        dit_stages<R, 2 * H, ZHI>(u);
    }
}

// Stages whose butterflies take the 8-instruction form: with the 6-instruction
// form in every stage the error against FP64 was 1-3 % above that of separate
// products and sums at 512-4096 points, 5 % at 16384; so it is 0.5-1 % below.
__host__ __device__ constexpr bool full_stage(int radix, int h) { return radix == 32 || h >= 8; }

// stage H with the pass's twiddles; tw[k] = w^(R/2H) * exp(-2*pi*i*k/2H), k < max(H/2, 1)
template <int R, int H, int BASE, int K>
__device__ __forceinline__ void dit_tw_bfly(float2* u, const float2* tw)
{
    if constexpr (BASE < R) {
        if constexpr (K < H) {
            constexpr bool FULL = full_stage(R, H);
            if constexpr (H > 1 && K >= H / 2)
                bfly_tw<true, FULL>(u[BASE + K], u[BASE + K + H], tw[K - H / 2]);
            else
                bfly_tw<false, FULL>(u[BASE + K], u[BASE + K + H], tw[K]);
            dit_tw_bfly<R, H, BASE, K + 1>(u, tw);
        } else {
            dit_tw_bfly<R, H, BASE + 2 * H, 0>(u, tw);
        }
    }
}

template <int R>
__device__ __forceinline__ void bit_reverse(float2* u)
{
    constexpr int bits = (R == 2) ? 1 : (R == 4) ? 2 : (R == 8) ? 3 : (R == 16) ? 4 : 5;
    float2 t[R];
#pragma unroll
    for (int i = 0; i < R; ++i) t[i] = u[bitrev_small(i, bits)];
#pragma unroll
    for (int i = 0; i < R; ++i) u[i] = t[i];
}

// R-point DFT of u[r] * w^r from the pass's row q (tw_row), R = 16 or 32
template <int R>
__device__ __forceinline__ void dft_twiddled(float2 (&u)[R], const float4* q)
{
    static_assert(R == 16 || R == 32, "radix");
    bit_reverse<R>(u);
    auto entry = [&](int e) { return e % 2 ? make_float2(q[e / 2].z, q[e / 2].w) : make_float2(q[e / 2].x, q[e / 2].y); };
    if constexpr (R == 16) {
        const float2 w1 = entry(0), w2 = entry(1), w4 = entry(2), w8 = entry(3);
        dit_tw_bfly<R, 1, 0, 0>(u, &w8);
        dit_tw_bfly<R, 2, 0, 0>(u, &w4);
        const float2 t4[2] = {w2, twc<4>(w2)};
        dit_tw_bfly<R, 4, 0, 0>(u, t4);
        const float2 t8[4] = {w1, twc<2>(w1), twc<4>(w1), twc<6>(w1)};
        dit_tw_bfly<R, 8, 0, 0>(u, t8);
    } else {
        const float2 t1 = entry(0), t2 = entry(1);
        dit_tw_bfly<R, 1, 0, 0>(u, &t1);
        dit_tw_bfly<R, 2, 0, 0>(u, &t2);
        const float2 t4[2] = {entry(2), entry(3)};
        dit_tw_bfly<R, 4, 0, 0>(u, t4);
        const float2 t8[4] = {entry(4), entry(5), entry(6), entry(7)};
        dit_tw_bfly<R, 8, 0, 0>(u, t8);
        const float2 t16[8] = {entry(8),  entry(9),  entry(10), entry(11),
                               entry(12), entry(13), entry(14), entry(15)};
        dit_tw_bfly<R, 16, 0, 0>(u, t16);
    }
}

// forward 3-point DFT in place, W = exp(-2*pi*i/3): X1 = t2 - i*t3,
// X2 = t2 + i*t3 with t2 = x0 - (x1 + x2)/2, t3 = sin(pi/3) * (x1 - x2)
__device__ __forceinline__ void dft3(float2& x0, float2& x1, float2& x2)
{
    const float h = 0.86602540378443864676f;
    const float2 t1 = cadd(x1, x2);
    const float2 t2 = make_float2(__builtin_fmaf(-0.5f, t1.x, x0.x), __builtin_fmaf(-0.5f, t1.y, x0.y));
    const float2 t3 = make_float2(h * (x1.x - x2.x), h * (x1.y - x2.y));
    x0 = cadd(x0, t1);
    x1 = make_float2(t2.x + t3.y, t2.y - t3.x);
    x2 = make_float2(t2.x - t3.y, t2.y + t3.x);
}

// ZHI: inputs u[R/2 + 1 ..] are zero (the zero-padded half of a Bluestein
// line in its first pass).  R = 12 is the prime-factor (Good-Thomas) 3 x 4
// DFT: no twiddles; input n = (4*n1 + 3*n2) mod 12, output k = (4*k1 + 9*k2)
// mod 12 (k1 = k mod 3, k2 = k mod 4).
template <int R, bool ZHI = false>
__device__ __forceinline__ void dft_fwd(float2* u)
{
    if constexpr (R == 12) {
        static_assert(!ZHI, "no zero-input pruning for radix 12 (never a first pass)");
        float2 a0[4] = {u[0], u[3], u[6], u[9]};
        float2 a1[4] = {u[4], u[7], u[10], u[1]};
        float2 a2[4] = {u[8], u[11], u[2], u[5]};
        dft_fwd<4>(a0);
        dft_fwd<4>(a1);
        dft_fwd<4>(a2);
#pragma unroll
        for (int k2 = 0; k2 < 4; ++k2) {
            dft3(a0[k2], a1[k2], a2[k2]);
            u[(9 * k2) % 12] = a0[k2];
            u[(4 + 9 * k2) % 12] = a1[k2];
            u[(8 + 9 * k2) % 12] = a2[k2];
        }
    } else {
        static_assert(R >= 1 && R <= 32 && (R & (R - 1)) == 0, "radix");
        if constexpr (R > 1) {
            bit_reverse<R>(u);
            dit_stages<R, 1, ZHI>(u);
        }
    }
}

// ---------------------------------------------------------------------------
// the job of one axis pass
// ---------------------------------------------------------------------------
struct AxisJob {
    const float2* src;     // input image base
    float2* dst;           // output image base (may equal src)
    int64_t es;            // element stride (complex elements)
    int64_t ls;            // line stride
    int n;                 // logical line length
    int count;             // number of lines
    int inverse;           // 0 forward, 1 inverse
    float scale;           // 1/n for the inverse, 1 otherwise
    // Bluestein tables of the job's direction (c = exp(-i*pi*k^2/n)):
    const float2* chirp;      // load: c (forward) or conj(c) (inverse), k < n
    const float2* dtab;       // middle: D or conj(D), D = FFT_M(conj(c) embedded) / M
    const float2* chirp_out;  // store: conj(c) (forward) or c/n (inverse), k < n
    const float2* tw;      // twiddle block of the line's FFT shape
    // smooth lengths (smooth_device.hpp): threads per line and passes
    int tpl;
    int npass;
};

// Pass of a smooth length: GEN_MAX_PASS of these head the length's block, then
// for every pass after the first ns rows of four twiddles (tw_power).
struct GenPass {
    int radix;
    int ns;          // Stockham stride: the product of the earlier radices
    int nbf;         // butterflies, n / radix
    uint32_t magic;  // ceil(2^32 / ns): j / ns = umulhi(j, magic) for j < 4096
};
constexpr int GEN_MAX_PASS = 8;
constexpr int GEN_TABLE = GEN_MAX_PASS * (int)sizeof(GenPass) / (int)sizeof(float2);  // in float2
// shape code of such lengths, and the longest
constexpr int GEN_SHAPE = 60;
constexpr int GEN_MAX_N = 4096;

// ---------------------------------------------------------------------------
// image input and output of the view path: the luminance of an RGBA pixel
// becomes the complex input (src/gpu/dft/code/dft_copy_input.comp:37-54) and
// |X| * scale the R32F output (dft_copy_output.comp:34-48)
// ---------------------------------------------------------------------------
enum : int { IO_LUM = 1, IO_MAG = 2 };
enum : int { PIXEL_RGBA32F = 0, PIXEL_RGBA8 = 1 };
struct ImageIO {
    const void* img;  // RGBA pixel at the rectangle's origin
    int64_t iel;      // pixel stride along a line
    int64_t ils;      // pixel stride between lines
    int fmt;          // PIXEL_*
    float mscale;     // 1/(w*h)
    float* mag;       // R32F output at the rectangle's origin
    int64_t mel;      // float stride along a line
    int64_t mls;      // float stride between lines
};

// 0.2126 r + 0.7152 g + 0.0722 b (dft_copy_input.comp:37-40), fixed rounding order
__host__ __device__ __forceinline__ float luminance_rgb(float r, float g, float b)
{
    return __builtin_fmaf(0.0722f, b, __builtin_fmaf(0.7152f, g, 0.2126f * r));
}

// UNORM: c / 255, correctly rounded (one step of residual correction; equal to
// the division for all 256 values), in 3 instructions where a division takes about ten
__device__ __forceinline__ float unorm8(uint32_t c)
{
    const float r = 1.0f / 255.0f, x = (float)c, q = x * r;
    return __builtin_fmaf(__builtin_fmaf(-q, 255.0f, x), r, q);
}
__device__ __forceinline__ float luminance_rgba8(uint32_t c)
{
    return luminance_rgb(unorm8(c & 0xffu), unorm8((c >> 8) & 0xffu), unorm8((c >> 16) & 0xffu));
}

__device__ __forceinline__ float image_luminance(const ImageIO& io, int64_t idx)
{
    if (io.fmt == PIXEL_RGBA8) return luminance_rgba8(static_cast<const uint32_t*>(io.img)[idx]);
    const float4 c = static_cast<const float4*>(io.img)[idx];
    return luminance_rgb(c.x, c.y, c.z);
}

// out[i] = luminance of pixel index(i), i < N.  The format is uniform: one
// branch around all the loads, which are in flight together (a branch per
// pixel made every load a latency of its own).
template <int N, class Index>
__device__ __forceinline__ void load_luminance(const ImageIO& io, const Index& index, float (&out)[N])
{
    typedef float vec3 __attribute__((ext_vector_type(3)));
    if (io.fmt == PIXEL_RGBA8) {
        auto img = (const __attribute__((address_space(1))) uint32_t*)io.img;
        uint32_t px[N];
#pragma unroll
        for (int i = 0; i < N; ++i) px[i] = img[index(i)];
#pragma unroll
        for (int i = 0; i < N; ++i) out[i] = luminance_rgba8(px[i]);
    } else {
        auto img = (const __attribute__((address_space(1))) float*)io.img;
        vec3 px[N];
#pragma unroll
        for (int i = 0; i < N; ++i) {
            auto p = img + 4 * index(i);
            px[i] = vec3{p[0], p[1], p[2]};
        }
#pragma unroll
        for (int i = 0; i < N; ++i) out[i] = luminance_rgb(px[i].x, px[i].y, px[i].z);
    }
}

__device__ __forceinline__ float cabs_scaled(float2 y, float s)
{
    return __builtin_sqrtf(__builtin_fmaf(y.x, y.x, y.y * y.y)) * s;
}

// Global accesses.  The pointers of a batch job come from memory, where the
// compiler cannot tell global from LDS addresses and would use flat
// instructions, whose loads and stores also count as LDS traffic and are
// waited for at every exchange: the address space is stated.
typedef float vec2 __attribute__((ext_vector_type(2)));
typedef float vec4 __attribute__((ext_vector_type(4)));
#define MDFT_GLOBAL __attribute__((address_space(1)))
__device__ __forceinline__ float2 load_global(const float2* p)
{
    const vec2 x = *(const MDFT_GLOBAL vec2*)p;
    return make_float2(x.x, x.y);
}
__device__ __forceinline__ void store_global(float2* p, float2 x) { *(MDFT_GLOBAL vec2*)p = vec2{x.x, x.y}; }
// two adjacent elements (global accesses need no more than 4-byte alignment)
typedef float vec4_8 __attribute__((ext_vector_type(4), aligned(8)));
__device__ __forceinline__ void load_pair(const float2* p, float2& a, float2& b)
{
    const vec4 x = *(const MDFT_GLOBAL vec4_8*)p;
    a = make_float2(x.x, x.y);
    b = make_float2(x.z, x.w);
}
__device__ __forceinline__ void store_pair(float2* p, float2 a, float2 b)
{
    *(MDFT_GLOBAL vec4_8*)p = vec4{a.x, a.y, b.x, b.y};
}
// At a uniform address (p must not depend on the lane) plus a 32-bit element
// index: the address is kept in scalar registers, so every slot's access takes
// its offset from one vector register; left to itself the compiler adds each
// slot's offset to a 64-bit vector address, two or three VALU instructions and
// two registers a slot.
__device__ __forceinline__ float2 load_at(const float2* p, uint32_t i)
{
    auto g = (const MDFT_GLOBAL char*)p;
    asm("" : "+s"(g));
    const vec2 x = *(const MDFT_GLOBAL vec2*)(g + i * 8u);
    return make_float2(x.x, x.y);
}
__device__ __forceinline__ float4 load4_at(const float2* p, uint32_t bytes)
{
    auto g = (const MDFT_GLOBAL char*)p;
    asm("" : "+s"(g));
    const vec4 x = *(const MDFT_GLOBAL vec4*)(g + bytes);
    return make_float4(x.x, x.y, x.z, x.w);
}
__device__ __forceinline__ void store_at(float2* p, uint32_t i, float2 x)
{
    auto g = (MDFT_GLOBAL char*)p;
    asm("" : "+s"(g));
    *(MDFT_GLOBAL vec2*)(g + i * 8u) = vec2{x.x, x.y};
}
// a value the compiler knows nothing about
template <class V>
__device__ __forceinline__ V opaque(V x)
{
    asm("" : "+v"(x));
    return x;
}

// ---------------------------------------------------------------------------
// FFT of the tile held in registers
// ---------------------------------------------------------------------------
// Barrier around an LDS exchange.  When every line of a tile lies inside one
// wave (row mapping with TPL <= 64), an exchange never crosses waves, and the
// LDS operations of one wave are performed in order, so a wave-level
// code-motion barrier replaces the workgroup barrier: waves of the tile then
// run their passes independently.
template <bool WAVE>
__device__ __forceinline__ void exchange_sync()
{
    if constexpr (WAVE) {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    } else {
        __syncthreads();
    }
}

// Twiddle rows of pass P for the thread's butterflies are loaded one pass
// ahead (pass 1's with the tile's input), so the table latency overlaps the
// LDS exchange instead of following it.
// float4s of a row a radix-R butterfly reads
template <int R, bool FULL = false>
__host__ __device__ constexpr int tw_quads()
{
    return R <= 2 ? 1 : tw_row(R, FULL) / 2;
}

template <int S, int THREADS, int P>
struct TwLoad {
    using C = LineCfg<S, THREADS>;
    static constexpr int R = radix_of(S, P);
    static constexpr int Q = tw_quads<R, full_rows(S)>();
    static constexpr int NB = C::EPT / R;
    static constexpr int NS = ns_of(S, P);
    static_assert(NB * Q <= C::EPT / 2, "twiddle registers");
    __device__ __forceinline__ static void run(float4 (&w)[C::EPT / 2], int t, const float2* tw)
    {
#pragma unroll
        for (int b = 0; b < NB; ++b) {
            const int k = (t + b * C::TPL) & (NS - 1);
            // the second float4 of a row is an immediate offset away
#pragma unroll
            for (int r2 = 0; r2 < Q; ++r2)
                w[b * Q + r2] = load4_at(tw + tw_pass_off(S, P), uint32_t(k) * uint32_t(8 * tw_row(R, full_rows(S))) + 16u * r2);
        }
    }
};

// the R twiddles of one butterfly (wt[0] unused) from its row: w^1..w^4
// loaded, w^(4a+b) = w^(4a) * w^b, w^(4a) = w^(4a-4) * w^4 (at most four
// roundings from the FP64-generated entries)
template <int R, int r>
__device__ __forceinline__ void expand_products(float2 (&wt)[R])
{
    if constexpr (r < R) {
        if constexpr (r % 4 == 0)
            wt[r] = cmul(wt[r - 4], wt[4]);
        else
            wt[r] = cmul(wt[r - r % 4], wt[r % 4]);
        expand_products<R, r + 1>(wt);
    }
}

template <int R, bool FULL = false>
__device__ __forceinline__ void expand_twiddles(float2 (&wt)[R], const float4* q)
{
    if constexpr (FULL) {
        static_assert(R == 8 || R == 12, "radix");
#pragma unroll
        for (int e = 0; e < (R == 8 ? 7 : 8); ++e)
            wt[tw_power(R, e, true)] = e % 2 ? make_float2(q[e / 2].z, q[e / 2].w) : make_float2(q[e / 2].x, q[e / 2].y);
        if constexpr (R == 12) {
            wt[7] = cmul(wt[4], wt[3]);
            wt[9] = cmul(wt[8], wt[1]);
            wt[11] = cmul(wt[8], wt[3]);
        }
        return;
    }
    wt[1] = make_float2(q[0].x, q[0].y);
    if constexpr (R > 2) {
        wt[2] = make_float2(q[0].z, q[0].w);
        if constexpr (R > 3) wt[3] = make_float2(q[1].x, q[1].y);
    }
    if constexpr (R > 4) {
        wt[4] = make_float2(q[1].z, q[1].w);
        expand_products<R, 5>(wt);
    }
}

// ZIN (first pass only): slots EPT/2 + 1 .. EPT of every thread are zero.
// PF: the first PF slots of a table (pfs, indexed by line position) are
// loaded into pf one pass before the last, so their latency overlaps the
// last exchange and butterflies; slots PF .. PFL-1 at the start of the last
// pass, after its exchange (with one pass, all PFL at its start).
template <int S, int THREADS, bool COLS, int P, bool ZIN = false, int PF = 0, int PFL = 0, int EL = 0>
struct FftPass {
    using C = LineCfg<S, THREADS>;
    static constexpr bool WAVE = !COLS && C::TPL <= 64;
    static constexpr int R = radix_of(S, P);
    static constexpr int NB = C::EPT / R;
    static constexpr int NS = ns_of(S, P);
    static constexpr bool LAST = (P == C::NPASS - 1);
    static_assert(NB * R == C::EPT, "the radix divides the points per thread");

    using Regs = float2 (&)[C::L][C::EPT];  // the thread's lines

    // Stockham positions of this pass's outputs, component c
    template <int c>
    __device__ __forceinline__ static void scatter(const float2 (&v)[C::EPT], int t, float* plane)
    {
#pragma unroll
        for (int b = 0; b < NB; ++b) {
            const int j = t + b * C::TPL;
            const int k = j & (NS - 1);
            const int q0 = lds_pos<S, THREADS, COLS, P>((j - k) * R + k);
            // the layout keeps the R outputs' offsets linear: f(base) + f(r*NS)
#pragma unroll
            for (int r = 0; r < R; ++r)
                plane[q0 + lds_pos<S, THREADS, COLS, P>(r * NS)] = c == 0 ? v[b + NB * r].x : v[b + NB * r].y;
        }
    }

    // the next pass's operands: the thread's fixed positions t + i*TPL (the
    // offset of slot i is a compile-time constant, an LDS immediate)
    template <int c>
    __device__ __forceinline__ static void gather(float2 (&v)[C::EPT], int t, const float* plane)
    {
        const int q0 = lds_pos<S, THREADS, COLS, P>(t);
#pragma unroll
        for (int i = 0; i < C::EPT; ++i) {
            const float x = plane[q0 + lds_pos<S, THREADS, COLS, P>(i * C::TPL)];
            if constexpr (c == 0)
                v[i].x = x;
            else
                v[i].y = x;
        }
    }

    __device__ __forceinline__ static void exchange(Regs v, int t, float* re, float* im)
    {
#pragma unroll
        for (int l = 0; l < C::L; ++l) {
            exchange_sync<WAVE>();  // the previous exchange's reads are done
            if constexpr (C::SPLIT) {
                scatter<0>(v[l], t, re);
                exchange_sync<WAVE>();
                gather<0>(v[l], t, re);
                exchange_sync<WAVE>();
                scatter<1>(v[l], t, re);
                exchange_sync<WAVE>();
                gather<1>(v[l], t, re);
            } else {
                scatter<0>(v[l], t, re);
                scatter<1>(v[l], t, im);
                exchange_sync<WAVE>();
                gather<0>(v[l], t, re);
                gather<1>(v[l], t, im);
            }
        }
    }

    template <class Epi>
    __device__ __forceinline__ static void run(Regs v, int t, float* re, float* im, const float2* tw,
                                               float4 (&w)[C::EPT / 2], const float2* pfs, float2 (&pf)[C::EPT],
                                               const Epi& epi)
    {
        static_assert(PF <= C::EPT && PFL <= C::EPT, "prefetch slots");
        if constexpr ((PF > 0 || PFL > 0) && C::NPASS == 1) {
#pragma unroll
            for (int i = 0; i < (PFL > PF ? PFL : PF); ++i) pf[i] = load_at(pfs + i * C::TPL, uint32_t(t));
        }
        if constexpr (LAST && P > 0 && PFL > PF) {
#pragma unroll
            for (int i = PF; i < PFL; ++i) pf[i] = load_at(pfs + i * C::TPL, uint32_t(t));
        }
        // butterfly b reads and writes only the slots b + NB*r: update in place
#pragma unroll
        for (int b = 0; b < NB; ++b) {
            float2 u[R];
            float2 tab[R];
            if constexpr (LAST && C::SPLIT && EL > 0) {
#pragma unroll
                for (int r = 0; r < R; ++r)
                    if (b + NB * r < EL) tab[r] = load_at(pfs + (b + NB * r) * C::TPL, uint32_t(t));
            }
#pragma unroll
            for (int l = 0; l < C::L; ++l) {
#pragma unroll
                for (int r = 0; r < R; ++r) u[r] = v[l][b + NB * r];
                if constexpr (P > 0) {
                    // the same for the thread's lines
                    constexpr int Q = tw_quads<R, full_rows(S)>();
                    float4 q[Q];
#pragma unroll
                    for (int r2 = 0; r2 < Q; ++r2) q[r2] = w[b * Q + r2];
                    if constexpr (R == 16 || R == 32) {
                        dft_twiddled<R>(u, q);
                    } else {
                        float2 wt[R];
                        expand_twiddles<R, full_rows(S)>(wt, q);
#pragma unroll
                        for (int r = 1; r < R; ++r) u[r] = cmul(u[r], wt[r]);
                        dft_fwd<R>(u);
                    }
                } else {
                    // ZIN: slot b + NB*r holds a zero for r > R/2 (b + NB*(R/2 + 1) >= EPT/2 + 1)
                    dft_fwd<R, ZIN>(u);
                }
                static_assert(!ZIN || P == 0, "zero inputs only in the first pass");
#pragma unroll
                for (int r = 0; r < R; ++r) v[l][b + NB * r] = u[r];
            }
            if constexpr (LAST && C::SPLIT) {
#pragma unroll
                for (int r = 0; r < R; ++r) epi(b + NB * r, v[0][b + NB * r], tab[r]);
            }
            // one butterfly's operands at a time: without it the scheduler
            // starts the next one's loads early and spills
            if constexpr (C::SPLIT && NB > 1) __builtin_amdgcn_sched_barrier(0);
        }
        if constexpr (!LAST) {
            TwLoad<S, THREADS, P + 1>::run(w, t, tw);
            if constexpr (PF > 0 && P + 2 == C::NPASS) {
#pragma unroll
                for (int i = 0; i < PF; ++i) pf[i] = load_at(pfs + i * C::TPL, uint32_t(t));
            }
            exchange(v, t, re, im);
            FftPass<S, THREADS, COLS, P + 1, false, PF, PFL, EL>::run(v, t, re, im, tw, w, pfs, pf, epi);
        }
    }
};

// ZIN: the upper half of the line is zero apart from position M/2, so slots
// EPT/2 + 1 .. EPT of every thread hold zeros (the caller set them to
// constant zero).  PF > 0: pf[i] = pfs[t + i*TPL] for i < max(PF, PFL) on
// return, loaded during the FFT (pfs must be readable at every such
// position).
//
// Shapes with the split exchange have no registers for that: run_epi calls
// epi(i, v[i], pfs[t + i*TPL]) for every slot as the last pass finishes it,
// with the table entries of one butterfly loaded before its arithmetic (the
// entries of slots EL .. are not loaded).
struct NoEpilogue {
    __device__ __forceinline__ void operator()(int, float2&, float2) const {}
};
template <int S, int THREADS, bool COLS, bool ZIN = false, int PF = 0, int PFL = 0>
struct FftTile {
    using C = LineCfg<S, THREADS>;
    using Regs = float2 (&)[C::L][C::EPT];
    // no table: one line per thread
    __device__ __forceinline__ static void run(float2 (&v)[C::EPT], int t, int slot, float* lds, const float2* tw)
    {
        static_assert(PF == 0 && PFL == 0 && C::L == 1, "prefetch needs a destination");
        float2 pf[C::EPT];
        run_all<0>(reinterpret_cast<Regs>(v), t, slot, lds, tw, nullptr, pf, NoEpilogue{});
    }
    __device__ __forceinline__ static void run(Regs v, int t, int slot, float* lds, const float2* tw,
                                               const float2* pfs, float2 (&pf)[C::EPT])
    {
        run_all<0>(v, t, slot, lds, tw, pfs, pf, NoEpilogue{});
    }
    template <int EL, class Epi>
    __device__ __forceinline__ static void run_epi(Regs v, int t, int slot, float* lds, const float2* tw,
                                                   const float2* pfs, const Epi& epi)
    {
        static_assert(C::SPLIT && PF == 0 && PFL == 0, "split exchange only");
        float2 pf[C::EPT];
        run_all<EL>(v, t, slot, lds, tw, pfs, pf, epi);
    }

private:
    template <int EL, class Epi>
    __device__ __forceinline__ static void run_all(Regs v, int t, int slot, float* lds, const float2* tw,
                                                   const float2* pfs, float2 (&pf)[C::EPT], const Epi& epi)
    {
        constexpr int LST = C::template lstride<COLS>();
        float* re = lds + slot * LST;
        float* im = C::SPLIT ? re : re + C::SLOTS * LST;
        float4 w[C::EPT / 2];
        if constexpr (!C::SPLIT && C::NPASS > 1) TwLoad<S, THREADS, 1>::run(w, t, tw);
        FftPass<S, THREADS, COLS, 0, ZIN, PF, PFL, EL>::run(v, t, re, im, tw, w, pfs, pf, epi);
    }
};

// ---------------------------------------------------------------------------
// one tile of one axis pass: load (+chirp), FFT, [x D, FFT], store (+chirp)
// ---------------------------------------------------------------------------
// IO (image kernels only): IO_LUM loads luminance from io.img instead of
// complex values from job.src; IO_MAG stores |X| * io.mscale to io.mag
// instead of complex values to job.dst.
template <int S, int THREADS, bool BLUE, bool COLS, int IO = 0>
__device__ __forceinline__ void line_tile(const AxisJob& job, int tile, float* lds, int tid, ImageIO io = ImageIO{})
{
    using C = LineCfg<S, THREADS>;
    constexpr int L = C::L;
    static_assert(IO == 0 || L == 1 || (COLS && (IO & IO_LUM) == 0), "image input: one line per thread");
    const int slot = COLS ? (tid % C::SLOTS) : (tid / C::TPL);
    const int t = COLS ? (tid / C::SLOTS) : (tid % C::TPL);
    // the thread's lines: adjacent columns, or rows SLOTS apart
    auto line_of = [&](int l) { return tile * C::LPW + (COLS ? slot * L + l : l * C::SLOTS + slot); };
    auto valid = [&](int l) { return line_of(l) < job.count; };
    // two columns of a tile without a missing column: 16-byte accesses
    const bool pairs = COLS && L == 2 && (tile + 1) * C::LPW <= job.count;
    const int n = job.n;
    // Consecutive slots of a thread are TPL elements apart.  A column steps by
    // the image width: 64-bit addresses.  Rows are contiguous, and like the
    // tables they are addressed as a uniform base (of the tile's first line and
    // the slot) plus a 32-bit offset: a tile's rows span less than 2^25
    // elements, and one register serves every slot.
    const int64_t step = COLS ? int64_t(C::TPL) * job.es : int64_t(C::TPL);
    // (a line past the last one reads the tile's first line and stores nothing)
    int64_t base[L];
    uint32_t off[L];
#pragma unroll
    for (int l = 0; l < L; ++l) {
        base[l] = COLS ? int64_t(valid(l) ? line_of(l) : tile * C::LPW) * job.ls + int64_t(t) * job.es
                       : int64_t(tile) * C::LPW * job.ls;
        off[l] = COLS ? 0u : valid(l) ? uint32_t(line_of(l) - tile * C::LPW) * uint32_t(job.ls) + uint32_t(t) : uint32_t(t);
    }
    // direction enters as a sign mask: conjugation is one xor, and the
    // inverse's 1/n is a multiply by job.scale (exactly 1 for the forward)
    const uint32_t sgn = job.inverse ? 0x80000000u : 0u;
    // a direct line (2^k or 3 * 2^k points) fills the FFT (n == M); only Bluestein pads
    auto in_line = [&](int pos) { return !BLUE || pos < n; };
    // Bluestein: n <= M/2 + 1, so slot i holds a position of the line only
    // for i <= EPT/2 (slot EPT/2 only at t = 0 when n = M/2 + 1; for 3 * 2^k
    // lengths M >= 2n - 1, so i < EPT/2); the other slots are zero on input
    // and not stored on output.
    constexpr int LIVE = BLUE ? (is_f3(S) ? C::EPT / 2 : C::EPT / 2 + 1) : C::EPT;
    // the first FFT skips the zero half in the butterflies of its first pass
    constexpr bool ZIN = BLUE;

    // Every load is issued before the first wait: no load sits under a branch,
    // where the compiler waits for it before it goes on (nine latencies in a
    // row per Bluestein tile).  A slot past the end of its line reads the
    // thread's first slot and becomes zero afterwards; the chirp is readable at
    // every live slot (dir_tables_len).  The line fills more than a quarter (a
    // third for 3 * 2^k) of the FFT, so the first slots need no check.
    constexpr int SURE = BLUE ? (is_f3(S) ? C::EPT / 3 : C::EPT / 4) : C::EPT;
    // Rows of up to 16 points lie whole in one thread, whose loads a wave spreads
    // over 64 lines: in pairs they are half as many requests for the same cache
    // lines (2^20 rows of 16 points: 102 us by single elements, 56 in pairs).
    constexpr bool WHOLE_ROW = !BLUE && !COLS && C::TPL == 1 && IO == 0;
    float2 v[L][C::EPT];
    {
        float2 c[LIVE];
        if (pairs) {
            const float2* s = job.src + base[0];
#pragma unroll
            for (int i = 0; i < LIVE; ++i) {
                const bool in = i < SURE || t + i * C::TPL < n;
                // opaque: else the select becomes a branch around the load
                load_pair(i < SURE ? s + i * step : s + opaque(in ? i * step : 0), v[0][i], v[L - 1][i]);
            }
        } else if constexpr ((IO & IO_LUM) != 0) {
            const int64_t line = valid(0) ? line_of(0) : tile * C::LPW;
            float lum[LIVE];
            load_luminance<LIVE>(
                io,
                [&](int i) {
                    const int pos = i < SURE || t + i * C::TPL < n ? t + i * C::TPL : t;
                    return line * io.ils + int64_t(opaque(pos)) * io.iel;
                },
                lum);
#pragma unroll
            for (int i = 0; i < LIVE; ++i) v[0][i] = make_float2(lum[i], 0.0f);
        } else if constexpr (WHOLE_ROW) {
            const float2* s = job.src + int64_t(valid(0) ? line_of(0) : tile * C::LPW) * job.ls;
#pragma unroll
            for (int i = 0; i < C::EPT; i += 2) {
                load_pair(s + i, v[0][i], v[0][i + 1]);
                // in address order (any other: 2^22 rows of 4 points 41.3 us instead of 40.0)
                __builtin_amdgcn_sched_barrier(0);
            }
        } else {
#pragma unroll
            for (int i = 0; i < LIVE; ++i) {
                const bool in = i < SURE || t + i * C::TPL < n;
#pragma unroll
                for (int l = 0; l < L; ++l) {
                    const float2* s = job.src + base[l];
                    if constexpr (COLS) {
                        v[l][i] = load_global(i < SURE ? s + i * step : s + opaque(in ? i * step : 0));
                    } else {
                        v[l][i] = i < SURE ? load_at(s + i * step, off[l])
                                           : load_at(s, opaque(in ? off[l] + uint32_t(i * C::TPL) : off[l]));
                    }
                }
            }
        }
        if constexpr (BLUE) {
#pragma unroll
            for (int i = 0; i < LIVE; ++i) c[i] = load_at(job.chirp + i * C::TPL, uint32_t(t));
        }
#pragma unroll
        for (int l = 0; l < L; ++l) {
#pragma unroll
            for (int i = 0; i < C::EPT; ++i) {
                if (i >= LIVE) {
                    v[l][i] = make_float2(0.0f, 0.0f);
                } else if constexpr (BLUE) {
                    // forward x*c, inverse x*conj(c) (direction tables)
                    const bool in = i < SURE || t + i * C::TPL < n;
                    const float2 x = cmul(v[l][i], c[i]);
                    v[l][i] = in ? x : make_float2(0.0f, 0.0f);
                } else {
                    v[l][i] = cxor(v[l][i], sgn);  // conj for the inverse
                }
            }
        }
    }

    const float sc = job.scale;
    // The output's addresses: with two lines per thread worked out anew from
    // the thread index, since the input's would be kept (and spilled) through
    // both FFTs, 48 bytes of scratch traffic a thread.
    const int tid_o = L == 2 ? opaque(tid) : tid;
    const int slot_o = COLS ? (tid_o % C::SLOTS) : (tid_o / C::TPL);
    const int t_o = COLS ? (tid_o / C::SLOTS) : (tid_o % C::TPL);
    // finished slot i of the thread's lines into the output
    auto put = [&](int i, const float2 (&y)[L]) {
        const uint32_t pos = uint32_t(t_o + i * C::TPL);
        if (!in_line((int)pos)) return;
        const int first = tile * C::LPW + (COLS ? slot_o * L : slot_o);  // the thread's first line
        if constexpr (IO == 0 && L == 2) {
            if (pairs) {
                store_pair(job.dst + int64_t(first) * job.ls + int64_t(t_o) * job.es + i * step, y[0], y[L - 1]);
                return;
            }
        }
#pragma unroll
        for (int l = 0; l < L; ++l) {
            const int line = first + (COLS ? l : l * C::SLOTS);
            if (line >= job.count) continue;
            if constexpr ((IO & IO_MAG) != 0)
                io.mag[int64_t(line) * io.mls + int64_t(pos) * io.mel] = cabs_scaled(y[l], io.mscale);
            else if constexpr (COLS)
                store_global(job.dst + int64_t(line) * job.ls + int64_t(t_o) * job.es + i * step, y[l]);
            else
                store_at(job.dst + base[l] + i * step, off[l], y[l]);
        }
    };

    if constexpr (C::SPLIT) {
        if constexpr (BLUE) {
            // the products of the branch below, slot by slot in the last passes
            FftTile<S, THREADS, COLS, ZIN>::template run_epi<C::EPT>(
                v, t, slot, lds, job.tw, job.dtab, [&](int, float2& x, float2 d) { x = cmul_conj(x, d); });
            FftTile<S, THREADS, COLS>::template run_epi<LIVE>(v, t, slot, lds, job.tw, job.chirp_out,
                                                               [&](int i, float2& x, float2 c) {
                                                                   if (i < LIVE) put(i, {cmul_conj(x, c)});
                                                               });
        } else {
            FftTile<S, THREADS, COLS>::template run_epi<0>(
                v, t, slot, lds, job.tw, nullptr,
                [&](int i, float2& x, float2) { put(i, {cscale(cxor(x, sgn), sc)}); });
        }
    } else {
        // Bluestein: D arrives during the first FFT, its first half one pass
        // before the end and the rest at the start of the last pass (earlier
        // loads of all of D spill at the 128-VGPR cap; with two lines per thread
        // it all comes in the last pass), and the live slots of the output
        // chirp during the second
        constexpr int PFD = (BLUE && C::NPASS <= 3 && L == 1) ? C::EPT / 2 : 0;
        constexpr int PFDL = (BLUE && C::NPASS <= 3) ? C::EPT : 0;
        float2 pf[C::EPT];
        FftTile<S, THREADS, COLS, ZIN, PFD, PFDL>::run(v, t, slot, lds, job.tw, job.dtab, pf);

        if constexpr (BLUE) {
            // forward conj(v*D), inverse conj(v)*D = conj(v*conj(D)); the outer
            // conjugation turns the next forward FFT into the inverse one
#pragma unroll
            for (int i = 0; i < C::EPT; ++i) {
                const float2 d = i < PFDL ? pf[i] : load_at(job.dtab + i * C::TPL, uint32_t(t));
#pragma unroll
                for (int l = 0; l < L; ++l) v[l][i] = cmul_conj(v[l][i], d);
            }
            // the output chirp block is followed by readable entries up to
            // position M/2 + M/16 (dir_tables_len), so every live slot can be loaded
            constexpr int PFO = L == 1 ? LIVE : 0;
            FftTile<S, THREADS, COLS, false, PFO, LIVE>::run(v, t, slot, lds, job.tw, job.chirp_out, pf);
        }
        if constexpr (WHOLE_ROW) {
            if (!valid(0)) return;
            float2* o = job.dst + int64_t(line_of(0)) * job.ls;
#pragma unroll
            for (int i = 0; i < C::EPT; i += 2)
                store_pair(o + i, cscale(cxor(v[0][i], sgn), sc), cscale(cxor(v[0][i + 1], sgn), sc));
            return;
        }
#pragma unroll
        for (int i = 0; i < LIVE; ++i) {
            float2 y[L];
            // forward conj(v)*c = conj(v*conj(c)), inverse conj(v*c)/n = conj(v*(c/n))
#pragma unroll
            for (int l = 0; l < L; ++l) y[l] = BLUE ? cmul_conj(v[l][i], pf[i]) : cscale(cxor(v[l][i], sgn), sc);
            put(i, y);
        }
    }
}

// Workgroups are dealt to the 8 XCDs round-robin (block b runs on XCD b % 8).
// Give each XCD a contiguous range of tiles so neighbouring column tiles,
// which share cache lines, meet in the same L2.
__device__ __forceinline__ int xcd_remap(int bid, int nblocks)
{
    constexpr int NXCD = 8;
    const int xcd = bid % NXCD;
    const int local = bid / NXCD;
    const int q = nblocks / NXCD, r = nblocks % NXCD;
    return xcd < r ? xcd * (q + 1) + local : r * (q + 1) + (xcd - r) * q + local;
}

}  // namespace mdft
