// Sieve on the matrix cores for the all-pairs kernels.
//
// Whether |h_i - round(h_i)| < tol for the three rows h = UBI.g needs h only
// to a small fraction of tol, and only modulo 1.  v_mfma_f32_32x32x16_f16
// gives 32 peaks x 32 grains of one row from 16 products each, and with the
// f32 accumulator started at 1.5 2^23 its last bit is worth exactly 1.  With
// every product scaled by 2^16 the low 16 bits of the accumulator's own bit
// pattern are then the fraction of h in units of 2^-16: no subtraction,
// rounding or conversion is left for the vector ALU, which takes the maximum
// of three 16-bit fields, the minimum over four pairs, and compares that:
// three 16-bit instructions (2.4-2.8 cycles per wave each on their own;
// v_max3_u16 and v_min3_u16 take 8.4) and a quarter of a compare (4.2) per pair,
// 5.1 with the queues, the settling and the matrix instructions counted in,
// against 11 FP64 instructions (4.5) of the row sieve k_score_many_sieve.  The
// MFMA's 32 cycles per 1024 products overlap them.  Measured, 1000 grains x 10^6
// peaks, tol 0.05: 146 us against 386; with the queue pushes off 120, with the
// settling off 128.  Bound by vector issue: the vector ALU is busy 82% of the
// cycles and the matrix cores 25%, at 2.4 GHz and 3.3 waves per SIMD; where no
// pair passes, 88% of 24% fewer cycles, over constant data as over random
// (292 000 and 296 000 against 383 000).
//
// Splitting.  u and g are each held as hi + lo in f16 (22 bits), and the
// products hi hi + hi lo + lo hi use 9 of the 16 k slots:
//   k      0..2      3..5      6..8      9..15
//   peak   gh_j      gl_j      gh_j      p_0..p_6
//   grain  uh_j      uh_j      ul_j      q_0..q_6
// with u' = 2^6 u and g' = 2^10 g (so that the low parts are normal f16
// numbers) and p, q free for terms that depend on the grain's position.
//
// Certification.  With |u| < 900 and |g| < 30 (no overflow of f16) and
// A = sum_j |u_ij| max|g_j| <= GS_SIEVE_SPAN for every row:
//   hi + lo is within 2^-22 of u' (g') relative, or 2^-25 absolute where lo
//   is subnormal, the product lo lo that is left out is below 2^-22 |u' g'|:
//   together < 3 2^-22 A + 2^-31 (|u|_1 + |g|_1) 2^5 < 5e-5;
//   the products of two f16 numbers are exact in f32, and each of the 17
//   additions, of whatever order and of rounding or truncation, keeps the
//   accumulator in [2^23, 2^24) or below it and is therefore within one unit
//   of its last place, 2^-16 of h: < 2.6e-4.
// So h is within GS_SIEVE_ERR = 2^-11 = 4.9e-4, tested with r = tol + 2^-11
// (+ the reference's own rounding of h and t, 1e-12): a pair with
// fract(h + r) > 2r in any row has a reference drlv2 >= tol^2 and is not
// counted.  The others (the cube of side 2r, 0.1% of random pairs at tol
// 0.05, and the true hits) are settled one by one with the reference
// arithmetic, so the sieve decides nothing that arithmetic would not.
// A pair with a non-finite u or g has a NaN drlv2 and never counts: such peaks
// and grains are kept out of the bounds and given a finite stand-in, in the
// score the one that passes nothing (k_sieve_pack).  Larger A: up to GS_SIEVE_SPAN_WIDE the accumulator
// starts at 1.5 2^27 (its last bit 2^-12 of h) and the fields are shifted
// left by four first, error GS_SIEVE_ERR_WIDE = 2^-7 by the same count;
// beyond that, and beyond |u| and |g|, the tile is tested in f32 on the
// vector ALU (gs_tile32).
#pragma once
#include "gs_kernels.h"

typedef _Float16 gs_half8 __attribute__((ext_vector_type(8)));
typedef float gs_float16 __attribute__((ext_vector_type(16)));
typedef short gs_short2 __attribute__((ext_vector_type(2)));

#define GS_SIEVE_SPAN 60.0f
#define GS_SIEVE_SPAN_WIDE 1000.0f
#define GS_SIEVE_UMAX 900.0f
#define GS_SIEVE_GMAX 30.0f
#define GS_SIEVE_ERR 0x1p-11
#define GS_SIEVE_ERR_WIDE 0x1p-7
// The ball (gs_ball_tile) is the faster one from here (1000 x 10^6 at tol 0.1:
// sieve 207 us, ball 282; at 0.2 a quarter of all quads would pass the sieve),
// up to where (tol + sqrt(3) GS_SIEVE_ERR_WIDE)^2, 0.583 at 0.75, would come
// near a dead pair's S, 3/4.
#define GS_BALL_TOL_MIN 0.1
#define GS_BALL_TOL_MAX 0.75
#define GS_SIEVE_SETS 4    // 32-peak sets per wave (NB)
#define GS_SIEVE_SPLIT 64  // grain tiles of a block's split at most (its counters in LDS)

// v = hi + lo in f16, for a scaled value below the f16 range
GS_HD __forceinline__ void gs_split16(double v, _Float16& hi, _Float16& lo) {
    hi = (_Float16)(float)v;
    lo = (_Float16)(float)(v - (double)(float)hi);
}

// the sieve radius in units of 2^-16 (the threshold is twice it), 0x7fff
// with threshold 0xffff (every pair passes) where 2r would reach 1
GS_HD __forceinline__ void gs_sieve_units(double r, int& r16, int& thr) {
    if (r < 0.49) {
        r16 = (int)(r * 65536.0) + 2;
        thr = 2 * r16;
    } else {
        r16 = 0;
        thr = 0xffff;
    }
}

// the bounds of gs_ball_tile for tolerance tol and an error err per row, one
// unit of S outward each: lo = 2^32 (tol - sqrt(3) err)^2 (0: nothing is
// certain), lo + width = 2^32 (tol + sqrt(3) err)^2
GS_HD __forceinline__ void gs_ball_units(double tol, double err, unsigned& lo, unsigned& width) {
    const double e = 1.7320508075688774 * err + 1e-9;
    const double a = fmax(tol - e, 0.0) * 65536.0, b = (tol + e) * 65536.0;
    lo = (unsigned)fmax(a * a - 1.0, 0.0);
    width = (unsigned)(b * b + 2.0) - lo;
}

// A peak's 16 k slots, the half this lane holds (k = 8 half + j); p may be
// NULL (slots 9..15 zero)
__device__ __forceinline__ gs_half8 gs_peak_frag(double g0, double g1, double g2, const double* p,
                                                 int half) {
    _Float16 h[3], l[3];
    gs_split16(g0 * 1024.0, h[0], l[0]);
    gs_split16(g1 * 1024.0, h[1], l[1]);
    gs_split16(g2 * 1024.0, h[2], l[2]);
    gs_half8 f;
    f[0] = half ? h[2] : h[0];
    f[1] = half ? (p ? (_Float16)(float)p[0] : (_Float16)0) : h[1];
    f[2] = half ? (p ? (_Float16)(float)p[1] : (_Float16)0) : h[2];
    f[3] = half ? (p ? (_Float16)(float)p[2] : (_Float16)0) : l[0];
    f[4] = half ? (p ? (_Float16)(float)p[3] : (_Float16)0) : l[1];
    f[5] = half ? (p ? (_Float16)(float)p[4] : (_Float16)0) : l[2];
    f[6] = half ? (p ? (_Float16)(float)p[5] : (_Float16)0) : h[0];
    f[7] = half ? (p ? (_Float16)(float)p[6] : (_Float16)0) : h[1];
    return f;
}

// Both halves of a grain row's 16 k slots
__device__ __forceinline__ void gs_grain_frag(double u0, double u1, double u2, const double* q,
                                              gs_half8& a, gs_half8& b) {
    _Float16 h[3], l[3];
    gs_split16(u0 * 64.0, h[0], l[0]);
    gs_split16(u1 * 64.0, h[1], l[1]);
    gs_split16(u2 * 64.0, h[2], l[2]);
    a = (gs_half8){h[0], h[1], h[2], h[0], h[1], h[2], l[0], l[1]};
    b[0] = l[2];
#pragma unroll
    for (int i = 0; i < 7; i++) b[1 + i] = q ? (_Float16)(float)q[i] : (_Float16)0;
}

// LDS stores of this wave's lanes before, loads after
__device__ __forceinline__ void gs_wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

__device__ __forceinline__ bool gs_finite(double a) { return fabs(a) < __builtin_inf(); }

// the 16-bit fraction fields of the three rows of one pair: the largest
template <bool WIDE>
__device__ __forceinline__ unsigned short gs_sieve_field(float a, float b, float c) {
    unsigned short x = (unsigned short)__builtin_bit_cast(unsigned, a);
    unsigned short y = (unsigned short)__builtin_bit_cast(unsigned, b);
    unsigned short z = (unsigned short)__builtin_bit_cast(unsigned, c);
    if (WIDE) {
        x = (unsigned short)(x << 4);
        y = (unsigned short)(y << 4);
        z = (unsigned short)(z << 4);
    }
    unsigned short m = __builtin_elementwise_max(x, y);
    // two v_max_u16 (2.4 cycles each), not one v_max3_u16 (8.4 cycles)
    asm("" : "+v"(m));
    return __builtin_elementwise_max(m, z);
}

// One 32-peak x 32-grain tile.  Accumulator register i of a lane holds peak
// 8 (i / 4) + 4 (lane >> 5) + i % 4 and grain lane & 31, so registers 4 j ..
// 4 j + 3 are four consecutive peaks against one grain: the smallest of their
// four fields is compared (one compare and one branch for four pairs), and
// where it passes the quad is appended to the wave's queue, entry lp + 2 j.
// The queue's fill qn is wave-uniform; at most 256 entries are added, in
// order of j, then lane.
template <bool WIDE, class Entry>
__device__ __forceinline__ void gs_sieve_tile(gs_half8 pk, gs_half8 b0, gs_half8 b1, gs_half8 b2,
                                              gs_float16 c, unsigned short thr, unsigned lp,
                                              Entry* q, int& qn) {
    const gs_float16 h0 = __builtin_amdgcn_mfma_f32_32x32x16_f16(pk, b0, c, 0, 0, 0);
    const gs_float16 h1 = __builtin_amdgcn_mfma_f32_32x32x16_f16(pk, b1, c, 0, 0, 0);
    const gs_float16 h2 = __builtin_amdgcn_mfma_f32_32x32x16_f16(pk, b2, c, 0, 0, 0);
#pragma unroll
    for (int j = 0; j < 4; j++) {
        unsigned short f = gs_sieve_field<WIDE>(h0[4 * j], h1[4 * j], h2[4 * j]);
#pragma unroll
        for (int i = 4 * j + 1; i < 4 * j + 4; i++) {
            f = __builtin_elementwise_min(f, gs_sieve_field<WIDE>(h0[i], h1[i], h2[i]));
            asm("" : "+v"(f));  // as in gs_sieve_field: no v_min3_u16
        }
        const bool in = f <= thr;
        const unsigned long long m = __builtin_amdgcn_ballot_w64(in);
        if (m) {
            if (in) {
                const unsigned pos = __builtin_amdgcn_mbcnt_hi(
                    (unsigned)(m >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)m, 0u));
                (q + qn)[pos] = (Entry)(lp + 2 * j);
            }
            qn += __popcll(m);
        }
    }
}

// The same tile by the ball: with the accumulator started at 1.5 2^23 itself
// its low 16 bits, signed, are 2^16 (h - round(h)), and S, the sum of their
// three squares (at most 3 2^30, so it wraps nowhere as an unsigned number),
// is 2^32 drlv2 with each root off by GS_SIEVE_ERR at most.  By the triangle
// inequality S < lo counts for certain and S >= lo + width does not (lo,
// width of gs_ball_units); only a quad with a pair between them is queued.
// Returns how many pairs of the lane's grain count in the quads not queued.
// 11 vector instructions of 32 bits or less per pair (a byte permute, two
// 16-bit dot products, a mask, and the subtraction, carry and minimum of the
// two tests) against 14 of FP64 in k_score_many_fast.  Bound by their issue:
// 1000 grains x 10^6 peaks at tol 0.25 290 us against 611, 257 x 300007 40
// against 59.
template <bool WIDE, class Entry>
__device__ __forceinline__ int gs_ball_tile(gs_half8 pk, gs_half8 b0, gs_half8 b1, gs_half8 b2,
                                            gs_float16 c, unsigned lo, unsigned width, unsigned lp,
                                            Entry* q, int& qn) {
    const gs_float16 h0 = __builtin_amdgcn_mfma_f32_32x32x16_f16(pk, b0, c, 0, 0, 0);
    const gs_float16 h1 = __builtin_amdgcn_mfma_f32_32x32x16_f16(pk, b1, c, 0, 0, 0);
    const gs_float16 h2 = __builtin_amdgcn_mfma_f32_32x32x16_f16(pk, b2, c, 0, 0, 0);
    int n = 0;
#pragma unroll
    for (int j = 0; j < 4; j++) {
        unsigned w = 0xffffffffu;
        int n4 = 0;
#pragma unroll
        for (int i = 4 * j; i < 4 * j + 4; i++) {
            unsigned x = __builtin_bit_cast(unsigned, (float)h0[i]);
            unsigned y = __builtin_bit_cast(unsigned, (float)h1[i]);
            unsigned z = __builtin_bit_cast(unsigned, (float)h2[i]);
            if (WIDE) {
                x <<= 4;
                y <<= 4;
                z <<= 4;
            }
            const gs_short2 xy = __builtin_bit_cast(gs_short2, __builtin_amdgcn_perm(y, x, 0x05040100u));
            const gs_short2 z0 = __builtin_bit_cast(gs_short2, z & 0xffffu);
            const unsigned S = (unsigned)__builtin_amdgcn_sdot2(
                xy, xy, __builtin_amdgcn_sdot2(z0, z0, 0, false), false);
            n4 += S < lo;
            w = min(w, S - lo);
        }
        const bool in = w < width;
        const unsigned long long m = __builtin_amdgcn_ballot_w64(in);
        if (m) {
            if (in) {
                const unsigned pos = __builtin_amdgcn_mbcnt_hi(
                    (unsigned)(m >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)m, 0u));
                (q + qn)[pos] = (Entry)(lp + 2 * j);
                n4 = 0;
            }
            qn += __popcll(m);
        }
        n += n4;
    }
    return n;
}

// ---------------------------------------------------------------------------
// Tiles outside the f16 ranges, in f32 on the vector ALU: a lane holds one
// grain of the tile (lane & 31) and goes through the wave's peaks, the lower
// half of the wave through the even quads and the upper half through the odd
// ones, with the queue and the entries of gs_sieve_tile.
// Certification, v = 2^-24 (half a unit in the last place), A = max over rows
// of |u|_1, times max |g|: u and g are rounded once (2 v A), the three FMAs
// round a partial sum of at most A + 1 each: h is within 5.1 v A + 3.1 v,
// below gs_err32 = 2^-21 A + 10^-6, which also covers v_fract_f32 and the
// rounding of r.  Used while A <= 2^16 (gs_err32 < 0.032) and the factors
// are far from the ends of f32; beyond that every pair of the grain passes.
// A grain that is not finite passes nothing; a peak that is not finite is NaN
// here, which fails every comparison.
// 14 f32 instructions per pair (ball 21), three 16-byte LDS reads per quad.
// 1000 grains x 10^6 peaks with cells of 300 to 1200 A: 392 us at tol 0.05,
// 525 at 0.25; k_score_many_sieve and k_score_many_fast take 449 and 713, and
// with the reference arithmetic for every pair of the tile it was 1287 and 1413.
struct gs_grain32 {
    float u[9];  // zero where the range above does not hold
    float a;     // A, infinite there
    bool live;   // all nine finite
};

__device__ __forceinline__ gs_grain32 gs_load_grain32(const double* __restrict__ u, bool on,
                                                      float gmax) {
    gs_grain32 w;
    double s[3], big = 0.0;
#pragma unroll
    for (int i = 0; i < 3; i++) {
        s[i] = fabs(u[3 * i]) + fabs(u[3 * i + 1]) + fabs(u[3 * i + 2]);
        big += s[i];
    }
    w.live = on && gs_finite(u[0]) && gs_finite(u[1]) && gs_finite(u[2]) && gs_finite(u[3]) &&
             gs_finite(u[4]) && gs_finite(u[5]) && gs_finite(u[6]) && gs_finite(u[7]) &&
             gs_finite(u[8]);
    const double top = fmax(s[0], fmax(s[1], s[2])) * (double)gmax * (1.0 + 0x1p-20);
    const bool fits = w.live && big < 0x1p100 && gmax < 0x1p100f && top <= 65536.0;
    w.a = fits ? (float)top : __builtin_inff();
#pragma unroll
    for (int i = 0; i < 9; i++) w.u[i] = fits ? (float)u[i] : 0.0f;
    return w;
}

// a component of a peak: within the range above or at its end, so that it
// gives no NaN against a grain of zeros
__device__ __forceinline__ float gs_clamp32(double v) {
    return fminf(fmaxf((float)v, -0x1p100f), 0x1p100f);
}

#define GS_ALL32 2.0f  // hi of a grain whose every pair passes

__device__ __forceinline__ float gs_err32(float a) { return 0x1p-21f * a + 1e-6f; }

// the largest of the fractions of h_i + r
__device__ __forceinline__ float gs_cube32(const float* u, float x, float y, float z, float r) {
    const float h0 = __builtin_fmaf(u[2], z, __builtin_fmaf(u[1], y, __builtin_fmaf(u[0], x, r)));
    const float h1 = __builtin_fmaf(u[5], z, __builtin_fmaf(u[4], y, __builtin_fmaf(u[3], x, r)));
    const float h2 = __builtin_fmaf(u[8], z, __builtin_fmaf(u[7], y, __builtin_fmaf(u[6], x, r)));
    return fmaxf(fmaxf(__builtin_amdgcn_fractf(h0), __builtin_amdgcn_fractf(h1)),
                 __builtin_amdgcn_fractf(h2));
}

// drlv2 - 3/4, as gs_drlv2_fract
__device__ __forceinline__ float gs_drlv2_32(const float* u, float x, float y, float z) {
    const float h0 = __builtin_fmaf(u[2], z, __builtin_fmaf(u[1], y, __builtin_fmaf(u[0], x, 0.5f)));
    const float h1 = __builtin_fmaf(u[5], z, __builtin_fmaf(u[4], y, __builtin_fmaf(u[3], x, 0.5f)));
    const float h2 = __builtin_fmaf(u[8], z, __builtin_fmaf(u[7], y, __builtin_fmaf(u[6], x, 0.5f)));
    const float f0 = __builtin_amdgcn_fractf(h0), f1 = __builtin_amdgcn_fractf(h1),
                f2 = __builtin_amdgcn_fractf(h2);
    float t = __builtin_fmaf(f0, f0, -f0);
    t = __builtin_fmaf(f1, f1, t) - f1;
    return __builtin_fmaf(f2, f2, t) - f2;
}

// the entries of the lanes with `in` to the end of the wave's queue
template <class Entry>
__device__ __forceinline__ void gs_push(bool in, Entry e, Entry* q, int& qn) {
    const unsigned long long m = __builtin_amdgcn_ballot_w64(in);
    if (m) {
        if (in) {
            const unsigned pos = __builtin_amdgcn_mbcnt_hi(
                (unsigned)(m >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)m, 0u));
            (q + qn)[pos] = e;
        }
        qn += __popcll(m);
    }
}

// 32 peaks (x, y, z: theirs, 16-byte aligned) against the tile.  Sieve: a quad
// is queued unless the fraction of every pair exceeds hi = 2 r (r in lo).
// Ball: queued if the drlv2 - 3/4 of a pair lies in [lo, hi); returns how many
// pairs lie below lo in the quads that are not.
template <bool BALL, class Entry>
__device__ __forceinline__ int gs_tile32(const float* x, const float* y, const float* z,
                                         const gs_grain32& w, float lo, float hi, int half,
                                         unsigned lp, Entry* q, int& qn) {
    int n = 0;
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const int pk = 8 * j + 4 * half;
        bool in;
        int n4 = 0;
        if constexpr (BALL) {
            // s - lo as a bit pattern: negative ones and NaN lie beyond hi - lo
            unsigned d = 0xffffffffu;
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const float s = gs_drlv2_32(w.u, x[pk + i], y[pk + i], z[pk + i]);
                n4 += s < lo;
                d = min(d, __builtin_bit_cast(unsigned, s - lo));
            }
            in = d < __builtin_bit_cast(unsigned, hi - lo);
        } else {
            float f = gs_cube32(w.u, x[pk], y[pk], z[pk], lo);
#pragma unroll
            for (int i = 1; i < 4; i++)
                f = fminf(f, gs_cube32(w.u, x[pk + i], y[pk + i], z[pk + i], lo));
            in = f <= hi;
        }
        if (in) n4 = 0;
        gs_push(in, (Entry)(lp + 2 * j), q, qn);
        n += n4;
    }
    return n;
}

// lo and hi of gs_tile32 for the lane's grain at tolerance tol and error e of
// a row: everything passes beyond the range (e infinite), nothing where the
// grain is not finite
template <bool BALL>
__device__ __forceinline__ void gs_units32(const gs_grain32& w, double tol, float e, float& lo,
                                           float& hi) {
    if constexpr (BALL) {
        // the roots are off by sqrt(3) e, the sum's own rounding is below 10^-6
        const float d = 1.7320509f * e, t = (float)tol, a = fmaxf(t - d, 0.0f);
        lo = fminf(a * a, 4.0f) - 0.750002f;
        hi = fminf((t + d) * (t + d), 4.0f) - 0.749998f;
        if (!w.live) lo = hi = -2.0f;  // below every drlv2 - 3/4
    } else {
        const float r = (float)tol + e;
        lo = r < 0.49f ? r : 0.0f;
        hi = r < 0.49f ? 2.0f * r + 1e-6f : GS_ALL32;
        if (!w.live) hi = -1.0f;
    }
}

__device__ __forceinline__ gs_float16 gs_splat16(float v) {
    return (gs_float16){v, v, v, v, v, v, v, v, v, v, v, v, v, v, v, v};
}

// ---------------------------------------------------------------------------
// Counters.  Atomics on one address from all over the chip go one after the
// other, so the pairs are counted in private copies of the K counters, copy
// blockIdx % copies for a block, which a last launch sums: a multiple of 8, so
// that each copy is the business of one XCD: 64 up to 512 grains, then 32768
// counters in all, and from 2049 grains on 8.  The assignment of 500 grains
// over 200 003 peaks took 112 us with one copy and 36 with 64, the score of
// 24 x 10^6 31 us and 21, of 100 x 10^6 49 and 38; of 500 x 3 10^5 both took 43,
// and from there the score counts in place (147 us against 152 at 1000 x 10^6,
// the sum's launch).
#define GS_SCORE_COPIES_MAX 256
inline int gs_copies(int K) {
    const int c = 4096 / (K > 0 ? K : 1);
    return 8 * (c < 1 ? 1 : c > 8 ? 8 : c);
}

__global__ __launch_bounds__(GS_BLOCK) void k_sum_copies(const int* __restrict__ priv, int copies,
                                                         int K, int* __restrict__ counts) {
    const int g = blockIdx.x * GS_BLOCK + threadIdx.x;
    if (g >= K) return;
    int s = 0;
#pragma unroll 8
    for (int c = 0; c < copies; c++) s += priv[(size_t)c * K + g];  // a multiple of 8
    counts[g] = s;
}

// ---------------------------------------------------------------------------
// The grains' fragments, packed once per call into the caller's workspace:
// tile t (grains 32 t .. 32 t + 31; "dead" past K and where any of the nine u
// is not finite, as a peak is past the list and where g is not finite: zeros,
// and 1/2 of h in all three rows from the p, q slots, which passes no sieve
// and, as S = 3/4, no ball up to GS_BALL_TOL_MAX) has
// 3 x 64 x 16 bytes, row-major by UBI row, lane l holding column l & 31 and k
// slots 8 (l >> 5) .. + 7, then one float per tile, the largest row sum of
// |u|.  Also clears the counters (so that no separate fill is launched).
inline long long gs_sieve_tiles(long long K) { return (K + 31) / 32; }
inline long long gs_sieve_ws_bytes(long long K) { return gs_sieve_tiles(K) * (3 * 64 * 16 + 16) + 16; }

__global__ __launch_bounds__(128) void k_sieve_pack(const double* __restrict__ ubis, int K,
                                                    gs_half8* __restrict__ frag,
                                                    float* __restrict__ span,
                                                    int* __restrict__ counts, int copies) {
    __shared__ float lspan[128];  // largest row sums
    __shared__ unsigned long long lfin[2];  // bit per lane: the thread's row is finite
    const int tl = blockIdx.x, t = threadIdx.x;
    const int row = t / 32, col = t & 31;
    double u0 = 0.0, u1 = 0.0, u2 = 0.0;
    float sp = 0.0f;
    if (t < 96) {  // one grain row each
        const double* u = ubis + 9 * (size_t)min(32 * tl + col, K - 1) + 3 * row;
        u0 = u[0];
        u1 = u[1];
        u2 = u[2];
    }
    if (32 * tl + (t & 31) < K)
        for (int c = t / 32; c < copies; c += 4) counts[(size_t)c * K + 32 * tl + (t & 31)] = 0;
    const unsigned long long fin = __ballot(gs_finite(u0) && gs_finite(u1) && gs_finite(u2));
    if ((t & (GS_WAVE - 1)) == 0) lfin[t / GS_WAVE] = fin;
    __syncthreads();
    if (t < 96) {
        // all three rows: a pair with one row at 1/2 and the others free has
        // S >= 1/4 only, which the ball counts as certain from tol 1/2 on
        const bool live = 32 * tl + col < K &&
                          (lfin[0] >> col & lfin[0] >> (32 + col) & lfin[1] >> col & 1);
        float a = (float)(fabs(u0) + fabs(u1) + fabs(u2));
        if (!live) {
            u0 = u1 = u2 = 0.0;
            a = 0.0f;
        }
        const double q[7] = {live ? 1.0 : 0.0, live ? 0.0 : 32768.0, 0.0, 0.0, 0.0, 0.0, 0.0};
        sp = a * (1.0f + 0x1p-20f);
        gs_half8* f = frag + (3 * (size_t)tl + row) * GS_WAVE;
        gs_half8 lo, hi;
        gs_grain_frag(u0, u1, u2, q, lo, hi);
        f[col] = lo;
        f[col + 32] = hi;
    }
    lspan[t] = sp;
    __syncthreads();
    if (t == 0) {
        float a = lspan[0];
        for (int i = 1; i < 96; i++) a = fmaxf(a, lspan[i]);
        span[tl] = a;
    }
}

// ---------------------------------------------------------------------------
// score (and list extraction) for K UBIs x ng g-vectors.  A wave owns NB sets
// of 32 peaks, their fragments in LDS, and goes through the block's split of
// grain tiles, whose fragments it reads from the workspace one tile ahead.
// Quads of pairs that may pass go to a per-wave LDS queue (entry: grain of
// the split << 5 | quad of the wave's peaks), and whenever it holds 64 they
// are settled, one quad per lane, by gs_drlv2.
// SELECT: cursor = counts; a pair that counts takes a slot of its grain and,
// when idx is given, writes its peak number there (see k_select_many).
// BALL: gs_ball_tile in the place of the sieve.
template <bool SELECT, bool BALL>
__global__ __launch_bounds__(GS_BLOCK, 4) void k_score_mfma(
    const double* __restrict__ ubis, int K, int tsplit, int nsplit, const double* __restrict__ gv,
    int ng, double tolsq, const gs_half8* __restrict__ frag, const float* __restrict__ span,
    int* __restrict__ priv, int copies, const long long* __restrict__ off, int* __restrict__ idx) {
    int* counts = priv + (size_t)(blockIdx.x % copies) * K;
    constexpr int NW = GS_BLOCK / GS_WAVE;
    constexpr int NB = GS_SIEVE_SETS;
    static_assert(8 * NB <= 32, "a queue entry holds 5 bits of quad");
    static_assert(32 * GS_SIEVE_SPLIT <= 2048, "and 11 bits of grain");
    static_assert(GS_SIEVE_SPLIT <= 64, "a mask holds the tiles left to f32");
    __shared__ __align__(16) gs_half8 lpk[NW][NB][GS_WAVE];
    __shared__ __align__(16) float lf[NW][3][32 * NB];  // the peaks for gs_tile32
    __shared__ int lcnt[32 * GS_SIEVE_SPLIT];
    __shared__ unsigned short lq[NW][GS_WAVE + 256];
    const int tile = gs_xcd_remap(blockIdx.x, gridDim.x);
    const int chunk = tile / nsplit;
    const int split = tile - chunk * nsplit;
    const int t0 = split * tsplit;
    const int t1 = min((K + 31) / 32, t0 + tsplit);
    const int g0 = 32 * t0;
    const int lane = threadIdx.x & (GS_WAVE - 1);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / GS_WAVE);
    const int half = lane >> 5;
    for (int i = threadIdx.x; i < 32 * (t1 - t0); i += GS_BLOCK) lcnt[i] = 0;
    // this wave's peaks: k0 .. k0 + 32 NB - 1
    const long long k0 = (long long)chunk * (NW * NB * 32) + wave * (NB * 32);
    float gmax = 0.0f;
    for (int s = 0; s < NB; s++) {
        long long k = k0 + 32 * s + (lane & 31);
        bool live = k < ng;
        k = live ? k : (long long)ng - 1;
        double x = gv[3 * k], y = gv[3 * k + 1], z = gv[3 * k + 2];
        live = live && gs_finite(x) && gs_finite(y) && gs_finite(z);
        if (!live) x = y = z = 0.0;
        const double p[7] = {live ? 0.0 : 32768.0, 1.0, 0.0, 0.0, 0.0, 0.0, 0.0};
        gmax = fmaxf(gmax, (float)fmax(fabs(x), fmax(fabs(y), fabs(z))));
        lpk[wave][s][lane] = gs_peak_frag(x, y, z, p, half);
    }
    for (int o = 1; o < 32; o <<= 1) gmax = fmaxf(gmax, __shfl_xor(gmax, o, GS_WAVE));
    gmax = __builtin_bit_cast(
        float, __builtin_amdgcn_readfirstlane(__builtin_bit_cast(int, gmax * (1.0f + 0x1p-20f))));
    const double tol = sqrt(tolsq) * (1.0 + 1e-15) + 1e-12;
    int r16, thr, r16w, thrw;
    gs_sieve_units(tol + GS_SIEVE_ERR, r16, thr);
    gs_sieve_units(tol + GS_SIEVE_ERR_WIDE, r16w, thrw);
    unsigned lo = 0, width = 0, low = 0, widthw = 0;
    if (BALL) {
        r16 = r16w = 0;
        gs_ball_units(tol, GS_SIEVE_ERR, lo, width);
        gs_ball_units(tol, GS_SIEVE_ERR_WIDE, low, widthw);
    }
    unsigned short* q = lq[wave];
    int qn = 0;
    unsigned long long left = 0;  // the split's tiles that the loop over them leaves out
    const auto hit = [&](int gl, long long k) {
        if constexpr (SELECT) {
            const int g = g0 + gl;
            const int slot = atomicAdd(&counts[g], 1);
            if (idx && slot < off[g + 1] - off[g]) idx[off[g] + slot] = (int)k;
        } else {
            atomicAdd(&lcnt[gl], 1);
        }
    };
    const auto settle = [&](unsigned e) {
        const int gl = e >> 5;
        if (g0 + gl >= K) return;
        const gs_ubi u = gs_load_ubi(ubis + 9 * (size_t)(g0 + gl));
        const long long k = k0 + 4 * (e & 31);
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const long long ki = min(k + i, (long long)ng - 1);
            if (gs_drlv2(u, gv[3 * ki], gv[3 * ki + 1], gv[3 * ki + 2]) < tolsq && k + i < ng)
                hit(gl, k + i);
        }
    };
    const auto drain = [&] {
        while (qn >= GS_WAVE) {
            qn -= GS_WAVE;
            __builtin_amdgcn_wave_barrier();
            settle(q[qn + lane]);
            __builtin_amdgcn_wave_barrier();
        }
    };
    __syncthreads();
    const gs_half8* f = frag + 3 * (size_t)t0 * GS_WAVE + lane;
    gs_half8 n0 = f[0], n1 = f[GS_WAVE], n2 = f[2 * GS_WAVE];
    const gs_float16 c = gs_splat16(12582912.0f + r16);  // 1.5 2^23
    for (int t = t0; t < t1; t++) {
        const gs_half8 b0 = n0, b1 = n1, b2 = n2;
        const float sp = span[t] * gmax;
        const bool fits = span[t] < GS_SIEVE_UMAX && gmax < GS_SIEVE_GMAX;
        if (t + 1 < t1) {  // the next tile's fragments, in flight during this one
            f += 3 * GS_WAVE;
            n0 = f[0];
            n1 = f[GS_WAVE];
            n2 = f[2 * GS_WAVE];
        }
        // entry of quad j, set s: lane part + 8 s + 2 j
        const unsigned lp = ((32 * (t - t0) + (lane & 31)) << 5) | half;
        int n = 0;  // BALL: the certain pairs of the lane's grain
        if (fits && sp <= GS_SIEVE_SPAN) {
#pragma unroll 1
            for (int s = 0; s < NB; s++) {
                if constexpr (BALL)
                    n += gs_ball_tile<false>(lpk[wave][s][lane], b0, b1, b2, c, lo, width,
                                             lp + 8 * s, q, qn);
                else
                    gs_sieve_tile<false>(lpk[wave][s][lane], b0, b1, b2, c, thr, lp + 8 * s, q, qn);
                drain();
            }
        } else if (fits && sp <= GS_SIEVE_SPAN_WIDE) {
            const gs_float16 cw = gs_splat16(201326592.0f + r16w);  // 1.5 2^27
#pragma unroll 1
            for (int s = 0; s < NB; s++) {
                if constexpr (BALL)
                    n += gs_ball_tile<true>(lpk[wave][s][lane], b0, b1, b2, cw, low, widthw,
                                            lp + 8 * s, q, qn);
                else
                    gs_sieve_tile<true>(lpk[wave][s][lane], b0, b1, b2, cw, thrw, lp + 8 * s, q,
                                        qn);
                drain();
            }
        } else {
            left |= 1ull << (t - t0);
        }
        if (BALL && n) atomicAdd(&lcnt[32 * (t - t0) + (lane & 31)], n);
    }
    if (left) {  // the tiles outside the f16 ranges, here so that the loop above has the registers
        for (int p = lane; p < 32 * NB; p += GS_WAVE) {
            const long long k = min(k0 + p, (long long)ng - 1);
            const double x = gv[3 * k], y = gv[3 * k + 1], z = gv[3 * k + 2];
            const bool live = k0 + p < ng && gs_finite(x) && gs_finite(y) && gs_finite(z);
            lf[wave][0][p] = live ? gs_clamp32(x) : __builtin_nanf("");
            lf[wave][1][p] = gs_clamp32(y);
            lf[wave][2][p] = gs_clamp32(z);
        }
        gs_wave_sync();
        for (; left; left &= left - 1) {
            const int tl = __builtin_ctzll(left);
            const int g = g0 + 32 * tl + (lane & 31);
            const gs_grain32 w =
                gs_load_grain32(ubis + 9 * (size_t)min(g, K - 1), g < K, gmax);
            float l32, h32;
            gs_units32<BALL>(w, tol, gs_err32(w.a), l32, h32);
            const unsigned lp = ((32 * tl + (lane & 31)) << 5) | half;
            int n = 0;
#pragma unroll 1
            for (int s = 0; s < NB; s++) {
                n += gs_tile32<BALL>(lf[wave][0] + 32 * s, lf[wave][1] + 32 * s,
                                     lf[wave][2] + 32 * s, w, l32, h32, half, lp + 8 * s, q, qn);
                drain();
            }
            if (BALL && n) atomicAdd(&lcnt[32 * tl + (lane & 31)], n);
        }
    }
    __builtin_amdgcn_wave_barrier();
    if (lane < qn) settle(q[lane]);
    if constexpr (!SELECT) {
        __syncthreads();
        for (int i = threadIdx.x; i < 32 * (t1 - t0); i += GS_BLOCK) {
            const int c = lcnt[i];
            if (c && g0 + i < K) atomicAdd(&counts[g0 + i], c);
        }
    }
}
