// score_and_assign for all grains in order, behind the matrix-core sieve
// (gs_sieve.h): grain g gets label g, as refinegrains.assignlabels,
// indexer.fight_over_peaks and nb_utils.assign_peaks_to_grains call it.
//
// GEOM: every grain sees the peaks from its own position t (compute_gv per
// grain, k_gv_assign_many's loop).  With a, c the peak's constants there,
// G = ds (a - t)/|a - t| - c, and to second order in t/|a|
//     u.G = u.G0 - (ds/|a|)(u.t) + (ds/|a|) sum_jl u_j n_j n_l t_l,
// G0 = ds n - c, n = a/|a|: a dot product of peak terms and grain terms, which
// the k slots 9..14 of the sieve hold next to G0's split product.  As
// n.n = 1 the u.t term is folded into the diagonal:
//     p = (ds/|a|) (nx nx, ny ny, nz nz, nx ny, nx nz, ny nz)
//     q = (ux tx - u.t, uy ty - u.t, uz tz - u.t, ux ty + uy tx,
//          ux tz + uz tx, uy tz + uz ty)
// in single f16 numbers, p 2^(16 - y) and q 2^y, 2^y between 32 and 64 ds/|a| of
// a middling peak: p is then below 8192 in the waves whose peaks lie no nearer
// than a quarter of that, and q below 32768 for every grain that the radius lets
// through where they lie no farther than 2.5 times.  (From the largest |t| one
// grain far off made p too large for all: 777 x 10^5 121 us, 200 with one such
// grain in f32 and 441 in FP64; 121 this way.)
// Added to the sieve's error (L = max over rows of sum |q|, T = max |t|, A1 =
// max over rows of |u|_1, in the tile; amin = min |a| over the wave's peaks):
//   rounding of p and q: 1.01 2^-10 (ds/amin) L;
//   the remainder of the expansion: for x(s) = a - s t, |d2/ds2 x/|x|| =
//   |t_perp| sqrt(4 t_par^2 + t_perp^2)/|x|^2 <= 1.1548 |t|^2/|x|^2, so it is
//   below 0.5775 A1 ds T^2/(amin - T)^2.
// Terms that f16 may flush (p, q below 2^-14) move h by 2^-30 (sum |q| + sum p) <
// 2^-30 (32768 + 2 8192) = 4.6e-5, within the sieve's margin.  The expansion is
// used while p and sum |q| keep these limits, T <= amin/2 and the radius stays below GS_ASSIGN_RMAX; otherwise (grains far from the centre of a
// near detector) the tile is tested in f32 on the vector ALU, as in gs_tile32,
// with G itself from a, t and c.  Its error there, v = 2^-24, while |t| <= |a|/2
// (so |a| + |t| <= 3 |a - t|): a - t is within 4 v |a - t|, the square of its
// length 3 v and v_rsq_f32 2 v of the value, the scaling by ds 2 v more, so
// that with the rounding of c and the FMA a component of G is within 12.5 v ds;
// u, of row sum at most A1, and the three FMAs add 8 v A1 ds + 3 v: below
// 2^-19 A1 ds + 10^-6, used while A1 ds <= 2^16 and lengths and ds are far
// from the ends of f32; otherwise every pair of the grain passes.  Measured,
// 2000 grains x 10^6 peaks 8 mm from the detector, positions to 500 um: 1761 us
// against 2973 of k_gv_assign_many and 3498 with its FP64 loop for such tiles
// here; g-vectors given, cells of 300 to 1200 A: 813 against 2149 and 2259.
//
// Order.  The update rule is sequential in the grains of one peak: a pair is
// accepted if its drlv2 is below tol^2 and the peak's current drlv2, so the
// current drlv2 only falls and a pair the sieve drops changes nothing but a
// label equal to the grain's, which becomes -1.  With label g for grain g the
// latter can only be the label the peak came in with: at the end a peak that
// accepted no grain has -1 if its first label is a grain's.  A wave owns its
// peaks and queues the surviving quads in grain order (lanes of a push, then
// pushes); they are filtered (GEOM: the certified fast drlv2 against min(tol^2,
// current), 37 instructions; else the reference's own drlv2) into a second
// queue, 64 of which are decided at once with the reference arithmetic; pairs
// of one peak in one batch go through in lane order, which is grain order.
//
// Measured, labels, drlv2 and counts identical: 20 000 grains x 8 10^6 peaks
// with positions 23.9 ms against 191 of k_gv_assign_many (FP64 VALU, 92%
// busy), 777 x 10^5 45 us against 310; g-vectors given, 500 x 200 003 36 us
// against 230.  Per 32 x 32 tile: 51 vector instructions for the sieve, 20 for
// pushes, settling and the tile's constants (the accumulator start is rebuilt
// for each tile: kept across tiles in registers it made the compiler copy and
// spill it, 37.7 ms), 356 cycles in all.  Bound, as the score, by vector issue:
// the vector ALU is busy 80% of the cycles and the matrix cores 27%, at 2.9
// waves per SIMD and 2.2 GHz.
#pragma once
#include "gs_assign_gv.h"
#include "gs_sieve.h"

#define GS_ASSIGN_RMAX 0.2f
#define GS_ASSIGN_PMAX 8192.0f
#define GS_ASSIGN_QMAX 32768.0f

struct gs_tile_info {
    float span;  // largest row sum of |u|
    float lin;   // largest row sum of |q| (unscaled)
    float tmax;  // largest |t|
    float pad;
};

__device__ __forceinline__ float gs_uniform(float v) {
    return __builtin_bit_cast(float, __builtin_amdgcn_readfirstlane(__builtin_bit_cast(int, v)));
}

// Fragments and tile_info of every tile, the exponent y, the counters cleared.
// xl (GEOM): the ng peaks, ds = 1/wavelength; y is every block's own, from the
// median |xl| of the same 64 of them.
template <bool GEOM>
__global__ __launch_bounds__(128) void k_assign_pack(const double* __restrict__ ubis,
                                                     const double* __restrict__ trans, int K,
                                                     const double* __restrict__ xl, int ng,
                                                     double ds,
                                                     gs_half8* __restrict__ frag,
                                                     gs_tile_info* __restrict__ info,
                                                     int* __restrict__ yexp,
                                                     int* __restrict__ priv, int copies) {
    __shared__ __align__(16) float lspan[128], llin[128], lt[128];
    const int tl = blockIdx.x, t = threadIdx.x;
    const int row = t / 32, col = t & 31;
    const int g = min(32 * tl + col, K - 1);
    // everything that is read, on its way at once
    const double* u = ubis + 9 * (size_t)g + 3 * min(row, 2);
    double u0 = u[0], u1 = u[1], u2 = u[2], t0 = 0.0, t1 = 0.0, t2 = 0.0;
    float n2 = __builtin_inff();  // |xl|^2 of the thread's sample
    if constexpr (GEOM) {
        t0 = trans[3 * (size_t)g];
        t1 = trans[3 * (size_t)g + 1];
        t2 = trans[3 * (size_t)g + 2];
        const double* x = xl + 3 * ((long long)(t & 63) * ng / 64);
        const float s = (float)(x[0] * x[0] + x[1] * x[1] + x[2] * x[2]);
        n2 = s > 0.0f ? s : n2;  // NaN: not one either
    }
    if (32 * tl + (t & 31) < K)
        for (int c = t / 32; c < copies; c += 4) priv[(size_t)c * K + 32 * tl + (t & 31)] = 0;
    int y = 0;
    if constexpr (GEOM) {
        if (t < 64) lt[t] = n2;
        if (t == 0) lspan[0] = __builtin_inff();
        __syncthreads();
        if (t < 64) {
            int rank = 0, n = 0;
#pragma unroll
            for (int i = 0; i < 64; i++) {
                rank += lt[i] < n2 || (lt[i] == n2 && i < t);
                n += lt[i] < __builtin_inff();
            }
            if (rank == n / 2) lspan[0] = n2;
        }
        __syncthreads();
        const float r = 64.0f * fabsf((float)ds) / sqrtf(lspan[0]);
        int e = 0;
        if (r > 0.0f && r < __builtin_inff()) (void)frexpf(r, &e);
        y = max(-60, min(60, e - 1));
        if (tl == 0 && t == 0) *yexp = y;
        __syncthreads();
    }
    lspan[t] = llin[t] = lt[t] = 0.0f;
    if (t < 96) {  // one grain row each
        float a = (float)(fabs(u0) + fabs(u1) + fabs(u2));
        const float at = (float)(fabs(t0) + fabs(t1) + fabs(t2));
        if (!(a < __builtin_inff() && at < __builtin_inff())) {
            u0 = u1 = u2 = t0 = t1 = t2 = 0.0;  // never accepted, whatever passes
            a = 0.0f;
        }
        const double ut = u0 * t0 + u1 * t1 + u2 * t2;
        double q[7] = {u0 * t0 - ut, u1 * t1 - ut, u2 * t2 - ut, u0 * t1 + u1 * t0,
                       u0 * t2 + u2 * t0, u1 * t2 + u2 * t1, 0.0};
        double l = 0.0;
        for (int i = 0; i < 6; i++) l += fabs(q[i]);
        lspan[t] = a * (1.0f + 0x1p-20f);
        llin[t] = (float)l * (1.0f + 0x1p-20f);
        lt[t] = (float)sqrt(t0 * t0 + t1 * t1 + t2 * t2) * (1.0f + 0x1p-20f);
        if constexpr (GEOM)
            for (int i = 0; i < 6; i++) q[i] = ldexp(q[i], y);
        gs_half8* f = frag + (3 * (size_t)tl + row) * GS_WAVE;
        gs_half8 lo, hi;
        gs_grain_frag(u0, u1, u2, GEOM ? q : nullptr, lo, hi);
        f[col] = lo;
        f[col + 32] = hi;
    }
    __syncthreads();
    if (t < 32) {
        gs_tile_info w = {fmaxf(lspan[t], fmaxf(lspan[t + 32], lspan[t + 64])),
                          fmaxf(llin[t], fmaxf(llin[t + 32], llin[t + 64])),
                          fmaxf(lt[t], fmaxf(lt[t + 32], lt[t + 64])), 0.0f};
        for (int o = 16; o > 0; o >>= 1) {
            w.span = fmaxf(w.span, __shfl_xor(w.span, o, 32));
            w.lin = fmaxf(w.lin, __shfl_xor(w.lin, o, 32));
            w.tmax = fmaxf(w.tmax, __shfl_xor(w.tmax, o, 32));
        }
        if (t == 0) info[tl] = w;
    }
}

// NB 32 peaks per wave, all K grains.  FEW: at most 64 of them, counted in LDS:
// with many peaks of each their atomics went one after the other (16 grains x
// 4 10^6 peaks of theirs 577 us, 204 this way; as a branch at run time it cost
// 777 grains x 10^5 with positions a tenth).  gvx: the g-vectors, or with GEOM the
// lab positions (so, co, gp then given as for k_gv_assign_many).
template <bool GEOM, int NB, bool FEW>
__global__ __launch_bounds__(GS_BLOCK, 3) void k_assign_mfma(
    const double* __restrict__ gvx, const double* __restrict__ so_in,
    const double* __restrict__ co_in, int ng, gs_goniometer gp, const double* __restrict__ ubis,
    const double* __restrict__ trans, int K, double tolsq, const gs_half8* __restrict__ frag,
    const gs_tile_info* __restrict__ info, const int* __restrict__ yexp,
    double* __restrict__ drlv2, int* __restrict__ labels, int* __restrict__ priv, int copies) {
    int* counts = priv + (size_t)(blockIdx.x % copies) * K;  // this block's copy
    constexpr int NW = GS_BLOCK / GS_WAVE;
    constexpr int NP = 32 * NB;  // peaks per wave
    static_assert(NP <= 128, "a queue entry holds 5 bits of quad, 7 of peak");
    __shared__ __align__(16) gs_half8 lpk[NW][NB][GS_WAVE];
    __shared__ __align__(16) double la[NW][GEOM ? 3 : 1][GEOM ? NP : 2];  // a of each peak
    __shared__ __align__(16) float lf[NW][GEOM ? 2 : 3][NP];  // c_x, c_y (GEOM) or g, in f32
    __shared__ double ld[NW][NP];                           // current drlv2
    __shared__ int lg[NW][NP];                              // last accepted grain, or -1
    __shared__ unsigned lclaim[NW][NP];
    __shared__ int lcnt[FEW ? NW : 1][GS_WAVE];  // the wave's counts
    __shared__ unsigned lq1[NW][GS_WAVE + 256];  // grain << 5 | quad
    __shared__ unsigned lq2[NW][2 * GS_WAVE];    // grain << 7 | peak
    const int lane = threadIdx.x & (GS_WAVE - 1);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / GS_WAVE);
    const int half = lane >> 5;
    const long long k0 = ((long long)blockIdx.x * NW + wave) * NP;
    if (k0 >= ng) return;  // no barrier of the block below
    const double* mat = gp.mat;
    const double ds = 1. / gp.wvln;
    if (FEW) lcnt[wave][lane] = 0;
    unsigned* q1 = lq1[wave];
    unsigned* q2 = lq2[wave];

    float gmax = 0.0f;
    double n2min = __builtin_inf(), n2max = 0.0;
    for (int s = 0; s < NB; s++) {
        const int pk = 32 * s + (lane & 31);
        const long long k = min(k0 + pk, (long long)ng - 1);  // past ng: the last again
        double x = gvx[3 * k], y = gvx[3 * k + 1], z = gvx[3 * k + 2];
        double p[7] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
        if constexpr (GEOM) {
            double a[3], c[3];
            const double n2 = x * x + y * y + z * z;
            n2min = n2 == n2 ? fmin(n2min, n2) : n2min;
            n2max = n2 == n2 ? fmax(n2max, n2) : n2max;
            gs_scan_consts(x, y, z, so_in[k], co_in[k], mat, ds, a, c);
            if (half == 0) {
                lf[wave][0][pk] = (float)c[0];
                lf[wave][1][pk] = (float)c[1];
                la[wave][0][pk] = a[0];
                la[wave][1][pk] = a[1];
                la[wave][2][pk] = a[2];
            }
            const double r = 1.0 / sqrt(n2), w = ldexp(ds * r, 16 - *yexp);
            const double nx = a[0] * r, ny = a[1] * r, nz = a[2] * r;
            x = ds * nx - c[0];
            y = ds * ny - c[1];
            z = ds * nz - c[2];
            p[0] = w * nx * nx;
            p[1] = w * ny * ny;
            p[2] = w * nz * nz;
            p[3] = w * nx * ny;
            p[4] = w * nx * nz;
            p[5] = w * ny * nz;
        }
        if (!(gs_finite(x) && gs_finite(y) && gs_finite(z))) {
            x = 0.3137;  // never accepted (or the wave's n2min is 0: no tile is sieved)
            y = 0.2711;
            z = 0.1873;
            for (int i = 0; i < 6; i++) p[i] = 0.0;
        }
        gmax = fmaxf(gmax, (float)fmax(fabs(x), fmax(fabs(y), fabs(z))));
        lpk[wave][s][lane] = gs_peak_frag(x, y, z, GEOM ? p : nullptr, half);
        if (half == 0) {
            ld[wave][pk] = k0 + pk < ng ? drlv2[k] : -1.0;  // -1: accepts nothing
            lg[wave][pk] = -1;
            lclaim[wave][pk] = ~0u;
        }
    }
    for (int o = 1; o < 32; o <<= 1) {
        gmax = fmaxf(gmax, __shfl_xor(gmax, o, GS_WAVE));
        n2min = fmin(n2min, __shfl_xor(n2min, o, GS_WAVE));
        if (GEOM) n2max = fmax(n2max, __shfl_xor(n2max, o, GS_WAVE));
    }
    gmax = gs_uniform(gmax * (1.0f + 0x1p-20f));
    const float amin = gs_uniform((float)sqrt(n2min) * (1.0f - 0x1p-20f));
    const float dsa = GEOM ? gs_uniform((float)fabs(ds)) / amin * (1.0f + 0x1p-20f) : 0.0f;
    const float pmax = GEOM ? ldexpf(dsa, 16 - *yexp) : 0.0f;
    const float lmax = GEOM ? ldexpf(GS_ASSIGN_QMAX, -*yexp) : 0.0f;  // of sum |q|, unscaled
    const float tol = (float)(sqrt(tolsq) + 1e-9);
    gs_wave_sync();

    // one pair, decided with the reference arithmetic
    const auto exact = [&](int g, int pk) {
        const gs_ubi u = gs_load_ubi(ubis + 9 * (size_t)g);
        const long long k = k0 + pk;
        double x = gvx[3 * k], y = gvx[3 * k + 1], z = gvx[3 * k + 2];
        if constexpr (GEOM) {
            double m[9];
            for (int i = 0; i < 9; i++) m[i] = mat[i];
            const double* t = trans + 3 * (size_t)g;
            double g0, g1, g2;
            gs_gv_one(x, y, z, so_in[k], co_in[k], m, ds, t[0], t[1], t[2], g0, g1, g2);
            x = g0;
            y = g1;
            z = g2;
        }
        return gs_drlv2(u, x, y, z);
    };
    // can the pair be accepted (certified: true unless it certainly cannot)
    const auto maybe = [&](const gs_ubi& u, double t0, double t1, double t2, double win, int pk) {
        const double d = ld[wave][pk];
        const long long k = min(k0 + pk, (long long)ng - 1);
        if constexpr (GEOM) {
            const double a[3] = {la[wave][0][pk], la[wave][1][pk], la[wave][2][pk]};
            const double so = so_in[k], co = co_in[k];
            const double c[3] = {ds * (co * mat[0] + so * mat[1]),
                                 ds * (-so * mat[0] + co * mat[1]), ds * mat[2]};
            return !(gs_scan_fast_drlv2(u, a, c, t0, t1, t2, ds) >= fmin(tolsq, d) - 0.75 + win);
        } else {
            const double s = gs_drlv2(u, gvx[3 * k], gvx[3 * k + 1], gvx[3 * k + 2]);
            return s < tolsq && s < d;
        }
    };
    const auto window = [&](const gs_ubi& u, double t0, double t1, double t2) {
        return GEOM ? gs_scan_window(u, ds, tolsq, t0 * t0 + t1 * t1 + t2 * t2, n2min) : 0.0;
    };
    const auto accept = [&](int g, int pk, double se) {
        if (se < ld[wave][pk]) {
            ld[wave][pk] = se;
            lg[wave][pk] = g;
            if constexpr (FEW)
                atomicAdd(&lcnt[wave][g], 1);
            else
                atomicAdd(&counts[g], 1);
        }
    };
    int n1 = 0, n2 = 0;  // fills of the queues, wave-uniform
    // the first 64 (or n) entries of the second queue
    const auto settle2 = [&](int n) {
        gs_wave_sync();
        const unsigned e = q2[lane];
        const int g = e >> 7, pk = e & 127;
        double se = 0.0;
        bool todo = false;
        if (lane < n) {
            se = exact(g, pk);
            todo = se < tolsq;
        }
        while (__ballot(todo)) {  // at least the lowest lane leaves in each round
            if (todo) atomicMin(&lclaim[wave][pk], (unsigned)lane);
            gs_wave_sync();
            const bool mine = todo && lclaim[wave][pk] == (unsigned)lane;
            gs_wave_sync();
            if (mine) {
                accept(g, pk, se);
                lclaim[wave][pk] = ~0u;
            }
            todo = todo && !mine;
            gs_wave_sync();
        }
    };
    // 64 (or n) entries of the first queue from `at`
    const auto settle1 = [&](int at, int n) {
        gs_wave_sync();
        const unsigned e = q1[at + lane];
        const int g = min((int)(e >> 5), K - 1), quad = e & 31;
        const bool on = lane < n && (int)(e >> 5) < K;  // K and on: the repeated last grain
        const gs_ubi u = gs_load_ubi(ubis + 9 * (size_t)(on ? g : 0));
        double t0 = 0.0, t1 = 0.0, t2 = 0.0;
        if constexpr (GEOM) {
            const double* t = trans + 3 * (size_t)(on ? g : 0);
            t0 = t[0];
            t1 = t[1];
            t2 = t[2];
        }
        const double win = window(u, t0, t1, t2);
#pragma unroll 1
        for (int i = 0; i < 4; i++) {
            const int pk = on ? 4 * quad + i : 0;
            const bool cand = on && maybe(u, t0, t1, t2, win, pk) && k0 + pk < ng;
            const unsigned long long m = __ballot(cand);
            if (m) {
                if (cand) {
                    const unsigned pos = __builtin_amdgcn_mbcnt_hi(
                        (unsigned)(m >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)m, 0u));
                    q2[n2 + pos] = ((unsigned)g << 7) | pk;
                }
                n2 += __popcll(m);
                if (n2 >= GS_WAVE) {
                    settle2(GS_WAVE);
                    n2 -= GS_WAVE;
                    const unsigned rest = q2[GS_WAVE + lane];
                    gs_wave_sync();
                    q2[lane] = rest;
                    gs_wave_sync();
                }
            }
        }
    };
    const auto drain = [&] {  // whole batches of the first queue, the rest to its front
        if (n1 >= GS_WAVE) {
            int at = 0;
            for (; n1 - at >= GS_WAVE; at += GS_WAVE) settle1(at, GS_WAVE);
            const unsigned rest = q1[at + lane];  // in bounds: at <= 256
            gs_wave_sync();
            q1[lane] = rest;
            gs_wave_sync();
            n1 -= at;
        }
    };
    const auto flush = [&] {
        if (n1) settle1(0, n1);
        n1 = 0;
        if (n2) settle2(n2);
        n2 = 0;
    };

    const int tiles = (K + 31) / 32;
    const gs_half8* f = frag + lane;
    gs_half8 m0 = f[0], m1 = f[GS_WAVE], m2 = f[2 * GS_WAVE];
    // the sieve radius of a tile in units of 2^-16 (rounded up to a multiple
    // of 64), with GS_WIDE in the wide range; 0 where the tile is not sieved
    constexpr int GS_WIDE = 1 << 20;
    const auto radius = [&](int t) {
        const gs_tile_info w = info[t];
        const float sp = w.span * gmax + (GEOM ? dsa * w.lin : 0.0f);
        const bool wide = sp > GS_SIEVE_SPAN;
        float r = tol + (wide ? (float)GS_SIEVE_ERR_WIDE : (float)GS_SIEVE_ERR);
        if (GEOM) {
            const float part = w.tmax / (amin - w.tmax);
            r += 1.002f * (0x1.03p-10f * dsa * w.lin + 0.5775f * w.span * dsa * amin * part * part);
        }
        const bool fits = w.span < GS_SIEVE_UMAX && gmax < GS_SIEVE_GMAX &&
                          sp <= GS_SIEVE_SPAN_WIDE && r < GS_ASSIGN_RMAX &&
                          (!GEOM || (pmax <= GS_ASSIGN_PMAX && w.lin <= lmax && amin > 0.0f &&
                                     2.0f * w.tmax <= amin));
        return fits ? (((int)(r * 65536.0f) + 66) & ~63) | (wide ? GS_WIDE : 0) : 0;
    };
    // f32: everything that does not depend on the grain
    const float ds32 = GEOM ? (float)ds : 0.0f, cz32 = GEOM ? (float)(ds * mat[2]) : 0.0f;
    const bool range32 = GEOM && n2min > 0x1p-80 && n2max < 0x1p100 && fabs(ds) > 0x1p-60 &&
                         fabs(ds) < 0x1p60;
    int radii = 0;  // lane l: the radius of tile (t & ~63) + l
    for (int t = 0; t < tiles; t++) {
        const gs_half8 b0 = m0, b1 = m1, b2 = m2;
        if (t + 1 < tiles) {  // the next tile's fragments, in flight during this one
            f += 3 * GS_WAVE;
            m0 = f[0];
            m1 = f[GS_WAVE];
            m2 = f[2 * GS_WAVE];
        }
        if ((t & 63) == 0) radii = radius(min(t + lane, tiles - 1));
        const int want = __builtin_amdgcn_readlane(radii, t & 63);
        const bool wide = want & GS_WIDE;
        const unsigned lp = ((32u * t + (lane & 31)) << 5) | half;
        if (want) {
            const int ru = want & (GS_WIDE - 1);
            const gs_float16 c = gs_splat16((wide ? 201326592.0f : 12582912.0f) + (float)ru);
            const unsigned short thr = (unsigned short)(2 * ru);
#pragma unroll 1
            for (int s = 0; s < NB; s++) {
                const gs_half8 pk = lpk[wave][s][lane];
                if (!wide)
                    gs_sieve_tile<false>(pk, b0, b1, b2, c, thr, lp + 8 * s, q1, n1);
                else
                    gs_sieve_tile<true>(pk, b0, b1, b2, c, thr, lp + 8 * s, q1, n1);
                drain();
            }
        } else {  // a grain per lane in f32, the entries in the same order
            const int g = min(32 * t + (lane & 31), K - 1);
            const bool on = 32 * t + (lane & 31) < K;
            float lo, hi, t0 = 0.0f, t1 = 0.0f, t2 = 0.0f;
            gs_grain32 w;
            if constexpr (GEOM) {
                const double* tr = trans + 3 * (size_t)g;
                const float tt = (float)sqrt(tr[0] * tr[0] + tr[1] * tr[1] + tr[2] * tr[2]);
                w = gs_load_grain32(ubis + 9 * (size_t)g, on, fabsf(ds32));
                // a NaN |t| fails the comparison: every pair passes
                const bool fits = range32 && 2.0f * tt * (1.0f + 0x1p-20f) <= amin;
                t0 = (float)tr[0];
                t1 = (float)tr[1];
                t2 = (float)tr[2];
                gs_units32<false>(w, tol, fits ? 4.0f * gs_err32(w.a) : __builtin_inff(), lo, hi);
            } else {
                for (int p = lane; p < NP; p += GS_WAVE) {
                    const long long k = min(k0 + p, (long long)ng - 1);
                    const double x = gvx[3 * k], y = gvx[3 * k + 1], z = gvx[3 * k + 2];
                    const bool live = gs_finite(x) && gs_finite(y) && gs_finite(z);
                    lf[wave][0][p] = live ? gs_clamp32(x) : __builtin_nanf("");
                    lf[wave][1][p] = gs_clamp32(y);
                    lf[wave][GEOM ? 0 : 2][p] = gs_clamp32(z);
                }
                gs_wave_sync();
                w = gs_load_grain32(ubis + 9 * (size_t)g, on, gmax);
                gs_units32<false>(w, tol, gs_err32(w.a), lo, hi);
            }
#pragma unroll 1
            for (int s = 0; s < NB; s++) {
                if constexpr (GEOM) {
#pragma unroll 1
                    for (int j = 0; j < 4; j++) {
                        const int pk = 32 * s + 8 * j + 4 * half;
                        float f = 4.0f;
#pragma unroll
                        for (int i = pk; i < pk + 4; i++) {
                            const float e0 = (float)la[wave][0][i] - t0;
                            const float e1 = (float)la[wave][1][i] - t1;
                            const float e2 = (float)la[wave][2][i] - t2;
                            const float inv =
                                ds32 * __builtin_amdgcn_rsqf(__builtin_fmaf(
                                           e2, e2, __builtin_fmaf(e1, e1, e0 * e0)));
                            f = fminf(f, gs_cube32(w.u, __builtin_fmaf(e0, inv, -lf[wave][0][i]),
                                                   __builtin_fmaf(e1, inv, -lf[wave][1][i]),
                                                   __builtin_fmaf(e2, inv, -cz32), lo));
                        }
                        gs_push(f <= hi || hi == GS_ALL32, lp + 8 * s + 2 * j, q1, n1);
                    }
                } else {
                    gs_tile32<false>(lf[wave][0] + 32 * s, lf[wave][1] + 32 * s,
                                     lf[wave][2] + 32 * s, w, lo, hi, half, lp + 8 * s, q1, n1);
                }
                drain();
            }
        }
    }
    flush();
    gs_wave_sync();
    if constexpr (FEW)
        if (lane < K && lcnt[wave][lane]) atomicAdd(&counts[lane], lcnt[wave][lane]);
    for (int pk = lane; pk < NP; pk += GS_WAVE) {
        const long long k = k0 + pk;
        if (k < ng) {
            const int g = lg[wave][pk];
            if (g >= 0) {
                drlv2[k] = ld[wave][pk];
                labels[k] = g;
            } else {
                const int first = labels[k];
                if (first >= 0 && first < K) labels[k] = -1;
            }
        }
    }
}
