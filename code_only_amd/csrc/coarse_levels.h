// The levels of <= 16^3 cells of one periodic problem in one workgroup's LDS (gfx950), in either
// precision: the FMG part of mg_lin (mg.F90:142-215) from the coarsest level up to the first held
// one, or one V-cycle from that level down and back (the bottom of each finer level's V-cycle).
// Shared by the single-grid solver (n = 2^a) and the batched one (also n = 3 * 2^a, whose 3^3 level is
// solved exactly).
//
// Bound by latency: a 16^3 cycle is some 150 dependent steps of a few thousand cells.  So
//  * level widths are template parameters: decoding a cell is shifts and constants, and no step
//    waits for a load of its level's description;
//  * an even level is stored split by cell colour (i + j + k even first), each half [k][j][i / 2] with
//    the even j before the odd: the lanes of every step (one per 2 x 2 or 2^3 group of cells) read
//    consecutive words, where one array in cell order puts lane pairs on the same LDS banks;
//  * a smoothing call keeps each thread's 2 x 2 cells (y, z) of both colours and their source in
//    registers: a pass reads 4 LDS words per cell instead of 8 (the four cells share their y and z
//    neighbours), and which x neighbour a cell needs is known at compile time;
//  * the levels of <= 8^3 cells run in one wavefront, which needs no barrier between its steps (8^3:
//    four cells of a colour per lane), the 2^3 level with the 1^3 level under it in the registers of
//    every lane; 16^3 and 12^3 take the whole workgroup, one barrier per step;
//  * the restricted residual reads each 2^3 group of cells and its 24 outer neighbours once, and zeroes
//    the coarse level's u in the same step;
//  * the tricubic prolongation into 8^3 and larger runs as three separable passes with its weights
//    tabulated once per launch.
// Measured, FP64, 16^3: 57 us for the FMG, 18 us for a V-cycle (as launches of their own kernels: 290
// and 60 launches of 1.4-2 us); cycles per step of 16^3 / 8^3 / 4^3: down 6.9k / 3.8k / 2.7k, up 7.3k /
// 3.7k / 2.6k, the 2^3 bottom 3.3k.  Without the row order and the shared neighbours a 16^3 step took
// 10-13k; 1 024 threads with one cell each the same.  What is left is the latency of dependent LDS
// reads and FP64 adds, some 450 cycles per colour of a small level, and, where a kernel holds more than 256
// registers beside the levels' code, spills to scratch: the compiler reports none for the periodic k_coarse,
// 129 spilled registers for the FP64 one with zero ghosts, for 16^3 132 and 68 in k_cycle_small (FP64, FP32)
// and 149 and 274 in k_base_small (periodic, zero ghosts), 9 in kb_coarse<double>.
// Boundaries: periodic (ZERO false), or zero ghosts (ZERO: mg_boundary_fill0, with mg_boundary_extrap's
// odd continuation, (-1)^g times the clamped interior cell for g ghost coordinates, before a
// prolongation; mg.F90:735-771).
// Per-cell values come from relax_value, resid_value, restrict_value, trilinear_value and cubic4 in the
// order of the one-kernel-per-loop kernels, so both give the same bits.
#pragma once
#include "uniform_kernels.h"

namespace sg {

constexpr int kCoarseMaxN = 16;
constexpr int kCoarseThreads = 512;
constexpr int kWaveLevelN = 8;   // levels up to this width run in one wavefront
constexpr int kCoarseDepth = 5;  // 16, 8, 4, 2, 1

// 4-point cubic combination in the reference's order: (a0 v0 + a1 v1) + a2 v2 + a3 v3.
template <typename T> __device__ __forceinline__ T cubic4(const T w[4], T v0, T v1, T v2, T v3)
{
    T s = w[0] * v0 + w[1] * v1;
    s = s + w[2] * v2;
    s = s + w[3] * v3;
    return s;
}

constexpr int kCoarseCells = 16 * 16 * 16 + 8 * 8 * 8 + 4 * 4 * 4 + 2 * 2 * 2 + 1;  // >= 12^3 + 6^3 + 3^3
constexpr int kCubicTab = 16 + 8 + 4;   // >= 12 + 6: fine indices of the held levels with a cubic stencil

// what differs between problems with the same widths: h^2 and 1 / h^2 of the held levels, and the
// exact solve of a 3^3 coarsest level (Hartley basis, eigenvalues)
template <typename T> struct CoarseCoef {
    T h2[kCoarseDepth], h2i[kCoarseDepth];
    T q3[9], lam3[3];
};

// host: coefficients of the levels from the one with cell width h down
template <typename T> inline CoarseCoef<T> coarse_coef(double h)
{
    CoarseCoef<T> C{};
    for (int l = 0; l < kCoarseDepth; ++l) {
        const double hl = h * (double)(1 << l);
        C.h2[l] = (T)(hl * hl);
        C.h2i[l] = (T)(1.0 / (hl * hl));
    }
    return C;
}

template <typename T> struct CoarseLds {
    T u[kCoarseCells], r[kCoarseCells];
    T bx[8 * 8 * 16], bxy[8 * 16 * 16];   // separable tricubic passes into 16^3
    T tw[kCubicTab][4];                   // tricubic weights per fine index of a level, and its four
    int ti[kCubicTab][4];                 // coarse indices (wrapped)
};

// one held level of width N: its place in the LDS arrays
template <int N> struct CoarseLevel {
    static constexpr bool even = N % 2 == 0;
    static constexpr int len = N * N * N, nh = N / 2, pl = N * nh, half = N * pl;
    static constexpr int off = N == 16 || N == 12 ? 0 : N == 8 ? 4096 : N == 6 ? 1728 : N == 4 ? 4608
                                                  : N == 3 ? 1944 : N == 2 ? 4672 : 4680;
    static constexpr int tab = N == 16 || N == 12 ? 0 : N == 8 ? 16 : N == 6 ? 12 : 24;   // cubic table (N >= 4)
    // cell (i, j, k): split by colour when N is even, in cell order for 1^3 and 3^3
    static __device__ __forceinline__ int row(int j) { return (j & 1) * (N / 2) + (j >> 1); }
    static __device__ __forceinline__ int at(int i, int j, int k)
    {
        return even ? ((i + j + k) & 1) * half + (k * N + row(j)) * nh + (i >> 1) : (k * N + j) * N + i;
    }
    static __device__ __forceinline__ void decode(int t, int &i, int &j, int &k)
    {
        i = t % N;
        j = (t / N) % N;
        k = t / (N * N);
    }
};
constexpr int coarse_below(int n) { return n == 3 || n == 1 ? 0 : n / 2; }   // next level's width, 0: none

// The threads of a step: one wavefront (whose LDS accesses execute in order, so only the compiler has
// to keep it) or the workgroup.
template <bool WAVE> struct CoarseTeam {
    static constexpr int NT = WAVE ? kWave : kCoarseThreads;
    static __device__ __forceinline__ void sync()
    {
        if (WAVE) {
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            __builtin_amdgcn_wave_barrier();
        } else {
            __syncthreads();
        }
    }
};

// nsweep mg_relax calls (mg_poisson.F90:55-74) of the level of width N; resmax (nullable) receives
// max|resh2| of the last
template <typename T, int N, bool WAVE, bool ZERO>
__device__ __forceinline__ void coarse_relax(CoarseLds<T> &S, T h2, int nsweep, double *resmax)
{
    using C = CoarseTeam<WAVE>;
    using L = CoarseLevel<N>;
    static_assert(N >= 4 && N % 2 == 0, "2^3 and 1^3 levels: coarse_bottom");
    constexpr int nh = L::nh, pl = L::pl, half = L::half;
    T *const u = S.u + L::off;
    const T *const f = S.r + L::off;
    double amax = 0.0;
    if constexpr (N == 4) {
        // one cell per lane: 32 of a colour
        const int t = (int)threadIdx.x & (half - 1);
        const int ih = t % nh, rj = (t / nh) % N, k = t / pl, j = rj < N / 2 ? 2 * rj : 2 * (rj - N / 2) + 1;
        const int yp = t + (L::row(j + 1 == N ? 0 : j + 1) - rj) * nh, ym = t + (L::row(j == 0 ? N - 1 : j - 1) - rj) * nh;
        const int zp = k + 1 == N ? t + pl - half : t + pl, zm = k == 0 ? t - pl + half : t - pl;
        const int tp = ih + 1 == nh ? t + 1 - nh : t + 1, tm = ih == 0 ? t + nh - 1 : t - 1;
        const bool act = threadIdx.x < half;
        const T f1 = f[half + t], f0 = f[t];
        for (int q = 0; q < nsweep; ++q) {
            if (q == nsweep - 1) amax = 0.0;
#pragma unroll
            for (int ipass = 1; ipass <= 2; ++ipass) {
                T *own = u + (ipass == 1 ? half : 0);
                const T *oth = u + (ipass == 1 ? 0 : half);
                const bool odd = ((j + k + ipass) & 1) != 0;
                // i even: the x+ neighbour has the same i / 2, the x- one i / 2 - 1; i odd the reverse
                const T a = oth[t];
                T b = oth[odd ? tp : tm], vyp = oth[yp], vym = oth[ym], vzp = oth[zp], vzm = oth[zm];
                if (ZERO) {
                    if (odd ? ih + 1 == nh : ih == 0) b = T(0);
                    if (j + 1 == N) vyp = T(0);
                    if (j == 0) vym = T(0);
                    if (k + 1 == N) vzp = T(0);
                    if (k == 0) vzm = T(0);
                }
                T s;
                const T v = relax_value<T>(own[t], odd ? b : a, odd ? a : b, vyp, vym, vzp, vzm, ipass == 1 ? f1 : f0, h2, &s);
                if (act) own[t] = v;
                if (resmax) amax = fmax(amax, fabs((double)s));
                C::sync();
            }
        }
    } else {
        constexpr int nb = N / 2, lanes = nh * nb * nb;   // threads that own cells
        const int q0 = (int)threadIdx.x;
        constexpr int dy = nb * nh;                       // from an even row to the odd one above it
        const bool act = lanes == C::NT || q0 < lanes;
        const int q = act ? q0 : 0;
        const int ih = q % nh, J = (q / nh) % nb, K = q / (nh * nb);
        const int t = (2 * K * N + J) * nh + ih;           // cell (dj, dk) at t + dj dy + dk pl
        const int xp = ih + 1 == nh ? 1 - nh : 1, xm = ih == 0 ? nh - 1 : -1;
        const int ym = dy + (J == 0 ? dy - nh : -nh), yp = J + 1 == nb ? nh - dy : nh;   // rows 2 J - 1, 2 J + 2
        const int zm = K == 0 ? half - pl : -pl, zp = K + 1 == nb ? 2 * pl - half : 2 * pl;
        T ur[2][4], fr[2][4];   // colour (0: even), cell dj + 2 dk
#pragma unroll
        for (int c = 0; c < 2; ++c)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int o = c * half + t + (e & 1) * dy + (e >> 1) * pl;
                ur[c][e] = u[o];
                fr[c][e] = f[o];
            }
        for (int sw = 0; sw < nsweep; ++sw) {
            if (sw == nsweep - 1) amax = 0.0;
#pragma unroll
            for (int ipass = 1; ipass <= 2; ++ipass) {
                constexpr int kE = 4;
                const int c = ipass == 1 ? 1 : 0;
                const T *oth = u + (c ? 0 : half) + t;
                T a[4], b[4], yl[2], yh[2], zl[2], zh[2];   // other colour: same place, x side, outer y, outer z
#pragma unroll
                for (int e = 0; e < kE; ++e) {
                    const int dj = e & 1, dk = e >> 1, o = dj * dy + dk * pl;
                    const bool odd = ((dj + dk + ipass) & 1) != 0;   // i odd: its x+ neighbour is at ih + 1
                    a[e] = oth[o];
                    b[e] = oth[o + (odd ? xp : xm)];
                    if (ZERO && (odd ? ih + 1 == nh : ih == 0)) b[e] = T(0);
                }
#pragma unroll
                for (int d = 0; d < 2; ++d) {
                    yl[d] = oth[d * pl + ym];
                    yh[d] = oth[d * pl + yp];
                    zl[d] = oth[d * dy + zm];
                    zh[d] = oth[d * dy + zp];
                    if (ZERO) {
                        if (J == 0) yl[d] = T(0);
                        if (J + 1 == nb) yh[d] = T(0);
                        if (K == 0) zl[d] = T(0);
                        if (K + 1 == nb) zh[d] = T(0);
                    }
                }
#pragma unroll
                for (int e = 0; e < kE; ++e) {
                    const int dj = e & 1, dk = e >> 1;
                    const bool odd = ((dj + dk + ipass) & 1) != 0;
                    T s;
                    ur[c][e] = relax_value<T>(ur[c][e], odd ? b[e] : a[e], odd ? a[e] : b[e], dj ? yh[dk] : a[e + 1],
                                              dj ? a[e - 1] : yl[dk], dk ? zh[dj] : a[e + 2], dk ? a[e - 2] : zl[dj],
                                              fr[c][e], h2, &s);
                    if (act) u[c * half + t + dj * dy + dk * pl] = ur[c][e];
                    if (resmax && act) amax = fmax(amax, fabs((double)s));
                }
                C::sync();
            }
        }
    }
    if (resmax) {
        if (WAVE) {
            amax = wave_max(amax);
            if (threadIdx.x == 0) atomic_max_nonneg(resmax, amax);
        } else {
            block_atomic_max(resmax, amax);
        }
    }
}

// A V-cycle of the 2^3 level over the 1^3 one, every lane of the wavefront on the same eight values in
// registers (a step of two or one cell per lane would be all LDS latency).  Cell o = i + 2 j + 4 k.
template <typename T, bool ZERO>
__device__ __forceinline__ void coarse_bottom(CoarseLds<T> &S, T h2, T h2i, T h2b, int npre, int npost, double *resmax)
{
    using L = CoarseLevel<2>;
    T u[8], f[8];
#pragma unroll
    for (int o = 0; o < 8; ++o) {
        const int c = L::off + L::at(o & 1, (o >> 1) & 1, o >> 2);
        u[o] = S.u[c];
        f[o] = S.r[c];
    }
    double amax = 0.0;
    // neighbours of cell o along axis bit m: the other cell of the pair on both sides, or it and a zero
    auto hi = [&](int o, int m) { return ZERO && (o & m) ? T(0) : u[o ^ m]; };
    auto lo = [&](int o, int m) { return ZERO && !(o & m) ? T(0) : u[o ^ m]; };
    auto sweep = [&]() {
        amax = 0.0;
#pragma unroll
        for (int ipass = 1; ipass <= 2; ++ipass)
#pragma unroll
            for (int o = 0; o < 8; ++o) {
                if ((((o & 1) + ((o >> 1) & 1) + (o >> 2)) & 1) != (ipass & 1)) continue;
                T s;
                u[o] = relax_value<T>(u[o], hi(o, 1), lo(o, 1), hi(o, 2), lo(o, 2), hi(o, 4), lo(o, 4), f[o], h2, &s);
                if (resmax) amax = fmax(amax, fabs((double)s));
            }
    };
    for (int p = 0; p < npre; ++p) sweep();
    T r[8];
#pragma unroll
    for (int o = 0; o < 8; ++o)
        r[o] = resid_value<T>(u[o], hi(o, 1), lo(o, 1), hi(o, 2), lo(o, 2), hi(o, 4), lo(o, 4), f[o], h2i);
    const T fb = restrict_value<T>(r[0], r[1], r[2], r[4], r[3], r[5], r[6], r[7]);
    T ub = T(0);
#pragma unroll
    for (int it = 0; it < 2; ++it) {
        const T g = ZERO ? T(0) : ub;
        T s;
        ub = relax_value<T>(ub, g, g, g, g, g, g, fb, h2b, &s);
    }
    const T n1 = ZERO ? -ub : ub;   // the 1^3 level's neighbour across one face; two ghosts undo the sign
    const T e = trilinear_value<T>(ub, n1, n1, n1, ub, ub, ub, n1);
#pragma unroll
    for (int o = 0; o < 8; ++o) u[o] = u[o] + e;
    for (int p = 0; p < npost; ++p) sweep();
    CoarseTeam<true>::sync();
    if (threadIdx.x == 0) {
#pragma unroll
        for (int o = 0; o < 8; ++o) S.u[L::off + L::at(o & 1, (o >> 1) & 1, o >> 2)] = u[o];
        if (resmax && npost > 0) atomic_max_nonneg(resmax, amax);
    }
    CoarseTeam<true>::sync();
}

// mg_slvsml (mg.F90:540-546) of a 3^3 coarsest level: the exact periodic solve u = Q3 (Lambda^+ (Q3
// rhs)), Q the symmetric orthonormal Hartley basis, Lambda = (lam_i + lam_j) + lam_k with the zero mode
// dropped; one output per lane and pass, accumulated k = 0, 1, 2 in order (as the CPU restatement).
template <typename T> __device__ __forceinline__ void coarse_exact3(CoarseLds<T> &S, const CoarseCoef<T> &P)
{
    using L = CoarseLevel<3>;
    T *g = S.u + L::off;
    const int c = (int)threadIdx.x < 27 ? (int)threadIdx.x : 26;
    const int i = c % 3, j = (c / 3) % 3, k = c / 9;
    T v = S.r[L::off + c];
    for (int pass = 0; pass < 6; ++pass) {
        CoarseTeam<true>::sync();
        if (threadIdx.x < 27) g[c] = v;
        CoarseTeam<true>::sync();
        const int axis = pass % 3, m = axis == 0 ? i : (axis == 1 ? j : k), st = axis == 0 ? 1 : (axis == 1 ? 3 : 9);
        const int base = c - m * st;
        T acc = T(0);
#pragma unroll
        for (int e = 0; e < 3; ++e) acc = acc + P.q3[m * 3 + e] * g[base + e * st];
        v = acc;
        if (pass == 2) {
            const T den = (P.lam3[i] + P.lam3[j]) + P.lam3[k];
            v = den != T(0) ? v / den : T(0);
        }
    }
    CoarseTeam<true>::sync();
    if (threadIdx.x < 27) g[c] = v;
    CoarseTeam<true>::sync();
}

// the 1^3 level alone (mg_slvsml: two sweeps from zero), one cell
template <typename T, bool ZERO> __device__ __forceinline__ void coarse_single(CoarseLds<T> &S, T h2)
{
    if (threadIdx.x == 0) {
        T ub = T(0), s;
        const T fb = S.r[CoarseLevel<1>::off];
        for (int it = 0; it < 2; ++it) {
            const T g = ZERO ? T(0) : ub;
            ub = relax_value<T>(ub, g, g, g, g, g, g, fb, h2, &s);
        }
        S.u[CoarseLevel<1>::off] = ub;
    }
    CoarseTeam<true>::sync();
}

// residual of the level of width N (mg_poisson.F90:17-27) restricted into the next one's right-hand
// side (restriction.F90:132-147), whose u is zeroed
template <typename T, int N, bool WAVE, bool ZERO>
__device__ __forceinline__ void coarse_resid_restrict(CoarseLds<T> &S, T h2i)
{
    using C = CoarseTeam<WAVE>;
    using L = CoarseLevel<N>;
    using K = CoarseLevel<N / 2>;
    const T *u = S.u + L::off, *f = S.r + L::off;
#pragma unroll
    for (int q0 = 0; q0 < K::len; q0 += C::NT) {
        const int q = q0 + (int)threadIdx.x;
        if (K::len % C::NT == 0 || q < K::len) {
            int cx, cy, cz;
            K::decode(q, cx, cy, cz);
            const int i = 2 * cx, j = 2 * cy, k = 2 * cz;
            const int im = i == 0 ? N - 1 : i - 1, ip = i + 2 == N ? 0 : i + 2;
            const int jm = j == 0 ? N - 1 : j - 1, jp = j + 2 == N ? 0 : j + 2;
            const int km = k == 0 ? N - 1 : k - 1, kp = k + 2 == N ? 0 : k + 2;
            T v[8], xo[8], yo[8], zo[8];   // the group, and each cell's neighbour outside it per axis
#pragma unroll
            for (int o = 0; o < 8; ++o) {
                const int a = o & 1, b = (o >> 1) & 1, d = o >> 2;
                v[o] = u[L::at(i + a, j + b, k + d)];
                xo[o] = u[L::at(a ? ip : im, j + b, k + d)];
                yo[o] = u[L::at(i + a, b ? jp : jm, k + d)];
                zo[o] = u[L::at(i + a, j + b, d ? kp : km)];
                if (ZERO) {
                    if (a ? i + 2 == N : i == 0) xo[o] = T(0);
                    if (b ? j + 2 == N : j == 0) yo[o] = T(0);
                    if (d ? k + 2 == N : k == 0) zo[o] = T(0);
                }
            }
            T r[8];
#pragma unroll
            for (int o = 0; o < 8; ++o) {
                const int a = o & 1, b = (o >> 1) & 1, d = o >> 2;
                r[o] = resid_value<T>(v[o], a ? xo[o] : v[o ^ 1], a ? v[o ^ 1] : xo[o], b ? yo[o] : v[o ^ 2],
                                      b ? v[o ^ 2] : yo[o], d ? zo[o] : v[o ^ 4], d ? v[o ^ 4] : zo[o],
                                      f[L::at(i + a, j + b, k + d)], h2i);
            }
            const int c = K::at(cx, cy, cz);
            S.r[K::off + c] = restrict_value<T>(r[0], r[1], r[2], r[4], r[3], r[5], r[6], r[7]);
            S.u[K::off + c] = T(0);
        }
    }
    C::sync();
}

// right-hand side of the level of width N restricted into the next one's
template <typename T, int N, bool WAVE> __device__ __forceinline__ void coarse_restrict(CoarseLds<T> &S)
{
    using C = CoarseTeam<WAVE>;
    using L = CoarseLevel<N>;
    using K = CoarseLevel<N / 2>;
#pragma unroll
    for (int q0 = 0; q0 < K::len; q0 += C::NT) {
        const int q = q0 + (int)threadIdx.x;
        if (K::len % C::NT == 0 || q < K::len) {
            int cx, cy, cz;
            K::decode(q, cx, cy, cz);
            auto F = [&](int a, int b, int d) { return S.r[L::off + L::at(2 * cx + a, 2 * cy + b, 2 * cz + d)]; };
            S.r[K::off + K::at(cx, cy, cz)] = restrict_value<T>(F(0, 0, 0), F(1, 0, 0), F(0, 1, 0), F(0, 0, 1), F(1, 1, 0),
                                                                F(1, 0, 1), F(0, 1, 1), F(1, 1, 1));
        }
    }
    C::sync();
}

// interior cell and factor that coarse index c (-1 .. n) stands for
template <typename T, bool ZERO> __device__ __forceinline__ int coarse_ghost(int c, int n, T &sign)
{
    sign = T(1);
    if (!ZERO) return wrap_g(c, n);
    if (c < 0 || c >= n) sign = T(-1);
    return c < 0 ? 0 : (c >= n ? n - 1 : c);
}

// trilinear prolongation into the level of width N (interpolation.F90:226-245), added to u
// (mg_addint) or stored: one thread per coarse cell forms its 2^3 fine cells from the 27 coarse cells
// around it
template <typename T, int N, bool WAVE, bool ADD, bool ZERO> __device__ __forceinline__ void coarse_linear(CoarseLds<T> &S)
{
    using C = CoarseTeam<WAVE>;
    using L = CoarseLevel<N>;
    using K = CoarseLevel<N / 2>;
    constexpr int nc = N / 2;
    T *const u = S.u + L::off;
#pragma unroll
    for (int q0 = 0; q0 < K::len; q0 += C::NT) {
        const int q = q0 + (int)threadIdx.x;
        if (K::len % C::NT == 0 || q < K::len) {
            int cx, cy, cz;
            K::decode(q, cx, cy, cz);
            int ix[3], iy[3], iz[3];
            T sx[3], sy[3], sz[3];
#pragma unroll
            for (int e = 0; e < 3; ++e) {
                ix[e] = coarse_ghost<T, ZERO>(cx + e - 1, nc, sx[e]);
                iy[e] = coarse_ghost<T, ZERO>(cy + e - 1, nc, sy[e]);
                iz[e] = coarse_ghost<T, ZERO>(cz + e - 1, nc, sz[e]);
            }
            T c[3][3][3];
#pragma unroll
            for (int d = 0; d < 3; ++d)
#pragma unroll
                for (int b = 0; b < 3; ++b)
#pragma unroll
                    for (int a = 0; a < 3; ++a) {
                        c[d][b][a] = S.u[K::off + K::at(ix[a], iy[b], iz[d])];
                        if (ZERO && (a != 1 || b != 1 || d != 1)) c[d][b][a] = (sx[a] * sy[b] * sz[d]) * c[d][b][a];
                    }
#pragma unroll
            for (int o = 0; o < 8; ++o) {
                const int i = o & 1, j = (o >> 1) & 1, k = o >> 2, x = 2 * i, y = 2 * j, z = 2 * k;   // toward the cell
                const T v = trilinear_value<T>(c[1][1][1], c[1][1][x], c[1][y][1], c[z][1][1], c[z][y][1], c[z][1][x],
                                               c[1][y][x], c[z][y][x]);
                T &w = u[L::at(2 * cx + i, 2 * cy + j, 2 * cz + k)];
                w = ADD ? w + v : v;
            }
        }
    }
    C::sync();
}

// FMG prolongation into the level of width N (mg.F90:608-633): tricubic, trilinear where the coarse
// grid with ghosts is narrower than 4
template <typename T, int N, bool WAVE, bool ZERO> __device__ __forceinline__ void coarse_fmg_interp(CoarseLds<T> &S)
{
    using C = CoarseTeam<WAVE>;
    using L = CoarseLevel<N>;
    using K = CoarseLevel<N / 2>;
    constexpr int nc = N / 2;
    if constexpr (nc + 2 < 4) {
        coarse_linear<T, N, WAVE, false, ZERO>(S);
        return;
    } else {
        const T(*tw)[4] = S.tw + L::tab;
        const int(*ti)[4] = S.ti + L::tab;
        const T *uc = S.u + K::off;
        T *u = S.u + L::off;
        if constexpr (N < 8) {
            for (int q = threadIdx.x; q < L::len; q += C::NT) {
                int i, j, k;
                L::decode(q, i, j, k);
                T bz[4];
                for (int kq = 0; kq < 4; ++kq) {
                    T by[4];
#pragma unroll
                    for (int jq = 0; jq < 4; ++jq) {
                        T x[4];
#pragma unroll
                        for (int e = 0; e < 4; ++e) x[e] = uc[K::at(ti[i][e], ti[j][jq], ti[k][kq])];
                        by[jq] = cubic4<T>(tw[i], x[0], x[1], x[2], x[3]);
                    }
                    bz[kq] = cubic4<T>(tw[j], by[0], by[1], by[2], by[3]);
                }
                u[L::at(i, j, k)] = cubic4<T>(tw[k], bz[0], bz[1], bz[2], bz[3]);
            }
        } else {
            for (int q = threadIdx.x; q < nc * nc * N; q += C::NT) {   // bx[kc][jc][i]
                const int i = q % N, jc = (q / N) % nc, kc = q / (N * nc);
                S.bx[q] = cubic4<T>(tw[i], uc[K::at(ti[i][0], jc, kc)], uc[K::at(ti[i][1], jc, kc)],
                                    uc[K::at(ti[i][2], jc, kc)], uc[K::at(ti[i][3], jc, kc)]);
            }
            C::sync();
            for (int q = threadIdx.x; q < nc * N * N; q += C::NT) {    // bxy[kc][j][i]
                int i, j, kc;
                L::decode(q, i, j, kc);
                const T *col = S.bx + kc * nc * N + i;
                S.bxy[q] = cubic4<T>(tw[j], col[ti[j][0] * N], col[ti[j][1] * N], col[ti[j][2] * N], col[ti[j][3] * N]);
            }
            C::sync();
            for (int q = threadIdx.x; q < L::len; q += C::NT) {
                int i, j, k;
                L::decode(q, i, j, k);
                const T *p = S.bxy + j * N + i;
                u[L::at(i, j, k)] = cubic4<T>(tw[k], p[ti[k][0] * N * N], p[ti[k][1] * N * N], p[ti[k][2] * N * N],
                                              p[ti[k][3] * N * N]);
            }
        }
        C::sync();
    }
}

// The schedule runs as a loop over steps, each level's code once in it: written out as nested cycles the
// FP64 kernel of 16^3 was 85 KB of straight-line code, more than the instruction cache, and a cold launch
// waited for it line by line.  Depth v counts the held levels from 0; depth B is the bottom (2^3 with the
// 1^3 under it, or 3^3).
constexpr int coarse_bottom_depth(int n) { return n <= 3 ? 0 : 1 + coarse_bottom_depth(n / 2); }

// a step of a V-cycle on depth v: down (smoothing, restricted residual), up (prolongated correction,
// smoothing) or the bottom
enum CoarseStep { kStepDown, kStepUp, kStepBottom };

template <typename T, int N, int D, bool ZERO>
__device__ __forceinline__ void coarse_step(CoarseLds<T> &S, const CoarseCoef<T> &P, int v, CoarseStep kind, int npre,
                                            int npost, double *resmax)
{
    constexpr bool WAVE = N <= kWaveLevelN;
    if (v == D) {
        if constexpr (WAVE) {
            if (threadIdx.x >= kWave) return;
        }
        if constexpr (N == 3) {
            coarse_exact3<T>(S, P);
        } else if constexpr (N == 2) {
            coarse_bottom<T, ZERO>(S, P.h2[D], P.h2i[D], P.h2[D + 1], npre, npost, resmax);
        } else {
            if (kind == kStepUp) coarse_linear<T, N, WAVE, true, ZERO>(S);
            coarse_relax<T, N, WAVE, ZERO>(S, P.h2[D], kind == kStepUp ? npost : npre,
                                           kind == kStepUp && npost > 0 ? resmax : nullptr);
            if (kind == kStepDown) coarse_resid_restrict<T, N, WAVE, ZERO>(S, P.h2i[D]);
        }
        return;
    }
    if constexpr (N > 3) coarse_step<T, N / 2, D + 1, ZERO>(S, P, v, kind, npre, npost, resmax);
}

// the right-hand sides of depths 1 .. B (and 1^3), and the coarsest level's solution
template <typename T, int N, int D, bool ZERO> __device__ __forceinline__ void coarse_start(CoarseLds<T> &S, const CoarseCoef<T> &P)
{
    constexpr bool WAVE = N <= kWaveLevelN;
    if constexpr (WAVE) {
        if (threadIdx.x >= kWave) return;
    }
    if constexpr (N == 3) {
        coarse_exact3<T>(S, P);
    } else {
        coarse_restrict<T, N, WAVE>(S);
        if constexpr (N == 2) coarse_single<T, ZERO>(S, P.h2[D + 1]);
        else coarse_start<T, N / 2, D + 1, ZERO>(S, P);
    }
}

// FMG prolongation into depth v
template <typename T, int N, int D, bool ZERO> __device__ __forceinline__ void coarse_prolong(CoarseLds<T> &S, int v)
{
    constexpr bool WAVE = N <= kWaveLevelN;
    if (v == D) {
        if constexpr (WAVE) {
            if (threadIdx.x >= kWave) return;
        }
        if constexpr (N != 3) coarse_fmg_interp<T, N, WAVE, ZERO>(S);
        return;
    }
    if constexpr (N > 3) coarse_prolong<T, N / 2, D + 1, ZERO>(S, v);
}

// depths run by one wavefront start here
constexpr int coarse_wave_depth(int n) { return n <= kWaveLevelN ? 0 : 1 + coarse_wave_depth(n / 2); }

// FMG over the held levels from the right-hand side of width N in S.r (mg.F90:142-215), or one V-cycle
// from the u there (mg.F90:179-210).  Every thread of the workgroup; S.u of width N is ready afterwards.
template <typename T, int N, bool ZERO>
__device__ __forceinline__ void coarse_run(CoarseLds<T> &S, const CoarseCoef<T> &P, bool fmg, int ncycle, int npre,
                                           int npost, double *resmax)
{
    constexpr int B = coarse_bottom_depth(N), W = coarse_wave_depth(N);
    constexpr bool three = N % 3 == 0;
    bool wave = W == 0;   // the last step ran in one wavefront: the next of the workgroup meets it first
    if (fmg) {
        coarse_start<T, N, 0, ZERO>(S, P);
        wave = true;
    }
    // a 3^3 bottom is exact: its FMG stage has no cycles
    for (int ml = fmg ? (three ? B - 1 : B) : 0; ml >= 0; --ml) {
        if (fmg) {
            if (ml < W && wave) __syncthreads();
            coarse_prolong<T, N, 0, ZERO>(S, ml);
            wave = ml >= W;
        }
        for (int jc = 0; jc < (fmg ? ncycle : 1); ++jc) {
            const int nstep = 2 * (B - ml) + 1;
            for (int q = 0; q < nstep; ++q) {
                const int v = q <= B - ml ? ml + q : 2 * B - ml - q;
                const CoarseStep kind = v == B ? kStepBottom : (q < B - ml ? kStepDown : kStepUp);
                if (v < W && wave) __syncthreads();
                coarse_step<T, N, 0, ZERO>(S, P, v, kind, npre, npost,
                                           ml == 0 && q == nstep - 1 && jc == (fmg ? ncycle : 1) - 1 ? resmax : nullptr);
                wave = v >= W;
            }
        }
    }
    if (W == 0 || wave) __syncthreads();
}

// tricubic stencils of the levels from width N whose coarse grid is wide enough, one fine index per
// lane (q).  A ghost cell's factor goes into its weight: w (-v) = (-w) v in every operation.
template <typename T, int N, bool ZERO> __device__ __forceinline__ void coarse_tables(CoarseLds<T> &S, int q)
{
    constexpr int M = coarse_below(N);
    if constexpr (M >= 2) {
        const int f = q - CoarseLevel<N>::tab;
        if (f >= 0 && f < N) {
            int idx[4];
            double a[4];
            cubic_stencil(f, -1, M, idx, a);
            for (int e = 0; e < 4; ++e) {
                T sign;
                S.ti[q][e] = coarse_ghost<T, ZERO>(idx[e], M, sign);
                S.tw[q][e] = sign * (T)a[e];
            }
        }
        coarse_tables<T, M, ZERO>(S, q);
    }
}

// mode 0: FMG over all held levels from the right-hand side of the first (mg.F90:142-215 restricted to
// them); mode 1: one V-cycle from it with zero initial guess (mg.F90:179-210).  rhs_in, u_out: dense
// N^3 arrays.  Every thread of a kCoarseThreads workgroup calls it.
template <typename T, int N, bool ZERO = false>
__device__ __forceinline__ void coarse_solve(CoarseLds<T> &S, const CoarseCoef<T> &P, const T *__restrict__ rhs_in,
                                             T *__restrict__ u_out, int mode, int ncycle, int npre, int npost)
{
    using L = CoarseLevel<N>;
    for (int c = threadIdx.x; c < L::len; c += kCoarseThreads) {
        int i, j, k;
        L::decode(c, i, j, k);
        const int d = L::off + L::at(i, j, k);
        S.r[d] = rhs_in[c];
        if (mode == 1) S.u[d] = T(0);
    }
    if (mode == 0 && threadIdx.x >= kCoarseThreads - 64) coarse_tables<T, N, ZERO>(S, (int)threadIdx.x - (kCoarseThreads - 64));
    __syncthreads();
    coarse_run<T, N, ZERO>(S, P, mode == 0, ncycle, npre, npost, nullptr);
    for (int c = threadIdx.x; c < L::len; c += kCoarseThreads) {
        int i, j, k;
        L::decode(c, i, j, k);
        u_out[c] = S.u[L::off + L::at(i, j, k)];
    }
}

} // namespace sg
