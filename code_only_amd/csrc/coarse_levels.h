// The levels of <= 16^3 cells of one periodic problem in one workgroup's LDS (gfx950), in either
// precision: the FMG part of mg_lin (mg.F90:142-215) from the coarsest level up to the first held
// one, or one V-cycle from that level down and back (the bottom of each finer level's V-cycle).
// Shared by the single-grid solver (n = 2^a) and the batched one (also n = 3 * 2^a, whose 3^3 level is
// solved exactly).
//
// Bound by latency: a 16^3 cycle is some 150 dependent steps of a few thousand cells.  So
//  * level widths are template parameters: decoding a cell is shifts and constants, and no step
//    waits for a load of its level's description;
//  * an even level is stored split by cell colour (i + j + k even first), each half [k][j][i / 2]: a
//    colour pass reads its six neighbours, its source and its own values with consecutive lanes on
//    consecutive words, where one array in cell order puts every lane pair on the same LDS bank;
//  * the levels of <= 6^3 cells run in one wavefront, which needs no barrier between its steps; the
//    others keep the whole workgroup, one barrier per step;
//  * the restricted residual reads each 2^3 group of cells and its 24 outer neighbours once, and zeroes
//    the coarse level's u in the same step;
//  * the tricubic prolongation into 8^3 and larger runs as three separable passes with its weights
//    tabulated once per launch.
// Boundaries: periodic (ZERO false), or zero ghosts (ZERO: mg_boundary_fill0, with mg_boundary_extrap's
// odd continuation, (-1)^g times the clamped interior cell for g ghost coordinates, before a
// prolongation; mg.F90:735-771).
// Per-cell values come from relax_value, resid_value, restrict_value, trilinear_value and cubic4 in the
// order of the one-kernel-per-loop kernels, so both give the same bits.
#pragma once
#include "uniform_kernels.h"

namespace sg {

constexpr int kCoarseMaxN = 16;
constexpr int kCoarseThreads = 1024;
constexpr int kWaveLevelN = 6;   // levels up to this width run in one wavefront
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

// one held level of width N: its place in the LDS arrays, depth D below the first held level
template <int N> struct CoarseLevel {
    static constexpr bool even = N % 2 == 0;
    static constexpr int len = N * N * N, nh = N / 2, pl = N * nh, half = N * pl;
    static constexpr int off = N == 16 || N == 12 ? 0 : N == 8 ? 4096 : N == 6 ? 1728 : N == 4 ? 4608
                                                  : N == 3 ? 1944 : N == 2 ? 4672 : 4680;
    static constexpr int tab = N == 16 || N == 12 ? 0 : N == 8 ? 16 : N == 6 ? 12 : 24;   // cubic table (N >= 4)
    // cell (i, j, k): split by colour when N is even, in cell order for 1^3 and 3^3
    static __device__ __forceinline__ int at(int i, int j, int k)
    {
        return even ? ((i + j + k) & 1) * half + (k * N + j) * nh + (i >> 1) : (k * N + j) * N + i;
    }
    static __device__ __forceinline__ void decode(int t, int &i, int &j, int &k)
    {
        i = t % N;
        j = (t / N) % N;
        k = t / (N * N);
    }
};
constexpr int coarse_below(int n) { return n == 3 || n == 1 ? 0 : n / 2; }   // next level's width, 0: none

// Exact periodic solve of a 3^3 coarsest level (one thread): u = Q3 (Lambda^+ (Q3 rhs)), Q the
// symmetric orthonormal Hartley basis, Lambda = (lam_i + lam_j) + lam_k with the zero mode dropped;
// every output of an axis pass is accumulated k = 0, 1, 2 in order.  The FP64 instantiation rounds as
// the CPU restatement does.
template <typename T> __device__ __forceinline__ void exact3_pass(T *g, const T *Q, int axis)
{
    for (int b = 0; b < 3; ++b)
        for (int a = 0; a < 3; ++a) {
            T x[3], y[3];
            for (int k = 0; k < 3; ++k) {
                const int q = axis == 0 ? (b * 3 + a) * 3 + k : axis == 1 ? (b * 3 + k) * 3 + a : (k * 3 + b) * 3 + a;
                x[k] = g[q];
            }
            for (int m = 0; m < 3; ++m) {
                T acc = T(0);
                for (int k = 0; k < 3; ++k) acc = acc + Q[m * 3 + k] * x[k];
                y[m] = acc;
            }
            for (int m = 0; m < 3; ++m) {
                const int q = axis == 0 ? (b * 3 + a) * 3 + m : axis == 1 ? (b * 3 + m) * 3 + a : (m * 3 + b) * 3 + a;
                g[q] = y[m];
            }
        }
}

template <typename T> __device__ __forceinline__ void exact3(T *u, const T *rhs, const T *Q, const T *lam)
{
    T g[27];
    for (int c = 0; c < 27; ++c) g[c] = rhs[c];
    for (int a = 0; a < 3; ++a) exact3_pass<T>(g, Q, a);
    for (int k = 0; k < 3; ++k)
        for (int j = 0; j < 3; ++j)
            for (int i = 0; i < 3; ++i) {
                const T den = (lam[i] + lam[j]) + lam[k];
                T &v = g[(k * 3 + j) * 3 + i];
                v = den != T(0) ? v / den : T(0);
            }
    for (int a = 0; a < 3; ++a) exact3_pass<T>(g, Q, a);
    for (int c = 0; c < 27; ++c) u[c] = g[c];
}


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

// one mg_relax call (mg_poisson.F90:55-74); a 1^3 level's cell belongs to the second pass
template <typename T, int N, bool WAVE, bool ZERO>
__device__ __forceinline__ void coarse_relax(CoarseLds<T> &S, T h2, double *resmax)
{
    using C = CoarseTeam<WAVE>;
    using L = CoarseLevel<N>;
    T *u = S.u + L::off;
    const T *f = S.r + L::off;
    double amax = 0.0;
    T s;
    if constexpr (N == 1) {
        if (threadIdx.x == 0) {
            const T g = ZERO ? T(0) : u[0];
            u[0] = relax_value<T>(u[0], g, g, g, g, g, g, f[0], h2, &s);
        }
        C::sync();
        return;
    } else {
        constexpr int nh = L::nh, pl = L::pl, half = L::half;
#pragma unroll
        for (int ipass = 1; ipass <= 2; ++ipass) {
            T *own = u + (ipass == 1 ? half : 0);
            const T *oth = u + (ipass == 1 ? 0 : half), *fo = f + (ipass == 1 ? half : 0);
#pragma unroll
            for (int t0 = 0; t0 < half; t0 += C::NT) {
                const int t = t0 + (int)threadIdx.x;
                if (half % C::NT == 0 || t < half) {
                    const int ih = t % nh, j = (t / nh) % N, k = t / pl;
                    const bool odd = ((j + k + ipass) & 1) != 0;
                    // i even: the x+ neighbour has the same i / 2, the x- one i / 2 - 1; i odd the reverse
                    const int side = odd ? (ih + 1 == nh ? t + 1 - nh : t + 1) : (ih == 0 ? t + nh - 1 : t - 1);
                    const int yp = j + 1 == N ? t + nh - pl : t + nh, ym = j == 0 ? t - nh + pl : t - nh;
                    const int zp = k + 1 == N ? t + pl - half : t + pl, zm = k == 0 ? t - pl + half : t - pl;
                    const T a = oth[t];
                    T b = oth[side], vyp = oth[yp], vym = oth[ym], vzp = oth[zp], vzm = oth[zm];
                    if (ZERO) {
                        if (odd ? ih + 1 == nh : ih == 0) b = T(0);
                        if (j + 1 == N) vyp = T(0);
                        if (j == 0) vym = T(0);
                        if (k + 1 == N) vzp = T(0);
                        if (k == 0) vzm = T(0);
                    }
                    own[t] = relax_value<T>(own[t], odd ? b : a, odd ? a : b, vyp, vym, vzp, vzm, fo[t], h2, &s);
                    amax = fmax(amax, fabs((double)s));
                }
            }
            C::sync();
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
// (mg_addint) or stored
template <typename T, int N, bool WAVE, bool ADD, bool ZERO> __device__ __forceinline__ void coarse_linear(CoarseLds<T> &S)
{
    using C = CoarseTeam<WAVE>;
    using L = CoarseLevel<N>;
    using K = CoarseLevel<N / 2>;
    constexpr int nc = N / 2;
#pragma unroll
    for (int q0 = 0; q0 < L::len; q0 += C::NT) {
        const int q = q0 + (int)threadIdx.x;
        if (L::len % C::NT == 0 || q < L::len) {
            // in storage order: colour, k, j, i / 2
            const int p = q / L::half, h = q % L::half;
            const int ic = h % nc, j = (h / nc) % N, k = h / L::pl, i = 2 * ic + ((j + k + p) & 1);
            const int jc = j >> 1, kc = k >> 1;
            T sx, sy, sz;
            const int ic1 = coarse_ghost<T, ZERO>(ic + 2 * (i & 1) - 1, nc, sx), jc1 = coarse_ghost<T, ZERO>(jc + 2 * (j & 1) - 1, nc, sy),
                      kc1 = coarse_ghost<T, ZERO>(kc + 2 * (k & 1) - 1, nc, sz);
            auto V = [&](int a, int b, int d) { return S.u[K::off + K::at(a, b, d)]; };
            T c[8] = {V(ic, jc, kc), V(ic1, jc, kc), V(ic, jc1, kc), V(ic, jc, kc1),
                      V(ic, jc1, kc1), V(ic1, jc, kc1), V(ic1, jc1, kc), V(ic1, jc1, kc1)};
            if (ZERO) {
                c[1] = sx * c[1];
                c[2] = sy * c[2];
                c[3] = sz * c[3];
                c[4] = (sy * sz) * c[4];
                c[5] = (sx * sz) * c[5];
                c[6] = (sx * sy) * c[6];
                c[7] = (sx * sy * sz) * c[7];
            }
            const T v = trilinear_value<T>(c[0], c[1], c[2], c[3], c[4], c[5], c[6], c[7]);
            T &w = S.u[L::off + q];
            w = ADD ? w + v : v;
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
        if constexpr (WAVE) {
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

// One V-cycle from the level of width N (depth D below the first held one) down and back.  Levels of
// <= kWaveLevelN run in wavefront 0 (WAVE); the workgroup meets it at a barrier.  mg_slvsml
// (mg.F90:540-546) at the bottom: two sweeps of a 1^3 level, the exact solve of a 3^3 one.
template <typename T, int N, int D, bool WAVE, bool ZERO>
__device__ __forceinline__ void coarse_cycle(CoarseLds<T> &S, const CoarseCoef<T> &P, int npre, int npost, double *resmax)
{
    static_assert(WAVE == (N <= kWaveLevelN), "levels of <= kWaveLevelN run in one wavefront");
    if constexpr (N == 1) {
        for (int it = 0; it < 2; ++it) coarse_relax<T, 1, true, ZERO>(S, P.h2[D], nullptr);
    } else if constexpr (N == 3) {
        if (threadIdx.x == 0) exact3<T>(S.u + CoarseLevel<3>::off, S.r + CoarseLevel<3>::off, P.q3, P.lam3);
        CoarseTeam<true>::sync();
    } else {
        for (int p = 0; p < npre; ++p) coarse_relax<T, N, WAVE, ZERO>(S, P.h2[D], nullptr);
        coarse_resid_restrict<T, N, WAVE, ZERO>(S, P.h2i[D]);
        constexpr int M = coarse_below(N);
        constexpr bool MW = M <= kWaveLevelN;
        if constexpr (MW && !WAVE) {
            if (threadIdx.x < kWave) coarse_cycle<T, M, D + 1, true, ZERO>(S, P, npre, npost, nullptr);
            __syncthreads();
        } else {
            coarse_cycle<T, M, D + 1, MW, ZERO>(S, P, npre, npost, nullptr);
        }
        coarse_linear<T, N, WAVE, true, ZERO>(S);
        for (int p = 0; p < npost; ++p) coarse_relax<T, N, WAVE, ZERO>(S, P.h2[D], p == npost - 1 ? resmax : nullptr);
    }
}

// FMG from the coarsest level up to the level of width N (mg.F90:142-215)
template <typename T, int N, int D, bool WAVE, bool ZERO>
__device__ __forceinline__ void coarse_fmg(CoarseLds<T> &S, const CoarseCoef<T> &P, int ncycle, int npre, int npost,
                                           double *resmax)
{
    if constexpr (N == 1 || N == 3) {
        if (threadIdx.x < N * N * N) S.u[CoarseLevel<N>::off + threadIdx.x] = T(0);
        CoarseTeam<true>::sync();
        coarse_cycle<T, N, D, true, ZERO>(S, P, npre, npost, nullptr);
    } else {
        constexpr int M = coarse_below(N);
        constexpr bool MW = M <= kWaveLevelN;
        coarse_restrict<T, N, WAVE>(S);
        if constexpr (MW && !WAVE) {
            if (threadIdx.x < kWave) coarse_fmg<T, M, D + 1, true, ZERO>(S, P, ncycle, npre, npost, nullptr);
            __syncthreads();
        } else {
            coarse_fmg<T, M, D + 1, MW, ZERO>(S, P, ncycle, npre, npost, nullptr);
        }
        coarse_fmg_interp<T, N, WAVE, ZERO>(S);
        for (int jc = 0; jc < ncycle; ++jc)
            coarse_cycle<T, N, D, WAVE, ZERO>(S, P, npre, npost, jc == ncycle - 1 ? resmax : nullptr);
    }
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
// N^3 arrays.  resmax receives max|resh2| of the last smoothing of the first level when non-null.
// Every thread of a kCoarseThreads workgroup calls it.
template <typename T, int N, bool ZERO = false>
__device__ __forceinline__ void coarse_solve(CoarseLds<T> &S, const CoarseCoef<T> &P, const T *__restrict__ rhs_in,
                                             T *__restrict__ u_out, int mode, int ncycle, int npre, int npost,
                                             double *resmax)
{
    using L = CoarseLevel<N>;
    constexpr bool W = N <= kWaveLevelN;
    for (int c = threadIdx.x; c < L::len; c += kCoarseThreads) {
        int i, j, k;
        L::decode(c, i, j, k);
        const int d = L::off + L::at(i, j, k);
        S.r[d] = rhs_in[c];
        if (mode == 1) S.u[d] = T(0);
    }
    if (mode == 0 && threadIdx.x >= kCoarseThreads - 64) coarse_tables<T, N, ZERO>(S, (int)threadIdx.x - (kCoarseThreads - 64));
    __syncthreads();
    if (!W || threadIdx.x < kWave) {
        if (mode == 0) coarse_fmg<T, N, 0, W, ZERO>(S, P, ncycle, npre, npost, resmax);
        else coarse_cycle<T, N, 0, W, ZERO>(S, P, npre, npost, resmax);
    }
    if (W) __syncthreads();
    for (int c = threadIdx.x; c < L::len; c += kCoarseThreads) {
        int i, j, k;
        L::decode(c, i, j, k);
        u_out[c] = S.u[L::off + L::at(i, j, k)];
    }
}

} // namespace sg
