// Streaming form of the fused sweep: NS full red-black sweeps (mg_poisson.F90:55-74) of one launch,
// optionally from u = 0, with the trilinear correction added on load, or ending with the residual
// restricted to the coarse grid, as k_sweep_tile (fast_kernels.h).
//
// A workgroup owns an SX x SY column of the grid and a chunk of ZC planes, and marches up it.  A thread
// owns one pair of x neighbours, (even x, odd x), of the column and its halo, on every plane: one cell of
// each colour, which it holds by colour -- ur (first colour, i + j + k odd, the reference's ipass 1) and
// ub -- on the R planes in flight, the source (fr, fb) beside them.  So of a cell's six neighbours one x
// neighbour and both z neighbours are the thread's own registers; the other three have the same colour
// and sit in LDS planes that hold one colour each, at the thread's own index, the index of the row above
// and below, and one pair to the left or right by the parity of the row and plane.  Step p:
//   plane p + 1 + LATE + PD fetched into registers; plane p + 1 (fetched PD steps before) put: its
//   correction added (PROLONG), sorted by colour, ub to LDS;
//   colour pass h = 0 .. 2 NS - 1 on plane p - h: in-plane neighbours from LDS as the step before left
//   them, z neighbours from the registers, of which the one above was formed earlier in this step;
//   plane p - 2 NS + 1 is final and is stored; RESID: the residual of plane p - 2 NS;
//   one barrier.
// Every plane's LDS arrays are written in one step and read in the next, by different colour passes on
// different planes within a step, so one barrier a step orders all of it.  No cell is masked: a cell
// nearer the halo's rim than its pass needs takes meaningless values that no core cell reads (pass h is
// right from margin h + 1 on; H = 2 NS, with RESID one more).  The march is unrolled by R, so the slots
// are constants.  LATE (PROLONG): plane p + 2 is put at the end of step p, which takes the correction's
// chain of sums off the front of the first colour pass.
// max|resh2| of the last sweep is kept in FP32 only when asked for (the max of the FP32 values, widened
// once, equals the max of their widened values).  Every cell update sees the same operands in the same
// order as the two-launch colour passes, so the values are those of the tile kernel, bit for bit.
//
// Bound by the latency of a step (two sweeps of a plane, about 2 500 cycles at the one workgroup of 14 to
// 16 wavefronts per CU that 256^3 makes): counters find the vector units issuing 51-56 % of a launch, the
// wavefronts waiting 42-60 % of their cycles, LDS bank conflicts under 3 %, and 243 MB moved in 74 us at
// 256^3, two thirds of a large copy's rate.  One sweep per launch read u and the source and wrote u four
// times per V(2,2) visit, with nine LDS accesses per update instead of four and two barriers per plane and
// sweep.  One V(2,2) visit of one grid, FP32, before -> with two sweeps here, us: 512^3 1749 -> 1140, 256^3
// 213 -> 146, 128^3 (tile 32 x 16 x 16) 54 -> 40; FP64: 512^3 3358 -> 2457, 256^3 426 -> 357, 128^3 64 -> 55.
#pragma once
#include <utility>

#include "uniform_kernels.h"

namespace sg {

template <int SX_, int SY_, int ZC_> struct StreamShape {
    static constexpr int SX = SX_, SY = SY_, ZC = ZC_;
};

template <class SS, int NS, bool PROLONG, bool RESID, typename T> struct StreamGeom {
    static constexpr int LATE = PROLONG ? 1 : 0;
    // planes fetched ahead.  Two: 512^3 plain 573 us against 624 with one, 598 with three (registers);
    // one where the late put already leaves a step: PROLONG 569 us against 619 with two
    static constexpr int PD = PROLONG ? 1 : 2;
    static constexpr int H = 2 * NS + (RESID ? 1 : 0);          // halo in y and z
    static constexpr int HX = (H + 1) / 2 * 2;                  // in x: whole pairs
    static constexpr int PX = SS::SX / 2 + HX, PY = SS::SY + 2 * H, PP = PX * PY;
    static constexpr int NT = (PP + 63) / 64 * 64;              // one thread per pair
    static constexpr int LAG = 2 * NS - 1;                      // plane p - LAG is final after step p
    // ring: planes p - LAG - 1 (RESID: - 2) .. p + 1 + LATE + PD, even so that a slot keeps its parity
    static constexpr int R = (LAG + 3 + LATE + PD + (RESID ? 1 : 0) + 1) / 2 * 2;
    static constexpr int PAD = PX + 1, LP = NT + 2 * PAD;       // one colour of a plane in LDS
    static constexpr int lds_bytes = (int)sizeof(T) * (2 * R * LP + (RESID ? SS::SX * SS::SY : 0));
    static constexpr bool fits = NT <= 1024 && lds_bytes + 1024 <= 163840;
};

template <typename T> struct Pair { T x, y; };

template <class F, int... U> __device__ __forceinline__ void pair_steps(F &step, std::integer_sequence<int, U...>)
{
    (void)(step(std::integral_constant<int, U>{}) && ...);
}

// Body for column and chunk t of an n^3 level (n even, divisible by the shape, n > 2 H); called by every
// thread of a workgroup of StreamGeom::NT with the same t.  u, f and uc rows are aligned to pairs.
template <class SS, int NS, bool ZERO, bool PROLONG, bool RESID, typename T>
__device__ __forceinline__ void sweep_stream(const T *__restrict__ uin, T *__restrict__ uout, const T *__restrict__ f,
                                            int n, T h2, T h2i, const T *__restrict__ uc, T *__restrict__ rc,
                                            double *resmax, int t)
{
    using G = StreamGeom<SS, NS, PROLONG, RESID, T>;
    constexpr int SX = SS::SX, SY = SS::SY, ZC = SS::ZC, H = G::H, HX = G::HX, PX = G::PX, R = G::R, LP = G::LP,
                  LAG = G::LAG, LATE = G::LATE, PD = G::PD;
    static_assert(SX % 2 == 0 && SY % 2 == 0 && ZC % 2 == 0 && R % 2 == 0, "stream shape");
    static_assert(!PROLONG || H % 2 == 0, "the coarse planes start on an even fine plane");
    __shared__ T sr[R * LP], sb[R * LP];
    __shared__ T sx[RESID ? SX * SY : 1];
    const int ntx = n / SX, nty = n / SY;
    const int x0 = t % ntx * SX, y0 = t / ntx % nty * SY, z0 = t / (ntx * nty) * ZC;
    const int nc = n >> 1, tid = (int)threadIdx.x;
    const int q = tid < G::PP ? tid : G::PP - 1;
    const int xp = q % PX, l = q / PX;
    const int gx = wrapn(x0 - HX + 2 * xp, n), gy = wrapn(y0 - H + l, n);
    const unsigned off = (unsigned)(gy * n + gx) * (unsigned)sizeof(T);   // within a plane
    const bool core = tid < G::PP && 2 * xp >= HX && 2 * xp < HX + SX && l >= H && l < H + SY;
    const bool want = resmax != nullptr;
    T amax = T(0);
    // e: the first colour sits on the odd cell of this row's pairs, on planes of even parity
    const bool e = ((H + l) & 1) == 0;
    T *const R0 = sr + G::PAD + tid, *const B0 = sb + G::PAD + tid;
    const int xs = e ? 1 : -1;
    T *const RX[2] = {R0 - xs, R0 + xs}, *const BX[2] = {B0 + xs, B0 - xs};   // by plane parity

    T ur[R], ub[R], fr[R], fb[R];   // first colour / second colour of the pair on each plane of the ring
#pragma unroll
    for (int i = 0; i < R; ++i) ur[i] = ub[i] = fr[i] = fb[i] = T(0);

    const int zlo = z0 - H, zhi = z0 + ZC + H - 1, zend = z0 + ZC - 1 + LAG + (RESID ? 1 : 0);
    auto fetch = [&](int k, int s) {   // raw: (even x, odd x)
        const long base = (long)wrapn(k, n) * n * n;
        Pair<T> v = {T(0), T(0)};
        if (!ZERO) v = *reinterpret_cast<const Pair<T> *>(reinterpret_cast<const char *>(uin + base) + off);
        ur[s] = v.x;
        ub[s] = v.y;
        const Pair<T> w = *reinterpret_cast<const Pair<T> *>(reinterpret_cast<const char *>(f + base) + off);
        fr[s] = w.x;
        fb[s] = w.y;
    };
    // coarse columns of the pair: rows jc and jc1 (toward the cell), columns ic - 1, ic, ic + 1
    T cw[2][6], cn[6];
    unsigned co[6];
    if (PROLONG) {
        const int ic = gx >> 1, jc = gy >> 1, jc1 = wrapn(jc + 2 * (gy & 1) - 1, nc);
        const int im = wrapn(ic - 1, nc), ip = wrapn(ic + 1, nc);
        const int c[6] = {jc * nc + im, jc * nc + ic, jc * nc + ip, jc1 * nc + im, jc1 * nc + ic, jc1 * nc + ip};
#pragma unroll
        for (int i = 0; i < 6; ++i) co[i] = (unsigned)c[i] * (unsigned)sizeof(T);
    }
    auto fetch_coarse = [&](int c, T (&o)[6]) {
        const T *p = uc + (long)wrapn(c, nc) * nc * nc;
#pragma unroll
        for (int i = 0; i < 6; ++i) o[i] = *reinterpret_cast<const T *>(reinterpret_cast<const char *>(p) + co[i]);
    };
    // plane k (parity par) of slot s from raw to colours, the correction added, second colour to LDS
    auto put = [&](int k, int s, int par) {
        T a = ur[s], b = ub[s];
        if (PROLONG) {
            if (par) {
#pragma unroll
                for (int i = 0; i < 6; ++i) { cw[0][i] = cw[1][i]; cw[1][i] = cn[i]; }
                fetch_coarse((k >> 1) + 2, cn);
            }
            const T *A = cw[par ? 0 : 1], *B = cw[par ? 1 : 0];
            a = a + trilinear_value<T>(A[1], A[0], A[4], B[1], B[4], B[0], A[3], B[3]);
            b = b + trilinear_value<T>(A[1], A[2], A[4], B[1], B[4], B[2], A[5], B[5]);
        }
        const bool d = par ? !e : e;
        const T fa = fr[s], fo = fb[s];
        ur[s] = d ? b : a;
        ub[s] = d ? a : b;
        fr[s] = d ? fo : fa;
        fb[s] = d ? fa : fo;
        B0[s * LP] = ub[s];
    };

    if (PROLONG) {   // zlo is even: put(zlo) reads coarse planes zlo / 2 - 1 and zlo / 2
        fetch_coarse((zlo >> 1) - 1, cw[0]);
        fetch_coarse(zlo >> 1, cw[1]);
        fetch_coarse((zlo >> 1) + 1, cn);
    }
    constexpr int P0 = H & 1;   // parity of zlo
#pragma unroll
    for (int i = 0; i < 1 + LATE + PD; ++i) fetch(zlo + i, i);
    put(zlo, 0, P0);
    if (LATE) put(zlo + 1, 1, P0 ^ 1);
    T ro[2][2];   // RESID: the pair's residuals on the last even and odd plane
    // coarse cell of the planes kq - 1, kq: the thread of the even row takes its own four residuals and the
    // odd row's from sx.  r[a + 2 b + 4 dz] in restriction.F90's operand order 000 100 010 001 110 101 011 111
    auto restrict_pair = [&](int kq) {
        if (!core || ((l - H) & 1) || kq < z0 || kq >= z0 + ZC) return;
        const T *w = sx + 4 * ((l - H) / 2 * (SX / 2) + xp - HX / 2);
        rc[((long)(kq >> 1) * nc + (gy >> 1)) * nc + (gx >> 1)] =
            restrict_value<T>(ro[0][0], ro[0][1], w[0], ro[1][0], w[1], ro[1][1], w[2], w[3]);
    };
    __syncthreads();
    int pb = zlo;
    auto step = [&](auto uc_) -> bool {   // plane p = pb + uu; uniform per workgroup
        constexpr int uu = decltype(uc_)::value;
        const int p = pb + uu;
        if (p > zend) return false;
        auto S = [](int delta) constexpr { return ((uu + delta) % R + R) % R; };
        auto PAR = [](int delta) constexpr { return (P0 + uu + delta + 64) & 1; };
        if (p + 1 + LATE + PD <= zhi) fetch(p + 1 + LATE + PD, S(1 + LATE + PD));
        if (RESID && PAR(-LAG - 2) == 1) restrict_pair(p - LAG - 2);
        if (!LATE) put(p + 1, S(1), PAR(1));
#pragma unroll
        for (int h = 0; h < 2 * NS; ++h) {
            const int s = S(-h), sm = S(-h - 1), sp = S(-h + 1), par = PAR(-h);
            T w;
            if (h % 2 == 0) {
                ur[s] = relax_value<T>(ur[s], ub[s], BX[par][s * LP], B0[s * LP + PX], B0[s * LP - PX], ub[sp], ub[sm],
                                       fr[s], h2, &w);
                R0[s * LP] = ur[s];
            } else {
                ub[s] = relax_value<T>(ub[s], ur[s], RX[par][s * LP], R0[s * LP + PX], R0[s * LP - PX], ur[sp], ur[sm],
                                       fb[s], h2, &w);
                B0[s * LP] = ub[s];
            }
            if (h >= 2 * NS - 2 && want && core && p - h >= z0 && p - h < z0 + ZC) amax = fmax(amax, fabs(w));
        }
        const int ks = p - LAG;
        if (core && ks >= z0 && ks < z0 + ZC) {
            const int s = S(-LAG);
            const bool d = PAR(-LAG) ? !e : e;
            Pair<T> v;
            v.x = d ? ub[s] : ur[s];
            v.y = d ? ur[s] : ub[s];
            *reinterpret_cast<Pair<T> *>(reinterpret_cast<char *>(uout + (long)ks * n * n) + off) = v;
        }
        if (RESID) {
            const int s = S(-LAG - 1), sm = S(-LAG - 2), sp = S(-LAG), par = PAR(-LAG - 1);
            const T rr = resid_value<T>(ur[s], ub[s], BX[par][s * LP], B0[s * LP + PX], B0[s * LP - PX], ub[sp], ub[sm],
                                        fr[s], h2i);
            const T rb = resid_value<T>(ub[s], ur[s], RX[par][s * LP], R0[s * LP + PX], R0[s * LP - PX], ur[sp], ur[sm],
                                        fb[s], h2i);
            const bool d = par ? !e : e;
            ro[par][0] = d ? rb : rr;
            ro[par][1] = d ? rr : rb;
            if (par == 1 && core && ((l - H) & 1)) {
                T *w = sx + 4 * ((l - H) / 2 * (SX / 2) + xp - HX / 2);
                w[0] = ro[0][0]; w[1] = ro[0][1]; w[2] = ro[1][0]; w[3] = ro[1][1];
            }
        }
        if (LATE && p + 2 <= zhi) put(p + 2, S(2), PAR(2));
        __syncthreads();
        return true;
    };
    for (; pb <= zend; pb += R) pair_steps(step, std::make_integer_sequence<int, R>{});
    if (RESID) restrict_pair(z0 + ZC - 1);
    if (want) block_atomic_max(resmax, (double)amax);
}

template <class SS, int NS, bool ZERO, bool PROLONG, bool RESID, typename T>
__global__ void __launch_bounds__((StreamGeom<SS, NS, PROLONG, RESID, T>::NT))
k_sweep_stream(const T *__restrict__ uin, T *__restrict__ uout, const T *__restrict__ f, int n, T h2, T h2i,
               const T *__restrict__ uc, T *__restrict__ rc, double *resmax)
{
    const int ntiles = (n / SS::SX) * (n / SS::SY) * (n / SS::ZC);
    const int t = xcd_tile(ntiles);
    if (t >= ntiles) return;
    sweep_stream<SS, NS, ZERO, PROLONG, RESID, T>(uin, uout, f, n, h2, h2i, uc, rc, resmax, t);
}

} // namespace sg
