// Kernels of the batched uniform solve: many independent periodic n^3 problems (n = 2^a or
// 3 * 2^a, each with its own h) advanced together, one launch per step of the multigrid schedule.
//
// A launch carries a list of items (problem p, level l, first workgroup, workgroup count), sorted
// by first workgroup; every workgroup finds its item by binary search, so one launch covers the
// same step of all problems whatever their sizes.  Per-(problem, level) data -- array pointers by
// code, n, h -- sit in a device table indexed p * kBLev + l.  A per-problem activity flag lets a
// problem that has converged drop out of every later launch without changing the launch sequence
// (which can then be replayed as a graph).
//
// Per-cell arithmetic is that of the single-grid kernels (relax_value, resid_value,
// restrict_value, trilinear/tricubic values, the fused sweep and cubic tile bodies, the coarse
// kernel's level operations), so a power-of-two problem solved in a batch has the same values as
// solved alone.  Index arithmetic is general (division by n through a multiply-high reciprocal):
// n need not be a power of two.
#pragma once
#include "exact_planes.h"
#include "fast_kernels.h"

namespace sg {
namespace batch {

constexpr int kMaxProb = 4096;
constexpr int kBLev = 12;        // levels per problem (n <= 1024, so n^3 < 2^31)
constexpr int kThreads = 256;    // workgroup of the cell-per-thread kernels

// Codes of the per-level arrays: U, U1 (second buffer of the fused sweeps), RHS (shared with RHO).
enum { CU = 0, CU1 = 1, CRHS = 2, kCodes = 3 };

// t / d for 0 <= t < 2^31 as (umulhi(t, m) + t) >> s, m = floor(2^32 (2^s - d) / d) + 1,
// s = ceil(log2 d) (Granlund & Montgomery, "Division by invariant integers using multiplication").
struct FastDiv {
    unsigned d, m;
    int s;
};

inline FastDiv make_div(unsigned d)
{
    FastDiv f{d, 0u, 0};
    while ((1u << f.s) < d) ++f.s;
    f.m = (unsigned)((((unsigned long long)1 << 32) * (((unsigned long long)1 << f.s) - d)) / d + 1);
    return f;
}

__device__ __forceinline__ unsigned fdiv(unsigned t, const FastDiv &f) { return (__umulhi(t, f.m) + t) >> f.s; }

template <typename T> struct PL {
    T *a[kCodes];
    int n;        // cells per side
    int lc;       // first level held by the coarse kernel (problem-wide)
    int lb;       // level of the exact-coarse cycle's bottom (problem-wide)
    FastDiv dn;   // division by n
    T h2, h2i;
};

struct Item {
    int p, l, blk0, nblk;
};

template <typename T> struct BL {
    const Item *items;
    int nitems;
    const PL<T> *pl;
    const int *active;
    bool exact;   // the cycle ends at lb, not lc
};

__device__ __forceinline__ int find_item(const Item *it, int n, int b)
{
    int lo = 0, hi = n - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (it[mid].blk0 <= b) lo = mid;
        else hi = mid - 1;
    }
    return lo;
}

// Workgroup b of a grid of 8 * ceil(total / 8) workgroups, dealt round-robin over the 8 XCDs:
// XCD x works through the contiguous range [x * per, (x + 1) * per) of the logical workgroups, so
// neighbouring tiles of a problem share one L2.  Returns -1 for the padding.
__device__ __forceinline__ int xcd_block(int total)
{
    const int per = (int)(gridDim.x / 8);
    const int b = (int)blockIdx.x;
    const int v = (b % 8) * per + b / 8;
    return v < total ? v : -1;
}

template <typename T> struct Cell {
    const Item *it;
    const PL<T> *q;
    int lb;  // workgroup index inside the item
};

template <typename T> __device__ __forceinline__ bool locate(const BL<T> &L, int b, Cell<T> &c)
{
    if (b < 0) return false;
    const Item &it = L.items[find_item(L.items, L.nitems, b)];
    if (!L.active[it.p]) return false;
    c.it = &it;
    c.q = L.pl + it.p * kBLev + it.l;
    c.lb = b - it.blk0;
    return true;
}

__device__ __forceinline__ int wrp(int i, int n) { return i + 1 == n ? 0 : i + 1; }
__device__ __forceinline__ int wrm(int i, int n) { return i == 0 ? n - 1 : i - 1; }

__device__ __forceinline__ void decode(unsigned t, const FastDiv &dn, int n, int &i, int &j, int &k)
{
    const unsigned r1 = fdiv(t, dn);
    i = (int)(t - r1 * (unsigned)n);
    const unsigned r2 = fdiv(r1, dn);
    j = (int)(r1 - r2 * (unsigned)n);
    k = (int)r2;
}

// restriction.F90:132-147: item level l is the coarse level, its source level l - 1.
template <typename T>
__global__ void __launch_bounds__(kThreads) kb_restrict(BL<T> L, int cdst, int csrc)
{
    Cell<T> c;
    if (!locate(L, (int)blockIdx.x, c)) return;
    const PL<T> &q = *c.q, &qf = *(c.q - 1);
    const int nc = q.n, nf = qf.n;
    const unsigned t = (unsigned)c.lb * kThreads + threadIdx.x;
    if (t >= (unsigned)nc * nc * nc) return;
    int ic, jc, kc;
    decode(t, q.dn, nc, ic, jc, kc);
    const T *uf = qf.a[csrc];
    const int i = 2 * ic, j = 2 * jc, k = 2 * kc;
    auto F = [&](int a, int b, int d) { return uf[((k + d) * nf + (j + b)) * nf + (i + a)]; };
    q.a[cdst][t] = restrict_value<T>(F(0, 0, 0), F(1, 0, 0), F(0, 1, 0), F(0, 0, 1), F(1, 1, 0), F(1, 0, 1),
                                     F(0, 1, 1), F(1, 1, 1));
}

// ---- FP64 outer step (mg.F90:84-90 per problem) ---------------------------------------------

struct Outer {
    double *psi[kMaxProb];
    double *alt[kMaxProb];       // second phi buffer (ping-pong of the fused update)
    const double *src[kMaxProb];
    double h2i[kMaxProb];        // 1 / h^2 of the finest level, as the CPU restatement forms it
};

// Norm partials of the source of level-0 items: per workgroup max|f| and sum f^2.
__global__ void __launch_bounds__(kThreads) kb_src_norms(BL<double> L, const Outer *O, double *pmax, double *psum)
{
    Cell<double> c;
    if (!locate(L, (int)blockIdx.x, c)) return;
    const int n = c.q->n;
    const unsigned t = (unsigned)c.lb * kThreads + threadIdx.x;
    double mx = 0.0, sm = 0.0;
    if (t < (unsigned)n * n * n) {
        const double v = O->src[c.it->p][t];
        mx = fabs(v);
        sm = v * v;
    }
    block_max_sum(mx, sm);
    if (threadIdx.x == 0) { pmax[blockIdx.x] = mx; psum[blockIdx.x] = sm; }
}

// pout = pin + e (UPD) and r = f - L pout stored as Te into level 0's RHS, with per-workgroup norm
// partials of r.  pin / pout are psi / alt of the problem by the parity (0: psi -> alt).  Neighbour
// values are pin + e formed on the fly, exactly the values pout receives.  e: level 0 array `ce`
// (U when the problem has no fine level).
template <typename Te, bool UPD>
__global__ void __launch_bounds__(kThreads)
kb_outer_resid(BL<Te> L, const Outer *O, int parity, int ce, double *pmax, double *psum)
{
    Cell<Te> c;
    if (!locate(L, (int)blockIdx.x, c)) return;
    const PL<Te> &q = *c.q;
    const int p = c.it->p, n = q.n;
    const double *pin = parity ? O->alt[p] : O->psi[p];
    double *pout = parity ? O->psi[p] : O->alt[p];
    const Te *e = q.a[q.lc == 0 ? CU : ce];  // a problem held by the coarse kernel alone keeps e in U
    const unsigned t = (unsigned)c.lb * kThreads + threadIdx.x;
    double mx = 0.0, sm = 0.0;
    if (t < (unsigned)n * n * n) {
        int i, j, k;
        decode(t, q.dn, n, i, j, k);
        auto P = [&](int x) -> double { return UPD ? pin[x] + (double)e[x] : pin[x]; };
        const int row = (k * n + j) * n;
        const double pc = P((int)t);
        const double rv = resid_value<double>(pc, P(row + wrp(i, n)), P(row + wrm(i, n)), P((k * n + wrp(j, n)) * n + i),
                                              P((k * n + wrm(j, n)) * n + i), P((wrp(k, n) * n + j) * n + i),
                                              P((wrm(k, n) * n + j) * n + i), O->src[p][t], O->h2i[p]);
        q.a[CRHS][t] = (Te)rv;
        if (UPD) pout[t] = pc;
        mx = fabs(rv);
        sm = rv * rv;
    }
    block_max_sum(mx, sm);
    if (threadIdx.x == 0) { pmax[blockIdx.x] = mx; psum[blockIdx.x] = sm; }
}

// The same outer step marching along z: workgroup b of an item owns a kOzX x kOzY patch of (i, j)
// columns and zc planes of that problem (n % 32 == 0, n % zc == 0).  Each thread forms its cell
// of the next plane (and, on the patch edge, one x and/or y halo cell: the periodic neighbours)
// while the current plane sits in a double-buffered LDS plane with a one-cell halo, the z
// neighbours in registers: every value of pin + e is loaded once per patch instead of once per
// stencil use.  Same operands, in the same order, as kb_outer_resid, so the same values.
constexpr int kOzX = 32, kOzY = 8;

template <typename Te, bool UPD>
__global__ void __launch_bounds__(kOzX * kOzY)
kb_outer_resid_z(BL<Te> L, int total, const Outer *O, int parity, int ce, int zc, double *pmax, double *psum)
{
    constexpr int TX = kOzX, TY = kOzY, SP = TX + 2;
    __shared__ double sp[2][(TY + 2) * SP];
    Cell<Te> c;
    // XCD-aware numbering: neighbouring patches (consecutive in x) share an XCD, so the cache
    // lines an x-halo cell pulls in are the ones its neighbour loads anyway
    const int wb = xcd_block(total);
    if (!locate(L, wb, c)) return;   // uniform per workgroup
    const PL<Te> &q = *c.q;
    const int p = c.it->p, n = q.n;
    const double *pin = parity ? O->alt[p] : O->psi[p];
    double *pout = parity ? O->psi[p] : O->alt[p];
    const Te *e = q.a[q.lc == 0 ? CU : ce];
    const double *f = O->src[p];
    Te *r = q.a[CRHS];
    const int nbx = n / TX, nby = n / TY;
    const int bx = c.lb % nbx, by = (c.lb / nbx) % nby, bz = c.lb / (nbx * nby);
    const int tx = (int)threadIdx.x % TX, ty = (int)threadIdx.x / TX;
    const int i = bx * TX + tx, j = by * TY + ty, z0 = bz * zc;
    auto at = [&](int ii, int jj, int kk) { return (kk * n + jj) * n + ii; };
    auto wrapz = [&](int a) { return a < 0 ? a + n : (a >= n ? a - n : a); };
    auto P = [&](int x) -> double { return UPD ? pin[x] + (double)e[x] : pin[x]; };
    const bool hx = tx == 0 || tx == TX - 1, hy = ty == 0 || ty == TY - 1;
    const int ih = tx == 0 ? wrapz(i - 1) : wrapz(i + 1), jh = ty == 0 ? wrapz(j - 1) : wrapz(j + 1);
    const int sx = tx == 0 ? (ty + 1) * SP : (ty + 1) * SP + TX + 1;
    const int sy = ty == 0 ? tx + 1 : (TY + 1) * SP + tx + 1;
    const int sc = (ty + 1) * SP + tx + 1;
    double zm = P(at(i, j, wrapz(z0 - 1))), zcen = P(at(i, j, z0));
    double vx = hx ? P(at(ih, j, z0)) : 0.0, vy = hy ? P(at(i, jh, z0)) : 0.0;
    double fc = f[at(i, j, z0)];
    double mx = 0.0, sm = 0.0;
    for (int k = z0; k < z0 + zc; ++k) {
        double *s = sp[k & 1];
        s[sc] = zcen;
        if (hx) s[sx] = vx;
        if (hy) s[sy] = vy;
        const int kn = wrapz(k + 1);
        const double zp = P(at(i, j, kn));
        double vxn = 0.0, vyn = 0.0, fn = 0.0;
        if (k + 1 < z0 + zc) {
            if (hx) vxn = P(at(ih, j, kn));
            if (hy) vyn = P(at(i, jh, kn));
            fn = f[at(i, j, kn)];
        }
        const int cc = at(i, j, k);
        __syncthreads();
        const double rv = resid_value<double>(zcen, s[sc + 1], s[sc - 1], s[sc + SP], s[sc - SP], zp, zm, fc, O->h2i[p]);
        r[cc] = (Te)rv;
        if (UPD) pout[cc] = zcen;
        mx = fmax(mx, fabs(rv));
        sm += rv * rv;
        zm = zcen;
        zcen = zp;
        vx = vxn;
        vy = vyn;
        fc = fn;
    }
    block_max_sum(mx, sm);
    if (threadIdx.x == 0) { pmax[wb] = mx; psum[wb] = sm; }
}

// Per-problem second stage of a norm: workgroup w reduces item w's partials in order.
__global__ void __launch_bounds__(1024) kb_norm_final(const Item *items, const int *active, const double *pmax,
                                                     const double *psum, double *out)
{
    const Item it = items[blockIdx.x];
    if (!active[it.p]) return;
    double mx = 0.0, sm = 0.0;
    for (int q = threadIdx.x; q < it.nblk; q += blockDim.x) {
        mx = fmax(mx, pmax[it.blk0 + q]);
        sm += psum[it.blk0 + q];
    }
    block_max_sum(mx, sm);
    if (threadIdx.x == 0) { out[2 * it.p] = mx; out[2 * it.p + 1] = sm; }
}

// ---- fused inner solve (FP32: mixed, FP64: plain) -----------------------------------------------------------------

// The coarse array of level l + 1 that a level-l kernel reads: U where l + 1 is the level of the problem's
// coarse-grid solve, else the fused sweeps' current buffer `cur` (that of the problems whose bottom lies below).
template <typename T> __device__ __forceinline__ const T *coarse_src(const BL<T> &L, const PL<T> &q, int l, int cur)
{
    const PL<T> &qc = *(&q + 1);
    return qc.a[(l + 1 == (L.exact ? q.lb : q.lc)) ? CU : cur];
}

// ns fused sweeps of level l of every item (the fused sweep body of the single-grid solver).
template <class TL, int NS, bool ZERO, bool PROLONG, bool RESID, bool FS, typename T>
__global__ void __launch_bounds__(TL::NT) kb_sweep(BL<T> L, int total, int cin, int cout, int cuc)
{
    Cell<T> c;
    if (!locate(L, xcd_block(total), c)) return;
    const PL<T> &q = *c.q;
    const int l = c.it->l;
    sweep_tile<TL, NS, ZERO, PROLONG, RESID, FS, T>(q.a[cin], q.a[cout], q.a[CRHS], q.n, q.h2, q.h2i,
                                                 PROLONG ? coarse_src(L, q, l, cuc) : nullptr,
                                                 RESID ? (&q + 1)->a[CRHS] : nullptr, nullptr, c.lb);
}

// The streaming form of the same sweeps.
template <class SS, int NS, bool ZERO, bool PROLONG, bool RESID, typename T>
__global__ void __launch_bounds__((StreamGeom<SS, NS, PROLONG, RESID, T>::NT))
kb_stream(BL<T> L, int total, int cin, int cout, int cuc)
{
    Cell<T> c;
    if (!locate(L, xcd_block(total), c)) return;
    const PL<T> &q = *c.q;
    const int l = c.it->l;
    sweep_stream<SS, NS, ZERO, PROLONG, RESID, T>(q.a[cin], q.a[cout], q.a[CRHS], q.n, q.h2, q.h2i,
                                           PROLONG ? coarse_src(L, q, l, cuc) : nullptr,
                                           RESID ? (&q + 1)->a[CRHS] : nullptr, nullptr, c.lb);
}

// FMG tricubic prolongation into U of level l from level l + 1 (tile body of the single-grid
// solver).
template <int FX, int FY, int FZ, int NT, typename T>
__global__ void __launch_bounds__(NT) kb_interp_cubic_tile(BL<T> L, int total, int cuc)
{
    Cell<T> c;
    if (!locate(L, xcd_block(total), c)) return;
    const PL<T> &q = *c.q;
    interp_cubic_tile<FX, FY, FZ, NT, T>(q.a[CU], coarse_src(L, q, c.it->l, cuc), q.n, c.lb);
}

// Levels of <= 16^3 cells of one problem, resident in one workgroup's LDS (coarse_levels.h).
template <typename T> struct CoarseDesc {
    int n;                  // width of the first held level
    CoarseCoef<T> coef;
    int exact;              // it lies below the problem's level 0: exact solve available (FP32)
    float qx[kCoarseMaxN * kCoarseMaxN], lamx[kCoarseMaxN];  // its Hartley basis and eigenvalues
    const float *qp, *invp; // plane-parallel exact solve of the problem's bottom level (n <= 64):
                            // Hartley basis and 1 / Lambda (device), or null
};

// One workgroup per item (level l = the problem's first coarse level, <= 16^3 cells).  mode 0: FMG over
// the held levels from level 0's RHS (mg.F90:142-215 restricted to them); mode 1: one V-cycle from
// held level 0 with zero initial guess (mg.F90:179-210).  One launch for all widths: each is a kernel
// body of its own, and the problems run side by side.
template <typename T>
__global__ void __launch_bounds__(kCoarseThreads)
kb_coarse(BL<T> L, const CoarseDesc<T> *descs, int mode, int ncycle, int npre, int npost)
{
    Cell<T> c;
    if (!locate(L, (int)blockIdx.x, c)) return;
    __shared__ CoarseLds<T> S;
    const CoarseDesc<T> &D = descs[c.it->p];
    const T *f = c.q->a[CRHS];
    T *u = c.q->a[CU];
    switch (D.n) {
    case 16: coarse_solve<T, 16>(S, D.coef, f, u, mode, ncycle, npre, npost); break;
    case 12: coarse_solve<T, 12>(S, D.coef, f, u, mode, ncycle, npre, npost); break;
    case 8: coarse_solve<T, 8>(S, D.coef, f, u, mode, ncycle, npre, npost); break;
    case 6: coarse_solve<T, 6>(S, D.coef, f, u, mode, ncycle, npre, npost); break;
    case 4: coarse_solve<T, 4>(S, D.coef, f, u, mode, ncycle, npre, npost); break;
    case 3: coarse_solve<T, 3>(S, D.coef, f, u, mode, ncycle, npre, npost); break;
    default: coarse_solve<T, 2>(S, D.coef, f, u, mode, ncycle, npre, npost); break;
    }
}

// The exact solve of the first held level (coarse_exact) of every item.
static __global__ void __launch_bounds__(kCoarseExactThreads) kb_coarse_exact(BL<float> L, const CoarseDesc<float> *descs)
{
    Cell<float> c;
    if (!locate(L, (int)blockIdx.x, c)) return;
    const CoarseDesc<float> &D = descs[c.it->p];
    __shared__ float g[kCoarseMaxN * kCoarseMaxN * (kCoarseMaxN + 1)], q[kCoarseMaxN * kCoarseMaxN + kCoarseMaxN];
    coarse_exact(g, q, D.qx, D.lamx, c.q->a[CRHS], c.q->a[CU], D.n);
}

// Plane-parallel exact solve (exact_planes.h, whole form) of each item's level: workgroup b of an
// item works on plane (k_exact_xy) or row (k_exact_z) b of that problem's level.
__global__ void __launch_bounds__(kPlaneThreads) kb_exact_xy(BL<float> L, int total, const CoarseDesc<float> *descs, int cin,
                                                             int cout)
{
    Cell<float> c;
    if (!locate(L, xcd_block(total), c)) return;
    exact_xy(c.q->a[cin], c.q->a[cout], descs[c.it->p].qp, c.q->n, c.lb);
}

__global__ void __launch_bounds__(kPlaneThreads) kb_exact_z(BL<float> L, int total, const CoarseDesc<float> *descs, int cw)
{
    Cell<float> c;
    if (!locate(L, xcd_block(total), c)) return;
    const CoarseDesc<float> &D = descs[c.it->p];
    exact_z(c.q->a[cw], D.qp, D.invp, c.q->n, c.lb);
}

} // namespace batch
} // namespace sg
