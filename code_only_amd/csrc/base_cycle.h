// The base grid's mg_cycle (vmg_slvsml, vmg.F90:387-432 -> mg_cycle, mg.F90:42-94) on dense n^3 grids
// with the fused kernels of the uniform tier, periodic or with zero ghosts (coarse_levels.h): the same
// values as the one-workgroup k_base_mg (base_mg.h).
//
//  * n <= 16 (base grids of up to 8^3 blocks): k_base_small, the whole defect-correction loop with its
//    stopping test in one launch.
//  * larger: per iteration one restriction, the levels of <= 16^3 cells in k_coarse, and per V-cycle
//    visit of a finer level two launches of two fused sweeps (32^3: 64 workgroups of an 8^3 tile); the
//    host reads the stopping test's two maxima once per iteration, while the update runs.
// One iteration on 32^3 took about 30 launches (each colour, residual, ghost fill a launch of its own,
// 3-5 us) around three single-workgroup stretches of 176 us on ghosted arrays: 1.3 ms per call of two
// iterations, now 0.38 ms (sphere hierarchy of 20 480 blocks, staged FP64 solve 105 -> 82 ms); on 8^3
// 0.42 ms per call, now 0.028 ms.
#pragma once
#include "amr_kernels.h"
#include "fast_kernels.h"

namespace sg {
namespace amr {

// base block and cell of grid position (i, j, k); inv: base block number by block position
__device__ __forceinline__ long base_cell(const int *inv, int nb, int i, int j, int k)
{
    const int b = inv[((k >> 1) * nb + (j >> 1)) * nb + (i >> 1)];
    return (long)b * Blk<2>::LEN + Blk<2>::gi(i & 1, j & 1, k & 1);
}

template <int N, bool ZERO>
__global__ void __launch_bounds__(kCoarseThreads)
k_base_small(double *Au, const double *__restrict__ Arhs, const int *__restrict__ inv, CoarseCoef<double> P, double h,
             double tol, int maxit)
{
    using L = CoarseLevel<N>;
    constexpr int IT = (L::len + kCoarseThreads - 1) / kCoarseThreads;
    __shared__ CoarseLds<double> S;
    __shared__ double psi[L::len];
    __shared__ double s_max[2];   // max|residual| of the first iteration, max|resh2| of the last sweep
    double src[IT];
    long cell[IT];
#pragma unroll
    for (int m = 0; m < IT; ++m) {
        const int c = (int)threadIdx.x + m * kCoarseThreads;
        src[m] = 0.0;
        cell[m] = 0;
        if (L::len % kCoarseThreads == 0 || c < L::len) {
            int i, j, k;
            L::decode(c, i, j, k);
            cell[m] = base_cell(inv, N / 2, i, j, k);
            psi[L::at(i, j, k)] = Au[cell[m]];
            src[m] = Arhs[cell[m]];
        }
    }
    if (threadIdx.x >= kCoarseThreads - 64) coarse_tables<double, N, ZERO>(S, (int)threadIdx.x - (kCoarseThreads - 64));
    if (threadIdx.x == 0) s_max[0] = 0.0;
    __syncthreads();
    for (int it = 0;;) {
        double mx = 0.0;
#pragma unroll
        for (int m = 0; m < IT; ++m) {
            const int c = (int)threadIdx.x + m * kCoarseThreads;
            if (L::len % kCoarseThreads == 0 || c < L::len) {
                int i, j, k;
                L::decode(c, i, j, k);
                auto U = [&](int a, int b, int d) -> double {
                    if (ZERO && (a < 0 || a >= N || b < 0 || b >= N || d < 0 || d >= N)) return 0.0;
                    return psi[L::at((a + N) % N, (b + N) % N, (d + N) % N)];
                };
                const double r = resid_value<double>(U(i, j, k), U(i + 1, j, k), U(i - 1, j, k), U(i, j + 1, k), U(i, j - 1, k),
                                                     U(i, j, k + 1), U(i, j, k - 1), src[m], P.h2i[0]);
                S.r[L::off + L::at(i, j, k)] = r;
                mx = fmax(mx, fabs(r));
            }
        }
        if (it >= maxit) break;
        if (it == 0) block_atomic_max(&s_max[0], mx);
        if (threadIdx.x == 0) s_max[1] = 0.0;
        __syncthreads();
        coarse_run<double, N, ZERO>(S, P, true, 2, 2, 2, &s_max[1]);
        __syncthreads();
#pragma unroll
        for (int m = 0; m < IT; ++m) {
            const int c = (int)threadIdx.x + m * kCoarseThreads;
            if (L::len % kCoarseThreads == 0 || c < L::len) psi[c] = psi[c] + S.u[L::off + c];
        }
        const double rhomax = s_max[0], resmaxg = s_max[1] / (h * h);
        __syncthreads();
        ++it;
        if ((rhomax > 0 ? resmaxg / rhomax : 0.0) < tol) break;
    }
#pragma unroll
    for (int m = 0; m < IT; ++m) {
        const int c = (int)threadIdx.x + m * kCoarseThreads;
        if (L::len % kCoarseThreads == 0 || c < L::len) {
            int i, j, k;
            L::decode(c, i, j, k);
            Au[cell[m]] = psi[L::at(i, j, k)];
        }
    }
}

// base blocks -> dense grids, the two maxima cleared
static __global__ void k_base_in(double *psi, double *src, const double *Au, const double *Arhs, const int *inv, int n,
                                 double *acc)
{
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t < 2) acc[t] = 0.0;
    if (t >= n * n * n) return;
    const long q = base_cell(inv, n / 2, t % n, (t / n) % n, t / (n * n));
    psi[t] = Au[q];
    src[t] = Arhs[q];
}

static __global__ void k_base_out(double *Au, const double *psi, const int *inv, int n)
{
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t < n * n * n) Au[base_cell(inv, n / 2, t % n, (t / n) % n, t / (n * n))] = psi[t];
}

// psi_out = psi_in + e (UPD) and r = src - L psi_out; amax (nullable) receives max|r|
template <bool UPD, bool ZERO>
__global__ void __launch_bounds__(256) k_base_resid(const double *__restrict__ pin, const double *__restrict__ e,
                                                    double *__restrict__ pout, const double *__restrict__ src,
                                                    double *__restrict__ r, int n, double h2i, double *amax)
{
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    double m = 0.0;
    if (t < n * n * n) {
        const int i = t % n, j = (t / n) % n, k = t / (n * n);
        auto U = [&](int a, int b, int d) -> double {
            if (ZERO && (a < 0 || a >= n || b < 0 || b >= n || d < 0 || d >= n)) return 0.0;
            const int q = (wrapn(d, n) * n + wrapn(b, n)) * n + wrapn(a, n);
            return UPD ? pin[q] + e[q] : pin[q];
        };
        const double c = U(i, j, k);
        const double v = resid_value<double>(c, U(i + 1, j, k), U(i - 1, j, k), U(i, j + 1, k), U(i, j - 1, k),
                                             U(i, j, k + 1), U(i, j, k - 1), src[t], h2i);
        if (UPD) pout[t] = c;
        r[t] = v;
        m = fabs(v);
    }
    if (amax) block_atomic_max(amax, m);
}

// the two maxima into pinned host memory; the sweep's is cleared for the next iteration
static __global__ void k_base_publish(double *acc, double *host)
{
    host[0] = acc[0];
    host[1] = acc[1];
    acc[1] = 0.0;
}

} // namespace amr
} // namespace sg
