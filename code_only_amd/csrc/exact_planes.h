// Exact solve of a periodic level of n^3 cells (n <= 64) spread over the chip, for the FP32 inner
// solve of the mixed-precision path: the coarse-grid problem L u = f that the V-cycles below this
// level approximate (mg.F90:142-210) is solved exactly instead.
//
// The 7-point operator separates; the symmetric orthonormal Hartley basis Q of the periodic second
// difference, Q[m n + k] = (cos a + sin a) / sqrt(n), a = 2 pi ((m k) mod n) / n, diagonalises it
// along each axis with eigenvalues lam[m] = (2 cos(2 pi m / n) - 2) / h^2, so
//     u = Q_xyz (Lambda^-1 (Q_xyz f)),  Lambda = (lam_i + lam_j) + lam_k,
// the zero mode set to zero (the zero-mean solution).  Three launches:
//   xy  (plane k):  x pass, then y pass             f -> w
//   z   (row j):    z pass, times 1 / Lambda, z pass w -> w
//   xy  (plane k):  x pass, then y pass             w -> u
//
// Sixteen lines to sixteen frequencies are one 16 x 16 tile of a matrix product, formed by one wavefront
// on the matrix cores in FP32 (v_mfma_f32_16x16x4f32, FP32 products and sums).  Lane group g = lane / 16
// holds the values k = 16 c + 4 g + r of its row, one 16-byte load per c, and instruction (c, r) adds the
// four products k = 16 c + 4 g + r.  The instructions of one tile are independent chains of two (ep_tile),
// added pairwise: four times shorter sums than one chain per half line, and a smaller error.  The division
// by Lambda is a product with 1 / Lambda, tabulated once per level (formed in double precision, zero for
// the zero mode).  A width that is no multiple of 16 (24) is padded with zeros.
//
// Q and the lines go from global memory straight into the registers that feed the matrix cores; only the
// plane between two passes goes through LDS.  Two launch forms of the same tiles, so the same bits:
// * whole (the batched solver): one workgroup of four wavefronts per plane (row); wavefront w takes the
//   lines 16 w .. 16 w + 15 to all frequencies, then the outputs 16 w .. of the second pass.  Bound by
//   latency: the launch's 1 712 planes (32 us) are on the chip at once, each one chain load, product, LDS,
//   product, store; counters find the wavefronts waiting 45 % of their cycles and the matrix cores busy 25 %
//   of the launch (8 us).
// * split (k_exact_*_split; the single-grid solver): n / 16 workgroups per plane (row), each with 16 of
//   the first transform's frequencies (columns), which it takes through both passes alone.  Bound by the
//   launch and the chain load, product, LDS, product, store: one level's n planes alone would leave most
//   of the chip idle.
// Measured against multiply-add chains over lines and Q staged in LDS: split, 64^3, three launches 24.1
// -> 14.7 us; whole, the 48-problem batch, per launch (average over its plane counts) xy 27.3 -> 20.3 and
// z 31.7 -> 20.6 us.  Root mean square error of the solution against 64-bit sums, n = 64: 2.7 .. 4.2e-7 ->
// 1.5 .. 2.4e-7 (n = 24, 32, 48: 1.7 .. 3.0e-7 -> 0.8 .. 2.0e-7).
#pragma once
#include <hip/hip_runtime.h>

namespace sg {

constexpr int kPlaneMaxN = 64;
constexpr int kPlaneThreads = 256;
constexpr int kPlanePitch = kPlaneMaxN + 4;   // rows of 272 bytes: 16-byte accesses of 16 rows spread over the banks
constexpr int kPlaneChunks = kPlaneMaxN / 16;

typedef float ep_v4 __attribute__((ext_vector_type(4)));

// Workgroups per plane (row) of the split form, each owning 16 frequencies: n % 16 == 0.
__host__ __device__ constexpr int plane_groups(int n) { return n / 16; }

// lane's operand of the 16 rows from row0 of M (row-major, `pitch` floats per row, n x n valid): its row
// row0 + lane % 16, values k = 16 c + 4 (lane / 16) + r in o[c][r]
__device__ __forceinline__ void ep_rows(ep_v4 (&o)[kPlaneChunks], const float *M, int pitch, int row0, int n)
{
    const int lane = (int)threadIdx.x % 64, row = row0 + lane % 16, k0 = 4 * (lane / 16);
#pragma unroll
    for (int c = 0; c < kPlaneChunks; ++c) {
        const int k = 16 * c + k0;
        o[c] = ep_v4{0.f, 0.f, 0.f, 0.f};
        if (row < n && k < n) o[c] = *reinterpret_cast<const ep_v4 *>(M + (long)row * pitch + k);
    }
}

// tile[4 (lane / 16) + r][lane % 16] = sum_k a-row[..] b-row[lane % 16] over the operands' k: two chains
// per 16 values of k, (c, r < 2) and (c, r >= 2), added pairwise
__device__ __forceinline__ ep_v4 ep_tile(const ep_v4 (&a)[kPlaneChunks], const ep_v4 (&b)[kPlaneChunks])
{
    ep_v4 s[kPlaneChunks][2];
#pragma unroll
    for (int c = 0; c < kPlaneChunks; ++c) s[c][0] = s[c][1] = ep_v4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int r = 0; r < 2; ++r)
#pragma unroll
        for (int c = 0; c < kPlaneChunks; ++c)
#pragma unroll
            for (int h = 0; h < 2; ++h)
                s[c][h] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[c][2 * h + r], b[c][2 * h + r], s[c][h], 0, 0, 0);
    static_assert(kPlaneChunks == 4, "the sum below");
    return ((s[0][0] + s[0][1]) + (s[1][0] + s[1][1])) + ((s[2][0] + s[2][1]) + (s[3][0] + s[3][1]));
}

// lane's operand of 16 columns of the (k, i) plane of row j: its column i, values w[k][j][i]
__device__ __forceinline__ void ep_column(ep_v4 (&o)[kPlaneChunks], const float *w, int j, int i, int n)
{
    const int k0 = 4 * ((int)threadIdx.x % 64 / 16);
    const long nn = (long)n * n;
#pragma unroll
    for (int c = 0; c < kPlaneChunks; ++c) {
        const int k = 16 * c + k0;
        o[c] = ep_v4{0.f, 0.f, 0.f, 0.f};
        if (i < n && k < n) {
            const float *p = w + k * nn + (long)j * n + i;
            o[c] = ep_v4{p[0], p[nn], p[2 * nn], p[3 * nn]};
        }
    }
}

// x pass of lines j0 .. j0 + 15 to the frequencies mi0 ..: Xs[mi][j] (rows of kPlanePitch)
__device__ __forceinline__ void ep_x(float *Xs, const ep_v4 (&line)[kPlaneChunks], const float *Q, int n, int j0, int mi0,
                                     int xrow0)
{
    const int lane = (int)threadIdx.x % 64;
    ep_v4 q[kPlaneChunks];
    ep_rows(q, Q, n, mi0, n);
    const ep_v4 v = ep_tile(line, q);   // rows j, column mi
    *reinterpret_cast<ep_v4 *>(Xs + (xrow0 + lane % 16) * kPlanePitch + j0 + 4 * (lane / 16)) = v;
}

// Plane k = `plane` of the dense n^3 array in (i fastest): x pass then y pass, into out.
__device__ __forceinline__ void exact_xy(const float *__restrict__ in, float *__restrict__ out, const float *Q, int n,
                                         int plane)
{
    __shared__ __align__(16) float Xs[kPlaneMaxN * kPlanePitch];
    const int wave = (int)threadIdx.x / 64, lane = (int)threadIdx.x % 64, nt = (n + 15) / 16;
    const long base = (long)plane * n * n;
    ep_v4 line[kPlaneChunks], q[kPlaneChunks];
    if (wave < nt) {
        ep_rows(line, in + base, n, 16 * wave, n);
        ep_rows(q, Q, n, 16 * wave, n);   // the y pass's frequencies, ahead
        for (int t = 0; t < nt; ++t) ep_x(Xs, line, Q, n, 16 * wave, 16 * t, 16 * t);
    }
    __syncthreads();
    if (wave >= nt) return;
    for (int t = 0; t < nt; ++t) {
        ep_v4 x[kPlaneChunks];
        ep_rows(x, Xs, kPlanePitch, 16 * t, 16 * nt);
        const ep_v4 v = ep_tile(q, x);   // rows mj, column mi
        const int mi = 16 * t + lane % 16, mj = 16 * wave + 4 * (lane / 16);
        if (mi < n && mj < n)
#pragma unroll
            for (int r = 0; r < 4; ++r) out[base + (long)(mj + r) * n + mi] = v[r];
    }
}

// Row j of the dense n^3 array w: the (k, i) plane, z pass, product with 1 / Lambda (inv, dense n^3 like
// w), z pass, back into w.
__device__ __forceinline__ void exact_z(float *__restrict__ w, const float *Q, const float *inv, int n, int j)
{
    __shared__ __align__(16) float Zs[kPlaneMaxN * kPlanePitch];   // [i][mk]
    const int wave = (int)threadIdx.x / 64, lane = (int)threadIdx.x % 64, nt = (n + 15) / 16;
    const long nn = (long)n * n;
    const int m0 = 16 * wave + 4 * (lane / 16);
    ep_v4 q[kPlaneChunks];
    if (wave < nt) {
        ep_rows(q, Q, n, 16 * wave, n);   // frequencies of the first pass, outputs of the second
        for (int t = 0; t < nt; ++t) {
            const int i = 16 * t + lane % 16;
            ep_v4 col[kPlaneChunks], d = {0.f, 0.f, 0.f, 0.f};
            ep_column(col, w, j, i, n);
            if (i < n && m0 < n)
#pragma unroll
                for (int r = 0; r < 4; ++r) d[r] = inv[(m0 + r) * nn + (long)j * n + i];
            const ep_v4 v = ep_tile(q, col);   // rows mk, column i
            *reinterpret_cast<ep_v4 *>(Zs + i * kPlanePitch + m0) = ep_v4{v[0] * d[0], v[1] * d[1], v[2] * d[2], v[3] * d[3]};
        }
    }
    __syncthreads();
    if (wave >= nt) return;
    for (int t = 0; t < nt; ++t) {
        ep_v4 z[kPlaneChunks];
        ep_rows(z, Zs, kPlanePitch, 16 * t, 16 * nt);
        const ep_v4 v = ep_tile(q, z);   // rows k, column i
        const int i = 16 * t + lane % 16;
        if (i < n && m0 < n)
#pragma unroll
            for (int r = 0; r < 4; ++r) w[(m0 + r) * nn + (long)j * n + i] = v[r];
    }
}

// Workgroup wg = plane * G + g, G = plane_groups(n): the x frequencies 16 g .. 16 g + 15 of the plane
// through the x and y passes.
__device__ __forceinline__ void exact_xy_split(const float *__restrict__ in, float *__restrict__ out, const float *Q,
                                               int n, int wg)
{
    __shared__ __align__(16) float Xs[16 * kPlanePitch];
    const int wave = (int)threadIdx.x / 64, lane = (int)threadIdx.x % 64, nt = n / 16;
    const int G = plane_groups(n), plane = wg / G, g = wg % G;
    const long base = (long)plane * n * n;
    ep_v4 line[kPlaneChunks], q[kPlaneChunks], x[kPlaneChunks];
    if (wave < nt) {
        ep_rows(line, in + base, n, 16 * wave, n);
        ep_rows(q, Q, n, 16 * wave, n);
        ep_x(Xs, line, Q, n, 16 * wave, 16 * g, 0);
    }
    __syncthreads();
    if (wave >= nt) return;
    ep_rows(x, Xs, kPlanePitch, 0, 16 * nt);
    const ep_v4 v = ep_tile(q, x);
    const int mi = 16 * g + lane % 16, mj = 16 * wave + 4 * (lane / 16);
#pragma unroll
    for (int r = 0; r < 4; ++r) out[base + (long)(mj + r) * n + mi] = v[r];
}

// Workgroup wg = row * G + g: the columns 16 g .. 16 g + 15 of row j through both z passes, in place.
__device__ __forceinline__ void exact_z_split(float *__restrict__ w, const float *Q, const float *inv, int n, int wg)
{
    __shared__ __align__(16) float Zs[16 * kPlanePitch];   // [i][mk]
    const int wave = (int)threadIdx.x / 64, lane = (int)threadIdx.x % 64, nt = n / 16;
    const int G = plane_groups(n), j = wg / G, i = 16 * (wg % G) + lane % 16;
    const long nn = (long)n * n;
    const int m0 = 16 * wave + 4 * (lane / 16);
    ep_v4 q[kPlaneChunks], z[kPlaneChunks];
    if (wave < nt) {
        ep_v4 col[kPlaneChunks], d;
        ep_column(col, w, j, i, n);
        ep_rows(q, Q, n, 16 * wave, n);
#pragma unroll
        for (int r = 0; r < 4; ++r) d[r] = inv[(m0 + r) * nn + (long)j * n + i];
        const ep_v4 v = ep_tile(q, col);
        *reinterpret_cast<ep_v4 *>(Zs + (lane % 16) * kPlanePitch + m0) =
            ep_v4{v[0] * d[0], v[1] * d[1], v[2] * d[2], v[3] * d[3]};
    }
    __syncthreads();
    if (wave >= nt) return;
    ep_rows(z, Zs, kPlanePitch, 0, 16 * nt);
    const ep_v4 v = ep_tile(q, z);
#pragma unroll
    for (int r = 0; r < 4; ++r) w[(m0 + r) * nn + (long)j * n + i] = v[r];
}

// XCD-aware numbering: the hardware deals consecutive workgroups round-robin to the 8 XCDs; the
// G workgroups of one plane (which all read that plane and Q) get consecutive numbers on one XCD.
__device__ __forceinline__ int ep_xcd_block()
{
    const int nb = (int)gridDim.x, b = (int)blockIdx.x;
    return nb % 8 == 0 ? (b % 8) * (nb / 8) + b / 8 : b;
}

static __global__ void __launch_bounds__(kPlaneThreads) k_exact_xy_split(const float *in, float *out, const float *Q,
                                                                         int n)
{
    exact_xy_split(in, out, Q, n, ep_xcd_block());
}

static __global__ void __launch_bounds__(kPlaneThreads) k_exact_z_split(float *w, const float *Q, const float *inv, int n)
{
    exact_z_split(w, Q, inv, n, ep_xcd_block());
}

// 1 / ((lam_i + lam_j) + lam_k) for the dense n^3 grid (0 where the sum is 0), host, double.
inline void exact_inverse_table(int n, const double *lam, float *inv)
{
    for (int k = 0; k < n; ++k)
        for (int j = 0; j < n; ++j)
            for (int i = 0; i < n; ++i) {
                const double den = (lam[i] + lam[j]) + lam[k];
                inv[((size_t)k * n + j) * n + i] = den != 0.0 ? (float)(1.0 / den) : 0.f;
            }
}

} // namespace sg
