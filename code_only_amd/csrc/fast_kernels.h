// Fused kernels of the inner solve (gfx950), in FP32 (mixed precision) and FP64 (plain).
//
//  * k_sweep_tile: one full red-black sweep (mg_poisson.F90:55-74, both colours) of a TX*TY*TZ
//    tile held in LDS with an H-cell halo, optionally
//      - starting from u = 0 (the zero fill of mg.F90:189 folded into the load),
//      - adding the trilinear coarse-grid correction on load (mg_addint, mg.F90:727-731), the
//        coarse tile staged in LDS first,
//      - finishing with the residual (mg_poisson.F90:17-27) restricted to the coarse grid
//        (restriction.F90:132-147), which needs H = 3.
//    Reads u from one buffer and writes the tile core to another: a workgroup's halo is then
//    never a value another workgroup has already updated.  The redundant halo updates repeat the
//    owner's arithmetic exactly, so the result equals the two-launch colour sweep bit for bit.
//    Tile shape and workgroup size are template parameters; the host picks one per level size by
//    timing (all shapes give identical values).
//  * k_sweep_stream: the same, two sweeps per launch, marching up a column (pair_stream.h).
//  * k_interp_cubic_tile: the FMG tricubic prolongation (interpolation.F90:98-217) as the
//    reference's three separable passes, on an LDS-staged coarse tile.
//  * k_coarse: every level of <= 16^3 cells in one workgroup's LDS (coarse_levels.h): the FMG part of
//    mg_lin (mg.F90:142-215) from the coarsest level up to the first fine level, or one V-cycle from
//    that level down and back (the bottom of each fine-level V-cycle); k_coarse_exact: in both places,
//    the exact solve of the first level of <= 16^3 cells by Hartley transforms (coarse_exact).
//
// Every cell value is produced by the same helpers (relax_value, resid_value, restrict_value,
// trilinear_value, cubic_stencil) as the one-kernel-per-loop path, in the same order, so the fused
// solve reproduces the unfused FP32 solve exactly.
#pragma once
#include <cmath>

#include "coarse_levels.h"
#include "pair_stream.h"
#include "uniform_kernels.h"

namespace sg {

template <int TX_, int TY_, int TZ_, int NT_> struct Tile {
    static constexpr int TX = TX_, TY = TY_, TZ = TZ_, NT = NT_;
};

// Tile shapes the autotuners choose from (all give identical values), each with 1 or 2 sweeps
// per launch.
using Tile0 = Tile<32, 16, 16, 1024>;
using Tile1 = Tile<16, 8, 8, 1024>;
using Tile2 = Tile<16, 8, 8, 256>;
using Tile3 = Tile<64, 8, 8, 512>;
using Tile4 = Tile<8, 8, 8, 512>;
constexpr int kNumTiles = 5;
constexpr int kMaxSweepsPerLaunch = 2;
static const int kTileDims[kNumTiles][4] = {
    {32, 16, 16, 1024}, {16, 8, 8, 1024}, {16, 8, 8, 256}, {64, 8, 8, 512}, {8, 8, 8, 512}};

inline bool tile_fits(int cfg, int n)
{
    const int *d = kTileDims[cfg];
    return n >= d[0] && n >= d[1] && n >= d[2] && n % d[0] == 0 && n % d[1] == 0 && n % d[2] == 0;
}

// One colour of the sweep over the LDS region shrunk by margin M: cells with
// (gx + gy + gz) % 2 == colour, where colour 1 is the reference's first pass (ipass = 1).  The
// source values are fetched for all of a thread's cells before any update.
template <class TL, int LX, int LY, int LZ, int M, int H, bool FS, typename T, bool ZB>
__device__ __forceinline__ void tile_colour(T *su, const T *sf, const T *__restrict__ f, int n, int x0,
                                            int y0, int z0, int colour, T h2, double &amax)
{
    constexpr int RX = (LX - 2 * M) / 2, RY = LY - 2 * M, RZ = LZ - 2 * M;
    constexpr int CNT = RX * RY * RZ;
    constexpr int IT = (CNT + TL::NT - 1) / TL::NT;
    static_assert((LX - 2 * M) % 2 == 0, "region x extent must be even");
    static_assert(IT <= 32, "too many cells per thread");
    T fv[IT];
    int cv[IT];
    unsigned core = 0u;
#pragma unroll
    for (int it = 0; it < IT; ++it) {
        const int q = threadIdx.x + it * TL::NT;
        cv[it] = -1;
        fv[it] = T(0);
        if (CNT % TL::NT == 0 || q < CNT) {
            const int xh = q % RX;
            const int y = M + (q / RX) % RY;
            const int z = M + q / (RX * RY);
            const int d = (colour + x0 + M + y0 + y + z0 + z) & 1;
            const int x = M + 2 * xh + d;
            cv[it] = (z * LY + y) * LX + x;
            if (ZB && ((unsigned)(x0 + x) >= (unsigned)n || (unsigned)(y0 + y) >= (unsigned)n ||
                       (unsigned)(z0 + z) >= (unsigned)n)) {
                cv[it] = -1;
                continue;
            }
            if (x >= H && x < H + TL::TX && y >= H && y < H + TL::TY && z >= H && z < H + TL::TZ) core |= 1u << it;
            if (FS) {
                fv[it] = sf[cv[it]];
            } else {
                const int gi = wrapn(x0 + x, n), gj = wrapn(y0 + y, n), gk = wrapn(z0 + z, n);
                fv[it] = f[(gk * n + gj) * n + gi];
            }
        }
    }
#pragma unroll
    for (int it = 0; it < IT; ++it) {
        const int c = cv[it];
        if (c >= 0) {
            T s;
            su[c] = relax_value<T>(su[c], su[c + 1], su[c - 1], su[c + LX], su[c - LX], su[c + LX * LY],
                                   su[c - LX * LY], fv[it], h2, &s);
            if (core & (1u << it)) amax = fmax(amax, fabs((double)s));
        }
    }
}

// Sweeps S .. NS-1 of a multi-sweep tile: sweep s updates the first colour on margin 2s+1 and the
// second on margin 2s+2.  Only the last sweep feeds the max|resh2| (one mg_relax call's Resmaxg).
template <class TL, int LX, int LY, int LZ, int H, int S, int NS, bool FS, typename T, bool ZB> struct TileSweeps {
    static __device__ __forceinline__ void run(T *su, const T *sf, const T *__restrict__ f, int n, int x0,
                                               int y0, int z0, T h2, double &amax)
    {
        double dummy = 0.0;
        double &acc = (S == NS - 1) ? amax : dummy;
        tile_colour<TL, LX, LY, LZ, 2 * S + 1, H, FS, T, ZB>(su, sf, f, n, x0, y0, z0, 1, h2, acc);
        __syncthreads();
        tile_colour<TL, LX, LY, LZ, 2 * S + 2, H, FS, T, ZB>(su, sf, f, n, x0, y0, z0, 0, h2, acc);
        __syncthreads();
        TileSweeps<TL, LX, LY, LZ, H, S + 1, NS, FS, T, ZB>::run(su, sf, f, n, x0, y0, z0, h2, amax);
    }
};
template <class TL, int LX, int LY, int LZ, int H, int NS, bool FS, typename T, bool ZB>
struct TileSweeps<TL, LX, LY, LZ, H, NS, NS, FS, T, ZB> {
    static __device__ __forceinline__ void run(T *, const T *, const T *__restrict__, int, int, int, int, T, double &)
    {
    }
};

// LDS bytes of the largest variant of a (tile, sweeps, staging) choice: the residual variant has
// the widest halo, the prolongation variant adds the staged coarse tile.
template <class TL, int NS, bool FS, typename T = float> constexpr int sweep_lds_bytes()
{
    constexpr int H1 = 2 * NS + 1, H2 = 2 * NS;
    constexpr int r1 = (TL::TX + 2 * H1) * (TL::TY + 2 * H1) * (TL::TZ + 2 * H1) * (FS ? 2 : 1);
    constexpr int r2 = (TL::TX + 2 * H2) * (TL::TY + 2 * H2) * (TL::TZ + 2 * H2) * (FS ? 2 : 1) +
                       ((TL::TX + 2 * H2) / 2 + 2) * ((TL::TY + 2 * H2) / 2 + 2) * ((TL::TZ + 2 * H2) / 2 + 2);
    return (int)sizeof(T) * (r1 > r2 ? r1 : r2) + 1024;
}
template <class TL, int NS, bool FS, typename T = float> constexpr bool sweep_fits_lds()
{
    return sweep_lds_bytes<TL, NS, FS, T>() <= 163840;
}


// NS full sweeps (temporal blocking: halo 2 per sweep, +1 for the residual).  FS stages the source
// on the same LDS region as u, loaded together with u, so the colour passes touch LDS only.
// Body of the fused sweep for tile t of an n^3 level (n even, divisible by the tile extents);
// called by every thread of a workgroup with the same t.  ZB: zero ghosts instead of periodic ones
// (coarse_levels.h): cells outside the grid hold zero and are never updated, a coarse cell outside
// its grid is the odd continuation.
template <class TL, int NS, bool ZERO, bool PROLONG, bool RESID, bool FS, typename T = float, bool ZB = false>
__device__ __forceinline__ void sweep_tile(const T *__restrict__ uin, T *__restrict__ uout,
                                           const T *__restrict__ f, int n, T h2, T h2i,
                                           const T *__restrict__ uc, T *__restrict__ rc, double *resmax, int t)
{
    constexpr int H = 2 * NS + (RESID ? 1 : 0);
    constexpr int TX = TL::TX, TY = TL::TY, TZ = TL::TZ, NT = TL::NT;
    constexpr int LX = TX + 2 * H, LY = TY + 2 * H, LZ = TZ + 2 * H;
    constexpr int CX = LX / 2 + 2, CY = LY / 2 + 2, CZ = LZ / 2 + 2;  // staged coarse region
    static_assert(!RESID || H >= 3, "residual needs a 3-cell halo");
    static_assert(H % 2 == 0 || !PROLONG, "prolongation staging assumes an even tile origin");
    __shared__ T su[LX * LY * LZ];
    __shared__ T sf[FS ? LX * LY * LZ : 1];
    __shared__ T sc[PROLONG ? CX * CY * CZ : 1];
    const int ntx = n / TX, nty = n / TY;
    const int tx = t % ntx, ty = (t / ntx) % nty, tz = t / (ntx * nty);
    const int x0 = tx * TX - H, y0 = ty * TY - H, z0 = tz * TZ - H;
    const int nc = n >> 1;

    {
        // one batch of global loads: u and (FS) the source on tile + halo, (PROLONG) the coarse
        // cells x0/2 - 1 .. x0/2 + LX/2 (x0 even) that the trilinear correction reads
        constexpr int CNT = LX * LY * LZ, IT = (CNT + NT - 1) / NT;
        constexpr int CNTC = CX * CY * CZ, ITC = PROLONG ? (CNTC + NT - 1) / NT : 1;
        T v[IT];
        T fvl[FS ? IT : 1];
        T cvl[ITC];
        if (!ZERO || FS) {
#pragma unroll
            for (int it = 0; it < IT; ++it) {
                const int q = threadIdx.x + it * NT;
                if (CNT % NT == 0 || q < CNT) {
                    const int x = q % LX, y = (q / LX) % LY, z = q / (LX * LY);
                    const int g = (wrapn(z0 + z, n) * n + wrapn(y0 + y, n)) * n + wrapn(x0 + x, n);
                    if (!ZERO) v[it] = uin[g];
                    if (!ZERO && ZB && ((unsigned)(x0 + x) >= (unsigned)n || (unsigned)(y0 + y) >= (unsigned)n ||
                                        (unsigned)(z0 + z) >= (unsigned)n))
                        v[it] = T(0);
                    if (FS) fvl[FS ? it : 0] = f[g];
                }
            }
        }
        if (PROLONG) {
            const int cx0 = x0 / 2 - 1, cy0 = y0 / 2 - 1, cz0 = z0 / 2 - 1;
#pragma unroll
            for (int it = 0; it < ITC; ++it) {
                const int q = threadIdx.x + it * NT;
                if (CNTC % NT == 0 || q < CNTC) {
                    const int x = q % CX, y = (q / CX) % CY, z = q / (CX * CY);
                    T sx, sy, sz;
                    const int a = coarse_ghost<T, ZB>(cx0 + x, nc, sx), b = coarse_ghost<T, ZB>(cy0 + y, nc, sy),
                              d = coarse_ghost<T, ZB>(cz0 + z, nc, sz);
                    cvl[it] = uc[(d * nc + b) * nc + a];
                    if (ZB) cvl[it] = (sx * sy * sz) * cvl[it];
                }
            }
#pragma unroll
            for (int it = 0; it < ITC; ++it) {
                const int q = threadIdx.x + it * NT;
                if (CNTC % NT == 0 || q < CNTC) sc[q] = cvl[it];
            }
        }
#pragma unroll
        for (int it = 0; it < IT; ++it) {
            const int q = threadIdx.x + it * NT;
            if (CNT % NT == 0 || q < CNT) {
                su[q] = ZERO ? T(0) : v[it];
                if (FS) sf[q] = fvl[FS ? it : 0];
            }
        }
    }
    __syncthreads();
    if (PROLONG) {
        // u += trilinear(coarse) on tile + halo (mg_addint, mg.F90:727-731)
        constexpr int CNT = LX * LY * LZ, IT = (CNT + NT - 1) / NT;
#pragma unroll
        for (int it = 0; it < IT; ++it) {
            const int q = threadIdx.x + it * NT;
            if (CNT % NT == 0 || q < CNT) {
                const int x = q % LX, y = (q / LX) % LY, z = q / (LX * LY);
                // local coarse index of the parent: floor(x/2) + 1; neighbour toward the cell
                const int ic = (x >> 1) + 1, jc = (y >> 1) + 1, kc = (z >> 1) + 1;
                const int ic1 = ic + 2 * (x & 1) - 1, jc1 = jc + 2 * (y & 1) - 1, kc1 = kc + 2 * (z & 1) - 1;
                auto C = [&](int a, int b, int d) { return sc[(d * CY + b) * CX + a]; };
                if (ZB && ((unsigned)(x0 + x) >= (unsigned)n || (unsigned)(y0 + y) >= (unsigned)n ||
                           (unsigned)(z0 + z) >= (unsigned)n))
                    continue;
                su[q] = su[q] + trilinear_value<T>(C(ic, jc, kc), C(ic1, jc, kc), C(ic, jc1, kc), C(ic, jc, kc1),
                                                       C(ic, jc1, kc1), C(ic1, jc, kc1), C(ic1, jc1, kc),
                                                       C(ic1, jc1, kc1));
            }
        }
        __syncthreads();
    }
    double amax = 0.0;
    TileSweeps<TL, LX, LY, LZ, H, 0, NS, FS, T, ZB>::run(su, sf, f, n, x0, y0, z0, h2, amax);
    {
        constexpr int CNT = TX * TY * TZ, IT = (CNT + NT - 1) / NT;
#pragma unroll
        for (int it = 0; it < IT; ++it) {
            const int q = threadIdx.x + it * NT;
            if (CNT % NT == 0 || q < CNT) {
                const int x = q % TX, y = (q / TX) % TY, z = q / (TX * TY);
                const int gi = x0 + H + x, gj = y0 + H + y, gk = z0 + H + z;
                uout[(gk * n + gj) * n + gi] = su[((z + H) * LY + (y + H)) * LX + (x + H)];
            }
        }
    }
    if (RESID) {
        // residual of the 8 fine cells of each coarse cell of the tile, restricted
        constexpr int QX = TX / 2, QY = TY / 2, QZ = TZ / 2;
        constexpr int CNT = QX * QY * QZ, IT = (CNT + NT - 1) / NT;
        T fv[IT][8];
#pragma unroll
        for (int it = 0; it < IT; ++it) {
            const int q = threadIdx.x + it * NT;
            if (CNT % NT == 0 || q < CNT) {
                const int cx = q % QX, cy = (q / QX) % QY, cz = q / (QX * QY);
#pragma unroll
                for (int o = 0; o < 8; ++o) {
                    const int a = o & 1, b = (o >> 1) & 1, d = (o >> 2) & 1;
                    if (FS) {
                        fv[it][o] = sf[((H + 2 * cz + d) * LY + (H + 2 * cy + b)) * LX + (H + 2 * cx + a)];
                    } else {
                        const int gi = x0 + H + 2 * cx + a, gj = y0 + H + 2 * cy + b, gk = z0 + H + 2 * cz + d;
                        fv[it][o] = f[(gk * n + gj) * n + gi];
                    }
                }
            }
        }
#pragma unroll
        for (int it = 0; it < IT; ++it) {
            const int q = threadIdx.x + it * NT;
            if (CNT % NT == 0 || q < CNT) {
                const int cx = q % QX, cy = (q / QX) % QY, cz = q / (QX * QY);
                T r[8];
#pragma unroll
                for (int o = 0; o < 8; ++o) {
                    const int a = o & 1, b = (o >> 1) & 1, d = (o >> 2) & 1;
                    const int c = ((H + 2 * cz + d) * LY + (H + 2 * cy + b)) * LX + (H + 2 * cx + a);
                    r[o] = resid_value<T>(su[c], su[c + 1], su[c - 1], su[c + LX], su[c - LX], su[c + LX * LY],
                                              su[c - LX * LY], fv[it][o], h2i);
                }
                // restriction.F90:140-143 order: 000 100 010 001 110 101 011 111
                const int gci = tx * QX + cx, gcj = ty * QY + cy, gck = tz * QZ + cz;
                rc[(gck * nc + gcj) * nc + gci] =
                    restrict_value<T>(r[0], r[1], r[2], r[4], r[3], r[5], r[6], r[7]);
            }
        }
    }
    if (resmax) block_atomic_max(resmax, amax);
}

template <class TL, int NS, bool ZERO, bool PROLONG, bool RESID, bool FS, typename T = float, bool ZB = false>
__global__ void __launch_bounds__(TL::NT)
k_sweep_tile(const T *__restrict__ uin, T *__restrict__ uout, const T *__restrict__ f, int n, T h2,
             T h2i, const T *__restrict__ uc, T *__restrict__ rc, double *resmax)
{
    const int ntiles = (n / TL::TX) * (n / TL::TY) * (n / TL::TZ);
    const int t = xcd_tile(ntiles);
    if (t >= ntiles) return;  // uniform per workgroup, before any barrier
    sweep_tile<TL, NS, ZERO, PROLONG, RESID, FS, T, ZB>(uin, uout, f, n, h2, h2i, uc, rc, resmax, t);
}

// Streaming shapes (pair_stream.h) the autotuners choose from beside the tiles, with two sweeps per launch
// (one where a single sweep is left): column SX x SY, chunk of ZC planes.  A longer chunk spends less on
// its halo planes, a shorter one makes more workgroups: 512^3 is fastest with 128 planes, 256^3 with 64.
// A shape's number is public (sg_uniform_set_tile) and fixes the widths it takes, the multiples of its
// largest extent: shapes are appended, never renumbered.  Numbers 1, 3 and 6 named shapes that are no longer
// built and run the shape of the same column family that takes the same widths (Stream0, Stream5, Stream5);
// 2 and 4 named columns of 64 x 32 and 128 x 16, whose pairs exceed a workgroup, and take their widths
// (4 also 64).
using Stream0 = StreamShape<64, 16, 32>;
using Stream2 = StreamShape<64, 16, 64>;
using Stream4 = StreamShape<32, 32, 64>;
using Stream5 = StreamShape<32, 16, 16>;
using Stream7 = StreamShape<32, 32, 32>;
using Stream8 = StreamShape<16, 16, 16>;
using Stream9 = StreamShape<64, 16, 128>;
using Stream10 = StreamShape<32, 16, 64>;
using Stream11 = StreamShape<16, 8, 8>;
constexpr int kNumStream = 12;
static const int kStreamDims[kNumStream][3] = {
    {64, 16, 32}, {64, 16, 32}, {64, 16, 64}, {32, 16, 16},  {32, 32, 64}, {32, 16, 16},
    {32, 16, 16}, {32, 32, 32}, {16, 16, 16}, {64, 16, 128}, {32, 16, 64}, {16, 8, 8}};

// sweep configurations: 0 .. kNumTiles-1 tiles, kNumTiles .. kNumTiles+kNumStream-1 streams
constexpr int kNumCfg = kNumTiles + kNumStream;
constexpr int kNumCand = kNumTiles * kMaxSweepsPerLaunch * 2 + kNumStream;
static_assert(kNumCand <= 32, "autotuner timing tables hold 32 candidates");

// whether the autotuners time configuration cfg (not the second numbers of a shape)
inline bool cfg_timed(int cfg) { return cfg != kNumTiles + 1 && cfg != kNumTiles + 3 && cfg != kNumTiles + 6; }

inline bool cfg_fits(int cfg, int n)
{
    if (cfg < kNumTiles) return tile_fits(cfg, n);
    const int *d = kStreamDims[cfg - kNumTiles];
    return n >= d[0] && n >= d[1] && n >= d[2] && n % d[0] == 0 && n % d[1] == 0 && n % d[2] == 0;
}


// Whether a sweep kernel is instantiated for T: FP32 (autotuned), every shape that fits the LDS; FP64,
// the shapes of fp64_sweep_shape.
template <class TL, int NS, bool FS, typename T> constexpr bool sweep_built()
{
    if (sizeof(T) == sizeof(float)) return sweep_fits_lds<TL, NS, FS, T>();
    return !FS && ((TL::TX == 16 && TL::NT == 1024) || TL::TX == 8);
}
template <class SS, typename T> constexpr bool stream_built()
{
    return sizeof(T) == sizeof(float) || (SS::SX == 32 && SS::SY == 16);
}
template <class SS, typename T> constexpr bool stream_built_fits()
{
    return !stream_built<SS, T>() || (StreamGeom<SS, 2, true, false, T>::fits && StreamGeom<SS, 2, false, true, T>::fits);
}
template <class TL, int NS, bool FS, typename T> constexpr bool sweep_built_fits()
{
    return !sweep_built<TL, NS, FS, T>() || sweep_fits_lds<TL, NS, FS, T>();
}
static_assert(sweep_built_fits<Tile1, 2, false, double>() && sweep_built_fits<Tile4, 2, false, double>() &&
                  stream_built_fits<Stream5, double>() && stream_built_fits<Stream10, double>(),
              "FP64 sweep shapes exceed the LDS");
static_assert(stream_built_fits<Stream0, float>() && stream_built_fits<Stream5, float>() &&
                  stream_built_fits<Stream7, float>() && stream_built_fits<Stream8, float>(),
              "FP32 streaming shapes exceed the LDS or a workgroup");

// The FP64 sweep shape of a launch, always of two sweeps where two are left, over levels whose widths are
// all multiples of `unit` (64, 32, 16 or 8) with `cells` cells in all: the largest shape that still makes
// 256 workgroups, one per CU, since a workgroup's halo costs less the larger its shape; below that the
// levels are bound by latency.  One V(2,2) visit of one grid, us: 512^3 stream 32 x 16 z64 2457 (one sweep
// per launch in 64 x 16 z64 3062); 256^3 357 (374); 128^3 stream 32 x 16 z16 55, tile 32 x 16 x 16 with
// one sweep 64; 64^3 tile 16 x 8 x 8 20.3, stream 16 x 8 z8 25.4, tile 8^3 22.1; 32^3 tile 8^3 14.6, tile
// 16 x 8 x 8 18.1.
constexpr long kSweepCUs = 256;
inline int fp64_sweep_shape(int unit, long cells)
{
    if (unit >= 64 && cells >= kSweepCUs * 32 * 16 * 64) return kNumTiles + 10;
    if (unit >= 32 && cells >= kSweepCUs * 32 * 16 * 16) return kNumTiles + 5;
    return unit >= 16 && cells >= kSweepCUs * 16 * 8 * 8 ? 1 : 4;
}

template <class TL, typename T> inline bool built(int ns, bool fs)
{
    if (ns == 2) return fs ? sweep_built<TL, 2, true, T>() : sweep_built<TL, 2, false, T>();
    return fs ? sweep_built<TL, 1, true, T>() : sweep_built<TL, 1, false, T>();
}

// whether (tile shape, sweeps per launch, staging) is instantiated
template <typename T> inline bool cand_ok(int cfg, int ns, bool fs)
{
    switch (cfg) {
    case 0: return built<Tile0, T>(ns, fs);
    case 1: return built<Tile1, T>(ns, fs);
    case 2: return built<Tile2, T>(ns, fs);
    case 3: return built<Tile3, T>(ns, fs);
    default: return built<Tile4, T>(ns, fs);
    }
}

// whether configuration cfg with (ns, fs) exists: streams hold the source in registers (fs = 0)
template <typename T> inline bool cfg_ok(int cfg, int ns, bool fs)
{
    if (cfg < kNumTiles) return cand_ok<T>(cfg, ns, fs);
    if (ns < 1 || ns > kMaxSweepsPerLaunch || fs) return false;
    switch (cfg - kNumTiles) {
    case 0:
    case 1: return stream_built<Stream0, T>();
    case 2: return stream_built<Stream2, T>();
    case 4: return stream_built<Stream4, T>();
    case 3:
    case 5:
    case 6: return stream_built<Stream5, T>();
    case 7: return stream_built<Stream7, T>();
    case 8: return stream_built<Stream8, T>();
    case 9: return stream_built<Stream9, T>();
    case 10: return stream_built<Stream10, T>();
    case 11: return stream_built<Stream11, T>();
    default: return false;
    }
}

// autotuner candidate index -> (cfg, ns, fs)
inline void cand_decode(int cand, int &cfg, int &ns, bool &fs)
{
    constexpr int nt = kNumTiles * kMaxSweepsPerLaunch * 2;
    if (cand < nt) {
        cfg = cand / (2 * kMaxSweepsPerLaunch);
        ns = 1 + (cand / 2) % kMaxSweepsPerLaunch;
        fs = cand % 2;
    } else {
        cfg = kNumTiles + (cand - nt);
        ns = kMaxSweepsPerLaunch;
        fs = false;
    }
}

// FMG tricubic prolongation uf = P3 uc (interpolation.F90:98-217) on an LDS tile: the coarse cells
// any stencil of the fine tile can touch are staged, then the x, y and z passes run on LDS exactly
// as the reference's bufx / bufxy sweeps.  Fine tile FX*FY*FZ, nf >= FX, nf % FY == nf % FZ == 0.
// T = float (mixed path) or double (plain path): the weights are rounded to T as k_interp_cubic
// rounds them, and every value is formed in the same operand order, so both give its results.
template <int FX, int FY, int FZ, int NT, typename T = float, bool ZB = false>
__device__ __forceinline__ void interp_cubic_tile(T *__restrict__ uf, const T *__restrict__ uc, int nf, int t)
{
    constexpr int CX = FX / 2 + 4, CY = FY / 2 + 4, CZ = FZ / 2 + 4;
    __shared__ T sc[CX * CY * CZ];
    __shared__ T bx[CZ * CY * FX];
    __shared__ T bxy[CZ * FY * FX];
    const int nc = nf >> 1;
    const int ntx = nf / FX, nty = nf / FY;
    const int tx = t % ntx, ty = (t / ntx) % nty, tz = t / (ntx * nty);
    const int fx0 = tx * FX, fy0 = ty * FY, fz0 = tz * FZ;
    const int bxo = fx0 / 2 - 2, byo = fy0 / 2 - 2, bzo = fz0 / 2 - 2;  // ghosted coarse index of local 0
    {
        constexpr int CNT = CX * CY * CZ, IT = (CNT + NT - 1) / NT;
        T v[IT];
#pragma unroll
        for (int it = 0; it < IT; ++it) {
            const int q = threadIdx.x + it * NT;
            if (CNT % NT == 0 || q < CNT) {
                const int x = q % CX, y = (q / CX) % CY, z = q / (CX * CY);
                T sx, sy, sz;
                const int a = coarse_ghost<T, ZB>(bxo + x, nc, sx), b = coarse_ghost<T, ZB>(byo + y, nc, sy),
                          d = coarse_ghost<T, ZB>(bzo + z, nc, sz);
                v[it] = uc[(d * nc + b) * nc + a];
                if (ZB) v[it] = (sx * sy * sz) * v[it];
            }
        }
#pragma unroll
        for (int it = 0; it < IT; ++it) {
            const int q = threadIdx.x + it * NT;
            if (CNT % NT == 0 || q < CNT) sc[q] = v[it];
        }
    }
    // per-axis stencil tables (interpolation.F90:106-127), computed once per tile
    __shared__ int tix[FX][4], tiy[FY][4], tiz[FZ][4];
    __shared__ T twx[FX][4], twy[FY][4], twz[FZ][4];
    if (threadIdx.x < FX + FY + FZ) {
        const int q = threadIdx.x;
        int idx[4];
        double a[4];
        if (q < FX) {
            cubic_stencil(fx0 + q, -1, nc, idx, a);
            for (int e = 0; e < 4; ++e) { tix[q][e] = idx[e] - bxo; twx[q][e] = (T)a[e]; }
        } else if (q < FX + FY) {
            cubic_stencil(fy0 + q - FX, -1, nc, idx, a);
            for (int e = 0; e < 4; ++e) { tiy[q - FX][e] = idx[e] - byo; twy[q - FX][e] = (T)a[e]; }
        } else {
            cubic_stencil(fz0 + q - FX - FY, -1, nc, idx, a);
            for (int e = 0; e < 4; ++e) { tiz[q - FX - FY][e] = idx[e] - bzo; twz[q - FX - FY][e] = (T)a[e]; }
        }
    }
    __syncthreads();
    // x pass: bx(fx, jc, kc) over the staged coarse y, z range
    for (int q = threadIdx.x; q < CZ * CY * FX; q += NT) {
        const int x = q % FX, r = q / FX;
        const T *row = sc + r * CX;
        bx[q] = cubic4<T>(twx[x], row[tix[x][0]], row[tix[x][1]], row[tix[x][2]], row[tix[x][3]]);
    }
    __syncthreads();
    // y pass: bxy(fx, fy, kc)
    for (int q = threadIdx.x; q < CZ * FY * FX; q += NT) {
        const int x = q % FX, y = (q / FX) % FY, z = q / (FX * FY);
        const T *col = bx + z * CY * FX + x;
        bxy[q] = cubic4<T>(twy[y], col[tiy[y][0] * FX], col[tiy[y][1] * FX], col[tiy[y][2] * FX],
                               col[tiy[y][3] * FX]);
    }
    __syncthreads();
    // z pass: uf(fx, fy, fz)
    for (int q = threadIdx.x; q < FZ * FY * FX; q += NT) {
        const int x = q % FX, y = (q / FX) % FY, z = q / (FX * FY);
        const T *p = bxy + y * FX + x;
        constexpr int PL = FY * FX;
        uf[((fz0 + z) * nf + (fy0 + y)) * nf + (fx0 + x)] =
            cubic4<T>(twz[z], p[tiz[z][0] * PL], p[tiz[z][1] * PL], p[tiz[z][2] * PL], p[tiz[z][3] * PL]);
    }
}

template <int FX, int FY, int FZ, int NT, typename T = float, bool ZB = false>
__global__ void __launch_bounds__(NT) k_interp_cubic_tile(T *__restrict__ uf, const T *__restrict__ uc, int nf)
{
    const int ntiles = (nf / FX) * (nf / FY) * (nf / FZ);
    const int t = xcd_tile(ntiles);
    if (t >= ntiles) return;
    interp_cubic_tile<FX, FY, FZ, NT, T, ZB>(uf, uc, nf, t);
}

// ------------------------------------------------------------------------------------------------
// Single-workgroup solvers of the first level of <= 16^3 cells (of a grid of n = 2^a > 16: the 16^3 one):
// the reference's cycles from there down (coarse_levels.h), or its exact solve.
// ------------------------------------------------------------------------------------------------
template <typename T, bool ZERO = false>
__global__ void __launch_bounds__(kCoarseThreads)
k_coarse(const T *__restrict__ rhs_in, T *__restrict__ u_out, CoarseCoef<T> P, int mode, int ncycle, int npre, int npost)
{
    __shared__ CoarseLds<T> S;
    coarse_solve<T, kCoarseMaxN, ZERO>(S, P, rhs_in, u_out, mode, ncycle, npre, npost);
}

// mg_cycle (mg.F90:42-94) of a grid held by the coarse levels alone (N <= 16) in one launch: FP64
// residual and update around the inner solve in T, both stopping tests.  A 16^3 solve of 4 iterations
// is 4 inner solves of 57 us; as launches (inner solve, update + residual, norm) with a host read of the
// norms per iteration it took 400 us, this 300 us.  psi stays in LDS, its source and the
// cells' places in registers.  rec (pinned host memory): what the host's statistics need.
struct SmallRecord {
    double fmax, fsum;             // max|f|, sum f^2
    double rmax, rsum, resmax;     // last residual's max and sum of squares; last max|resh2|
    int iterations, status;
    double hist[SG_HIST];          // max|r| per iteration
};

template <typename T, int N>
__global__ void __launch_bounds__(kCoarseThreads)
k_cycle_small(double *__restrict__ psi_io, const double *__restrict__ src, CoarseCoef<T> P, double h, double h2i,
              double tol, int maxit, int stop_mode, int ncycle, int npre, int npost, SmallRecord *rec)
{
    using L = CoarseLevel<N>;
    constexpr int IT = (L::len + kCoarseThreads - 1) / kCoarseThreads;
    constexpr bool full = L::len % kCoarseThreads == 0;
    __shared__ CoarseLds<T> S;
    __shared__ double psi[L::len];
    __shared__ double s_norm[5];   // max|f|, sum f^2, max|r|, sum r^2, max|resh2|
    double f[IT];
    double mx = 0.0, sm = 0.0;
#pragma unroll
    for (int m = 0; m < IT; ++m) {
        const int c = (int)threadIdx.x + m * kCoarseThreads;
        f[m] = 0.0;
        if (full || c < L::len) {
            int i, j, k;
            L::decode(c, i, j, k);
            psi[L::at(i, j, k)] = psi_io[c];
            f[m] = src[c];
            mx = fmax(mx, fabs(f[m]));
            sm += f[m] * f[m];
        }
    }
    if (threadIdx.x >= kCoarseThreads - 64) coarse_tables<T, N, false>(S, (int)threadIdx.x - (kCoarseThreads - 64));
    block_max_sum(mx, sm);
    if (threadIdx.x == 0) {
        s_norm[0] = mx;
        s_norm[1] = sm;
        s_norm[4] = 0.0;
    }
    __syncthreads();
    int it = 0, status = SG_ERR_NOT_CONVERGED;
    double rhomax = 0.0;
    for (;;) {
        mx = sm = 0.0;
#pragma unroll
        for (int m = 0; m < IT; ++m) {
            const int c = (int)threadIdx.x + m * kCoarseThreads;
            if (full || c < L::len) {
                int i, j, k;
                L::decode(c, i, j, k);
                auto U = [&](int a, int b, int d) { return psi[L::at((a + N) % N, (b + N) % N, (d + N) % N)]; };
                const double r = resid_value<double>(U(i, j, k), U(i + 1, j, k), U(i - 1, j, k), U(i, j + 1, k), U(i, j - 1, k),
                                                     U(i, j, k + 1), U(i, j, k - 1), f[m], h2i);
                S.r[L::off + L::at(i, j, k)] = (T)r;
                mx = fmax(mx, fabs(r));
                sm += r * r;
            }
        }
        block_max_sum(mx, sm);
        if (threadIdx.x == 0) {
            s_norm[2] = mx;
            s_norm[3] = sm;
        }
        __syncthreads();
        // every thread takes the same decision, in the order of the host's loop
        const double fm = s_norm[0], rm = s_norm[2], resmaxg = s_norm[4] / (h * h);
        const double rel = fm > 0 ? rm / fm : 0.0;
        if (it == 0) rhomax = rm;
        if (threadIdx.x == 0 && it < SG_HIST) rec->hist[it] = rm;
        if (!isfinite(rm) || !isfinite(s_norm[3])) { status = SG_ERR_NONFINITE; break; }
        if (stop_mode == SG_STOP_TRUE_RESIDUAL && rel < tol) { status = SG_OK; break; }
        if (it > 0 && stop_mode == SG_STOP_REFERENCE && (rhomax > 0 ? resmaxg / rhomax : 0.0) < tol) { status = SG_OK; break; }
        if (it >= maxit) break;
        __syncthreads();
        if (threadIdx.x == 0) s_norm[4] = 0.0;
        __syncthreads();
        coarse_run<T, N, false>(S, P, true, ncycle, npre, npost,
                                stop_mode == SG_STOP_REFERENCE ? &s_norm[4] : (double *)nullptr);
        __syncthreads();
#pragma unroll
        for (int m = 0; m < IT; ++m) {
            const int c = (int)threadIdx.x + m * kCoarseThreads;
            if (full || c < L::len) psi[c] = psi[c] + (double)S.u[L::off + c];
        }
        ++it;
        __syncthreads();
    }
#pragma unroll
    for (int m = 0; m < IT; ++m) {
        const int c = (int)threadIdx.x + m * kCoarseThreads;
        if (full || c < L::len) {
            int i, j, k;
            L::decode(c, i, j, k);
            psi_io[c] = psi[L::at(i, j, k)];
        }
    }
    if (threadIdx.x == 0) {
        rec->fmax = s_norm[0];
        rec->fsum = s_norm[1];
        rec->rmax = s_norm[2];
        rec->rsum = s_norm[3];
        rec->resmax = s_norm[4];
        rec->iterations = it;
        rec->status = status;
    }
}

struct CoarseExact {
    int n;                                                 // cells per side, <= 16
    float Q[kCoarseMaxN * kCoarseMaxN], lam[kCoarseMaxN];  // Hartley basis and eigenvalues
};

// Hartley basis of the periodic 3-point second difference on n cells, Q[m n + k] =
// (cos a + sin a) / sqrt(n) with a = 2 pi ((m k) mod n) / n, and its eigenvalues
// lam[m] = (2 cos(2 pi m / n) - 2) / h^2 (host; the CPU restatement forms them the same way).
inline void hartley_basis(int n, double h, double *Q, double *lam)
{
    const double pi = 3.14159265358979323846;
    for (int m = 0; m < n; ++m) {
        for (int k = 0; k < n; ++k) {
            const double a = 2.0 * pi * (double)((m * k) % n) / (double)n;
            Q[m * n + k] = (std::cos(a) + std::sin(a)) / std::sqrt((double)n);
        }
        lam[m] = (2.0 * std::cos(2.0 * pi * (double)m / (double)n) - 2.0) / (h * h);
    }
}

// ---- exact solve of a periodic level of n^3 cells (n <= 16) in one workgroup ---------------------
// The coarse-grid problem L u = f that the V-cycle bottom and the FMG start approximate (mg.F90:
// 142-210 below the first fine level) is solved exactly instead: the 7-point operator separates,
// the symmetric orthonormal Hartley basis Q diagonalises the periodic second difference along
// each axis, so u = Q (Lambda^-1 (Q f)) with Lambda = (lam_i + lam_j) + lam_k and the zero mode set
// to zero (the zero-mean solution).  Three axis passes serve as forward and inverse transform.
// The grid sits in LDS with row pitch n + 1.  Thread t works on grid line t / 4 and owns the
// outputs m = t % 4 + 4 r (r < 4) of every line it is given: its four rows of Q stay in registers
// for all six passes, and the four threads of a line sit in adjacent lanes, so the line's reads
// are broadcasts.  Each output is accumulated k = 0 .. n-1 in order with fused multiply-adds.
constexpr int kCeParts = 4;
constexpr int kCoarseExactThreads = 1024;
static_assert(kCoarseMaxN * kCoarseMaxN * kCeParts <= kCoarseExactThreads, "one thread per (line, part)");
static_assert(kCoarseMaxN <= 4 * kCeParts, "four outputs per thread");

__device__ inline void ce_basis(float (&q)[4][kCoarseMaxN], const float *Q, int n)
{
    const int part = threadIdx.x % kCeParts;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const int m = part + kCeParts * r;
#pragma unroll
        for (int k = 0; k < kCoarseMaxN; ++k) q[r][k] = (m < n && k < n) ? Q[m * n + k] : 0.f;
    }
}

__device__ inline void ce_pass(float *g, const float (&q)[4][kCoarseMaxN], int n, int axis)
{
    const int P = n + 1;
    const int line = threadIdx.x / kCeParts, part = threadIdx.x % kCeParts;
    const int a = line % n, b = line / n;
    int base, stride;
    if (axis == 0) { base = (b * n + a) * P; stride = 1; }        // line (j, k) = (a, b)
    else if (axis == 1) { base = b * n * P + a; stride = P; }     // line (i, k)
    else { base = b * P + a; stride = n * P; }                    // line (i, j)
    const bool act = line < n * n;
    float x[kCoarseMaxN];
#pragma unroll
    for (int k = 0; k < kCoarseMaxN; ++k) x[k] = (act && k < n) ? g[base + k * stride] : 0.f;
    __syncthreads();
    if (act) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int m = part + kCeParts * r;
            if (m < n) {
                float acc = 0.f;
#pragma unroll
                for (int k = 0; k < kCoarseMaxN; ++k)
                    if (k < n) acc = __builtin_fmaf(q[r][k], x[k], acc);
                g[base + m * stride] = acc;
            }
        }
    }
    __syncthreads();
}

// u_out := exact solution for rhs_in (dense n^3 arrays, i fastest).  g: n^2 (n + 1) floats of LDS,
// s: n^2 + n floats of LDS for the basis (staged there once, then read into registers as
// broadcasts) and the eigenvalues; Qg, lamg: basis and eigenvalues (any address space).
__device__ inline void coarse_exact(float *g, float *s, const float *Qg, const float *lamg, const float *rhs_in,
                                    float *u_out, int n)
{
    const int P = n + 1, n3 = n * n * n;
    float *Qs = s, *lam = s + n * n;
    for (int t = threadIdx.x; t < n * n; t += kCoarseExactThreads) Qs[t] = Qg[t];
    for (int t = threadIdx.x; t < n; t += kCoarseExactThreads) lam[t] = lamg[t];
    for (int c = threadIdx.x; c < n3; c += kCoarseExactThreads) {
        const int i = c % n, j = (c / n) % n, k = c / (n * n);
        g[(k * n + j) * P + i] = rhs_in[c];
    }
    __syncthreads();
    float q[4][kCoarseMaxN];
    ce_basis(q, Qs, n);
    for (int a = 0; a < 3; ++a) ce_pass(g, q, n, a);
    for (int c = threadIdx.x; c < n3; c += kCoarseExactThreads) {
        const int i = c % n, j = (c / n) % n, k = c / (n * n);
        const float den = (lam[i] + lam[j]) + lam[k];
        float &v = g[(k * n + j) * P + i];
        v = den != 0.f ? v / den : 0.f;
    }
    __syncthreads();
    for (int a = 0; a < 3; ++a) ce_pass(g, q, n, a);
    for (int c = threadIdx.x; c < n3; c += kCoarseExactThreads) {
        const int i = c % n, j = (c / n) % n, k = c / (n * n);
        u_out[c] = g[(k * n + j) * P + i];
    }
}

static __global__ void __launch_bounds__(kCoarseExactThreads)
k_coarse_exact(const float *__restrict__ rhs_in, float *__restrict__ u_out, CoarseExact E)
{
    __shared__ float g[kCoarseMaxN * kCoarseMaxN * (kCoarseMaxN + 1)], q[kCoarseMaxN * kCoarseMaxN + kCoarseMaxN];
    coarse_exact(g, q, E.Q, E.lam, rhs_in, u_out, E.n);
}

} // namespace sg
