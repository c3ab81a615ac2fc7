// nlse3d.hip -- 3D NLSE RK4 stage kernels on MI355X.
//
// Replaces NLSE3D_STEP and add_cube of src/NLSEmagic3D/NLSE3D_TAKE_STEPS_CD.c
// (:28-223) and NLSE3D_TAKE_STEPS_2SHOC.c (:28-412), with the chunk loop of
// :308-322 / :507-521 on the host.  Element (i, j, k) is at (i*N + j)*M + k:
// i < L slowest, k < M contiguous.
// By default two stages per launch on plane-marching tiles (nlse3d_cdpair.h,
// nlse3d_shocpair.h).  One stage per launch (on request, and on small MSD
// grids):
//   CD:    one fused kernel per RK4 stage (7-point stencil + BC + update).
//   2SHOC: one plane-marching kernel per RK4 stage that keeps D on chip
//          (nlse3d_march.h); for MSD boundaries, whose partner can lie in
//          another plane and row, a D pass (D = Lap_CD(Y)/h^2 with its
//          boundary values, written to a scratch field) and a fused F +
//          update pass that reads D's six neighbours and Y's twelve edge
//          neighbours.
// Neighbour reads of the per-point kernels go through the L1/L2 caches: a
// wavefront covers 64 consecutive k, so every plane and row neighbour is a
// coalesced line read.
#include "nlse3d_cdpair.h"
#include "nlse3d_march.h"
#include "nlse3d_shocpair.h"
#include "nlse_common.h"
#include "nlse_launch.h"

namespace nlse {

struct Grid3 {
    int N, M, L;
    long si, sj;  // strides of i and j
};

template <typename T>
__device__ __forceinline__ c2<T> d3_int(const c2<T>* __restrict__ y, long p, const Grid3& g, const Coefs<T>& c)
{
    // NLSE3D_TAKE_STEPS_2SHOC.c:62-69
    const c2<T> a = y[p + g.si], b = y[p - g.si], d = y[p + g.sj], e = y[p - g.sj], f = y[p + 1], h = y[p - 1],
                m = y[p];
    return mk<T>(c.lh2 * (a.x + b.x + d.x + e.x + f.x + h.x - 6 * m.x),
                 c.lh2 * (a.y + b.y + d.y + e.y + f.y + h.y - 6 * m.y));
}

template <typename T, int METHOD>
__device__ __forceinline__ c2<T> f3_int(const c2<T>* __restrict__ y, const c2<T>* __restrict__ D,
                                        const T* __restrict__ V, long p, const Grid3& g, const Coefs<T>& c)
{
    const c2<T> m = y[p];
    const T w = V[p] - c.s * (m.x * m.x + m.y * m.y);
    if (METHOD == 1) {
        // NLSE3D_TAKE_STEPS_CD.c:59-71
        const c2<T> a = y[p + g.si], b = y[p - g.si], d = y[p + g.sj], e = y[p - g.sj], f = y[p + 1],
                    h = y[p - 1];
        return mk<T>(-c.ah2 * (a.y + b.y + d.y + e.y + f.y + h.y - 6 * m.y) + w * m.y,
                     c.ah2 * (a.x + b.x + d.x + e.x + f.x + h.x - 6 * m.x) - w * m.x);
    } else {
        // NLSE3D_TAKE_STEPS_2SHOC.c:239-259; edge neighbours in source order
        const long si = g.si, sj = g.sj;
        const long e12[12] = {si + sj, sj + 1, si + 1, -si - sj, -sj - 1, -si - 1,
                              si - sj, sj - 1, si - 1, -si + sj, -sj + 1, -si + 1};
        c2<T> es = y[p + e12[0]];
#pragma unroll
        for (int t = 1; t < 12; ++t) {
            const c2<T> q = y[p + e12[t]];
            es.x = es.x + q.x;
            es.y = es.y + q.y;
        }
        const c2<T> da = D[p + si], db = D[p - si], dd = D[p + sj], de = D[p - sj], df = D[p + 1], dh = D[p - 1],
                    dm = D[p];
        return mk<T>(c.a_12 * (da.y + db.y + dd.y + de.y + df.y + dh.y - 10 * dm.y) - c.a_6h2 * (es.y - 12 * m.y)
                         + w * m.y,
                     -c.a_12 * (da.x + db.x + dd.x + de.x + df.x + dh.x - 10 * dm.x)
                         + c.a_6h2 * (es.x - 12 * m.x) - w * m.x);
    }
}

__device__ __forceinline__ bool interior3(int i, int j, int k, const Grid3& g)
{
    return i > 0 && i < g.L - 1 && j > 0 && j < g.N - 1 && k > 0 && k < g.M - 1;
}

__device__ __forceinline__ long partner3(int i, int j, int k, const Grid3& g)
{
    return ((long)clamp_in(i, g.L) * g.N + clamp_in(j, g.N)) * g.M + clamp_in(k, g.M);
}

// D with its boundary values (NLSE3D_TAKE_STEPS_2SHOC.c:56-230)
template <typename T>
__global__ __launch_bounds__(256) void d3_kernel(const c2<T>* __restrict__ y, c2<T>* __restrict__ D,
                                                 const T* __restrict__ V, Coefs<T> c, Grid3 g, int BC)
{
    const int k = blockIdx.x * 64 + (threadIdx.x & 63);
    const int j = blockIdx.y * 4 + (threadIdx.x >> 6);
    const int i = blockIdx.z;
    if (k >= g.M || j >= g.N) return;
    const long p = ((long)i * g.N + j) * g.M + k;
    c2<T> d;
    if (interior3(i, j, k, g)) {
        d = d3_int<T>(y, p, g, c);
    } else if (BC == BC_DIRICHLET) {
        d = dir_d<T>(y[p], V[p], c);
    } else if (BC == BC_MSD) {
        const long q = partner3(i, j, k, g);
        d = msd_d<T>(d3_int<T>(y, q, g, c), y[q], V[q], y[p], V[p], c);
    } else {
        d = mk<T>(0, 0);
    }
    D[p] = d;
}

// F with its boundary values, then the RK4 stage update
template <typename T, int METHOD>
__global__ __launch_bounds__(256) void f3_kernel(const c2<T>* __restrict__ y, const c2<T>* u, c2<T>* __restrict__ acc,
                                                 c2<T>* yout, const c2<T>* __restrict__ D, const T* __restrict__ V,
                                                 Coefs<T> c, Grid3 g, int BC, int stage, c2<T>* ulo)
{
    const int k = blockIdx.x * 64 + (threadIdx.x & 63);
    const int j = blockIdx.y * 4 + (threadIdx.x >> 6);
    const int i = blockIdx.z;
    if (k >= g.M || j >= g.N) return;
    const long p = ((long)i * g.N + j) * g.M + k;
    c2<T> f;
    if (interior3(i, j, k, g)) {
        f = f3_int<T, METHOD>(y, D, V, p, g, c);
    } else if (BC == BC_MSD) {
        const long q = partner3(i, j, k, g);
        f = msd_f<T>(f3_int<T, METHOD>(y, D, V, q, g, c), y[q], y[p]);
    } else if (BC == BC_LAP0) {
        f = lap0_f<T>(y[p], V[p], c.s);
    } else {
        f = mk<T>(0, 0);
    }
    const c2<T> uu = (stage == 1) ? y[p] : u[p];
    rk4_epilogue<T>(stage, c, f, uu, acc, yout, yout, p, ulo);
}

// 2SHOC stage with D on chip: one workgroup per (j tile, k tile, i chunk);
// consecutive tiles of a chunk go to the same XCD
template <typename T, int TJ, int NW>
__global__ __launch_bounds__(NW * 64) void march3d_kernel(const c2<T>* __restrict__ yin, const c2<T>* u,
                                                      c2<T>* __restrict__ acc, c2<T>* yout, const T* __restrict__ V,
                                                      Coefs<T> c, March3 g, int BC, int stage, c2<T>* ulo)
{
    __shared__ March3Lds<T, TJ> sm;
    const int t = (blockIdx.x & 7) * g.per_xcd + (blockIdx.x >> 3);
    if (t >= g.tj * g.tk * g.ti) return;
    const int kt = t % g.tk, rest = t / g.tk;
    const int jt = rest % g.tj, ci = rest / g.tj;
    march3d_tile<T, TJ, NW>(sm, ci * g.IC, jt * TJ, kt * March3Cfg<TJ>::W, g, yin, u, acc, yout, V, c, BC, stage,
                            ulo);
}

template <typename T, int TJ, int NW>
static hipError_t launch_march3d(const StageArgs<T>& a, int IC, hipStream_t st)
{
    March3 g;
    g.N = a.N;
    g.M = a.M;
    g.L = a.L;
    g.IC = IC;
    g.ioff = g.joff = g.koff = 0;
    g.tj = (a.N + TJ - 1) / TJ;
    g.tk = (a.M + March3Cfg<TJ>::W - 1) / March3Cfg<TJ>::W;
    g.ti = (a.L + IC - 1) / IC;
    g.per_xcd = (g.tj * g.tk * g.ti + 7) / 8;
    hipLaunchKernelGGL((march3d_kernel<T, TJ, NW>), dim3(8 * g.per_xcd), dim3(NW * 64), 0, st, a.yin, a.u, a.acc,
                       a.yout, a.V, a.c, g, a.BC, a.stage, a.ulo);
    return hipGetLastError();
}

// whether the extended tile (owned points plus H on each side) of a pair
// launch reaches the grid's boundary
template <int TJ, int W, int H>
__device__ __forceinline__ bool pair_edge(const March3& g, int i0, int j0, int k0)
{
    return i0 - H <= 0 || i0 + g.IC + H >= g.L || j0 - H <= 0 || j0 + TJ + H >= g.N || k0 - H <= 0 ||
           k0 + W + H >= g.M;
}

// CD, two stages per launch (stages 1-2 or 3-4) on plane-marching tiles
template <typename T, int FIRST, int TJ, int NW, bool MSD>
__global__ __launch_bounds__(NW * 64) void cdpair3d_kernel(const c2<T>* __restrict__ yin, const c2<T>* u,
                                                           c2<T>* __restrict__ acc, c2<T>* __restrict__ yout,
                                                           const T* __restrict__ V, Coefs<T> c, March3 g, int BC,
                                                           c2<T>* ulo)
{
    __shared__ CdPairLds<T, TJ, MSD> sm;
    const int t = (blockIdx.x & 7) * g.per_xcd + (blockIdx.x >> 3);
    if (t >= g.tj * g.tk * g.ti) return;
    const int kt = t % g.tk, rest = t / g.tk;
    const int jt = rest % g.tj, ci = rest / g.tj;
    const int i0 = ci * g.IC - g.ioff, j0 = jt * TJ - g.joff, k0 = kt * 60 - g.koff;
    if (MSD && pair_edge<TJ, 60, 2>(g, i0, j0, k0))
        cdpair_tile<T, FIRST, TJ, NW, MSD>(sm, i0, j0, k0, g, yin, u, acc, yout, V, c, BC, ulo);
    else
        cdpair_tile<T, FIRST, TJ, NW, false>(sm, i0, j0, k0, g, yin, u, acc, yout, V, c, BC, ulo);
}

// 2SHOC, two stages per launch on plane-marching tiles
template <typename T, int FIRST, int TJ, bool MSD>
__global__ __launch_bounds__((TJ + 4) * 64) void shocpair3d_kernel(const c2<T>* __restrict__ yin, const c2<T>* u,
                                                                   c2<T>* __restrict__ acc, c2<T>* __restrict__ yout,
                                                                   const T* __restrict__ V, Coefs<T> c, March3 g,
                                                                   int BC, c2<T>* ulo)
{
    using Lds = ShocPairLds<T, TJ, MSD>;
    __shared__ Lds sm;
    const int t = (blockIdx.x & 7) * g.per_xcd + (blockIdx.x >> 3);
    if (t >= g.tj * g.tk * g.ti) return;
    const int kt = t % g.tk, rest = t / g.tk;
    const int jt = rest % g.tj, ci = rest / g.tj;
    const int i0 = ci * g.IC - g.ioff, j0 = jt * TJ - g.joff, k0 = kt * 56 - g.koff;
    if (MSD && pair_edge<TJ, 56, 4>(g, i0, j0, k0))
        ShocPair<T, FIRST, TJ, MSD, Lds>(sm, i0, j0, k0, g, yin, u, acc, yout, V, c, BC, ulo).run();
    else
        ShocPair<T, FIRST, TJ, false, Lds>(sm, i0, j0, k0, g, yin, u, acc, yout, V, c, BC, ulo).run();
}

// Planes per chunk of a pair launch with `cols` tiles per plane, H halo planes
// per chunk and steps in groups of G.  A workgroup (one per CU) takes about
// as long as its steps plus two for its first loads, so a launch takes
// rounds(chunks) * (steps(chunk) + 2): short chunks fill the chip on small
// grids, long ones spend less on halo planes.  Chunks of 32 planes stay where
// nothing is 7 % better by this count (on grids of several rounds the count
// is only good to a few per cent).  Time per step, chunks of 32 -> this rule:
// 64^3 CD FP64 79 -> 22 us, 2SHOC FP64 112 -> 33; 97 x 120 x 111 CD FP64
// 92 -> 47, 2SHOC FP64 121 -> 70; 192^3 CD FP64 223 -> 181, 2SHOC FP64
// 373 -> 317; 256^3 unchanged within 2 %.
static int pair_chunk(int cols, int L, int H, int G)
{
    const int cus = device_cus();
    auto cost = [&](int IC) -> long {
        const long wgs = (long)cols * ((L + IC - 1) / IC);
        return (wgs + cus - 1) / cus * ((IC + H + G - 1) / G * G + 2);
    };
    const int base = 32;
    int best = base;
    long bc = cost(base) * 93;  // hundredths
    for (int n = 1; n <= (L + 3) / 4; ++n) {
        const int IC = (L + n - 1) / n;
        if (IC < 4 || IC > 96) continue;
        const long k = cost(IC) * 100;
        if (k < bc) {
            bc = k;
            best = IC;
        }
    }
    return best;
}

// the tiles of a pair launch: TJ rows x W columns over chunks of planes (a
// halo of H on each side); MSD tiles own at least two points of the grid
// along every axis
static March3 pair_tiles(int N, int M, int L, int TJ, int W, int H, int G, bool msd)
{
    March3 g;
    g.N = N;
    g.M = M;
    g.L = L;
    g.joff = msd && N % TJ == 1;
    g.koff = msd && M % W == 1;
    g.tj = (N + g.joff + TJ - 1) / TJ;
    g.tk = (M + g.koff + W - 1) / W;
    g.IC = pair_chunk(g.tj * g.tk, L, 2 * H, G);
    g.ioff = msd && L % g.IC == 1;
    g.ti = (L + g.ioff + g.IC - 1) / g.IC;
    g.per_xcd = (g.tj * g.tk * g.ti + 7) / 8;
    return g;
}

template <typename T, int FIRST, bool MSD>
static hipError_t launch_shocpair3d(const StageArgs<T>& a, hipStream_t st)
{
    // the most rows whose register rings fit: TJ + 4 waves of 168 (12 waves),
    // 128 (16) or, for double MSD, 209 VGPRs (8)
    constexpr int TJ = std::is_same<T, double>::value ? (MSD ? 4 : 8) : 12;
    if ((long)a.N * a.M > 0x7fffffffL) return hipErrorInvalidValue;  // 32-bit offsets within a plane
    const March3 g = pair_tiles(a.N, a.M, a.L, TJ, 56, 4, 4, MSD);
    hipLaunchKernelGGL((shocpair3d_kernel<T, FIRST, TJ, MSD>), dim3(8 * g.per_xcd), dim3((TJ + 4) * 64), 0, st, a.yin,
                       a.u, a.acc, a.yout, a.V, a.c, g, a.BC, a.ulo);
    return hipGetLastError();
}

template <typename T, int FIRST, bool MSD>
static hipError_t launch_cdpair3d(const StageArgs<T>& a, hipStream_t st)
{
    // 12 owned rows on 16 waves, one extended row per wave: few registers
    // per wave (stages 3-4 in FP64: 117 VGPRs, against 208 with two rows per
    // wave) and j-halo rows re-read through L2 for 12 owned rows instead of
    // 4 (the halo re-reads dominate the HBM traffic beyond the 128 B per
    // point-step the pair needs)
    constexpr int TJ = 12, NW = TJ + 4;
    const March3 g = pair_tiles(a.N, a.M, a.L, TJ, 60, 2, 3, MSD);
    hipLaunchKernelGGL((cdpair3d_kernel<T, FIRST, TJ, NW, MSD>), dim3(8 * g.per_xcd), dim3(NW * 64), 0, st, a.yin,
                       a.u, a.acc, a.yout, a.V, a.c, g, a.BC, a.ulo);
    return hipGetLastError();
}

template <typename T>
hipError_t launch_pair3d(const StageArgs<T>& a, bool first, hipStream_t st)
{
    const bool msd = a.BC == BC_MSD;
    if (a.method == 2) {
        if (msd) return first ? launch_shocpair3d<T, 1, true>(a, st) : launch_shocpair3d<T, 3, true>(a, st);
        return first ? launch_shocpair3d<T, 1, false>(a, st) : launch_shocpair3d<T, 3, false>(a, st);
    }
    if (msd) return first ? launch_cdpair3d<T, 1, true>(a, st) : launch_cdpair3d<T, 3, true>(a, st);
    return first ? launch_cdpair3d<T, 1, false>(a, st) : launch_cdpair3d<T, 3, false>(a, st);
}

template hipError_t launch_pair3d<double>(const StageArgs<double>&, bool, hipStream_t);
template hipError_t launch_pair3d<float>(const StageArgs<float>&, bool, hipStream_t);

template <typename T>
hipError_t launch_stage3d(const StageArgs<T>& a, hipStream_t st)
{
    if (a.method == 2 && a.BC != BC_MSD && a.kernel != KERNEL_TILES) {
        // rows per tile: 4 or 8 (a.tile below 8 selects 4); planes per chunk 32
        if (a.tile < 8) return launch_march3d<T, 4, 4>(a, 32, st);
        return launch_march3d<T, 8, 4>(a, 32, st);
    }
    Grid3 g;
    g.N = a.N;
    g.M = a.M;
    g.L = a.L;
    g.sj = a.M;
    g.si = (long)a.N * a.M;
    dim3 grid((a.M + 63) / 64, (a.N + 3) / 4, a.L);
    if (a.method == 2) {
        hipLaunchKernelGGL((d3_kernel<T>), grid, dim3(256), 0, st, a.yin, a.dbuf, a.V, a.c, g, a.BC);
        hipLaunchKernelGGL((f3_kernel<T, 2>), grid, dim3(256), 0, st, a.yin, a.u, a.acc, a.yout, a.dbuf, a.V,
                           a.c, g, a.BC, a.stage, a.ulo);
    } else {
        hipLaunchKernelGGL((f3_kernel<T, 1>), grid, dim3(256), 0, st, a.yin, a.u, a.acc, a.yout,
                           (const c2<T>*)nullptr, a.V, a.c, g, a.BC, a.stage, a.ulo);
    }
    return hipGetLastError();
}

template hipError_t launch_stage3d<double>(const StageArgs<double>&, hipStream_t);
template hipError_t launch_stage3d<float>(const StageArgs<float>&, hipStream_t);

}  // namespace nlse
