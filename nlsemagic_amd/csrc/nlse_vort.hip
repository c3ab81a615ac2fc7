// nlse_vort.hip -- 3D vorticity of a resident state on MI355X.
//
// Replaces the reference's MEX post-processor rmc_vorticity3D
// (src/NLSEmagic3D/rmc_vorticity3D.c:24-354), which reads the state the 3D
// drivers produce:
//   V = Im(conj(U) grad U) / (2|U|^2 + veps)   (per point, :188-204)
//   w = curl V, W = |w|                        (:207-329)
// with central differences lh2*(A[+1] - A[-1]) at interior points and
// one-sided (2 lh2)*(A[+1] - A[0]) / (2 lh2)*(A[0] - A[-1]) normal to a face
// (the y- and z-faces also take the x-derivative one-sided forward, as the
// reference does).  All arithmetic is double, in the reference's operand
// order (FP contraction off, correctly rounded division and square root), so
// the result is bit-identical to the reference wherever the reference is
// defined: it never sets the gradient on edges and corners (two or more
// boundary indices); here it is 0 there, and the curl on edges and corners
// is 0 as in the reference's zero-initialised outputs.  Single-precision
// states are widened (hi + lo) to double first.
//
// One kernel, no scratch: a workgroup owns TJ rows (j) x 56 or 60 columns (k) and
// marches along i over a chunk of planes.  Lane l is column k0 - 2 + l;
// extended row e is row j0 - 2 + e.  At step p a row takes U of plane p
// (loaded two steps ahead), the rows next to the owned ones and the owned ones
// form the velocity of plane p-1, and the owned rows the curl of plane p-2;
// one barrier ends the step.  An owned row has a wave of its own, the four halo
// rows share one.  U of three planes and the velocity of three planes stay in
// registers (the i +- 1 neighbours), the k +- 1 neighbours come from adjacent
// lanes (DPP) and the j +- 1 neighbours from LDS copies of the previous step's
// U and of the two velocity components the y-differences read
// (double-buffered).  HBM traffic per point: U once (plus halo re-reads
// through L2) and the four outputs.
//
// Rows and planes inside the grid, in tiles without column 0 or M-1, run
// central differences only (uniform branch); the others select operands per
// lane, without branches.  At 256^3 the bytes a point needs take 159 us at the
// rate of a large copy (48 B: FP64, FP32 compensated) or 133 us (FP32, 40 B).  A
// call takes about the same in every precision: the four outputs and the plane
// step's chain of loads, differences and division bound it, not the state's
// bytes, of which repeated calls find a part in the 256 MB cache.  The time
// depends on the values (clock): a uniform state FP64 151 us, FP32 149, FP32c 158,
// four vortex rings 173, 163 and 179.  Per call, 16 rows on 16 waves with a branch
// per difference and loads widened at once -> this: uniform 256^3 FP64 244 -> 151
// us, FP32 275 -> 149, FP32c 333 -> 158; 201 x 180 x 190 FP64 150 -> 99; 64^3 FP64
// 68 -> 14; four rings of 256^3 in a run of 20 calls 258 -> 191.
#include "nlse2d_strip.h"
#include "nlse_host.h"

namespace nlse {

namespace {

struct Dims3 {
    int L, N, M;
    long si, sj;
};

// U as loaded: the values, with the low part of a compensated state; widened
// when its plane's step comes, so that a load stays in flight until then
template <typename T, bool COMP> struct Raw {
    c2<T> h, l;
    __device__ __forceinline__ double2 wide() const
    {
        double2 r = make_double2((double)h.x, (double)h.y);
        if constexpr (COMP) {
            r.x = r.x + (double)l.x;
            r.y = r.y + (double)l.y;
        }
        return r;
    }
};

struct VortMarch {
    int IC;                 // planes per chunk
    int kw;                 // owned columns, at most 60
    int tj, tk, ti;         // tiles along j, k and chunks along i
    int per_xcd;            // workgroups per XCD
};

template <int TJ>
struct VortLds {
    static constexpr int TE = TJ + 4;   // extended rows of U
    double2 u[2][TE][64];               // U of the last two planes
    double vx[2][TE - 2][64];           // velocity x and z of the last two planes, rows 1 .. TE-2
    double vz[2][TE - 2][64];
};

template <typename T, bool COMP, int TJ>
struct VortTile {
    static constexpr int TE = TJ + 4;
    // one extended row: level 0 loads, 1 also forms the velocity, 2 the curl
    // (rings: slot = (plane - first plane) mod 4)
    template <int LV> struct Row {
        int e, j;
        long ro;  // offset j * sj + k within a plane, clamped into the grid
        double2 U[4];
        double vx[4], vy[4], vz[4];
        Raw<T, COMP> n1, n2;  // the next two planes
    };
    VortLds<TJ>& sm;
    const c2<T>* u;
    const c2<T>* ulo;
    const double lh2, veps;
    const Dims3& g;
    double *wx, *wy, *wz, *W;
    const int i0, iend, j0, k, lane;
    const bool kout, kb, ktile;  // an owned column in the grid, a column on its boundary; the tile holds a boundary column (uniform)

    template <int LV> __device__ __forceinline__ void init(Row<LV>& R, int e) const
    {
        R.e = e;
        R.j = j0 - 2 + e;
        const int jc = R.j < 0 ? 0 : (R.j >= g.N ? g.N - 1 : R.j);
        R.ro = (long)jc * g.sj + (k < 0 ? 0 : (k >= g.M ? g.M - 1 : k));
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            R.U[s] = make_double2(0, 0);
            R.vx[s] = R.vy[s] = R.vz[s] = 0;
        }
    }
    template <int LV> __device__ __forceinline__ Raw<T, COMP> load(const Row<LV>& R, int pl) const
    {
        const long p = (long)(pl < 0 ? 0 : (pl >= g.L ? g.L - 1 : pl)) * g.si + R.ro;
        Raw<T, COMP> r;
        r.h = u[p];
        if constexpr (COMP) r.l = ulo[p];
        return r;
    }
    // differences of a along one axis: the operands of the point's kind,
    // (+1, -1) with lh2, or one-sided with 2 lh2
    struct Ops {
        bool p0, m0;  // the point itself in place of +1 / of -1
    };
    __device__ __forceinline__ double diff(Ops o, double ap, double a0, double am) const
    {
        const double c = (o.p0 || o.m0) ? lh2 * 2 : lh2;
        return c * ((o.p0 ? a0 : ap) - (o.m0 ? a0 : am));
    }
    // kinds at (i, j, this lane's k); false on edges and corners
    __device__ __forceinline__ bool kinds(int i, int j, Ops& x, Ops& y, Ops& z) const
    {
        const bool bi = i == 0 || i == g.L - 1, bj = j == 0 || j == g.N - 1;
        x = {i == g.L - 1 && !bj && !kb, i == 0 || bj || kb};
        if (i == g.L - 1 && (bj || kb)) x = {false, true};
        y = {bj && j != 0, j == 0};
        z = {kb && k != 0, k == 0};
        return (int)bi + (int)bj + (int)kb < 2;
    }

    template <int U4, int LV> __device__ __forceinline__ void step(Row<LV>& R, int p) const
    {
        constexpr int s0 = U4, s1 = (U4 + 3) & 3, s2 = (U4 + 2) & 3, s3 = (U4 + 1) & 3;  // planes p .. p-3
        constexpr int L0 = U4 & 1, L1 = L0 ^ 1;
        const int e = R.e, j = R.j;
        // (a) U of plane p, then the load of plane p+2
        R.U[s0] = R.n1.wide();
        sm.u[L0][e][lane] = R.U[s0];
        R.n1 = R.n2;
        R.n2 = load(R, p + 2);
        if constexpr (LV >= 1) {
            const bool jin = j > 0 && j < g.N - 1;
            // (b) the velocity of plane p-1
            const int q = p - 1;
            if (q >= 0 && q < g.L && j >= 0 && j < g.N) {
                const double2 c = R.U[s1], xp = R.U[s0], xm = R.U[s2];
                const double2 zp = lane_shift2<DPP_NEXT, double>(c), zm = lane_shift2<DPP_PREV, double>(c);
                const double2 yp = sm.u[L1][e + 1][lane], ym = sm.u[L1][e - 1][lane];
                double gxr, gxi, gyr, gyi, gzr, gzi;
                if (jin && !ktile && q > 0 && q < g.L - 1) {
                    gxr = lh2 * (xp.x - xm.x);
                    gxi = lh2 * (xp.y - xm.y);
                    gyr = lh2 * (yp.x - ym.x);
                    gyi = lh2 * (yp.y - ym.y);
                    gzr = lh2 * (zp.x - zm.x);
                    gzi = lh2 * (zp.y - zm.y);
                } else {
                    Ops ox, oy, oz;
                    const bool ok = kinds(q, j, ox, oy, oz);
                    gxr = ok ? diff(ox, xp.x, c.x, xm.x) : 0;
                    gxi = ok ? diff(ox, xp.y, c.y, xm.y) : 0;
                    gyr = ok ? diff(oy, yp.x, c.x, ym.x) : 0;
                    gyi = ok ? diff(oy, yp.y, c.y, ym.y) : 0;
                    gzr = ok ? diff(oz, zp.x, c.x, zm.x) : 0;
                    gzi = ok ? diff(oz, zp.y, c.y, zm.y) : 0;
                }
                const double l_U2 = 1 / (2 * c.x * c.x + 2 * c.y * c.y + veps);
                R.vx[s1] = (c.x * gxi - c.y * gxr) * l_U2;
                R.vy[s1] = (c.x * gyi - c.y * gyr) * l_U2;
                R.vz[s1] = (c.x * gzi - c.y * gzr) * l_U2;
                sm.vx[L1][e - 1][lane] = R.vx[s1];
                sm.vz[L1][e - 1][lane] = R.vz[s1];
            }
            if constexpr (LV == 2) {
                // (c) the curl of plane p-2 (velocity planes p-1, p-2, p-3 in s1, s2, s3)
                const int cp = p - 2;
                if (cp >= i0 && cp < iend && j < g.N) {
                    const double xyn = lane_shift<DPP_NEXT>(R.vy[s2]), xyp = lane_shift<DPP_PREV>(R.vy[s2]);
                    const double xxn = lane_shift<DPP_NEXT>(R.vx[s2]), xxp = lane_shift<DPP_PREV>(R.vx[s2]);
                    const double zyp = sm.vz[L0][e][lane], zym = sm.vz[L0][e - 2][lane];
                    const double xyp1 = sm.vx[L0][e][lane], xym1 = sm.vx[L0][e - 2][lane];
                    double vzx, vyx, vzy, vxy, vyz, vxz;
                    bool ok = true;
                    if (jin && !ktile && cp > 0 && cp < g.L - 1) {
                        vzx = lh2 * (R.vz[s1] - R.vz[s3]);
                        vyx = lh2 * (R.vy[s1] - R.vy[s3]);
                        vzy = lh2 * (zyp - zym);
                        vxy = lh2 * (xyp1 - xym1);
                        vyz = lh2 * (xyn - xyp);
                        vxz = lh2 * (xxn - xxp);
                    } else {
                        Ops ox, oy, oz;
                        ok = kinds(cp, j, ox, oy, oz);
                        vzx = diff(ox, R.vz[s1], R.vz[s2], R.vz[s3]);
                        vyx = diff(ox, R.vy[s1], R.vy[s2], R.vy[s3]);
                        vzy = diff(oy, zyp, R.vz[s2], zym);
                        vxy = diff(oy, xyp1, R.vx[s2], xym1);
                        vyz = diff(oz, xyn, R.vy[s2], xyp);
                        vxz = diff(oz, xxn, R.vx[s2], xxp);
                    }
                    double ox = vzy - vyz, oy = vxz - vzx, oz = vyx - vxy;
                    double on = sqrt(ox * ox + oy * oy + oz * oz);
                    if (!ok) ox = oy = oz = on = 0;
                    if (kout) {
                        const long pp = (long)cp * g.si + R.ro;
                        // streaming stores: the four outputs are not read
                        // again by this launch (3.8 % faster per call at 256^3)
                        if (wx) __builtin_nontemporal_store(ox, &wx[pp]);
                        if (wy) __builtin_nontemporal_store(oy, &wy[pp]);
                        if (wz) __builtin_nontemporal_store(oz, &wz[pp]);
                        if (W) __builtin_nontemporal_store(on, &W[pp]);
                    }
                }
            }
        }
    }
    // a wave's march over its rows: every wave runs the same steps and barriers
    template <typename... Rows> __device__ __forceinline__ void march(Rows&... R) const
    {
        const int pstart = i0 - 2;
        const int nstep = (iend - i0 + 4 + 3) & ~3;  // whole groups of four steps
        ((R.n1 = load(R, pstart)), ...);
        ((R.n2 = load(R, pstart + 1)), ...);
        for (int q0 = 0; q0 < nstep; q0 += 4) {
            static_for<0, 4>([&](auto uc) {
                constexpr int u4 = decltype(uc)::value;
                (step<u4>(R, pstart + q0 + u4), ...);
                __syncthreads();  // this step's LDS planes are complete; the previous step's may be overwritten
            });
        }
    }
};

// TJ owned rows on TJ + 1 waves
template <typename T, bool COMP, int TJ>
__global__ __launch_bounds__((TJ + 1) * 64) void vort_march_kernel(const c2<T>* __restrict__ u, const c2<T>* __restrict__ ulo,
                                                                   double lh2, double veps, Dims3 g, VortMarch vm,
                                                                   double* __restrict__ wx, double* __restrict__ wy,
                                                                   double* __restrict__ wz, double* __restrict__ W)
{
    constexpr int TE = TJ + 4;
    __shared__ VortLds<TJ> sm;
    const int t = (blockIdx.x & 7) * vm.per_xcd + (blockIdx.x >> 3);
    if (t >= vm.tj * vm.tk * vm.ti) return;
    const int kt = t % vm.tk, rest = t / vm.tk;
    const int jt = rest % vm.tj, ci = rest / vm.tj;
    const int i0 = ci * vm.IC, k0 = kt * vm.kw, lane = threadIdx.x & 63;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int k = k0 - 2 + lane;
    using Tile = VortTile<T, COMP, TJ>;
    const Tile tile{sm, u, ulo, lh2, veps, g, wx, wy, wz, W, i0, min(i0 + vm.IC, g.L), jt * TJ, k, lane,
                    k >= 0 && k < g.M && lane >= 2 && lane < 2 + vm.kw, k == 0 || k == g.M - 1, k0 - 2 <= 0 || k0 - 2 + 63 >= g.M - 1};
    if (w < TJ) {
        typename Tile::template Row<2> r;
        tile.init(r, 2 + w);
        tile.march(r);
    } else {
        typename Tile::template Row<1> a, b;
        typename Tile::template Row<0> c, d;
        tile.init(a, 1);
        tile.init(b, TE - 2);
        tile.init(c, 0);
        tile.init(d, TE - 1);
        tile.march(a, b, c, d);
    }
}

}  // namespace

// the vorticity into wx, wy, wz, W (device pointers; any output may be
// null).  Grids need >= 3 points along every axis (checked by the callers).
template <typename T>
hipError_t launch_vorticity3d(const c2<T>* u, const c2<T>* ulo, int L, int N, int M, double lh2, double veps,
                              double* wx, double* wy, double* wz, double* W, hipStream_t st)
{
    // 7 owned rows on 8 waves, two workgroups per CU (15 rows: 256^3
    // FP64 179 us, against 168, both with 60 columns)
    constexpr int TJ = 7;
    Dims3 g;
    g.L = L;
    g.N = N;
    g.M = M;
    g.sj = M;
    g.si = (long)N * M;
    VortMarch vm;
    vm.tj = (N + TJ - 1) / TJ;
    // 56 columns where they need no more tiles than 60: the rows of 448 bytes
    // that each workgroup then writes end on 64-byte lines where M is a
    // multiple of 8 (256^3: 169 -> 151 us; elsewhere equal)
    vm.kw = (M + 55) / 56 == (M + 59) / 60 ? 56 : 60;
    vm.tk = (M + vm.kw - 1) / vm.kw;
    // chunks of 16 planes (256^3: 8 planes 180 us, 12 planes 162, 16 planes 151); shorter
    // ones, down to 4 planes, where those would not fill the chip once and the
    // shorter ones still run in one round (64^3: 4 planes 14 us, 16 planes 22)
    const long slots = 2L * device_cus();
    auto wgs = [&](int IC) { return (long)vm.tj * vm.tk * ((L + IC - 1) / IC); };
    vm.IC = 16;
    while (vm.IC > 4 && wgs(vm.IC - 1) <= slots) --vm.IC;
    vm.ti = (L + vm.IC - 1) / vm.IC;
    const long tiles = (long)vm.tj * vm.tk * vm.ti;
    if (tiles > (1L << 30)) return hipErrorInvalidValue;
    vm.per_xcd = (int)((tiles + 7) / 8);
    if constexpr (std::is_same<T, float>::value) {
        if (ulo) {
            hipLaunchKernelGGL((vort_march_kernel<T, true, TJ>), dim3(8 * vm.per_xcd), dim3((TJ + 1) * 64), 0, st, u,
                               ulo, lh2, veps, g, vm, wx, wy, wz, W);
            return hipGetLastError();
        }
    }
    hipLaunchKernelGGL((vort_march_kernel<T, false, TJ>), dim3(8 * vm.per_xcd), dim3((TJ + 1) * 64), 0, st, u, ulo, lh2,
                       veps, g, vm, wx, wy, wz, W);
    return hipGetLastError();
}

template hipError_t launch_vorticity3d<double>(const double2*, const double2*, int, int, int, double, double, double*,
                                               double*, double*, double*, hipStream_t);
template hipError_t launch_vorticity3d<float>(const float2*, const float2*, int, int, int, double, double, double*,
                                              double*, double*, double*, hipStream_t);

}  // namespace nlse
