// nlse3d_cdpair.h -- two CD RK4 stages per launch in 3D, marching along i
// (device code).
//
// A workgroup of NW waves owns TJ rows (j) x 60 columns (k) and marches
// along i over a chunk of IC planes.  Lane l is column k0 - 2 + l; extended
// row e = 0 .. TJ+3 is row j0 - 2 + e and belongs to wave e mod NW in every
// phase.  At step p:
//   (a) plane p of the pair's input Y arrives (with V, and for stages 3-4
//       the base U and ktot), loaded one step ahead;
//   (b) the first stage of the pair at plane p-1, extended rows 1 .. TJ+2:
//       its i-neighbours are the wave's own rows of planes p and p-2
//       (registers), its j-neighbours come from the LDS copy of plane p-1
//       written at the previous step, its k-neighbours from adjacent lanes;
//   (c) the second stage at plane p-2, owned rows, from the first stage's
//       output the same way, then the update is written;
//   (d) one barrier.
// The first stage's output and its ktot contribution never leave the chip:
// per point a pair moves the bytes of one fused stage (stages 1-2: Y, V in;
// Y2, ktot out; stages 3-4: Y2, V, U, ktot in; U out).  Boundary points
// follow the local rules (Lap0 F, zero otherwise) or MSD (below).  The
// floating-point operations and their order are those of
// NLSE3D_TAKE_STEPS_CD.c:59-71 and the RK4 stage algebra (:300-321), so
// results are bit-identical to the per-stage kernel and to the reference.
//
// MSD (template flag): a boundary point's F is i om U, with om = Im(F/U) of
// its partner, each coordinate clamped into [1, n-2] (NLSE3D_TAKE_STEPS_CD.c:
// 103-167), so one real om per partner point serves the face, edge and corner
// points around it.  It travels from the partner to
//   - columns 0 and M-1 by DPP, in the row's own wave;
//   - plane 0 in the lane itself, at the step of plane 1 (plane 0 is finished
//     one step late: nothing reads it before the second stage of plane 1);
//   - plane L-1 through an LDS slot of the lane, one step later;
//   - rows 0 and N-1 through LDS: their waves finish them after a second
//     barrier, which only tiles that hold such a row take.
// The launch lays tiles out so that each owns at least two rows, columns and
// planes of the grid, which keeps a partner in its boundary point's tile.
// Measured per RK4 step (157 x 149 x 163 FP64): 270 us with one stage per
// launch, 124 us with two (Dirichlet 112 us); 256^3 FP64 1144 -> 480 us.  The
// second barrier and the division cost 0.2-0.3 us per plane in boundary tiles.
#pragma once

#include <type_traits>

#include "nlse2d_strip.h"
#include "nlse3d_march.h"

namespace nlse {

template <typename T, int TJ, bool MSD>
struct CdPairLds {
    static constexpr int TE = TJ + 4;
    c2<T> y[2][TE][64];   // the pair's input, last two planes (slot = step parity)
    c2<T> y1[2][TE][64];  // the first stage's output, last two planes
    // MSD, per stage of the pair: om of rows 1 and N-2 (this step), and of
    // each lane's point in plane L-2 (kept for the next step)
    T om[MSD ? 2 : 1][2][64];
    T oz[MSD ? 2 : 1][MSD ? TE : 1][64];
};

template <typename T, int FIRST, int TJ, int NW, bool MSD, typename Lds>
__device__ __forceinline__ void cdpair_tile(Lds& sm, int i0, int j0, int k0, const March3& g,
                                            const c2<T>* __restrict__ yin, const c2<T>* u, c2<T>* __restrict__ acc,
                                            c2<T>* __restrict__ yout, const T* __restrict__ V, const Coefs<T>& c,
                                            int BC, c2<T>* ulo)
{
    constexpr int TE = TJ + 4, RW = (TE + NW - 1) / NW;
    constexpr bool SECOND = (FIRST == 3);  // stages 3-4: base U and ktot come in, U goes out
    const int lane = threadIdx.x & 63;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    __builtin_assume(w >= 0 && w < NW);
    const int N = g.N, M = g.M, L = g.L;
    const int k = k0 - 2 + lane;
    const int kc = k < 0 ? 0 : (k >= M ? M - 1 : k);
    const bool kin = k >= 0 && k < M;
    const bool own_k = lane >= 2 && lane < 62 && kin;
    const bool kb = (k == 0 || k == M - 1);
    // MSD: the tile's lanes hold column 0 or M-1 / its rows 0 or N-1 (uniform)
    const int lM = M - 1 - k0 + 2, eN = N - 1 - j0 + 2;
    const bool kbc = MSD && ((2 - k0 >= 0 && 2 - k0 < 64) || (lM >= 0 && lM < 64));
    const bool jbc = MSD && ((2 - j0 >= 0 && 2 - j0 < TE) || (eN >= 0 && eN < TE));
    const long si = (long)N * M;
    const c2<T> z = mk<T>(0, 0);

    constexpr bool HAS_LO = SECOND && std::is_same<T, float>::value;
    // row offsets (j * M + k, clamped into the grid) of each extended row and
    // of the owned row whose U_lo it loads (rows outside 2 .. TE-3 load a copy
    // of the nearest owned row, so every wave issues the same loads)
    int jrow[RW];
    long rowoff[RW], rob[RW];
#pragma unroll
    for (int r = 0; r < RW; ++r) {
        const int e = NW * r + w;
        const int j = j0 - 2 + e;
        jrow[r] = j;
        auto off = [&](int ee) -> long {
            const int jj = j0 - 2 + ee;
            return (long)(jj < 0 ? 0 : (jj >= N ? N - 1 : jj)) * M + kc;
        };
        rowoff[r] = off(e);
        rob[r] = off(e < 2 ? 2 : (e > TE - 3 ? TE - 3 : e));
    }
    // register rings (slot = (plane - pstart) mod 3): the input Y and V of
    // planes p, p-1, p-2; the first stage's output and its ktot part of
    // planes p-1, p-2, p-3; for stages 3-4 the base U and ktot of planes
    // p, p-1, p-2
    c2<T> Yr[3][RW], Y1r[3][RW], Kr[3][RW], Br[SECOND ? 3 : 1][RW], Ar[SECOND ? 3 : 1][RW];
    T Vr[3][RW];
    c2<T> Yn[RW], Bn[RW], An[RW], Ln[RW];
    T Vn[RW];
#pragma unroll
    for (int s = 0; s < 3; ++s)
#pragma unroll
        for (int r = 0; r < RW; ++r) {
            Yr[s][r] = Y1r[s][r] = Kr[s][r] = z;
            Vr[s][r] = 0;
            if constexpr (SECOND) Br[s][r] = Ar[s][r] = z;
        }
#pragma unroll
    for (int r = 0; r < RW; ++r) Bn[r] = An[r] = z;

    const int pstart = i0 - 2;
    const int iend = min(i0 + g.IC, L);
    const int nstep = (iend - i0 + 4 + 2) / 3 * 3;  // whole groups of three steps
    // Every global load is issued on every step in the same order (clamped
    // planes and rows; values of planes and rows a step does not use are never
    // read), and the loads before the loop are those of a step, so the
    // compiler waits for each load by count instead of draining all of them
    // at each step.
    auto plane = [&](int pl, int lo, int hi) -> long { return (long)(pl < lo ? lo : (pl > hi ? hi : pl)) * si; };
    auto load_plane = [&](int pl) {
        const long pb = plane(pl, 0, L - 1);
#pragma unroll
        for (int r = 0; r < RW; ++r) {
            Yn[r] = yin[pb + rowoff[r]];
            Vn[r] = V[pb + rowoff[r]];
            if constexpr (SECOND) {
                Bn[r] = u[pb + rowoff[r]];
                An[r] = acc[pb + rowoff[r]];
            }
        }
    };
    // CD F at a grid point from its value, V and the six neighbours in the
    // reference's order (+i, -i, +j, -j, +k, -k), with the boundary rules
    auto fcd = [&](bool interior, c2<T> m, T v, c2<T> a, c2<T> b, c2<T> d, c2<T> e, c2<T> f, c2<T> h) {
        if (interior) {
            const T wv = v - c.s * (m.x * m.x + m.y * m.y);
            return mk<T>(-c.ah2 * (a.y + b.y + d.y + e.y + f.y + h.y - 6 * m.y) + wv * m.y,
                         c.ah2 * (a.x + b.x + d.x + e.x + f.x + h.x - 6 * m.x) - wv * m.x);
        }
        return (BC == BC_LAP0) ? lap0_f<T>(m, v, c.s) : z;
    };
    // the first stage's update of a point from its F: the running ktot and
    // the stage's output (b: its input value, or for stages 3-4 the base U; a: ktot)
    auto fin1 = [&](c2<T> f, c2<T> b, c2<T> a, c2<T>& y1, c2<T>& kk) {
        if constexpr (!SECOND) {
            // stage 1: ktot = K1, Y1 = U + k/2 K1 (the input is U)
            kk = f;
            y1 = mk<T>(b.x + c.k2 * f.x, b.y + c.k2 * f.y);
        } else {
            // stage 3: ktot = ktot + 2 K3, Y3 = U + k K3
            a.x = a.x + (T)2.0 * f.x;
            a.y = a.y + (T)2.0 * f.y;
            kk = a;
            y1 = mk<T>(b.x + c.k * f.x, b.y + c.k * f.y);
        }
    };
    // the second stage's update of the point pp from its F, ktot so far, base
    // U and (compensated) low part.  By reference without MSD: by value, stages 3-4
    // in FP32 take 66 registers instead of 64, and a CU holds one workgroup instead
    // of two (900 x 1001 x 3 CD FP32 per step 529 -> 445 us, 512 x 512 x 16 174 ->
    // 154, 3 x 1001 x 900 72 -> 66, 256^3 279 -> 273).  MSD has one either way, and
    // by reference FP32 compensated loses 7 % (256^3 357 -> 384).
    using Arg = std::conditional_t<MSD, c2<T>, const c2<T>&>;
    auto fin2 = [&](long pp, Arg f, Arg ktot, Arg base, Arg low) {
        c2<T> a = ktot, b = base;
        if constexpr (!SECOND) {
            // stage 2: ktot = K1 + 2 K2, Y2 = U + k/2 K2
            a.x = a.x + (T)2.0 * f.x;
            a.y = a.y + (T)2.0 * f.y;
            st_stream<T>(&acc[pp], a);
            st_stream<T>(&yout[pp], mk<T>(b.x + c.k2 * f.x, b.y + c.k2 * f.y));
        } else {
            // stage 4: U + k/6 (ktot + K4), compensated when a low part is kept
            a.x = a.x + (T)1.0 * f.x;
            a.y = a.y + (T)1.0 * f.y;
            if (HAS_LO && ulo) {
                c2<T> lo = low;
                comp_add<T>(b.x, lo.x, c.k6 * a.x);
                comp_add<T>(b.y, lo.y, c.k6 * a.y);
                st_stream<T>(&ulo[pp], lo);
                st_stream<T>(&yout[pp], b);
            } else {
                st_stream<T>(&yout[pp], mk<T>(b.x + c.k6 * a.x, b.y + c.k6 * a.y));
            }
        }
    };
    // MSD: the second stage at plane 0 (owned row r, at the step of plane 1):
    // its base U and low part come straight from memory, once per launch
    auto fin2_plane0 = [&](int r, T om, c2<T> y1, c2<T> kk) {
        if (!own_k) return;
        const long pp = rowoff[r];
        fin2(pp, msd_om<T>(om, y1), kk, SECOND ? u[pp] : yin[pp], (HAS_LO && ulo) ? ulo[pp] : z);
    };
    auto colq1 = [&](T v) { return msd_col<T>(v, k, M); };
    // U_lo of the next step's update plane p-1 (compensated stages 3-4; read
    // from U and unused when there is no low part)
    auto load_lo = [&](int p) {
        if constexpr (HAS_LO) {
            const c2<T>* const src = ulo ? ulo : u;
            const long pb = plane(p - 1, max(i0, 0), iend - 1);
#pragma unroll
            for (int r = 0; r < RW; ++r) Ln[r] = src[pb + rob[r]];
        }
    };
    load_plane(pstart);
    load_lo(pstart - 1);
    for (int q0 = 0; q0 < nstep; q0 += 3) {
        static_for<0, 3>([&](auto uc) {
            constexpr int u3 = decltype(uc)::value;
            const int st = q0 + u3;
            const int p = pstart + st;
            constexpr int a0 = u3, a1 = (u3 + 2) % 3, a2 = (u3 + 1) % 3;  // planes p, p-1, p-2 (p-3 -> a0)
            const int lnow = st & 1, lprev = lnow ^ 1;
            // (a) plane p of the input, then the loads of plane p+1
#pragma unroll
            for (int r = 0; r < RW; ++r) {
                const int e = NW * r + w;
                Yr[a0][r] = Yn[r];
                Vr[a0][r] = Vn[r];
                if constexpr (SECOND) {
                    Br[a0][r] = Bn[r];
                    Ar[a0][r] = An[r];
                }
                if (e < TE) sm.y[lnow][e][lane] = Yn[r];
            }
            load_plane(p + 1);
            // (b) the first stage at plane q = p-1 (i0-1 .. iend), extended rows 1 .. TE-2
            const int q = p - 1;
            if (q >= 0 && q < L && q >= i0 - 1 && q <= iend) {
#pragma unroll
                for (int r = 0; r < RW; ++r) {
                    const int e = NW * r + w;
                    if (e < 1 || e > TE - 2) continue;
                    const c2<T> m = Yr[a1][r];
                    const c2<T> fp = lane_shift2<DPP_NEXT, T>(m), fm = lane_shift2<DPP_PREV, T>(m);
                    const int j = jrow[r];
                    c2<T> y1 = z, kk = z;
                    if constexpr (!MSD) {
                        if (kin && j >= 0 && j < N) {
                            const bool in = q > 0 && q < L - 1 && j > 0 && j < N - 1 && k > 0 && k < M - 1;
                            const c2<T> f = fcd(in, m, Vr[a1][r], Yr[a0][r], Yr[a2][r], sm.y[lprev][e + 1][lane],
                                                sm.y[lprev][e - 1][lane], fp, fm);
                            fin1(f, SECOND ? Br[SECOND ? a1 : 0][r] : m, SECOND ? Ar[SECOND ? a1 : 0][r] : z, y1, kk);
                        }
                    } else {
                        // rows 0 and N-1 follow at (d), plane 0 with plane 1
                        if (j <= 0 || j >= N - 1 || q == 0) continue;
                        c2<T> f;
                        if (q < L - 1) {
                            f = fcd(true, m, Vr[a1][r], Yr[a0][r], Yr[a2][r], sm.y[lprev][e + 1][lane],
                                    sm.y[lprev][e - 1][lane], fp, fm);
                            const bool part = jbc && (j == 1 || j == N - 2);
                            if (kbc || part || q == 1 || q == L - 2) {  // uniform
                                T om = msd_rate<T>(f, m);
                                if (kbc) om = colq1(om);
                                if (kb) f = msd_om<T>(om, m);
                                if (part && j == 1) sm.om[0][0][lane] = om;
                                if (part && j == N - 2) sm.om[0][1][lane] = om;
                                if (q == L - 2) sm.oz[0][e][lane] = om;
                                if (q == 1) {
                                    const c2<T> y0 = Yr[a2][r];
                                    fin1(msd_om<T>(om, y0), SECOND ? Br[SECOND ? a2 : 0][r] : y0,
                                         SECOND ? Ar[SECOND ? a2 : 0][r] : z, Y1r[a2][r], Kr[a2][r]);
                                }
                            }
                        } else {
                            f = msd_om<T>(sm.oz[0][e][lane], m);
                        }
                        fin1(f, SECOND ? Br[SECOND ? a1 : 0][r] : m, SECOND ? Ar[SECOND ? a1 : 0][r] : z, y1, kk);
                    }
                    Y1r[a1][r] = y1;
                    Kr[a1][r] = kk;
                    sm.y1[lnow][e][lane] = y1;
                }
            }
            // (c) the second stage at plane p-2, owned rows 2 .. TE-3, and the update
            const int q2 = p - 2;
            if (q2 >= i0 && q2 < iend) {
#pragma unroll
                for (int r = 0; r < RW; ++r) {
                    const int e = NW * r + w;
                    if (e < 2 || e > TE - 3) continue;
                    const c2<T> m = Y1r[a2][r];
                    const c2<T> fp = lane_shift2<DPP_NEXT, T>(m), fm = lane_shift2<DPP_PREV, T>(m);
                    const int j = jrow[r];
                    if constexpr (!MSD) {
                        if (!own_k || j >= N) continue;
                        const bool in = q2 > 0 && q2 < L - 1 && j > 0 && j < N - 1 && k > 0 && k < M - 1;
                        const c2<T> f = fcd(in, m, Vr[a2][r], Y1r[a1][r], Y1r[a0][r], sm.y1[lprev][e + 1][lane],
                                            sm.y1[lprev][e - 1][lane], fp, fm);
                        fin2((long)q2 * si + (long)j * M + k, f, Kr[a2][r],
                             SECOND ? Br[SECOND ? a2 : 0][r] : Yr[a2][r], HAS_LO ? Ln[r] : z);
                    } else {
                        if (j <= 0 || j >= N - 1 || q2 <= 0) continue;
                        c2<T> f;
                        T om = 0;
                        if (q2 < L - 1) {
                            f = fcd(true, m, Vr[a2][r], Y1r[a1][r], Y1r[a0][r], sm.y1[lprev][e + 1][lane],
                                    sm.y1[lprev][e - 1][lane], fp, fm);
                            const bool part = jbc && (j == 1 || j == N - 2);
                            if (kbc || part || q2 == 1 || q2 == L - 2) {  // uniform
                                om = msd_rate<T>(f, m);
                                if (kbc) om = colq1(om);
                                if (kb) f = msd_om<T>(om, m);
                                if (part && j == 1) sm.om[1][0][lane] = om;
                                if (part && j == N - 2) sm.om[1][1][lane] = om;
                                if (q2 == L - 2) sm.oz[1][e][lane] = om;
                                if (q2 == 1) fin2_plane0(r, om, Y1r[a0][r], Kr[a0][r]);
                            }
                        } else {
                            f = msd_om<T>(sm.oz[1][e][lane], m);
                        }
                        if (own_k)
                            fin2((long)q2 * si + (long)j * M + k, f, Kr[a2][r],
                                 SECOND ? Br[SECOND ? a2 : 0][r] : Yr[a2][r], HAS_LO ? Ln[r] : z);
                    }
                }
            }
            // (d) MSD rows 0 and N-1 of both stages' planes, from the om their
            // partner rows left in LDS
            if constexpr (MSD) if (jbc) {
                __syncthreads();
#pragma unroll
                for (int r = 0; r < RW; ++r) {
                    const int e = NW * r + w;
                    const int j = jrow[r];
                    if ((j != 0 && j != N - 1) || e < 1 || e > TE - 2) continue;
                    const int side = j != 0;
                    if (q > 0 && q < L && q >= i0 - 1 && q <= iend) {
                        const T om = q < L - 1 ? sm.om[0][side][lane] : sm.oz[0][e][lane];
                        const c2<T> m = Yr[a1][r];
                        fin1(msd_om<T>(om, m), SECOND ? Br[SECOND ? a1 : 0][r] : m, SECOND ? Ar[SECOND ? a1 : 0][r] : z,
                             Y1r[a1][r], Kr[a1][r]);
                        sm.y1[lnow][e][lane] = Y1r[a1][r];
                        if (q == L - 2) sm.oz[0][e][lane] = om;
                        if (q == 1) {
                            const c2<T> y0 = Yr[a2][r];
                            fin1(msd_om<T>(om, y0), SECOND ? Br[SECOND ? a2 : 0][r] : y0,
                                 SECOND ? Ar[SECOND ? a2 : 0][r] : z, Y1r[a2][r], Kr[a2][r]);
                        }
                    }
                    if (e >= 2 && e <= TE - 3 && q2 > 0 && q2 >= i0 && q2 < iend) {
                        const T om = q2 < L - 1 ? sm.om[1][side][lane] : sm.oz[1][e][lane];
                        if (q2 == 1) fin2_plane0(r, om, Y1r[a0][r], Kr[a0][r]);
                        if (own_k)
                            fin2((long)q2 * si + (long)j * M + k, msd_om<T>(om, Y1r[a2][r]), Kr[a2][r],
                                 SECOND ? Br[SECOND ? a2 : 0][r] : Yr[a2][r], HAS_LO ? Ln[r] : z);
                        if (q2 == L - 2) sm.oz[1][e][lane] = om;
                    }
                }
            }
            load_lo(p);
            __syncthreads();  // this step's LDS planes are complete; the previous step's may be overwritten
        });
    }
}

}  // namespace nlse
