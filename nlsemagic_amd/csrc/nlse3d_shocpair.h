// nlse3d_shocpair.h -- two 2SHOC RK4 stages per launch in 3D, marching along
// i (device code).
//
// A workgroup owns TJ rows (j) x 56 columns (k) and marches along i over a
// chunk of IC planes.  Lane l is column k0 - 4 + l (four halo columns each
// side); extended row e = 0 .. TJ+7 is row j0 - 4 + e.  At step p, a row of
// level
//   0 (e = 0, TE-1)      (a) takes plane p of the pair's input Y (loaded one
//                            step ahead) to LDS;
//   1 (e = 1, TE-2)      (b) also forms D = Lap_CD(Y)/h^2 of the first stage
//                            at plane p-1;
//   2 (e = 2, TE-3)      (c) F of the first stage at plane p-2: its output Y1;
//   3 (e = 3, TE-4)      (d) D of the second stage, from Y1, at plane p-3;
//   4 (e = 4 .. TE-5)    (e) F of the second stage at plane p-4 and the
//                            update; these are the owned rows.
// One barrier per plane.  An owned row has a wave of its own, and so has a row
// of level 3; the three rows of levels 0-2 of a side share one wave, whose
// work is about that of a level-3 row.  TJ + 4 waves: each SIMD gets the same
// work (TJ / 4 owned rows and one halo wave).
//
// Where the values come from:
//   - the wave's own row of any plane, Y, Y1 and both D, from register rings
//     (slot = (plane - first plane) mod 4);
//   - rows j+-1 of a plane of Y or Y1: read from LDS once, in the D phase, and
//     kept in register rings for the two steps after it, where they are edge
//     neighbours of the F phase (k+-1 by DPP);
//   - D of rows j+-1 from LDS.
// So every LDS array holds two planes (one being written, one being read) and
// an owned row makes nine reads and five writes of 64 values per plane.
// Bound: VALU issue (per plane and SIMD about 620 wave-instructions of 4
// clocks, 2480 clocks of the 1.4 us a plane takes with one workgroup per CU),
// and at 256^3 the loads (1.75 us per plane).  Before, one row per wave on 12
// waves and 4 owned rows (FP64) kept four planes of every array in LDS: about
// 1760 clocks of LDS reads and writes per plane for half the rows.  Per RK4
// step at 256^3 (chunks as now): FP64 1014 -> 705 us, FP32c 548 -> 433 us;
// 128^3 FP64 194 -> 121 us.  12 waves (TJ = 8, FP64) leave 168 VGPRs, 16
// (TJ = 12, FP32) 128; TJ = 4 in FP64 and 8 in FP32 were slower at every size
// of 96^3 and more (256^3: 926 and 471 us).
//
// Per point a pair moves the bytes of one fused stage (stages 1-2: Y, V in;
// Y2, ktot out; stages 3-4: Y2, V, U, ktot in; U out); D, the first stage's
// output and its ktot never leave the chip.  Lanes and rows in the halo hold
// values no owned point depends on once their inputs reach beyond the tile
// (each stencil level loses one lane and one row on each side).  Boundary
// points follow the local rules (Dirichlet D, Lap0 F, zero otherwise) or MSD
// (below).  The floating-point operations and their order are those of
// NLSE3D_TAKE_STEPS_2SHOC.c:62-69, 239-259 and the RK4 stage algebra
// (:490-521), so results are bit-identical to one stage per launch and to
// the reference.
//
// MSD (template flag): F of a boundary point is i om U with om = Im(F/U) of
// its partner (each coordinate clamped into [1, n-2]), and its D is
// (A + (n1 - n)/a) U with A = Re(D conj U)/|U|^2 and n1 = s|U|^2 - V of the
// partner.  As in nlse3d_cdpair.h, the partner's values reach columns 0 and
// M-1 by DPP, plane 0 in the lane itself at the step of plane 1, plane L-1 one
// step later, and rows 0 and N-1 through LDS after a second barrier that only
// tiles holding such a row take.  Y1 of plane 0 reaches the neighbour rows
// through the slot of db that plane 0 leaves empty.  D on edges and corners is
// read by no point and left unset.  FP64 takes 4-row tiles there (8 waves, 209
// VGPRs, no spills; 8-row ones spilled 73 and were 10-15 % slower).  Per RK4
// step, one stage per launch / two: 97 x 120 x 111 FP32c 171 / 95 us,
// 157 x 149 x 163 FP64 642 / 371 us, 256^3 FP64 2944 / 1336 us.
//
// Every global load is issued on every step in the same order (clamped
// planes and rows; the values of planes and rows a step does not use are
// never read), and the load sequence before the loop is the one at the end
// of a step, so the compiler waits for each load by count instead of
// draining all of them at each step.  Offsets within a plane are 32-bit
// (N * M < 2^31).
#pragma once

#include <type_traits>

#include "nlse2d_strip.h"
#include "nlse3d_march.h"

namespace nlse {

template <typename T, int TJ, bool MSD>
struct ShocPairLds {
    static constexpr int TE = TJ + 8;
    c2<T> y[2][TE * 64];         // the pair's input, rows 0 .. TE-1
    c2<T> y1[2][(TE - 4) * 64];  // the first stage's output, rows 2 .. TE-3
    c2<T> da[2][(TE - 2) * 64];  // the first stage's D, rows 1 .. TE-2
    c2<T> db[2][(TE - 6) * 64];  // the second stage's D, rows 3 .. TE-4
    c2<T> kk[4][TJ * 64];        // the running ktot of owned rows (own lane only)
    // MSD, per stage of the pair: (A, n1) and om of rows 1 and N-2 (this
    // step); om of each lane's point in plane L-2 (kept for the next step)
    c2<T> an[MSD ? 2 : 1][2][MSD ? 64 : 1];
    T om[MSD ? 2 : 1][2][MSD ? 64 : 1];
    T oz1[MSD ? (TE - 4) * 64 : 1], oz2[MSD ? TJ * 64 : 1];
};

template <typename T, int FIRST, int TJ, bool MSD, typename Lds>
struct ShocPair {
    static constexpr int TE = TJ + 8;
    static constexpr bool SECOND = (FIRST == 3);
    static constexpr bool HAS_LO = SECOND && std::is_same<T, float>::value;

    // one extended row of this wave (members a level does not use cost nothing)
    template <int LV> struct Row {
        int e, j, ro;  // extended row, grid row, offset j * M + k within a plane (clamped into the grid)
        c2<T> Y[4];    // stage input of planes p .. p-3
        T V[4];        // V of planes p .. p-3
        c2<T> Xj[4], Xm[4];  // rows j+1, j-1 of the stage input, planes p-1 .. p-3
        c2<T> D[4];          // first stage's D, planes p-1 .. p-3
        c2<T> Y1[4];         // first stage's output, planes p-2 .. p-5
        c2<T> Bj[4], Bm[4];  // its rows j+1, j-1, planes p-3 .. p-5
        c2<T> D2[4];         // second stage's D, planes p-3 .. p-5
        // loaded ahead: the next input plane; the operands of the next step's
        // first-stage update (stages 3-4: U and ktot of plane p-1) and of its
        // second-stage update (U, V and U_lo of plane p-3)
        c2<T> Yn, Ua, Aa, Ub, Lb;
        T Vn, Vb;
        // MSD rows 0 and N-1: this step's operands, until the second barrier
        c2<T> ua, aa, ub, lb;
    };

    Lds& sm;
    const March3& g;
    const c2<T>* yin;
    const c2<T>* u;
    c2<T>* acc;
    c2<T>* yout;
    const T* V;
    const Coefs<T>& c;
    const int BC;
    c2<T>* ulo;
    const int i0, j0, k0, N, M, L, lane, k, kc, iend;
    const bool kb, own_k, kbc, jbc;
    const long si;

    __device__ __forceinline__ ShocPair(Lds& sm_, int i0_, int j0_, int k0_, const March3& g_, const c2<T>* yin_,
                                        const c2<T>* u_, c2<T>* acc_, c2<T>* yout_, const T* V_, const Coefs<T>& c_,
                                        int BC_, c2<T>* ulo_)
        : sm(sm_), g(g_), yin(yin_), u(u_), acc(acc_), yout(yout_), V(V_), c(c_), BC(BC_), ulo(ulo_), i0(i0_),
          j0(j0_), k0(k0_), N(g_.N), M(g_.M), L(g_.L), lane(threadIdx.x & 63), k(k0_ - 4 + lane),
          kc(k < 0 ? 0 : (k >= M ? M - 1 : k)), iend(min(i0_ + g_.IC, g_.L)), kb(k == 0 || k == M - 1),
          own_k(lane >= 4 && lane < 60 && k >= 0 && k < M),
          // MSD: the tile's lanes hold column 0 or M-1 / its rows 0 or N-1 (uniform)
          kbc(MSD && (has(4 - k0_, 64) || has(M - 1 - k0_ + 4, 64))),
          jbc(MSD && (has(4 - j0_, TE) || has(N - 1 - j0_ + 4, TE))), si((long)N * M)
    {
    }
    static __device__ __forceinline__ bool has(int x, int n) { return x >= 0 && x < n; }

    template <int LV> __device__ __forceinline__ void init(Row<LV>& R, int e) const
    {
        const c2<T> z = mk<T>(0, 0);
        R.e = e;
        R.j = j0 - 4 + e;
        R.ro = (R.j < 0 ? 0 : (R.j >= N ? N - 1 : R.j)) * M + kc;
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            R.Y[s] = R.Xj[s] = R.Xm[s] = R.D[s] = R.Y1[s] = R.Bj[s] = R.Bm[s] = R.D2[s] = z;
            R.V[s] = 0;
        }
    }
    __device__ __forceinline__ long plane(int pl, int lo, int hi) const
    {
        return (long)(pl < lo ? lo : (pl > hi ? hi : pl)) * si;
    }
    template <int LV> __device__ __forceinline__ void load_plane(Row<LV>& R, int pl) const
    {
        const long pb = plane(pl, 0, L - 1);
        R.Yn = (yin + pb)[R.ro];
        if constexpr (LV >= 1) R.Vn = (V + pb)[R.ro];
    }
    // U and ktot of plane pl (the first-stage update of stages 3-4)
    template <int LV> __device__ __forceinline__ void load_first(Row<LV>& R, int pl) const
    {
        if constexpr (SECOND && LV >= 2) {
            const long pa = plane(pl, 0, L - 1);
            R.Ua = (u + pa)[R.ro];
            R.Aa = (acc + pa)[R.ro];
        }
    }
    // U, V and the low part of plane pl (the second-stage update)
    template <int LV> __device__ __forceinline__ void load_second(Row<LV>& R, int pl) const
    {
        if constexpr (LV == 4) {
            const long pb = plane(pl, max(i0, 0), iend - 1);
            R.Ub = (u + pb)[R.ro];
            R.Vb = (V + pb)[R.ro];
            if constexpr (HAS_LO) R.Lb = ((ulo ? ulo : u) + pb)[R.ro];  // unused without a low part
        }
    }

    // D of an interior point (NLSE3D_TAKE_STEPS_2SHOC.c:62-69: i+1, i-1, j+1, j-1, k+1, k-1, centre)
    __device__ __forceinline__ c2<T> d_int(c2<T> m, c2<T> a, c2<T> b, c2<T> dj, c2<T> ej, c2<T> kn, c2<T> kp) const
    {
        return mk<T>(c.lh2 * (a.x + b.x + dj.x + ej.x + kn.x + kp.x - 6 * m.x),
                     c.lh2 * (a.y + b.y + dj.y + ej.y + kn.y + kp.y - 6 * m.y));
    }
    // F of an interior point (NLSE3D_TAKE_STEPS_2SHOC.c:239-259) from its
    // centre m, V, the sum of the twelve edge neighbours and the D values
    // (i+1, i-1, j+1, j-1, k+1, k-1, centre)
    __device__ __forceinline__ c2<T> f_int(c2<T> m, T vx, c2<T> es, c2<T> da, c2<T> db, c2<T> dd, c2<T> de, c2<T> df,
                                           c2<T> dh, c2<T> dm) const
    {
        const T wv = vx - c.s * (m.x * m.x + m.y * m.y);
        return mk<T>(c.a_12 * (da.y + db.y + dd.y + de.y + df.y + dh.y - 10 * dm.y) - c.a_6h2 * (es.y - 12 * m.y)
                         + wv * m.y,
                     -c.a_12 * (da.x + db.x + dd.x + de.x + df.x + dh.x - 10 * dm.x) + c.a_6h2 * (es.x - 12 * m.x)
                         - wv * m.x);
    }
    // the twelve edge neighbours, summed in source order: rows j+-1 of planes
    // i+1 (jn, mn), i (jc, mc) and i-1 (jp, mp), the row itself in planes i+1
    // (shifted: kn, kp) and i-1 (yp)
    __device__ __forceinline__ c2<T> edges(c2<T> jn, c2<T> mn, c2<T> jc, c2<T> mc, c2<T> jp, c2<T> mp, c2<T> kn,
                                           c2<T> kp, c2<T> yp) const
    {
        c2<T> es = jn;                                // (+1,+1, 0)
        auto add = [&](c2<T> v) {
            es.x = es.x + v.x;
            es.y = es.y + v.y;
        };
        add(lane_shift2<DPP_NEXT, T>(jc));            // ( 0,+1,+1)
        add(kn);                                      // (+1, 0,+1)
        add(mp);                                      // (-1,-1, 0)
        add(lane_shift2<DPP_PREV, T>(mc));            // ( 0,-1,-1)
        add(lane_shift2<DPP_PREV, T>(yp));            // (-1, 0,-1)
        add(mn);                                      // (+1,-1, 0)
        add(lane_shift2<DPP_PREV, T>(jc));            // ( 0,+1,-1)
        add(kp);                                      // (+1, 0,-1)
        add(jp);                                      // (-1,+1, 0)
        add(lane_shift2<DPP_NEXT, T>(mc));            // ( 0,-1,+1)
        add(lane_shift2<DPP_NEXT, T>(yp));            // (-1, 0,+1)
        return es;
    }
    // boundary values other than MSD's
    __device__ __forceinline__ c2<T> d_bnd(c2<T> m, T v) const
    {
        return (BC == BC_DIRICHLET) ? dir_d<T>(m, v, c) : mk<T>(0, 0);
    }
    __device__ __forceinline__ c2<T> f_bnd(c2<T> m, T v) const
    {
        return (BC == BC_LAP0) ? lap0_f<T>(m, v, c.s) : mk<T>(0, 0);
    }
    // MSD: (A, n1) of a partner, and D of a boundary point (value m, potential v) from it
    __device__ __forceinline__ c2<T> msd_an(c2<T> d, c2<T> m, T v) const
    {
        return mk<T>((d.x * m.x + d.y * m.y) / (m.x * m.x + m.y * m.y), nlin<T>(c.s, m, v));
    }
    __device__ __forceinline__ c2<T> msd_dd(c2<T> an, c2<T> m, T v) const
    {
        const T nb = nlin<T>(c.s, m, v);
        return mk<T>((an.x + c.l_a * (an.y - nb)) * m.x, (an.x + c.l_a * (an.y - nb)) * m.y);
    }
    // the first stage's update of a point from its F: the running ktot and
    // the stage's output (b: its input value, or for stages 3-4 the base U; a: ktot)
    __device__ __forceinline__ void fin1(c2<T> f, c2<T> b, c2<T> a, c2<T>& y1, c2<T>& kk) const
    {
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
    }
    // the second stage's update of the point pp from its F, ktot so far, base
    // U and (compensated) low part
    __device__ __forceinline__ void fin2(long pp, c2<T> f, c2<T> a, c2<T> b, c2<T> lo) const
    {
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
                comp_add<T>(b.x, lo.x, c.k6 * a.x);
                comp_add<T>(b.y, lo.y, c.k6 * a.y);
                st_stream<T>(&ulo[pp], lo);
                st_stream<T>(&yout[pp], b);
            } else {
                st_stream<T>(&yout[pp], mk<T>(b.x + c.k6 * a.x, b.y + c.k6 * a.y));
            }
        }
    }
    // MSD plane 0, at the step of plane 1: Y1 and ktot of the first stage (y0:
    // its input there), and the second stage's update
    template <int LV>
    __device__ __forceinline__ void plane0_first(const Row<LV>& R, T om, c2<T> y0, c2<T>& y1, c2<T>& kk) const
    {
        const c2<T> z = mk<T>(0, 0);
        fin1(msd_om<T>(om, y0), SECOND ? u[R.ro] : y0, SECOND ? acc[R.ro] : z, y1, kk);
    }
    template <int LV>
    __device__ __forceinline__ void plane0_second(const Row<LV>& R, T om, c2<T> y1, c2<T> kk) const
    {
        const c2<T> z = mk<T>(0, 0);
        if (own_k) fin2(R.ro, msd_om<T>(om, y1), kk, u[R.ro], (HAS_LO && ulo) ? ulo[R.ro] : z);
    }
    // planes each phase works on: D of the first stage on i0-3 .. iend+2, its
    // F on i0-2 .. iend+1, D of the second on i0-1 .. iend, its F on the
    // owned planes (each clipped to the grid)
    __device__ __forceinline__ bool in(int pl, int lo, int hi) const { return pl >= lo && pl <= hi && pl >= 0 && pl < L; }

    // the work of one row at step p (U4 = (p - first plane) mod 4)
    template <int U4, int LV> __device__ __forceinline__ void step(Row<LV>& R, int p) const
    {
        // slots of planes p, p-1, p-2, p-3 (p-4 shares p's, p-5 p-1's), and
        // the LDS slots of planes of p's parity and the other
        constexpr int s0 = U4, s1 = (U4 + 3) & 3, s2 = (U4 + 2) & 3, s3 = (U4 + 1) & 3;
        constexpr int L0 = U4 & 1, L1 = L0 ^ 1;
        const int e = R.e, j = R.j;
        const bool edge = MSD && (j == 0 || j == N - 1);  // follows after the second barrier
        const bool jin = j > 0 && j < N - 1;
        const bool part = jbc && (j == 1 || j == N - 2);
        // (a) plane p of the input, then the loads of plane p+1
        R.Y[s0] = R.Yn;
        if constexpr (LV >= 1) R.V[s0] = R.Vn;
        sm.y[L0][e * 64 + lane] = R.Yn;
        load_plane(R, p + 1);
        if constexpr (LV >= 1) {
            // (b) the first stage's D at plane p-1
            const int pd = p - 1;
            const c2<T> m = R.Y[s1];
            const c2<T> kn = lane_shift2<DPP_NEXT, T>(m), kp = lane_shift2<DPP_PREV, T>(m);
            R.Xj[s1] = sm.y[L1][(e + 1) * 64 + lane];
            R.Xm[s1] = sm.y[L1][(e - 1) * 64 + lane];
            if (in(pd, i0 - 3, iend + 2)) {
                const bool pin = pd > 0 && pd < L - 1;
                if (!MSD || (jin && pd > 0)) {
                    c2<T> dd = mk<T>(0, 0);
                    if (pin && jin) dd = d_int(m, R.Y[s0], R.Y[s2], R.Xj[s1], R.Xm[s1], kn, kp);
                    if constexpr (!MSD) {
                        if (!(pin && jin) || kb) dd = d_bnd(m, R.V[s1]);
                    } else if (!pin) {  // plane L-1 from plane L-2
                        dd = msd_dd(msd_an(R.D[s2], R.Y[s2], R.V[s2]), m, R.V[s1]);
                    } else if (kbc || part || pd == 1) {
                        const c2<T> an = msd_an(dd, m, R.V[s1]);
                        if (kbc) {
                            const c2<T> q = mk<T>(msd_col<T>(an.x, k, M), msd_col<T>(an.y, k, M));
                            if (kb) dd = msd_dd(q, m, R.V[s1]);
                        }
                        if (part && j == 1) sm.an[0][0][lane] = an;
                        if (part && j == N - 2) sm.an[0][1][lane] = an;
                        if (pd == 1) R.D[s2] = msd_dd(an, R.Y[s2], R.V[s2]);
                    }
                    R.D[s1] = dd;
                    sm.da[L1][(e - 1) * 64 + lane] = dd;
                }
            }
            if constexpr (LV >= 2) {
                // (c) the first stage's F at plane p-2, and Y1
                const int q = p - 2;
                if (MSD && edge) {
                    R.ua = R.Ua;
                    R.aa = R.Aa;
                }
                if (in(q, i0 - 2, iend + 1) && (!MSD || (jin && q > 0))) {
                    const c2<T> mq = R.Y[s2];
                    const bool pin = q > 0 && q < L - 1;
                    c2<T> f;
                    if (pin && jin) {
                        const c2<T> es = edges(R.Xj[s1], R.Xm[s1], R.Xj[s2], R.Xm[s2], R.Xj[s3], R.Xm[s3], kn, kp, R.Y[s3]);
                        const c2<T> dm = R.D[s2];
                        f = f_int(mq, R.V[s2], es, R.D[s1], R.D[s3], sm.da[L0][e * 64 + lane],
                                  sm.da[L0][(e - 2) * 64 + lane], lane_shift2<DPP_NEXT, T>(dm),
                                  lane_shift2<DPP_PREV, T>(dm), dm);
                    }
                    if constexpr (!MSD) {
                        if (!(pin && jin) || kb) f = f_bnd(mq, R.V[s2]);
                    } else if (!pin) {
                        f = msd_om<T>(sm.oz1[(e - 2) * 64 + lane], mq);
                    } else if (kbc || part || q == 1 || q == L - 2) {
                        T om = msd_rate<T>(f, mq);
                        if (kbc) om = msd_col<T>(om, k, M);
                        if (kb) f = msd_om<T>(om, mq);
                        if (part && j == 1) sm.om[0][0][lane] = om;
                        if (part && j == N - 2) sm.om[0][1][lane] = om;
                        if (q == L - 2) sm.oz1[(e - 2) * 64 + lane] = om;
                        if (q == 1) first_plane0<U4>(R, om);
                    }
                    c2<T> y1, kk;
                    fin1(f, SECOND ? R.Ua : mq, R.Aa, y1, kk);
                    R.Y1[s2] = y1;
                    sm.y1[L0][(e - 2) * 64 + lane] = y1;
                    if constexpr (LV == 4) sm.kk[s2][(e - 4) * 64 + lane] = kk;
                }
                load_first(R, p - 1);
            }
            if constexpr (LV >= 3) {
                // (d) the second stage's D at plane p-3, from Y1
                const int pd2 = p - 3;
                const c2<T> m1 = R.Y1[s3];
                const c2<T> bn = lane_shift2<DPP_NEXT, T>(m1), bp = lane_shift2<DPP_PREV, T>(m1);
                R.Bj[s3] = sm.y1[L1][(e - 1) * 64 + lane];
                R.Bm[s3] = sm.y1[L1][(e - 3) * 64 + lane];
                if (LV == 4 && MSD && p == 4) {  // Y1 of plane 0 came one step late, through db's empty slot
                    R.Bj[s0] = sm.db[L0][(e - 2) * 64 + lane];
                    R.Bm[s0] = sm.db[L0][(e - 4) * 64 + lane];
                }
                if (in(pd2, i0 - 1, iend) && (!MSD || (jin && pd2 > 0))) {
                    const bool pin = pd2 > 0 && pd2 < L - 1;
                    c2<T> dd = mk<T>(0, 0);
                    if (pin && jin) dd = d_int(m1, R.Y1[s2], R.Y1[s0], R.Bj[s3], R.Bm[s3], bn, bp);
                    if constexpr (!MSD) {
                        if (!(pin && jin) || kb) dd = d_bnd(m1, R.V[s3]);
                    } else if (!pin) {
                        dd = msd_dd(msd_an(R.D2[s0], R.Y1[s0], (V + (long)(L - 2) * si)[R.ro]), m1, R.V[s3]);
                    } else if (kbc || part || pd2 == 1) {
                        const c2<T> an = msd_an(dd, m1, R.V[s3]);
                        if (kbc) {
                            const c2<T> qa = mk<T>(msd_col<T>(an.x, k, M), msd_col<T>(an.y, k, M));
                            if (kb) dd = msd_dd(qa, m1, R.V[s3]);
                        }
                        if (part && j == 1) sm.an[1][0][lane] = an;
                        if (part && j == N - 2) sm.an[1][1][lane] = an;
                        if (pd2 == 1) R.D2[s0] = msd_dd(an, R.Y1[s0], V[R.ro]);
                    }
                    R.D2[s3] = dd;
                    sm.db[L1][(e - 3) * 64 + lane] = dd;
                }
                if constexpr (LV == 4) {
                    // (e) the second stage's F at plane p-4, and the update
                    // (Y1 planes: i+1 = p-3 in s3, i = p-4 in s0, i-1 = p-5 in s1)
                    const int q2 = p - 4;
                    if (MSD && edge) {
                        R.ub = R.Ub;
                        R.lb = R.Lb;
                    }
                    if (q2 >= i0 && q2 < iend && j >= 0 && j < N && (!MSD || (jin && q2 > 0))) {
                        const c2<T> mq = R.Y1[s0];
                        const bool pin = q2 > 0 && q2 < L - 1;
                        c2<T> f;
                        if (pin && jin) {
                            const c2<T> es =
                                edges(R.Bj[s3], R.Bm[s3], R.Bj[s0], R.Bm[s0], R.Bj[s1], R.Bm[s1], bn, bp, R.Y1[s1]);
                            const c2<T> dm = R.D2[s0];
                            f = f_int(mq, R.Vb, es, R.D2[s3], R.D2[s1], sm.db[L0][(e - 2) * 64 + lane],
                                      sm.db[L0][(e - 4) * 64 + lane], lane_shift2<DPP_NEXT, T>(dm),
                                      lane_shift2<DPP_PREV, T>(dm), dm);
                        }
                        if constexpr (!MSD) {
                            if (!(pin && jin) || kb) f = f_bnd(mq, R.Vb);
                        } else if (!pin) {
                            f = msd_om<T>(sm.oz2[(e - 4) * 64 + lane], mq);
                        } else if (kbc || part || q2 == 1 || q2 == L - 2) {
                            T om = msd_rate<T>(f, mq);
                            if (kbc) om = msd_col<T>(om, k, M);
                            if (kb) f = msd_om<T>(om, mq);
                            if (part && j == 1) sm.om[1][0][lane] = om;
                            if (part && j == N - 2) sm.om[1][1][lane] = om;
                            if (q2 == L - 2) sm.oz2[(e - 4) * 64 + lane] = om;
                            if (q2 == 1) plane0_second(R, om, R.Y1[s1], sm.kk[s1][(e - 4) * 64 + lane]);
                        }
                        if (own_k)  // kk: written at (c) two steps ago
                            fin2((long)q2 * si + R.ro, f, sm.kk[s0][(e - 4) * 64 + lane], R.Ub, R.Lb);
                    }
                    load_second(R, p - 3);
                }
            }
        }
    }
    // MSD plane 0 of the first stage, kept for the second
    template <int U4, int LV> __device__ __forceinline__ void first_plane0(Row<LV>& R, T om) const
    {
        constexpr int s3 = (U4 + 1) & 3, L1 = (U4 & 1) ^ 1;
        c2<T> y1, kk;
        plane0_first(R, om, R.Y[s3], y1, kk);
        R.Y1[s3] = y1;
        if constexpr (LV >= 3) sm.db[L1][(R.e - 3) * 64 + lane] = y1;
        if constexpr (LV == 4) sm.kk[s3][(R.e - 4) * 64 + lane] = kk;
    }
    // MSD rows 0 and N-1 of every phase's plane, from what their partner
    // rows left in LDS (plane 0 with plane 1)
    template <int U4, int LV> __device__ __forceinline__ void edge_row(Row<LV>& R, int p) const
    {
        constexpr int s0 = U4, s1 = (U4 + 3) & 3, s2 = (U4 + 2) & 3, s3 = (U4 + 1) & 3;
        constexpr int L0 = U4 & 1, L1 = L0 ^ 1;
        const int e = R.e, j = R.j;
        if (j != 0 && j != N - 1) return;
        const int side = j != 0;
        const int pa = p - 1, qa = p - 2, pb = p - 3, qb = p - 4;
        // every LDS value first, so their latencies overlap (unused where a
        // phase has no plane)
        c2<T> an1, an2, kk2;
        T om1 = 0, om2 = 0;
        if constexpr (LV >= 1) an1 = sm.an[0][side][lane];
        if constexpr (LV >= 2) om1 = qa < L - 1 ? sm.om[0][side][lane] : sm.oz1[(e - 2) * 64 + lane];
        if constexpr (LV >= 3) an2 = sm.an[1][side][lane];
        if constexpr (LV == 4) {
            om2 = qb < L - 1 ? sm.om[1][side][lane] : sm.oz2[(e - 4) * 64 + lane];
            kk2 = sm.kk[s0][(e - 4) * 64 + lane];
        }
        if constexpr (LV >= 1) {
            if (pa > 0 && pa < L - 1 && in(pa, i0 - 3, iend + 2))
                sm.da[L1][(e - 1) * 64 + lane] = msd_dd(an1, R.Y[s1], R.V[s1]);
        }
        if constexpr (LV >= 2) {
            if (qa > 0 && in(qa, i0 - 2, iend + 1)) {
                const c2<T> m = R.Y[s2];
                c2<T> y1, kk;
                fin1(msd_om<T>(om1, m), SECOND ? R.ua : m, R.aa, y1, kk);
                R.Y1[s2] = y1;
                sm.y1[L0][(e - 2) * 64 + lane] = y1;
                if constexpr (LV == 4) sm.kk[s2][(e - 4) * 64 + lane] = kk;
                if (qa == L - 2) sm.oz1[(e - 2) * 64 + lane] = om1;
                if (qa == 1) first_plane0<U4>(R, om1);
            }
        }
        if constexpr (LV >= 3) {
            if (pb > 0 && pb < L - 1 && in(pb, i0 - 1, iend))
                sm.db[L1][(e - 3) * 64 + lane] = msd_dd(an2, R.Y1[s3], R.V[s3]);
        }
        if constexpr (LV == 4) {
            if (qb > 0 && qb >= i0 && qb < iend) {
                if (qb == 1) plane0_second(R, om2, R.Y1[s1], sm.kk[s1][(e - 4) * 64 + lane]);
                if (own_k) fin2((long)qb * si + R.ro, msd_om<T>(om2, R.Y1[s0]), kk2, R.ub, R.lb);
                if (qb == L - 2) sm.oz2[(e - 4) * 64 + lane] = om2;
            }
        }
    }
    // a wave's march over its rows: every wave runs the same number of steps
    // and takes the same barriers
    template <typename... Rows> __device__ __forceinline__ void march(Rows&... R) const
    {
        const int pstart = i0 - 4;
        const int nstep = (iend - i0 + 8 + 3) & ~3;  // whole groups of four steps
        (load_plane(R, pstart), ...);
        (load_first(R, pstart - 2), ...);
        (load_second(R, pstart - 4), ...);
        for (int q0 = 0; q0 < nstep; q0 += 4) {
            static_for<0, 4>([&](auto uc) {
                constexpr int u4 = decltype(uc)::value;
                const int p = pstart + q0 + u4;
                (step<u4>(R, p), ...);
                if constexpr (MSD) if (jbc) {
                    __syncthreads();
                    (edge_row<u4>(R, p), ...);
                }
                __syncthreads();  // this step's LDS slots are complete; none is read at the step that writes it
            });
        }
    }
    __device__ __forceinline__ void run() const
    {
        const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
        if (w < TJ) {
            Row<4> r;
            init(r, 4 + w);
            march(r);
        } else if (w < TJ + 2) {
            Row<3> r;
            init(r, w == TJ ? 3 : TE - 4);
            march(r);
        } else {
            const bool low = w == TJ + 2;
            Row<2> r2;
            Row<1> r1;
            Row<0> r0;
            init(r2, low ? 2 : TE - 3);
            init(r1, low ? 1 : TE - 2);
            init(r0, low ? 0 : TE - 1);
            march(r2, r1, r0);
        }
    }
};

}  // namespace nlse
