// hc_fused.hpp -- the stage kernel's tile for Euler in FP64: the phases of StageTile (hc_stage.hpp)
// with the face arithmetic of hc_fused_flux.hpp and without the reference's operation order, which
// frees the phases of their branches:
//   1. load   : the state of the tile and a 2-cell halo into LDS, and the cell centres there; beyond a
//               non-periodic side the outermost cell again
//   2. qmetric: Q = sum over the four neighbours of dq (x) dx; a repeated cell adds zero, so every ring
//               cell takes the same straight-line path
//   3. faces  : increments d lim(g_c, g.n) from the directional weights w = X'^-1 n of the biased LSQ
//               factors (4 values a face instead of 6, and 4 operations a slope instead of 9).  Every
//               limiter but van Leer's (whose contexts keep StageTile) is homogeneous, d lim(a, b) = lim(d a, d b), so the weights hold the
//               distance d and the centred increment is the cell's share of the jump: 8 slots a face
//               for 10 (a 1000x901 AUSM+up box, bound by these bytes, 1376 -> 1242 us for 6 steps;
//               96 cylinders 13.87 -> 13.59 ms for 10)
//   4. cells  : R = F_left - F_right of the four faces (the wall flux of the far sides is stored
//               negated), then the Runge-Kutta accumulation and the update as StageTile has them
// Sums at the sides are in another order than the oracle's and products are fused: residuals agree to
// rounding of the face fluxes they are differences of, 2e-15 of the largest (vortex boxes of 64^2 to 400^2
// cells, every flux; relative to the residual itself that grows with the mesh, 3e-14 to 3e-13 there), and
// are the same bits in every tile shape, since every fused operation is explicit.
//
// Bound: latency of the load phase, then instruction issue (96 cylinders, a wavefront's 15.1k cycles: waits
// for the record and the tile 5.4k, metric 1.7k, faces 3.8k, cells 1.8k, barriers 2.4k; VALU busy 61 % at
// 4.2 waves a SIMD).  Against StageTile: the same 96 cylinders 18.9 -> 13.6 ms for 10 steps, a 2048x2048
// AUSM+up box 7.66 -> 2.99 ms for 4, a 256x512 cylinder 1.44 -> 0.97 ms for 20.
// Tried and slower: six waves with the fluxes stored over the state tile (spills off uniform geometry: 96
// cylinders 13.98 -> 15.07 ms), a persistent loop that loads the next tile during the cell phase (2048x2048
// 3.15 -> 3.76 ms).
#pragma once

#include "hc_fused_flux.hpp"
#include "hc_stage.hpp"

namespace hc {

// Off: byte offset into a plane of cells or faces: 32 bits where every plane is below 4 GiB, so that
// a load is a scalar base and one vector register; 64 bits otherwise.
template <int BASIS, int FLUX, int TI, int TJ, int NTHR, class Off, int UNI, int FOLD = 0> struct FusedTile {
    static constexpr int NV = 4, TILE_I = TI, TILE_J = TJ;
    static constexpr bool FOLDS = FOLD != 0;
    static constexpr int NC = TI * TJ, NT = NTHR;
    static constexpr int QH = TI + 4, QW = TJ + 4;   // state tile with a 2-cell halo
    static constexpr int MH = TI + 2, MW = TJ + 2;   // metric ring with a 1-cell halo
    static constexpr int NFI = (TI + 1) * TJ, NFJ = TI * (TJ + 1), NF = NFI + NFJ;
    static_assert(NF <= NT && NC <= NT && MH * MW <= NT, "one face, cell and metric per lane");
    // the i-faces fill whole wavefronts: the kind of a lane's face is wave-uniform
    static_assert(NFI % 64 == 0 && NT % 64 == 0, "wave-uniform face kind");
    static constexpr bool CPF = false, LPF = true, REREAD = true;
    static constexpr int CH = UNI ? 1 : QH, CW = UNI ? 1 : QW;

    struct Smem {
        double q[NV][QH][QW];
        double Q[NV][2][MH][MW];
        double F[NV + 1][NF];
        double gc[2][CH][CW];
    };
    struct Geo {
        double area, n0, n1, sl, wl0, wl1, wr0, wr1;
    };
    struct CellIn {
        double q0[NV], acc[NV], old[2][NV], vol, lam0;
    };

    HC_HD static double at(const double* p, Off o) { return *(const double*)((const char*)p + o); }
    // a value at a wave-uniform address, as a scalar load (geometry: written before the launch)
    HC_HD static double uniform(const double* p)
    {
#if defined(__HIP_DEVICE_COMPILE__)
        return *(const __attribute__((address_space(4))) double*)p;
#else
        return *p;
#endif
    }
    HC_HD static void put(double* p, Off o, double x) { *(double*)((char*)p + o) = x; }
    // byte offset of element r * w + c of a row-major plane
    HC_HD static Off offset(int r, int w, int c)
    {
#if defined(__HIP_DEVICE_COMPILE__)
        // rows and widths are below 2^24 where offsets are 32 bits wide (the launcher's rule)
        if constexpr (sizeof(Off) == 4) return Off((__umul24(r, w) + unsigned(c)) * 8u);
#endif
        return Off((long long)r * w + c) * 8;
    }

    // index of a halo cell: the periodic image, or the outermost cell beyond a non-periodic side; cells
    // further out than the halo of the last row are not read by any face and take any cell's values
    HC_HD static int halo(int g, int n, int per)
    {
        if (per) g = g < 0 ? g + n : g >= n ? g - n : g;
        return g < 0 ? 0 : g >= n ? n - 1 : g;
    }

    // whether the tile and its halo reach a periodic wrap (the same on every lane)
    HC_HD static bool wraps(const StageArgs<double>& a, int i0, int j0)
    {
        return (a.m.per_i && (i0 == 0 || i0 + TI + 1 >= a.m.ni)) || (a.m.per_j && (j0 == 0 || j0 + TJ + 1 >= a.m.nj));
    }

    // centre difference of the cells at state-tile positions pl, pr, left to right along i or j; across
    // a wrap the left cell's image, moved by the period: c_R - (c_L - period), the same bits from
    // either side of the wrap
    HC_HD static void centre_diff(const Smem& s, int pl, int pr, bool wrap, double px, double py, double& dx,
                                  double& dy)
    {
        const double* gc = &s.gc[0][0][0];
        dx = gc[pr] - (gc[pl] - (wrap ? px : 0.0));
        dy = gc[QH * QW + pr] - (gc[QH * QW + pl] - (wrap ? py : 0.0));
    }

    HC_HD static bool folded(const StageArgs<double>& a)
    {
#if defined(__HIP_DEVICE_COMPILE__)
        return FOLDS;
#else
        return a.fold_in != 0;
#endif
    }

    // updated() (hc_stage.hpp) with a cheaper finiteness check: 0 x finite = 0, and an infinity or NaN in
    // any variable leaves NaN
    HC_HD static void advance(const StageArgs<double>& a, const double* q0, const double* Rt, double fac, double* q1,
                              unsigned int& flag)
    {
        double qc[NV], nan = 0.0;
        to_conserved<double, LAW_EULER, BASIS>(a.sp, q0, qc);
        for (int v = 0; v < NV; ++v) qc[v] = qc[v] + Rt[v] * fac;
        from_conserved<double, LAW_EULER, BASIS>(a.sp, qc, q1);
        for (int v = 0; v < NV; ++v) nan = hc_fma(0.0, q1[v], nan);
        if (nan != nan) flag |= ST_NONFINITE;
        if (!(q1[2] > 0.0) || (BASIS == BASIS_PRIMITIVE && !(q1[3] > 0.0))) flag |= ST_NONPHYSICAL;
    }

    HC_HD static void load(const StageArgs<double>& a, Smem& s, int i0, int j0, int tid, unsigned int& flag)
    {
        for (int k = tid; k < QH * QW; k += NT) {
            const int li = k / QW, lj = k % QW;
            const int gi = halo(i0 - 2 + li, a.m.ni, a.m.per_i);
            const int gj = halo(j0 - 2 + lj, a.m.nj, a.m.per_j);
            const Off o = offset(gi, a.m.nj, gj);
            if (folded(a)) {
                double q0[NV], Rt[NV], q1[NV];
                for (int v = 0; v < NV; ++v) {
                    q0[v] = at(a.q0 + v * a.N, o);
                    Rt[v] = at(a.tmp_in + v * a.N, o);
                }
                const double vol = UNI ? uniform(a.m.cvol) : at(a.m.cvol, o);
                advance(a, q0, Rt, hc_div(a.beta_in * a.dt_in, vol), q1, flag);
                for (int v = 0; v < NV; ++v) s.q[v][li][lj] = q1[v];
                // a one-stage table: the update is the step's result
                if (a.mode == MODE_GLOBAL_STAGE0 && li >= 2 && li < TI + 2 && lj >= 2 && lj < TJ + 2 &&
                    i0 - 2 + li < a.m.ni && j0 - 2 + lj < a.m.nj)
                    for (int v = 0; v < NV; ++v) put(a.q_out + v * a.N, o, q1[v]);
            } else {
                for (int v = 0; v < NV; ++v) s.q[v][li][lj] = at(a.q_in + v * a.N, o);
            }
            if constexpr (!UNI) {
                s.gc[0][li][lj] = at(a.m.ccx, o);
                s.gc[1][li][lj] = at(a.m.ccy, o);
            }
        }
    }

    HC_HD static void qmetric(const StageArgs<double>& a, Smem& s, int i0, int j0, int tid)
    {
        if (tid >= MH * MW) return;
        const double* q = &s.q[0][0][0] + (tid / MW + 1) * QW + tid % MW + 1;
        double* Q = &s.Q[0][0][0][0] + tid;
        double dx[4], dy[4];
        const int nb[4] = {-QW, QW, -1, 1};
        if constexpr (UNI) {
            const double* b[2] = {a.m.fi, a.m.fj};
            const long long nf[2] = {a.m.nfi, a.m.nfj};
            for (int e = 0; e < 4; ++e) {
                dx[e] = uniform(b[e / 2] + FS_DX0 * nf[e / 2]);
                dy[e] = uniform(b[e / 2] + FS_DX1 * nf[e / 2]);
            }
        } else {
            const int c = int(q - &s.q[0][0][0]);
            if (wraps(a, i0, j0)) {
                const int ri = i0 - 1 + tid / MW, rj = j0 - 1 + tid % MW;
                const double px[2] = {a.m.period_i[0], a.m.period_j[0]}, py[2] = {a.m.period_i[1], a.m.period_j[1]};
                for (int e = 0; e < 4; ++e) {
                    // the edge's node line; 0 and the last one are the wrap
                    const int l = (e < 2 ? ri : rj) + e % 2, n = e < 2 ? a.m.ni : a.m.nj;
                    const bool wrap = (e < 2 ? a.m.per_i : a.m.per_j) && (l == 0 || l == n);
                    centre_diff(s, e % 2 ? c : c + nb[e], e % 2 ? c + nb[e] : c, wrap, px[e / 2], py[e / 2], dx[e],
                                dy[e]);
                }
            } else {
                for (int e = 0; e < 4; ++e)
                    centre_diff(s, e % 2 ? c : c + nb[e], e % 2 ? c + nb[e] : c, false, 0.0, 0.0, dx[e], dy[e]);
            }
        }
        for (int v = 0; v < NV; ++v) {
            const double c = q[v * QH * QW];
            double x = 0.0, y = 0.0;
            for (int e = 0; e < 4; ++e) {
                const double n = q[v * QH * QW + nb[e]];
                const double d = e % 2 ? n - c : c - n;
                x = hc_fma(d, dx[e], x);
                y = hc_fma(d, dy[e], y);
            }
            Q[(2 * v) * MH * MW] = x;
            Q[(2 * v + 1) * MH * MW] = y;
        }
    }

    // face k of the tile: i-faces k = li * TJ + lj, then j-faces
    HC_HD static bool kind_i(int k) { return wave_uniform(k) < NFI; }
    HC_HD static void pos(int k, bool isi, int& li, int& lj)
    {
        li = isi ? k / TJ : (k - NFI) / (TJ + 1);
        lj = isi ? k % TJ : (k - NFI) % (TJ + 1);
    }

    HC_HD static double slot(const double* b, Off o) { return UNI ? uniform(b) : at(b, o); }
    HC_HD static void slots(const double* b, long long nf, Off o, Geo& g)
    {
        g.area = slot(b + FS_AREA * nf, o);
        g.n0 = slot(b + FS_N0 * nf, o);
        g.n1 = slot(b + FS_N1 * nf, o);
        g.sl = slot(b + FS_XS * nf, o);
        g.wl0 = slot(b + FS_XL0 * nf, o);
        g.wl1 = slot(b + FS_XL1 * nf, o);
        g.wr0 = slot(b + FS_XR0 * nf, o);
        g.wr1 = slot(b + FS_XR1 * nf, o);
    }

    // the slots of the lane's face, loaded with the tile; lanes and faces beyond the tile or the mesh take
    // the last ones, so that every lane's registers are written
    HC_HD static void prefetch(const StageArgs<double>& a, int i0, int j0, int tid, Geo& g)
    {
        if (UNI) return;
        const int k = tid < NF ? tid : NF - 1;
        const bool isi = kind_i(k);
        int li, lj;
        pos(k, isi, li, lj);
        const int lmax = isi ? a.m.ni : a.m.nj, tmax = (isi ? a.m.nj : a.m.ni) - 1;
        int l = isi ? i0 + li : j0 + lj, t = isi ? j0 + lj : i0 + li;
        l = l < lmax ? l : (isi ? a.m.per_i : a.m.per_j) ? 0 : lmax;   // the wrap face is held on node line 0
        t = t < tmax ? t : tmax;
        slots(isi ? a.m.fi : a.m.fj, isi ? a.m.nfi : a.m.nfj, isi ? offset(l, a.m.nj, t) : offset(t, a.m.nj + 1, l), g);
    }

    HC_HD static void faces(const StageArgs<double>& a, Smem& s, int i0, int j0, int tid, unsigned int& flag, const Geo& pre)
    {
        if (tid >= NF) return;
        const int ni = a.m.ni, nj = a.m.nj;
        // both kinds' operands read before the selects: a select between addresses would keep the
        // arguments in memory
        const int per_i = a.m.per_i, per_j = a.m.per_j;
        const double pi0 = a.m.period_i[0], pi1 = a.m.period_i[1], pj0 = a.m.period_j[0], pj1 = a.m.period_j[1];
        const double *fi = a.m.fi, *fj = a.m.fj;
        const long long nfi = a.m.nfi, nfj = a.m.nfj;
        const bool isi = kind_i(tid);
        const double* base = isi ? fi : fj;
        const long long nf = isi ? nfi : nfj;
        const int per = isi ? per_i : per_j;
        const int bc0 = a.bc[0], bc1 = a.bc[1], bc2 = a.bc[2], bc3 = a.bc[3];
        int li, lj;
        pos(tid, isi, li, lj);
        const int l = isi ? i0 + li : j0 + lj;   // node line of the face
        const int t = isi ? j0 + lj : i0 + li;   // transverse cell index
        const int lmax = isi ? ni : nj;
        if (l > lmax || t >= (isi ? nj : ni)) return;
        const int pr = (li + 2) * QW + lj + 2, pl = pr - (isi ? QW : 1);   // right and left cell in the state tile
        const double* qs = &s.q[0][0][0];
        const double px = isi ? pi0 : pj0, py = isi ? pi1 : pj1;
        const bool wl = want_lambda(a);
        const bool two_sided = UNI || (l >= 1 && l < lmax) || per;
        // the few boundary faces after the others, which then hold no registers any more
        if (two_sided) {
            double F[NV], lam;
            Geo g = pre;
            if constexpr (UNI) slots(base, nf, Off(0), g);
            double ql[NV], qr[NV];
            for (int v = 0; v < NV; ++v) {
                ql[v] = qs[v * QH * QW + pl];
                qr[v] = qs[v * QH * QW + pr];
            }
            if (a.limiter != LIM_NOLIMIT1) {
                double dx, dy;
                if constexpr (UNI) {
                    dx = uniform(base + FS_DX0 * nf);
                    dy = uniform(base + FS_DX1 * nf);
                } else {
                    centre_diff(s, pl, pr, l == 0 || l == lmax, px, py, dx, dy);
                }
                const double* Qr = &s.Q[0][0][0][0] + (li + 1) * MW + lj + 1;
                const double* Ql = Qr - (isi ? MW : 1);
                double cl[NV], cr[NV], gl[NV], gr[NV], sl[NV], sr[NV];
                for (int v = 0; v < NV; ++v) {
                    const double dq = qr[v] - ql[v];
                    const int k0 = 2 * v * MH * MW, k1 = k0 + MH * MW;
                    cl[v] = dq * g.sl;
                    cr[v] = dq - cl[v];
                    gl[v] = hc_fma(hc_fma(-dq, dy, Ql[k1]), g.wl1, hc_fma(-dq, dx, Ql[k0]) * g.wl0);
                    gr[v] = hc_fma(hc_fma(-dq, dy, Qr[k1]), g.wr1, hc_fma(-dq, dx, Qr[k0]) * g.wr0);
                }
                fused_limit4(a.limiter, cl, gl, cr, gr, sl, sr);
                for (int v = 0; v < NV; ++v) {
                    ql[v] = ql[v] + sl[v];
                    qr[v] = qr[v] - sr[v];
                }
            }
            fused_flux<BASIS, FLUX>(a.sp, a.vscale, a.pscale, g.area, g.n0, g.n1, wl, ql, qr, F, lam);
            store(s, tid, wl, F, lam);
        }
        if (!UNI && !two_sided) {   // uniform geometry is periodic on all sides
            double F[NV], lam;
            // the interior cell is right of node line 0 and left of the last node line
            const bool first = l == 0;
            const int nc = first ? 0 : lmax - 1, pc = first ? pr : pl;
            double qi[NV];
            for (int v = 0; v < NV; ++v) qi[v] = qs[v * QH * QW + pc];
            boundary(a, (isi ? 0 : 2) + (first ? 0 : 1), first ? (isi ? bc0 : bc2) : (isi ? bc1 : bc3), base, nf,
                     isi ? offset(l, nj, t) : offset(t, nj + 1, l), qi, isi ? offset(nc, nj, t) : offset(t, nj, nc),
                     isi ? (long long)(first ? 0 : nj) + t : 2LL * nj + (first ? 0 : ni) + t, flag, F, lam);
            store(s, tid, wl, F, lam);
        }
    }

    HC_HD static void store(Smem& s, int k, bool wl, const double* F, double lam)
    {
        for (int v = 0; v < NV; ++v) s.F[v][k] = F[v];
        if (wl) s.F[NV][k] = lam;
    }

    // non-periodic boundary face, the flux from the left cell's side to the right's: ghost-cell flux
    // (ghostCellLoop.h:133-224) or wall flux (boundaryFluxLoop.h:150-261)
    HC_HD static void boundary(const StageArgs<double>& a, int bid, int type, const double* b, long long nf, Off of, const double* qi,
                               Off oc, long long row, unsigned int& flag, double* F, double& lam)
    {
        const double area = at(b + FS_AREA * nf, of), n0 = at(b + FS_N0 * nf, of), n1 = at(b + FS_N1 * nf, of);
        const bool far = bid == 1 || bid == 3;
        // the surface facing into the domain
        const FaceG<double> in{area, far ? -n0 : n0, far ? -n1 : n1};
        if (type == BC_WALL) {
            const FState s = fused_state<BASIS>(a.sp, qi);
            const double pa = (far ? -area : area) * s.p;
            F[0] = pa * in.n0;
            F[1] = pa * in.n1;
            F[2] = 0.0;
            F[3] = 0.0;
            lam = area * (hc_fabs(hc_fma(n0, s.u, n1 * s.v)) + hc_root(s.a2));
            return;
        }
        double qf[NV], qg[NV];
        for (int v = 0; v < NV; ++v) qf[v] = a.bref[row * NV + v];
        if (!ghost_value<double, LAW_EULER, BASIS>(a.sp, type, in, at(b + FS_CX * nf, of), at(b + FS_CY * nf, of),
                                                   at(a.m.ccx, oc), at(a.m.ccy, oc), qi, qf, qg))
            flag |= ST_BCNORMAL;
        double ql[NV], qr[NV];
        for (int v = 0; v < NV; ++v) {
            ql[v] = far ? qi[v] : qg[v];
            qr[v] = far ? qg[v] : qi[v];
        }
        fused_flux<BASIS, FLUX>(a.sp, a.vscale, a.pscale, area, n0, n1, true, ql, qr, F, lam);
    }

    // whether update u of the plan adds to an accumulator that the stage before left
    HC_HD static bool adds(const RkPlan& p, int u) { return u < p.nupd && !p.upd_first[u]; }

    // the spectral radii of the faces are summed where somebody reads the sum: stage 0 of a step whose
    // size comes from it, and stored residuals
    HC_HD static bool want_lambda(const StageArgs<double>& a)
    {
        return a.mode != MODE_FUSED || a.keep_res || (a.dt_mode == 1 && a.stage == 0);
    }

    // the cell phase's inputs, loaded once the lane's face is stored: in flight across the barrier
    HC_HD static void prefetch_cell(const StageArgs<double>& a, int i0, int j0, int tid, CellIn& ci)
    {
        const int i = i0 + tid / TJ, j = j0 + tid % TJ;
        if (tid >= NC || i >= a.m.ni || j >= a.m.nj || a.mode == MODE_RESIDUAL) return;
        const Off o = offset(i, a.m.nj, j);
        for (int v = 0; v < NV; ++v) ci.q0[v] = at(a.q0 + v * a.N, o);
        const RkPlan& p = a.plan;
        if (p.base >= 0)
            for (int v = 0; v < NV; ++v) ci.acc[v] = at(a.acc + ((long long)p.base * NV + v) * a.N, o);
#pragma unroll
        for (int u = 0; u < 2; ++u)
            if (adds(p, u))
                for (int v = 0; v < NV; ++v) ci.old[u][v] = at(a.acc + ((long long)p.upd_slot[u] * NV + v) * a.N, o);
        ci.vol = UNI ? uniform(a.m.cvol) : at(a.m.cvol, o);
        if (a.dt_mode == 1 && a.stage != 0) ci.lam0 = at(a.lam0, o);
    }

    HC_HD static void cells(const StageArgs<double>& a, const Smem& s, int i0, int j0, int tid, unsigned int& flag,
                            double& red, const CellIn& ci)
    {
        const int li = tid / TJ, lj = tid % TJ, i = i0 + li, j = j0 + lj;
        red = 0.0;
        if (tid >= NC || i >= a.m.ni || j >= a.m.nj) return;
        const int il = li * TJ + lj, ir = il + TJ, jl = NFI + li * (TJ + 1) + lj, jr = jl + 1;
        double R[NV];
        for (int v = 0; v < NV; ++v) R[v] = ((s.F[v][il] - s.F[v][ir]) + s.F[v][jl]) - s.F[v][jr];
        double lam = 0.0;
        if (want_lambda(a)) lam = ((s.F[NV][il] + s.F[NV][ir]) + s.F[NV][jl]) + s.F[NV][jr];
        const Off o = offset(i, a.m.nj, j);
        if (a.mode == MODE_RESIDUAL || a.keep_res) {
            double* r = a.res_out + ((long long)i * a.m.nj + j) * (NV + 1);
            for (int v = 0; v < NV; ++v) r[v] = R[v];
            r[NV] = lam;
            if (a.mode == MODE_RESIDUAL) return;
        }
        // Runge-Kutta accumulation (rungeKutta.h:176-197), in the reference's order
        const RkPlan& p = a.plan;
        double Rt[NV];
        for (int v = 0; v < NV; ++v) Rt[v] = (p.base >= 0 ? ci.acc[v] : 0.0) + R[v] * p.a_ss;
#pragma unroll
        for (int u = 0; u < 5; ++u) {
            if (u >= p.nupd) break;
            for (int v = 0; v < NV; ++v) {
                double* A = a.acc + ((long long)p.upd_slot[u] * NV + v) * a.N;
                double old = 0.0;
                if (!p.upd_first[u]) old = u < 2 ? ci.old[u < 2 ? u : 0][v] : at(A, o);
                put(A, o, old + R[v] * p.upd_coef[u]);
            }
        }
        if (a.mode == MODE_GLOBAL_STAGE0) {
            for (int v = 0; v < NV; ++v) put(a.tmp + v * a.N, o, Rt[v]);
            red = hc_div(lam, ci.vol);   // spectralRadius.h:33-35
            return;
        }
        double fac;
        if (a.dt_mode == 0) {
            fac = hc_div(p.beta * (folded(a) ? a.dt_in : a.dtslot[0]), ci.vol);
        } else {   // local steps (fixed ones keep the ordered tile)
            const double l0 = a.stage == 0 ? lam : ci.lam0;
            if (a.stage == 0) put(a.lam0, o, lam);
            fac = hc_div(p.beta * a.cfl, l0);
        }
        double qn[NV];
        advance(a, ci.q0, Rt, fac, qn, flag);
        for (int v = 0; v < NV; ++v) put(a.q_out + v * a.N, o, qn[v]);
    }
};

}   // namespace hc
