// 2D flux kernel in marching form: one wave per tile, lane = interface along
// the sweep, the lines of the tile visited one after another.
//
// The 2D flux of a line needs its two neighbour lines three times over (face
// conversion, transverse correction of the two-solve flux, flux correction).
// flux2d_kernel evaluates a 2D tile with all of them in LDS, so every halo line
// and interface is solved again by the neighbouring tiles (a 16 x 10 tile
// issues 1.6 first solves and 12.8 conservative conversions per cell) and its
// stages wait for each other at barriers.  Here a wave keeps the last two
// lines in registers and marches across the lines: each conservative
// conversion, face conversion and first solve is evaluated once per line (two
// halo lines per tile instead of 2 in 10, one halo interface in 63 instead of
// 1 in 16), there is no barrier, and no line but the current one is in flight
// in LDS.  The values are those of flux2d_kernel operation for operation.
//
// Bound by FP64 issue: 4.1e3 of the 5.5e3 cycles of a PPM/HLLC line are vector
// issue, a line costing 2.0e7 / (1024^2 / 63) wave instructions where the tiles
// spend 4.2e7.  Per launch (x, y sweep) at 1024^2 PPM/HLLC, tiles -> marching:
// 110, 119 -> 62, 69 us; at 2048^2 PLM/HLLC 307, 390 -> 200, 216 us; at 768^2
// WENO5/HLLD 141, 153 -> 98, 94 us (113, 108 with general divisions and
// roots; with one wave on a SIMD, the waves of a line's two solves run side by
// side).  Measured and left out: reading the
// states a whole line ahead (the registers spill, and a spill's reload waits
// for the loads before it), one wave per SIMD with all in registers (33 us of
// issue in 70), the line's values in LDS too, two lines per loop turn, and for
// MHD the next line's states a whole line ahead (100, 104 us).
#pragma once
#include "ah_kernels.h"

namespace ah {

// own cells of a tile: 63 of the 64 lanes are the left interface of one; LLF
// pairs each interface's radius with the next one's, which takes one more lane
template <int SOLVER>
constexpr int march_width() { return SOLVER == LLF ? 62 : 63; }

// waves that the registers leave room for on a SIMD
template <int MASK>
constexpr int march_waves() { return VS<MASK>::MHD ? 1 : 2; }

// lines of a tile
constexpr int MARCH_LINES_MIN = 3, MARCH_LINES_MAX = 24;

// Tile.pad of the marching kernel: own cells along the sweep, own lines
constexpr int march_pad(int width, int lines) { return (lines << 8) | width; }

// the next lane's value (0 in lane 63)
__device__ inline double lane_next(double x) {
    constexpr int WAVE_SHL1 = 0x130;
    const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(x), WAVE_SHL1, 0xf, 0xf, false);
    const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(x), WAVE_SHL1, 0xf, 0xf, false);
    return __hiloint2double(hi, lo);
}

// the five face-averaged quantities of one line that the correction differences across lines
template <int MASK>
struct MarchLine {
    V8<double> qm, qp, fm, fp, fa;
};

template <int MASK>
__device__ inline V8<double> sub8(const V8<double>& a, const V8<double>& b) {
    V8<double> d = zero8<double, MASK>();
#pragma unroll
    for (int c = 0; c < 8; ++c)
        if (VS<MASK>::live(c)) d.c[c] = a.c[c] - b.c[c];
    return d;
}

// x - K24 (dp - dm): the transverse correction of x with forward and backward differences
template <int MASK>
__device__ inline V8<double> corr8(const V8<double>& x, const V8<double>& dp, const V8<double>& dm) {
    V8<double> r = zero8<double, MASK>();
#pragma unroll
    for (int c = 0; c < 8; ++c)
        if (VS<MASK>::live(c)) r.c[c] = x.c[c] - K24 * (dp.c[c] - dm.c[c]);
    return r;
}

// CONV: 1 = point conversion of the interface states (PLM), 2 = 4th-order face
// conversion (PPM/WENO).  Grid: one 64-thread workgroup per tile, looping over
// the list beyond the grid.
template <int MASK, int SOLVER, int CONV, int AX>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(march_waves<MASK>())))
void flux2d_march_kernel(SweepArgs a) {
    using V = VS<MASK>;
    using Wave = typename std::conditional<SOLVER == HLLD, HlldWave<double>, HllcWave<double>>::type;
    constexpr int NV = V::NV;
    constexpr bool LAM = SOLVER == LLF;
    constexpr bool FAST = !V::MHD || SOLVER == HLLD;
    static_assert(CONV == 1 || CONV == 2, "the cell-centred form reads the stage input: flux2d_kernel");
    // x sweep: the lanes lie across the state's rows, so four lines of flux
    // differences are turned in LDS and written as 32-byte segments
    constexpr int TL = 4, TP = 68;
    __shared__ double turn[AX == 0 ? NV : 1][AX == 0 ? TL : 1][AX == 0 ? TP : 1];
    // differences of the five face-averaged quantities to the line before, one
    // column per lane: they are read once per line, and the 5 NV doubles in
    // registers would cost the second wave of the SIMD
    __shared__ double dback[5][NV][64];

    const int lane = threadIdx.x;
    const int ntiles_ = wave_uniform(a.ntiles_dev ? *a.ntiles_dev : a.ntiles);
    const double* wLg = reinterpret_cast<const double*>(a.wL);
    const double* wRg = reinterpret_cast<const double*>(a.wR);
    const double* bng = reinterpret_cast<const double*>(a.bn);
    const long long P = a.plane;
    for (int ti_ = blockIdx.x; ti_ < ntiles_; ti_ += gridDim.x) {
    const Tile tile = ld_const(a.tiles + ti_);
    const ProbDesc pd = ld_const(a.pd + tile.prob);
    ProbState* ps = a.ps + tile.prob;
    if (!ld_const(&ps->active)) continue;
    const int ns = AX == 0 ? pd.n0 : pd.n1, nt = AX == 0 ? pd.n1 : pd.n0;
    const bool edge = pd.bc == EDGE;
    const int s0 = tile.s0, t0 = tile.t0, width = tile.pad & 255, t1 = t0 + (tile.pad >> 8);
    const double gamma = pd.gamma;
    const long long off = pd.off;
    const int parity = a.parity_override >= 0 ? a.parity_override : ld_const(&ps->parity);
    const int sax = a.compat ? AX : (parity == 0 ? AX : 1 - AX);
    const int mom = a.compat ? sax + 1 : 1;  // the momentum HLLC's star state sets (solvers.py:127-128)
    const int k = s0 + lane;
    const int km = bcmap(k - 1, ns, pd.bc), kp = bcmap(k, ns, pd.bc);
    const bool own = lane < width;                                  // cell k is the tile's
    const bool jown = lane >= 1 && lane <= width && k <= ns;        // Jacobian position k is the tile's
    const DivDx bydx(pd.dx);
    int hit_;
    const double fdt = a.fuse_k2 ? step_dt(pd, *ps, 2, &hit_) : 0.0;

    auto line = [&](int t) { return bcmap(t, nt, pd.bc); };
    auto fetch = [&](int t, V8<double>& wm, V8<double>& wp) {
        const long long row = off + (long long)line(t) * ns;
        wm = load8<double, MASK>(wRg + row, P, km);
        wp = load8<double, MASK>(wLg + row, P, kp);
    };

    // lines at which the face averages are evaluated: the own ones and their
    // neighbours; beyond an edge the neighbour is the edge line itself
    const int c0 = edge && t0 == 0 ? 0 : t0 - 1;
    V8<double> wm, wp, dwm, dwp, dpm, dpp, hm, hp;
    // wave-uniform: the states of the line before and of this one are in the
    // range in which the short divisions and roots are exact
    bool okl = false, okw = false;
    double em_, ep_;  // energies of the states' conservative forms
    auto cons = [&](const V8<double>& w, double e) {
        V8<double> q = w;
        q.c[4] = e;
#pragma unroll
        for (int i = 1; i < 4; ++i)
            if (V::live(i)) q.c[i] = w.c[i] * w.c[0];
        return q;
    };
    {
        V8<double> lm, lp;
        fetch(c0 - 1, lm, lp);
        fetch(c0, wm, wp);
        fetch(c0 + 1, hm, hp);
        const V8<double> pm = prim_to_cons<double, MASK>(wm, gamma), pp = prim_to_cons<double, MASK>(wp, gamma);
        em_ = pm.c[4];
        ep_ = pp.c[4];
        if constexpr (CONV == 2) {
            dpm = sub8<MASK>(pm, prim_to_cons<double, MASK>(lm, gamma));
            dpp = sub8<MASK>(pp, prim_to_cons<double, MASK>(lp, gamma));
        }
        dwm = sub8<MASK>(wm, lm);
        dwp = sub8<MASK>(wp, lp);
        if constexpr (FAST) okl = __all(safe_states<MASK>(lm, lp, gamma));
    }
    MarchLine<MASK> x;      // face-averaged quantities of the line before
    V8<double> cwm, cwp;    // corrected interface states of the line before
    Wave wavx;              // HLLC, HLLD: the waves of its second solve in their place
    double lamx = 0.0, bnx = 0.0, lmax = 0.0;
    bool bad = false;
    if constexpr (FAST) okw = __all(safe_states<MASK>(wm, wp, gamma));
#pragma unroll 1
    for (int c = c0; c <= t1; ++c) {
        MarchLine<MASK> y;
        V8<double> ywm, ywp;
        Wave wavy;
        double lamy = 0.0, bny = 0.0;
        const bool past = edge && c == nt;  // beyond the edge: the line before again
        if (!past) {
            if constexpr (SOLVER == HLLD) bny = bng[off + (long long)line(c) * ns + kp];
            // transverse correction of the states; for PPM/WENO it is also the
            // point value the face conversion converts (fv.py:105-122)
            const V8<double> fwm = sub8<MASK>(hm, wm), fwp = sub8<MASK>(hp, wp);
            ywm = corr8<MASK>(wm, fwm, dwm);
            ywp = corr8<MASK>(wp, fwp, dwp);
            const bool town = c >= t0 && c < t1;
            double em_n, ep_n;
            V8<double> gm, gp;  // the differences of the conservative states to the next line
            bool ok = true;
            double ro = 0.0;
            // the first solve of line c in arithmetic R
            auto first = [&](auto tag) {
                using R = decltype(tag);
                const R gR = R(gamma);
                auto up = [](const V8<double>& v) { return cast8<R, double, MASK>(v); };
                const V8<R> hpm = prim_to_cons<R, MASK>(up(hm), gR), hpp = prim_to_cons<R, MASK>(up(hp), gR);
                Iface<R> s;
                s.wm = up(wm);
                s.wp = up(wp);
                const V8<double> qcm = cons(wm, em_), qcp = cons(wp, ep_);
                if constexpr (CONV == 1) {
                    s.qm = up(qcm);
                    s.qp = up(qcp);
                } else {
                    s.qm = prim_to_cons<R, MASK>(up(ywm), gR);
                    s.qp = prim_to_cons<R, MASK>(up(ywp), gR);
#pragma unroll
                    for (int i = 0; i < 8; ++i)
                        if (V::live(i)) {
                            gm.c[i] = double(hpm.c[i]) - qcm.c[i];
                            gp.c[i] = double(hpp.c[i]) - qcp.c[i];
                            s.qm.c[i] = s.qm.c[i] + R(K24 * (gm.c[i] - dpm.c[i]));
                            s.qp.c[i] = s.qp.c[i] + R(K24 * (gp.c[i] - dpp.c[i]));
                        }
                }
                em_n = double(hpm.c[4]);
                ep_n = double(hpp.c[4]);
                s.fm = phys_flux<R, MASK, AX>(s.wm, gR);
                s.fp = phys_flux<R, MASK, AX>(s.wp, gR);
                {
                    // spectral radius at Jacobian position k; beyond an edge the
                    // nearest interior position's (plm.py:84-86).  Only LLF
                    // needs it on the halo lines, but a branch there would part
                    // the chains that the block runs side by side
                    const V8<R> st = CONV == 1 ? arith_avg<R, MASK>(s.wp, s.wm) : roe_avg<R, MASK>(s.wp, s.wm);
                    double r = double(spectral_radius<R, MASK, AX>(st, gR));
                    ro = (town & jown) ? r : 0.0;
                    if constexpr (LAM) {
                        double rn = lane_next(r);
                        if (edge) {
                            if (k == 0) r = rn;
                            if (k >= ns) rn = r;
                        }
                        lamy = nmax(r, rn);
                    }
                }
                V8<R> F;
                if constexpr (SOLVER == HLLC) {
                    // the waves of both solves of the line: independent chains
                    // of divisions and roots, in flight together
                    const HllcWave<R> h1 = hllc_wave<R, MASK>(s.wm, s.wp, sax, gR);
                    F = hllc_flux<R, MASK>(h1, s.qm, s.qp, s.fm, s.fp, mom, a.compat != 0);
                    __builtin_amdgcn_sched_barrier(0);
                    const HllcWave<R> h2 = hllc_wave<R, MASK>(up(ywm), up(ywp), sax, gR);
                    wavy.k = double(h2.k);
                    wavy.sS = double(h2.sS);
                    wavy.mom = double(h2.mom);
                    wavy.en = double(h2.en);
                    wavy.sel = h2.sel;
                } else if constexpr (SOLVER == HLLD) {
                    auto both = [&](auto axis) {
                        constexpr int S = decltype(axis)::value;
                        bool ok2 = true;
                        const HlldWave<R> h1 = hlld_wave<R, MASK, S>(s.wm, s.wp, R(bny), gR, &ok);
                        const HlldWave<R> h2 = hlld_wave<R, MASK, S>(up(ywm), up(ywp), R(bny), gR, &ok2);
                        ok = ok && ok2;
                        auto dn = [](const V8<R>& v) { return cast8<double, R, MASK>(v); };
                        F = cast8<R, double, MASK>(hlld_flux<double, MASK, S>(wide(h1), bny, dn(s.qm), dn(s.qp), dn(s.fm), dn(s.fp)));
                        wavy = wide(h2);
                    };
                    if (sax == 0) both(std::integral_constant<int, 0>{});
                    else both(std::integral_constant<int, 1>{});
                } else {
                    F = riemann<R, MASK, SOLVER, AX>(s, R(lamy), sax, R(bny), gR, sax + 1, a.compat != 0);
                }
                y.qm = cast8<double, R, MASK>(s.qm);
                y.qp = cast8<double, R, MASK>(s.qp);
                y.fm = cast8<double, R, MASK>(s.fm);
                y.fp = cast8<double, R, MASK>(s.fp);
                y.fa = cast8<double, R, MASK>(F);
            };
            bool fast = false;
            if constexpr (FAST) {
                const bool okh = __all(safe_states<MASK>(hm, hp, gamma));
                fast = okl && okw && okh;
                if constexpr (V::MHD) fast = fast && __all(safe_states<MASK>(ywm, ywp, gamma) && safe_field(bny));
                else fast = fast && __all(safe_derived(ywm, ywp));
                okl = okw;
                okw = okh;
            }
            if (FAST && fast) {
                first(fd(0.0));
                if constexpr (V::MHD) fast = __all(ok);
            }
            if (!(FAST && fast)) first(0.0);
            bad = bad | !(ro <= 1.7976931348623157e308);
            lmax = ((ro > lmax) | (ro != ro)) ? ro : lmax;
            if constexpr (CONV == 2) {
                dpm = gm;
                dpp = gp;
            }
            em_ = em_n;
            ep_ = ep_n;
            wm = hm;
            wp = hp;
            dwm = fwm;
            dwp = fwp;
            // the states of the line after the next: in flight during the second solve
            if (c < t1) fetch(c + 2, hm, hp);
        } else {
            y = x;
        }
        if (c > c0) {
            // the flux of line c - 1 if it is the tile's, and the differences to line c
            const int t = c - 1;
            auto turnd = [&](int q, const V8<double>& yv, const V8<double>& xv) {
                // the line before's value corrected; leaves the difference of the pair behind
                V8<double> r = zero8<double, MASK>();
#pragma unroll
                for (int i = 0; i < 8; ++i)
                    if (V::live(i)) {
                        const double d = yv.c[i] - xv.c[i];
                        r.c[i] = xv.c[i] - K24 * (d - dback[q][V::slot(i)][lane]);
                        dback[q][V::slot(i)][lane] = d;
                    }
                return r;
            };
            auto keep = [&](int q, const V8<double>& yv, const V8<double>& xv) {
#pragma unroll
                for (int i = 0; i < 8; ++i)
                    if (V::live(i)) dback[q][V::slot(i)][lane] = yv.c[i] - xv.c[i];
            };
            if (t >= t0) {
                // what the end of the line reads: in flight during the second solve
                double ld[3][NV];
                const long long j0 = off + (long long)t * ns + k;
                if constexpr (AX == 1) {
                    if (own) {
#pragma unroll
                        for (int v = 0; v < NV; ++v) ld[0][v] = a.Dprev[v * P + j0];
                        if (a.fuse_k2) {
#pragma unroll
                            for (int v = 0; v < NV; ++v) {
                                ld[1][v] = a.fuse_u[v * P + j0];
                                ld[2][v] = a.fuse_k1[v * P + j0];
                            }
                        }
                    }
                }
                Iface<double> s;
                s.wm = cwm;
                s.wp = cwp;
                s.qm = turnd(0, y.qm, x.qm);
                s.qp = turnd(1, y.qp, x.qp);
                s.fm = turnd(2, y.fm, x.fm);
                s.fp = turnd(3, y.fp, x.fp);
                V8<double> F;
                if constexpr (SOLVER == HLLC)
                    F = hllc_flux<double, MASK>(wavx, s.qm, s.qp, s.fm, s.fp, mom, a.compat != 0);
                else if constexpr (SOLVER == HLLD)
                    F = sax == 0 ? hlld_flux<double, MASK, 0>(wavx, bnx, s.qm, s.qp, s.fm, s.fp)
                                 : hlld_flux<double, MASK, 1>(wavx, bnx, s.qm, s.qp, s.fm, s.fp);
                else F = riemann<double, MASK, SOLVER, AX>(s, lamx, sax, bnx, gamma, sax + 1, a.compat != 0);
#pragma unroll
                for (int i = 0; i < 8; ++i)
                    if (V::live(i)) {
                        const double d = y.fa.c[i] - x.fa.c[i];
                        F.c[i] = F.c[i] - K24 * (d - dback[4][V::slot(i)][lane]);
                        dback[4][V::slot(i)][lane] = d;
                    }
                // (the interface behind the last cell is the last tile's: a tile
                // before it may reach it too, with a lane that has no neighbour)
                if (a.flux_out && (own || (lane == width && k == ns))) {
#pragma unroll
                    for (int i = 0; i < 8; ++i)
                        if (V::live(i)) a.flux_out[V::slot(i) * a.flux_plane + (long long)k * nt + t] = F.c[i];
                }
                double df[NV];
#pragma unroll
                for (int i = 0; i < 8; ++i)
                    if (V::live(i)) df[V::slot(i)] = bydx(lane_next(F.c[i]) - F.c[i]);
                if constexpr (AX == 0) {
                    const int n = (t - t0) & (TL - 1);
#pragma unroll
                    for (int v = 0; v < NV; ++v) turn[v][n][lane] = df[v];
                    if (n == TL - 1 || t == t1 - 1) {
                        __builtin_amdgcn_wave_barrier();  // one wave: its LDS accesses are in order
                        const int tt = lane & (TL - 1);
#pragma unroll
                        for (int i = 0; i < TL; ++i) {
                            const int sl = (64 / TL) * i + lane / TL;
                            if (sl < width && tt <= n) {
                                const long long j = off + (long long)(s0 + sl) * pd.n1 + (t - n + tt);
#pragma unroll
                                for (int v = 0; v < NV; ++v) a.out[v * P + j] = turn[v][tt][sl];
                            }
                        }
                        __builtin_amdgcn_wave_barrier();
                    }
                } else if (own) {
#pragma unroll
                    for (int v = 0; v < NV; ++v) df[v] = -(ld[0][v] + df[v]);
                    if (a.fuse_k2) {
#pragma unroll
                        for (int v = 0; v < NV; ++v)
                            a.fuse_k2[v * P + j0] = .25 * (3 * ld[1][v] + ld[2][v] + fdt * df[v]);
                    } else {
#pragma unroll
                        for (int v = 0; v < NV; ++v) a.out[v * P + j0] = df[v];
                    }
                }
            } else {
                keep(0, y.qm, x.qm);
                keep(1, y.qp, x.qp);
                keep(2, y.fm, x.fm);
                keep(3, y.fp, x.fp);
                keep(4, y.fa, x.fa);
            }
        } else {
            // the first line; at a lower edge the line before it is itself
            // (elsewhere the difference is not read)
            auto start = [&](int q, const V8<double>& yv) {
#pragma unroll
                for (int i = 0; i < 8; ++i)
                    if (V::live(i)) {
                        dback[q][V::slot(i)][lane] = yv.c[i] - yv.c[i];
                    }
            };
            start(0, y.qm);
            start(1, y.qp);
            start(2, y.fm);
            start(3, y.fp);
            start(4, y.fa);
        }
        x = y;
        cwm = ywm;
        cwp = ywp;
        lamx = lamy;
        bnx = bny;
        wavx = wavy;
    }
    if (bad) atomicOr(&ps->fail_flag, 1);
    if (a.stage0) {
        unsigned long long b = (unsigned long long)__double_as_longlong(lmax);
        for (int o = 32; o > 0; o >>= 1) {
            const unsigned long long v = __shfl_xor(b, o, 64);
            b = v > b ? v : b;
        }
        if (lane == 0 && b != 0ull) atomicMax(&ps->eig[AX], b);
    }
    }
}

}  // namespace ah
