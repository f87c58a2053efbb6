// Instantiation of the sweep kernels for one arithmetic type R.  Included by
// the per-precision translation units with AH_INST_DIMS set to 1 or 2.
#pragma once
#include "ah_launch.h"

namespace ah {

template <class R, int MASK, int RECON, int SOLVER, bool SPLIT, int AUTH = AUTH_MC, int NTHR1 = 256>
inline void set1d(KernelSet* ks) {
    // cells per tile: the widest per-stage window (the q window, TS + 13)
    // fits one pass of the workgroup's threads, so no stage runs a second,
    // nearly empty round while the other waves wait at the barrier
    constexpr int TS = VS<MASK>::NV > 4 ? 128 : NTHR1 - 13;
    ks->sweep1d = [](const SweepArgs& a, int nb, hipStream_t s) {
        // HLLD's short divisions shorten a workgroup's chain and leave a SIMD
        // one or two waves: beyond two workgroups per CU the general form, with
        // its third wave, is faster.  1601-cell tubes (13 tiles each), us a step,
        // short / general: PPM 32 tubes 60.9 / 64.4, 48 86.7 / 82.1, 256 297 /
        // 272; WENO5 32 65.9 / 69.9, 48 91.3 / 88.8, 256 327 / 298 (before the
        // short form 318; WENO7 keeps it, 256 408 / 427).
        constexpr int SHORT_BLOCKS = 512;
        if constexpr (std::is_same<R, double>::value && !SPLIT && SOLVER == HLLD && (RECON == PPM || RECON == WENO5))
            if (nb > SHORT_BLOCKS)
                return launch_sweep(sweep1d_kernel<R, MASK, RECON, SOLVER, TS, SPLIT, AUTH, false>, a, nb, s, NTHR1);
        launch_sweep(sweep1d_kernel<R, MASK, RECON, SOLVER, TS, SPLIT, AUTH>, a, nb, s, NTHR1);
    };
    ks->ts1 = TS;
    ks->real_bytes = sizeof(R);
}

template <class R, int MASK, int RECON, int SOLVER, bool SPLIT>
inline void set2d(KernelSet* ks) {
    constexpr int CONV = RECON == PCM ? 0 : (RECON == PLM ? 1 : 2);
    constexpr int NVB = VS<MASK>::NV * (int)sizeof(R);
    // reconstruction tiles; with six or eight FP64 components (MHD) the
    // windows of 32 x 8 / 64 x 4 tiles take 56 KB of LDS (two workgroups per
    // CU), those of 32 x 7 / 64 x 3 under 53 KB (three)
    constexpr int RTS0 = 32, RTT0 = NVB > 32 ? 7 : 8, RTS1 = 64, RTT1 = NVB > 32 ? 3 : 4;
    // flux tile: (FTT + 2) x (FTS + 1) face solves and (FTT + 2) x (FTS + 2)
    // radii per tile each fit one pass of 256 threads; hydro 16 x 10 takes
    // 50.5 KB of LDS (three workgroups per CU), MHD 16 x 8 64 KB (two, as its
    // registers allow); measured on the 1024^2 shear layer against 16 x 12,
    // 16 x 8, 15 x 10, 15 x 14, 31 x 4, 31 x 6, 32 x 4, 24 x 8 and 40 x 4
    constexpr int FTS0 = 16, FTT0 = NVB > 32 ? 8 : 10, FTS1 = 16, FTT1 = NVB > 32 ? 8 : 10, FNT = 256;
    ks->recon[0] = [](const SweepArgs& a, int nb, hipStream_t s) {
        launch_sweep(recon2d_kernel<R, MASK, RECON, 0, RTS0, RTT0, SPLIT>, a, nb, s);
    };
    ks->recon[1] = [](const SweepArgs& a, int nb, hipStream_t s) {
        launch_sweep(recon2d_kernel<R, MASK, RECON, 1, RTS1, RTT1, SPLIT>, a, nb, s);
    };
    ks->flux[0] = [](const SweepArgs& a, int nb, hipStream_t s) {
        launch_sweep(flux2d_kernel<R, MASK, SOLVER, CONV, 0, FTS0, FTT0, SPLIT, FNT>, a, nb, s, FNT);
    };
    ks->flux[1] = [](const SweepArgs& a, int nb, hipStream_t s) {
        launch_sweep(flux2d_kernel<R, MASK, SOLVER, CONV, 1, FTS1, FTT1, SPLIT, FNT>, a, nb, s, FNT);
    };
    ks->rts[0] = RTS0;
    ks->rtt[0] = RTT0;
    ks->rts[1] = RTS1;
    ks->rtt[1] = RTT1;
    ks->fts[0] = FTS0;
    ks->ftt[0] = FTT0;
    ks->fts[1] = FTS1;
    ks->ftt[1] = FTT1;
    ks->real_bytes = sizeof(R);
    // constrained transport: FP64 translation units only (a split plan takes
    // these launchers from the FP64 kernel set; an instantiation here would
    // give the split unit's copy the same symbol, compiled with contraction)
    if constexpr (VS<MASK>::MHD && !SPLIT) {
        constexpr int TTS = 64, TTT = 8;
        ks->tts = TTS;
        ks->ttt = TTT;
        ks->trecon[0] = [](const MhdArgs& a, int nb, hipStream_t s) {
            if (nb > 0) hipLaunchKernelGGL((trecon_kernel<R, MASK, 0, TTS, TTT>), dim3(nb), dim3(64 * VS<MASK>::NV), 0, s, a);
        };
        ks->trecon[1] = [](const MhdArgs& a, int nb, hipStream_t s) {
            if (nb > 0) hipLaunchKernelGGL((trecon_kernel<R, MASK, 1, TTS, TTT>), dim3(nb), dim3(64 * VS<MASK>::NV), 0, s, a);
        };
        ks->corner = [](const MhdArgs& a, int nb, hipStream_t s) {
            if (nb > 0) hipLaunchKernelGGL((corner_kernel<R, MASK, TTS, TTT>), dim3(nb), dim3(256), 0, s, a);
        };
        ks->magL = [](const MhdArgs& a, int nb, hipStream_t s) {
            if (nb > 0) hipLaunchKernelGGL((magL_kernel<MASK>), dim3(nb), dim3(256), 0, s, a);
        };
        ks->bface = [](const MhdArgs& a, int nb, hipStream_t s) {
            if (nb > 0) hipLaunchKernelGGL((bface_kernel<R, MASK, TTS, TTT>), dim3(nb), dim3(256), 0, s, a);
        };
        ks->refine = [](const MhdArgs& a, int nb, hipStream_t s) {
            if (nb > 0) hipLaunchKernelGGL((refine_kernel<MASK, TTS, TTT>), dim3(nb), dim3(256), 0, s, a);
        };
        ks->copyB = [](const MhdArgs& a, double* dst, int nb, hipStream_t s) {
            if (nb > 0) hipLaunchKernelGGL((copyB_kernel<MASK>), dim3(nb), dim3(256), 0, s, a, dst);
        };
    }
}

template <class R, int MASK, int SOLVER, int DIMS, bool SPLIT>
inline bool by_recon(int recon, KernelSet* ks) {
    switch (recon) {
#define AH_CASE(RC)                                                     \
    case RC:                                                            \
        if constexpr (DIMS == 1) set1d<R, MASK, RC, SOLVER, SPLIT>(ks); \
        else set2d<R, MASK, RC, SOLVER, SPLIT>(ks);                     \
        return true;
        AH_CASE(PCM)
        AH_CASE(PLM)
        AH_CASE(PPM)
        AH_CASE(WENO3)
        AH_CASE(WENO5)
        AH_CASE(WENO7)
#undef AH_CASE
    }
    return false;
}

template <class R, int DIMS, bool SPLIT>
inline bool select_kernels(int mask, int recon, int solver, KernelSet* ks) {
    if constexpr (DIMS == 1) {
        if (mask == 0x13) {
            if (solver == LLF) return by_recon<R, 0x13, LLF, 1, SPLIT>(recon, ks);
            if (solver == HLLC) return by_recon<R, 0x13, HLLC, 1, SPLIT>(recon, ks);
            if constexpr (!SPLIT) {
                if (solver == DOTS) return by_recon<R, 0x13, DOTS, 1, SPLIT>(recon, ks);
                if (solver == LW) return by_recon<R, 0x13, LW, 1, SPLIT>(recon, ks);
            }
        }
        if (mask == 0xFF) {
            if (solver == LLF) return by_recon<R, 0xFF, LLF, 1, SPLIT>(recon, ks);
            if (solver == HLLC) return by_recon<R, 0xFF, HLLC, 1, SPLIT>(recon, ks);
            if (solver == HLLD) return by_recon<R, 0xFF, HLLD, 1, SPLIT>(recon, ks);
            if constexpr (!SPLIT) {
                if (solver == DOTS) return by_recon<R, 0xFF, DOTS, 1, SPLIT>(recon, ks);
                // entropy-stable: 1D only (as the reference), all 8 components, whose
                // non-finite values feed the reference's failure on the next step
                if (solver == ES) return by_recon<R, 0xFF, ES, 1, SPLIT>(recon, ks);
                // Lax-Wendroff with the hydrodynamic sound speed (transverse
                // velocities; the reference's own pick is hydrodynamic only)
                if (solver == LW) return by_recon<R, 0xFF, LW, 1, SPLIT>(recon, ks);
            }
        }
    } else {
        if (mask == 0x17) {
            if (solver == LLF) return by_recon<R, 0x17, LLF, 2, SPLIT>(recon, ks);
            if (solver == HLLC) return by_recon<R, 0x17, HLLC, 2, SPLIT>(recon, ks);
            if constexpr (!SPLIT) {
                if (solver == DOTS) return by_recon<R, 0x17, DOTS, 2, SPLIT>(recon, ks);
                if (solver == LW) return by_recon<R, 0x17, LW, 2, SPLIT>(recon, ks);
            }
        }
        if (mask == 0x77) {
            if (solver == LLF) return by_recon<R, 0x77, LLF, 2, SPLIT>(recon, ks);
            if (solver == HLLD) return by_recon<R, 0x77, HLLD, 2, SPLIT>(recon, ks);
            // HLLC on 2D MHD states: reachable from the reference's options
            // (a magnetic-2D configuration keeps 'hllc'; generic.py:266-269
            // resets it for 1D magnetic configurations only).  Osher-Solomon
            // is not: its dissipation couples v_z and B_z into the update, and
            // the reference's own 2D call raises (the reshape at
            // solvers.py:281 assumes 1D arrays)
            if (solver == HLLC) return by_recon<R, 0x77, HLLC, 2, SPLIT>(recon, ks);
            // Lax-Wendroff with the sound speed sqrt(gamma p / rho), as in 1D MHD
            if constexpr (!SPLIT) {
                if (solver == LW) return by_recon<R, 0x77, LW, 2, SPLIT>(recon, ks);
            }
        }
    }
    return false;
}

// 2D hydrodynamic PPM with author c or ph (FP64): replaces the reconstruction
// launchers of the FP64 kernel set (set2d's 32 x 8 and 64 x 4 tiles for four
// FP64 components) with the author's; the flux launchers stay
template <int AUTH>
inline void set2d_author(KernelSet* ks) {
    ks->recon[0] = [](const SweepArgs& a, int nb, hipStream_t s) {
        launch_sweep(recon2d_kernel<double, 0x17, PPM, 0, 32, 8, false, AUTH>, a, nb, s);
    };
    ks->recon[1] = [](const SweepArgs& a, int nb, hipStream_t s) {
        launch_sweep(recon2d_kernel<double, 0x17, PPM, 1, 64, 4, false, AUTH>, a, nb, s);
    };
}

// The 2D flux launches in marching form (FP64; LLF, HLLC, HLLD on point or
// 4th-order face conversion), beside the tile form; the plan picks one
template <int MASK, int SOLVER, int CONV>
inline bool set2d_march(KernelSet* ks) {
    ks->march[0] = [](const SweepArgs& a, int nb, hipStream_t s) {
        launch_sweep(flux2d_march_kernel<MASK, SOLVER, CONV, 0>, a, nb, s, 64);
    };
    ks->march[1] = [](const SweepArgs& a, int nb, hipStream_t s) {
        launch_sweep(flux2d_march_kernel<MASK, SOLVER, CONV, 1>, a, nb, s, 64);
    };
    ks->mw = march_width<SOLVER>();
    ks->march_waves = march_waves<MASK>();
    return true;
}

template <int MASK, int SOLVER>
inline bool set2d_march(int recon, KernelSet* ks) {
    return recon == PCM ? false : (recon == PLM ? set2d_march<MASK, SOLVER, 1>(ks) : set2d_march<MASK, SOLVER, 2>(ks));
}

// 2D hydrodynamics, one launch per sweep: the flux kernel reconstructs its
// own window (recon[] stays null, and the plan keeps no wL/wR planes).  The
// 16 x 8 tile takes 52 KB of LDS (the reconstruction windows share theirs
// with the face-average arrays): three workgroups per CU.
template <class R, int RECON, int SOLVER, bool SPLIT>
inline void set2d_fused(KernelSet* ks) {
    constexpr int CONV = RECON == PLM ? 1 : 2;
    constexpr int TS = 16, TT = 8, NT = 256;
    ks->flux[0] = [](const SweepArgs& a, int nb, hipStream_t s) {
        launch_sweep(flux2d_kernel<R, 0x17, SOLVER, CONV, 0, TS, TT, SPLIT, NT, RECON>, a, nb, s, NT);
    };
    ks->flux[1] = [](const SweepArgs& a, int nb, hipStream_t s) {
        launch_sweep(flux2d_kernel<R, 0x17, SOLVER, CONV, 1, TS, TT, SPLIT, NT, RECON>, a, nb, s, NT);
    };
    for (int ax = 0; ax < 2; ++ax) {
        ks->recon[ax] = nullptr;
        ks->fts[ax] = TS;
        ks->ftt[ax] = TT;
    }
    ks->real_bytes = sizeof(R);
}

template <class R, bool SPLIT>
inline bool select_kernels_2d_fused(int recon, int solver, KernelSet* ks) {
    if (recon == PLM && solver == LLF) set2d_fused<R, PLM, LLF, SPLIT>(ks);
    else if (recon == PLM && solver == HLLC) set2d_fused<R, PLM, HLLC, SPLIT>(ks);
    else if (recon == PPM && solver == LLF) set2d_fused<R, PPM, LLF, SPLIT>(ks);
    else if (recon == PPM && solver == HLLC) set2d_fused<R, PPM, HLLC, SPLIT>(ks);
    else return false;
    return true;
}

// 1D hydrodynamic PLM/PPM with LLF or HLLC on 115-cell tiles of 128-thread
// workgroups (two waves): the alternative tile shape the ensemble autotuner
// times against the 243-cell default
template <class R, bool SPLIT>
inline bool select_kernels_1d_small(int recon, int solver, KernelSet* ks) {
    if (recon == PLM && solver == LLF) set1d<R, 0x13, PLM, LLF, SPLIT, AUTH_MC, 128>(ks);
    else if (recon == PLM && solver == HLLC) set1d<R, 0x13, PLM, HLLC, SPLIT, AUTH_MC, 128>(ks);
    else if (recon == PPM && solver == LLF) set1d<R, 0x13, PPM, LLF, SPLIT, AUTH_MC, 128>(ks);
    else if (recon == PPM && solver == HLLC) set1d<R, 0x13, PPM, HLLC, SPLIT, AUTH_MC, 128>(ks);
    else return false;
    return true;
}

}  // namespace ah
