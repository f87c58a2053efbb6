// Snapshots of the state as the reference saves them every step
// (astrea.py:47): sim_variables.convert_conservative of the conservative grid
// -- the 4th-order cell conversion for PPM/WENO, the pointwise one otherwise
// (generic.py:250-255) -- transposed by ortho_axis (generic.py:264: the
// identity in 1D, (1, 0, 2) in 2D).  The conversion is the one the sweep
// kernels apply to their input (ho_cell_prim, Laplacians along x then y), so
// the snapshot equals the reference's to the last bit.
#pragma once
#include "ah_kernels.h"

namespace ah {

// Snapshots taken inside the step program, without the host: after a step of
// problem `prob`, when `mode` asks for it (1: every step, 2: steps whose dt
// was clamped to a checkpoint, astrea.py:74-78), the snapshot goes to slot
// ctl[0] % slots of a caller-owned ring and t to times[] of that slot.
// ctl[1] holds the step count of the last step looked at, so a launch after
// which the problem did not step (inactive, failed) captures nothing.
struct CaptureArgs {
    const ProbState* ps;
    double* ring;   // slots x cells x 8 doubles
    double* times;  // slots
    long long* ctl; // [0] snapshots taken, [1] steps at the last look; null: capture off
    long long cells;
    double t_end;   // states past t_end are not saved (the loop of astrea.py:45 ends there)
    int prob, mode, slots, pad;
};

__device__ inline bool capture_due(const CaptureArgs& c) {
    const ProbState& st = c.ps[c.prob];
    return st.steps != c.ctl[1] && (c.mode == 1 || st.ckpt != 0) && st.t <= c.t_end;
}

// One thread per cell, for snapshots of which that latency is all there is.
template <int MASK, int DIM, bool HO>
__global__ __launch_bounds__(256) void snapshot_cells_kernel(const double* X, long long P, long long off, int n0,
                                                             int n1, int bc, double gamma, double* out,
                                                             CaptureArgs cap) {
    using V = VS<MASK>;
    const long long cells = (long long)n0 * n1;
    const long long cell = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (cell >= cells) return;
    if (cap.ctl) {
        if (!capture_due(cap)) return;
        out = cap.ring + (cap.ctl[0] % cap.slots) * cells * 8;
    }
    const int i = (int)(cell / n1), j = (int)(cell % n1);
    auto Q = [&](int ii, int jj) {
        V8<double> q = zero8<double, MASK>();
#pragma unroll
        for (int c = 0; c < 8; ++c)
            if (V::live(c)) q.c[c] = X[V::slot(c) * P + off + (long long)ii * n1 + jj];
        return q;
    };
    const V8<double> q0 = Q(i, j);
    V8<double> w;
    if constexpr (HO) {
        const int im = bcmap(i - 1, n0, bc), ip = bcmap(i + 1, n0, bc);
        const V8<double> qxm = Q(im, j), qxp = Q(ip, j);
        V8<double> qym = zero8<double, MASK>(), qyp = qym;
        if constexpr (DIM == 2) {
            qym = Q(i, bcmap(j - 1, n1, bc));
            qyp = Q(i, bcmap(j + 1, n1, bc));
        }
        w = ho_cell_prim<MASK, DIM, false>(q0, qxm, qxp, qym, qyp, c2p<MASK, false>(q0, gamma),
                                           c2p<MASK, false>(qxm, gamma), c2p<MASK, false>(qxp, gamma),
                                           c2p<MASK, false>(qym, gamma), c2p<MASK, false>(qyp, gamma), gamma);
    } else {
        w = c2p<MASK, false>(q0, gamma);
    }
    const long long o = DIM == 2 ? ((long long)j * n0 + i) * 8 : (long long)i * 8;
#pragma unroll
    for (int c = 0; c < 8; ++c) out[o + c] = V::live(c) ? w.c[c] : 0.0;
}

// One workgroup per tile of 8 x 32 cells (2D) or 256 cells (1D).  The state is
// read along its rows, the snapshot is written along its own, transposed ones,
// eight values a cell: the tile's primitives are turned in LDS and written as
// 16-byte pieces, half a kilobyte of consecutive addresses per row.  The
// 4th-order conversion's window (one cell around the tile) is converted once
// per cell.  The snapshot is twice the state and not read here again, so its
// stores bypass the caches (plain ones: 110 us where these take 91).
// Bound by HBM: 2048^2 PPM 173 -> 93 us for 403 MB, 4.3 TB/s of a large copy's
// 4.8 (one thread per cell wrote 64-byte strides and converted five cells).
constexpr int SNAP_TI = 8, SNAP_TJ = 32;
template <int MASK, int DIM, bool HO>
__global__ __launch_bounds__(256) void snapshot_kernel(const double* X, long long P, long long off, int n0, int n1,
                                                       int bc, double gamma, double* out, CaptureArgs cap) {
    using V = VS<MASK>;
    constexpr int NV = V::NV;
    constexpr int TI = DIM == 2 ? SNAP_TI : 256, TJ = DIM == 2 ? SNAP_TJ : 1;  // cells along i0 (x) and i1 (y)
    constexpr int H = HO ? 1 : 0, HJ = DIM == 2 ? H : 0;
    constexpr int WI = TI + 2 * H, WJ = TJ + 2 * HJ;
    __shared__ double q_s[NV][WI][WJ];
    __shared__ double c_s[HO ? NV : 1][HO ? WI : 1][HO ? WJ : 1];
    __shared__ double w_s[NV][TJ][TI + (DIM == 2 ? 1 : 0)];
    const long long cells = (long long)n0 * n1;
    if (cap.ctl) {
        if (!capture_due(cap)) return;
        out = cap.ring + (cap.ctl[0] % cap.slots) * cells * 8;
    }
    const int ti = (n0 + TI - 1) / TI;
    const int i0 = (int)(blockIdx.x % ti) * TI, j0 = (int)(blockIdx.x / ti) * TJ;
    for (int k = threadIdx.x; k < WI * WJ; k += 256) {
        const int wi = k / WJ, wj = k % WJ;
        const long long g = off + (long long)bcmap(i0 - H + wi, n0, bc) * n1 + bcmap(j0 - HJ + wj, n1, bc);
        V8<double> q = zero8<double, MASK>();
#pragma unroll
        for (int c = 0; c < 8; ++c)
            if (V::live(c)) q.c[c] = X[V::slot(c) * P + g];
#pragma unroll
        for (int c = 0; c < 8; ++c)
            if (V::live(c)) q_s[V::slot(c)][wi][wj] = q.c[c];
        if constexpr (HO) {
            const V8<double> w = c2p<MASK, false>(q, gamma);
#pragma unroll
            for (int c = 0; c < 8; ++c)
                if (V::live(c)) c_s[V::slot(c)][wi][wj] = w.c[c];
        }
    }
    __syncthreads();
    {
        const int il = threadIdx.x / TJ, jl = threadIdx.x % TJ, wi = il + H, wj = jl + HJ;
        auto Q = [&](int a, int b) {
            V8<double> v = zero8<double, MASK>();
#pragma unroll
            for (int c = 0; c < 8; ++c)
                if (V::live(c)) v.c[c] = q_s[V::slot(c)][a][b];
            return v;
        };
        V8<double> w;
        if constexpr (HO) {
            auto C = [&](int a, int b) {
                V8<double> v = zero8<double, MASK>();
#pragma unroll
                for (int c = 0; c < 8; ++c)
                    if (V::live(c)) v.c[c] = c_s[V::slot(c)][a][b];
                return v;
            };
            const V8<double> z = zero8<double, MASK>();
            if constexpr (DIM == 2)
                w = ho_cell_prim<MASK, 2, false>(Q(wi, wj), Q(wi - 1, wj), Q(wi + 1, wj), Q(wi, wj - 1), Q(wi, wj + 1),
                                                 C(wi, wj), C(wi - 1, wj), C(wi + 1, wj), C(wi, wj - 1), C(wi, wj + 1),
                                                 gamma);
            else
                w = ho_cell_prim<MASK, 1, false>(Q(wi, wj), Q(wi - 1, wj), Q(wi + 1, wj), z, z, C(wi, wj),
                                                 C(wi - 1, wj), C(wi + 1, wj), z, z, gamma);
        } else {
            w = c2p<MASK, false>(Q(wi, wj), gamma);
        }
#pragma unroll
        for (int c = 0; c < 8; ++c)
            if (V::live(c)) w_s[V::slot(c)][jl][il] = w.c[c];
    }
    __syncthreads();
    // rows of the snapshot: cell (j, i) at (j n0 + i) 8, two components a piece
    const bool wide = ((unsigned long long)out & 15) == 0;
    for (int k = threadIdx.x; k < TI * TJ * 4; k += 256) {
        const int h = k & 3, il = (k >> 2) % TI, jl = (k >> 2) / TI;
        if (i0 + il >= n0 || j0 + jl >= n1) continue;
        using d2 = double __attribute__((ext_vector_type(2)));
        d2 v = {0.0, 0.0};
#pragma unroll
        for (int c = 0; c < 8; ++c)
            if (V::live(c) && (c >> 1) == h) v[c & 1] = w_s[V::slot(c)][jl][il];
        double* o = out + ((long long)(j0 + jl) * n0 + i0 + il) * 8 + 2 * h;
        if (wide) {
            __builtin_nontemporal_store(v, reinterpret_cast<d2*>(o));
        } else {
            __builtin_nontemporal_store(v.x, o);
            __builtin_nontemporal_store(v.y, o + 1);
        }
    }
}

// after the capture launch: record t of the slot and advance the counters
__global__ void capture_commit_kernel(CaptureArgs c) {
    if (blockIdx.x != 0 || threadIdx.x != 0) return;
    const ProbState& st = c.ps[c.prob];
    if (st.steps == c.ctl[1]) return;
    const bool due = (c.mode == 1 || st.ckpt != 0) && st.t <= c.t_end;
    c.ctl[1] = st.steps;
    if (!due) return;
    c.times[c.ctl[0] % c.slots] = st.t;
    c.ctl[0] += 1;
}

// start of a capture: nothing taken yet, the current step count already seen
__global__ void capture_init_kernel(CaptureArgs c) {
    if (blockIdx.x != 0 || threadIdx.x != 0) return;
    c.ctl[0] = 0;
    c.ctl[1] = c.ps[c.prob].steps;
}

}  // namespace ah
