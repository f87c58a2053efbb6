// Non-template control kernels: time step control (astrea.py:45-85), the
// Runge-Kutta stage combinations (evolvers.py:79-206) and the flux difference
// used by the parity entry point.  Included by ah_api.hip only.
#pragma once
#include "ah_kernels.h"

#include <utility>

namespace ah {

// ============================================================================
// Time control (astrea.py:45-85), one thread per problem.
// ============================================================================
__global__ void dt_kernel(const ProbDesc* pd, ProbState* ps, int nprob, int dims) {
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= nprob) return;
    ProbState& s = ps[p];
    if (!s.active) return;
    const ProbDesc d = pd[p];
    const double e0 = __longlong_as_double((long long)s.eig[0]);
    const double e1 = dims == 2 ? __longlong_as_double((long long)s.eig[1]) : e0;
    s.eig[0] = s.eig[1] = 0ull;
    if (!(e0 <= 1.7976931348623157e308) || !(e1 <= 1.7976931348623157e308) || s.fail_flag) {
        s.failed = 1;
        s.active = 0;
        return;
    }
    const double a0 = d.dx / e0, a1 = d.dx / e1;
    double dt = d.cfl * (dims == 2 ? (a1 < a0 ? a1 : a0) : a0);
    int hit = 0;
    if (s.t + dt >= d.chkpt * s.idx) {
        dt = d.chkpt * s.idx - s.t;
        s.idx += 1;
        hit = 1;
    }
    s.ckpt = hit;
    s.dt = dt;
}

__global__ void advance_kernel(const ProbDesc* pd, ProbState* ps, int nprob) {
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= nprob) return;
    ProbState& s = ps[p];
    if (!s.active) return;
    s.aflags = 0ull;
    const ProbDesc d = pd[p];
    if (s.fail_flag) {
        // the reference raises inside this step (LAPACK on a non-finite
        // Jacobian); the state and time stay those of the last good step
        s.failed = 1;
        s.active = 0;
        return;
    }
    s.t = s.t + s.dt;
    s.steps += 1;
    s.parity ^= 1;
    const bool more_time = (s.t <= d.t_end) && !(s.t == d.t_end);
    const bool more_steps = d.max_steps < 0 || s.steps < d.max_steps;
    s.active = more_time && more_steps;
}

// End of a step whose kernels evaluated dt themselves (step_dt): the state
// updates of dt_kernel and advance_kernel in one launch, with the same
// outcome -- a failure seen at stage 0 (non-finite radii) leaves dt and the
// checkpoint index as they were, a later one records this step's dt.
__device__ inline void finish_problem(const ProbDesc& d, ProbState& s, int dims) {
    s.aflags = 0ull;
    const double e0 = __longlong_as_double((long long)s.eig[0]);
    const double e1 = dims == 2 ? __longlong_as_double((long long)s.eig[1]) : e0;
    if (!(e0 <= 1.7976931348623157e308) || !(e1 <= 1.7976931348623157e308)) {
        s.eig[0] = s.eig[1] = 0ull;
        s.failed = 1;
        s.active = 0;
        return;
    }
    int hit;
    const double dt = step_dt(d, s, dims, &hit);
    s.eig[0] = s.eig[1] = 0ull;
    s.idx += hit;
    s.ckpt = hit;
    s.dt = dt;
    if (s.fail_flag) {
        s.failed = 1;
        s.active = 0;
        return;
    }
    s.t = s.t + s.dt;
    s.steps += 1;
    s.parity ^= 1;
    const bool more_time = (s.t <= d.t_end) && !(s.t == d.t_end);
    const bool more_steps = d.max_steps < 0 || s.steps < d.max_steps;
    s.active = more_time && more_steps;
}

__global__ void finish_kernel(const ProbDesc* pd, ProbState* ps, int nprob, int dims) {
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= nprob) return;
    ProbState& s = ps[p];
    if (!s.active) return;
    finish_problem(pd[p], s, dims);
}

__global__ void reset_kernel(const ProbDesc* pd, ProbState* ps, int nprob) {
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= nprob) return;
    ProbState s;
    s.t = 0.0;
    s.dt = 0.0;
    s.steps = 0;
    s.idx = 1;
    s.failed = 0;
    s.parity = 0;
    s.eig[0] = s.eig[1] = 0ull;
    s.fail_flag = 0;
    s.ckpt = 0;
    s.aflags = 0ull;
    const ProbDesc d = pd[p];
    s.active = (0.0 <= d.t_end) && !(0.0 == d.t_end) && d.max_steps != 0;
    ps[p] = s;
}

// ============================================================================
// Stage combinations of every Runge-Kutta scheme (evolvers.py:79-206),
// written in the reference's operation order.  regs[0] = U (state), regs[1..4]
// = k registers, regs[5..8] = saved L, L = this stage's L.
// ============================================================================
enum RkOp {
    OP_EULER = 0,
    OP_22_0, OP_22_1,
    OP_33_0, OP_33_1, OP_33_2,
    OP_43_0, OP_43_1, OP_43_2, OP_43_3,
    OP_RK4_0, OP_RK4_1, OP_RK4_2, OP_RK4_3,
    OP_53_0, OP_53_1, OP_53_2, OP_53_3, OP_53_4,
    OP_54_0, OP_54_1, OP_54_2, OP_54_3, OP_54_4,
    OP_104_FIRST, OP_104_ACC1, OP_104_K5, OP_104_K2FIRST, OP_104_ACC2, OP_104_FINAL,
    // SSPRK(10,4) with constrained transport refines the increment before
    // adding it (evolvers.py:89-90, 97-99): K4 := dt/6 L, refined, then added
    OP_104_INC, OP_104_ADD_U, OP_104_ADD_K1, OP_104_ADD_K3, OP_104_ADD_K2
};

struct CombineArgs {
    double* regs[9];
    const double* L;
    const ProbDesc* pd;
    ProbState* ps;
    const Tile* tiles;       // cell tiles: (problem, first cell, cell count)
    const int* ntiles_dev;
    long long plane;
    int nv;
    int live_dt;   // 1: dt from step_dt (no dt launch in this step program), 0: the stored dt
    int dims;
    // finish: this combination ends the step, and the block that combines a
    // problem's last tile also ends the problem's step (finish_problem); done
    // counts each problem's combined tiles (reset by that block), ct = cells
    // per tile
    int finish;
    int ct;
    unsigned* done;
};

// registers an operation reads (bit r: regs[r]), the one it writes, and the
// one it saves the stage's L in (-1: none)
constexpr int rk_reads(int op) {
    constexpr int U = 1, K1 = 2, K2 = 4, K3 = 8, K4 = 16, L5 = 32, L6 = 64, L7 = 128;
    switch (op) {
        case OP_22_1: case OP_33_1: return U | K1;
        case OP_33_2: return U | K2;
        case OP_43_1: case OP_53_1: return K1;
        case OP_43_2: return U | K2;
        case OP_43_3: return K3;
        case OP_RK4_3: return U | L5 | L6 | L7;
        case OP_53_2: return U | K2;
        case OP_53_3: return U | K1 | K3 | L5;
        case OP_53_4: return U | K1 | K2 | K4 | L5 | L6;
        case OP_54_1: return U | K1;
        case OP_54_2: return U | K2;
        case OP_54_3: return U | K3;
        case OP_54_4: return K2 | K3 | K4 | L5;
        case OP_104_ACC1: return K1;
        case OP_104_K5: return U | K1;
        case OP_104_K2FIRST: return K3;
        case OP_104_ACC2: return K2;
        case OP_104_INC: return 0;
        case OP_104_ADD_U: return U | K4;
        case OP_104_ADD_K1: return K1 | K4;
        case OP_104_ADD_K3: return K3 | K4;
        case OP_104_ADD_K2: return K2 | K4;
        case OP_104_FINAL: return U | K3 | K2;
    }
    return U;
}
constexpr int rk_writes(int op) {
    switch (op) {
        case OP_22_0: case OP_33_0: case OP_43_0: case OP_RK4_0: case OP_53_0: case OP_54_0: case OP_104_FIRST:
        case OP_104_ACC1: case OP_104_ADD_U: case OP_104_ADD_K1: return 1;
        case OP_33_1: case OP_43_1: case OP_RK4_1: case OP_53_1: case OP_54_1: case OP_104_K2FIRST: case OP_104_ACC2:
        case OP_104_ADD_K3: case OP_104_ADD_K2: return 2;
        case OP_43_2: case OP_RK4_2: case OP_53_2: case OP_54_2: case OP_104_K5: return 3;
        case OP_53_3: case OP_54_3: case OP_104_INC: return 4;
    }
    return 0;
}
constexpr int rk_saves(int op) {
    switch (op) {
        case OP_RK4_0: case OP_53_0: case OP_54_3: return 5;
        case OP_RK4_1: case OP_53_1: return 6;
        case OP_RK4_2: return 7;
    }
    return -1;
}
constexpr int RK_OPS = OP_104_ADD_K2 + 1;

// one value, from the registers' values r, the stage's L and dt
template <int OP>
__device__ inline double rk_value(const double (&r)[9], double L, double dt) {
    const double U = r[0], K1 = r[1], K2 = r[2], K3 = r[3], K4 = r[4];
    switch (OP) {
        case OP_EULER: return U + dt * L;
        case OP_22_0: return U + dt * L;
        case OP_22_1: return .5 * (U + K1 + dt * L);
        case OP_33_0: return U + dt * L;
        case OP_33_1: return .25 * (3 * U + K1 + dt * L);
        case OP_33_2: return (1.0 / 3.0) * (U + 2 * K2 + 2 * dt * L);
        case OP_43_0: return U + .5 * dt * L;
        case OP_43_1: return K1 + .5 * dt * L;
        case OP_43_2: return (1.0 / 6.0) * (4 * U + 2 * K2 + dt * L);
        case OP_43_3: return K3 + .5 * dt * L;
        case OP_RK4_0: return U + .5 * dt * L;
        case OP_RK4_1: return U + .5 * dt * L;
        case OP_RK4_2: return U + dt * L;
        case OP_RK4_3: return U + (1.0 / 6.0) * (dt * (r[5] + 2 * r[6] + 2 * r[7] + L));
        case OP_53_0: return U + .3772689151171 * dt * L;
        case OP_53_1: return K1 + .3772689151171 * dt * L;
        case OP_53_2: return .56656131914033 * U + .43343868085967 * K2 + .16352294089771 * dt * L;
        case OP_53_3:
            return .09299483444413 * U + .0000209036962 * K1 + .90698426185967 * K3 + .00071997378654 * dt * r[5] +
                   .34217696850008 * dt * L;
        case OP_53_4:
            return .0073613226092 * U + .20127980325145 * K1 + .00182955389682 * K2 + .78952932024253 * K4 +
                   (dt * (.0027771981946 * r[5] + .00001567934613 * r[6] + .29786487010104 * L));
        case OP_54_0: return U + .39175222657189 * dt * L;
        case OP_54_1: return .444370493651235 * U + .555629506348765 * K1 + .368410593050371 * dt * L;
        case OP_54_2: return .620101851488403 * U + .379898148511597 * K2 + .251891774271694 * dt * L;
        case OP_54_3: return .178079954393132 * U + .821920045606868 * K3 + .544974750228521 * dt * L;
        case OP_54_4:
            return .517231671970585 * K2 + .096059710526147 * K3 + .06369246866629 * dt * r[5] +
                   .386708617503269 * K4 + .226007483236906 * dt * L;
        case OP_104_FIRST: return U + (1.0 / 6.0) * dt * L;
        case OP_104_ACC1: return K1 + (1.0 / 6.0) * dt * L;
        case OP_104_K5: return 3.0 / 5.0 * U + 6.0 / 15.0 * K1 + 1.0 / 15.0 * dt * L;
        case OP_104_K2FIRST: return K3 + (1.0 / 6.0) * dt * L;
        case OP_104_ACC2: return K2 + (1.0 / 6.0) * dt * L;
        case OP_104_INC: return (1.0 / 6.0) * dt * L;
        case OP_104_ADD_U: return U + K4;
        case OP_104_ADD_K1: return K1 + K4;
        case OP_104_ADD_K3: return K3 + K4;
        case OP_104_ADD_K2: return K2 + K4;
        case OP_104_FINAL: return -11.0 / 35.0 * U + 5.0 / 7.0 * K3 + 3.0 / 5.0 * K2 + 1.0 / 10.0 * dt * L;
    }
    return 0.0;
}

// Four values per thread and turn: the next four components of one cell on
// tiles of 256 cells, four cells of one component on tiles of 1024.  All their
// loads leave before the first value is formed: the kernel is bound by memory
// bandwidth on large grids and by the length of its chain of loads on small
// ones (one value after another, a 128^2 tile of 4 x 4 values per thread took
// 12 us).  The tile's descriptor, the problem's and its time state are each
// read whole, so that the branch on the state costs one round trip, not four.
template <int OP, bool WIDE>
__global__ __launch_bounds__(256) void combine_kernel(CombineArgs a) {
    const long long n = a.plane;
    const int ntiles = wave_uniform(*a.ntiles_dev);
    for (int ti = blockIdx.x; ti < ntiles; ti += gridDim.x) {
        const Tile tl = ld_const(a.tiles + ti);
        const ProbState s = ld_const(a.ps + tl.prob);
        const ProbDesc d = ld_const(a.pd + tl.prob);
        if (!s.active) continue;
        if (!s.fail_flag) {
            int hit;
            const double dt = a.live_dt ? step_dt(d, s, a.dims, &hit) : s.dt;
            const long long base = d.off + tl.s0;
            auto four = [&](int v0, int dv, int c0, int dc) {
                double r[4][9], L[4];
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    const int v = v0 + u * dv, c = c0 + u * dc;
                    if (v < a.nv && c < tl.t0) {
                        const long long j = v * n + base + c;
                        L[u] = a.L[j];
#pragma unroll
                        for (int k = 0; k < 8; ++k)
                            if ((rk_reads(OP) >> k) & 1) r[u][k] = a.regs[k][j];
                    }
                }
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    const int v = v0 + u * dv, c = c0 + u * dc;
                    if (v < a.nv && c < tl.t0) {
                        const long long j = v * n + base + c;
                        if constexpr (rk_saves(OP) >= 0) a.regs[rk_saves(OP)][j] = L[u];
                        a.regs[rk_writes(OP)][j] = rk_value<OP>(r[u], L[u], dt);
                    }
                }
            };
            if constexpr (WIDE) {
                for (int v = 0; v < a.nv; ++v)
                    for (int c = threadIdx.x; c < tl.t0; c += 4 * 256) four(v, 0, c, 256);
            } else {
                for (int c = threadIdx.x; c < tl.t0; c += 256)
                    for (int v = 0; v < a.nv; v += 4) four(v, 1, c, 0);
            }
        }
        if (a.finish) {
            // every block that combines one of the problem's tiles counts it
            // once its threads have read the time state and written their
            // cells; the block that counts the last one ends the problem's
            // step.  No other block reads this problem's time state after
            // counting, so no fence orders the update against them; the next
            // launch sees it.
            __syncthreads();
            if (threadIdx.x == 0) {
                const long long cells = (long long)d.n0 * d.n1;
                const unsigned nt = (unsigned)((cells + a.ct - 1) / a.ct);
                if (atomicAdd(&a.done[tl.prob], 1u) == nt - 1) {
                    a.done[tl.prob] = 0u;
                    finish_problem(d, a.ps[tl.prob], a.dims);
                }
            }
        }
    }
}


using CombineLaunch = void (*)(const CombineArgs&, int nblocks, hipStream_t);
template <bool WIDE, int... OP>
inline CombineLaunch combine_launcher(int op, std::integer_sequence<int, OP...>) {
    static constexpr CombineLaunch table[] = {[](const CombineArgs& a, int nb, hipStream_t s) {
        hipLaunchKernelGGL((combine_kernel<OP, WIDE>), dim3(nb), dim3(256), 0, s, a);
    }...};
    return table[op];
}
inline CombineLaunch combine_launcher(int op, bool wide) {
    using Ops = std::make_integer_sequence<int, RK_OPS>;
    return wide ? combine_launcher<true>(op, Ops()) : combine_launcher<false>(op, Ops());
}

// L = -sum_a dF_a/dx from sweep-frame interface fluxes (evolvers.py:41-60)
__global__ void fluxdiff_kernel(const double* F0, const double* F1, double* L, int n0, int n1, int dims, int nv,
                                double dx, long long plane, long long fplane0, long long fplane1) {
    const long long ncell = (long long)n0 * n1;
    for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < ncell; i += (long long)gridDim.x * blockDim.x) {
        const int i0 = (int)(i / n1), i1 = (int)(i % n1);
        for (int v = 0; v < nv; ++v) {
            // axis 0: interfaces i0, i0+1 on line i1 (layout [k][t] with t = i1)
            const double d0 = (F0[v * fplane0 + (long long)(i0 + 1) * n1 + i1] - F0[v * fplane0 + (long long)i0 * n1 + i1]) / dx;
            if (dims == 1) {
                L[v * plane + i] = -d0;
            } else {
                const double d1 =
                    (F1[v * fplane1 + (long long)(i1 + 1) * n0 + i0] - F1[v * fplane1 + (long long)i1 * n0 + i0]) / dx;
                L[v * plane + i] = -(d0 + d1);
            }
        }
    }
}

}  // namespace ah
