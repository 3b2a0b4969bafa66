// va_kernels_impl.hpp -- generic (one lane per instance) HIP kernels of the batched
// explicit-RK forward sweep and discrete-adjoint reverse sweep, gfx950.
//
//   k_fwd       persistent forward: lanes pull instances from an atomic work
//               counter (lane refill), run odeint's controlled loop per lane and
//               store (t_n, y_n) rows -- lib/include/detail/runge_kutta.hpp:74-118
//               (fixed-step loop :36-72), StateStorage.hpp:28-35.
//   k_rev       persistent reverse: replays the stored rows backwards, recomputes
//               the stages and applies the RK adjoint recursion --
//               lib/include/detail/backpropagation.hpp:83-158,231-254,280-348.
//   k_plain_*   the plain GPU form: one launch per accepted step, no refill,
//               every row (t, h, y) stored [step][field][instance]; one reverse
//               launch per step, which recomputes the step's stages from y_n as
//               the reference's compute_intermediate_states does.
//
// Every lane runs a flattened state machine (one attempt / one reverse step per
// loop trip) so the wave stays converged on the arithmetic; the refill branch is
// the only divergent path.
#pragma once
#include "va_device.hpp"
#include "va_kernels.hpp"

namespace va {

enum { LANE_OK = 0, LANE_MAX_FAIL = 1, LANE_NONFINITE = 2, LANE_MAX_STEPS = 3 };
enum { COST_REFERENCE = 0, COST_SUM = 1, COST_SQUARED_NORM = 2, COST_LINEAR = 3 };

// Wait for this wave's outstanding vector-memory operations.  Placed at the end
// of a refill, it retires the instance's parameter loads there; otherwise the
// compiler cannot tell at the loop head whether a load is pending and waits
// for every outstanding operation -- including the trajectory stores, which
// count in the same in-order counter -- on each trip.  (gfx9 s_waitcnt
// encoding: vmcnt 0, expcnt and lgkmcnt left at their maxima.)
__device__ __forceinline__ void wait_vmem() { __builtin_amdgcn_s_waitcnt(0x0F70); }

template <int N>
__device__ __forceinline__ bool all_finite(const double *y)
{
    bool ok = true;
#pragma unroll
    for (int i = 0; i < N; ++i) ok = ok && (fabs(y[i]) <= 1.7976931348623157e308);
    return ok;
}

// ---------------------------------------------------------------------------
// Persistent forward
// ---------------------------------------------------------------------------
// What bounds it: one instance's chain of attempts where the batch leaves the
// chip idle, the instructions of an attempt where it does not.  A lone wave pays 4
// cycles for every instruction, so the loop holds one branch per attempt besides
// the accept, and nothing in it waits for memory: a refill retires its loads
// before the loop goes on (wait_vmem), and a step's row (t_n, h_n, y_n) is stored
// whole when the step is accepted and h_n is known, two 16-byte stores for N = 2.
// (With the waits on each step's stores and rows, here and in k_rev: solve of
// Van der Pol, B=1024, 2.67 ms, oscillator, B=2^20, 49.2 ms; without 2.10 and
// 34.4; with selects in the step control and, for Lone, the constants in vector
// registers 1.83 and 33.8.)
template <class Sys, class Tab, bool Adaptive, bool Lone>
__global__ void __launch_bounds__(256) k_fwd(FwdArgs a)
{
    if constexpr (Adaptive) load_ctrl_tables();
    constexpr int N = Sys::N;
    constexpr int F = N + 2;  // row (t_n, h_n, y_n)
    using R = RK<Sys, Tab, Lone>;
    const TabRegs<Tab, Lone> tc;
    const PowConsts<Lone && Adaptive> pc;
    const SolveParams sp = a.sp;
    const int64_t B = sp.B;
    const int32_t cap = (int32_t)sp.cap;  // va_problem.max_steps

    typename Sys::Params q;
    double y[N], k0[N] = {};  // k0 = f(y)
    double t = 0.0, dt = 0.0;
    int64_t b = 0;
    int32_t count = 0, rej = 0, tries = 0, st = LANE_OK;
    bool need = true;
    double *row = nullptr;  // row `count` of the instance

    // The head of the controlled loop at the point (t, y): false when the instance
    // is done (or has no room for another step), else dt clipped to end at t1.
    auto begin_step = [&]() {
        const bool more = Adaptive ? less_with_sign(t, sp.t1, dt)
                                   : less_eq_with_sign(t + sp.dt0, sp.t1, sp.dt0);
        if (more && count >= cap) st = LANE_MAX_STEPS;
        if constexpr (Adaptive)
            if (less_with_sign(sp.t1, t + dt, dt)) dt = sp.t1 - t;
        if constexpr (!Tab::FSAL) Sys::rhs(q, y, k0);
        tries = 0;
        return more && count < cap;
    };
    auto store_row = [&](double h) {
        row[0] = t;
        row[1] = h;
#pragma unroll
        for (int i = 0; i < N; ++i) row[2 + i] = y[i];
    };

    for (;;) {
        bool finish = false;
        if (need) {
            b = atomicAdd(a.counter, 1);
            if (b >= B) break;
            if (a.order) b = a.order[b];
            Sys::load(q, a.p, B, b, sp.kconst);
#pragma unroll
            for (int i = 0; i < N; ++i) y[i] = a.y[(int64_t)i * B + b];
            t = sp.t0;
            dt = sp.dt0;
            count = rej = 0;
            st = LANE_OK;
            need = false;
            row = a.traj + (size_t)b * (size_t)(sp.cap + 1) * F;
            wait_vmem();
            if constexpr (Tab::FSAL) Sys::rhs(q, y, k0);
            finish = !begin_step();
        }
        if (!finish) {
            const double h = Adaptive ? dt : sp.dt0;
            double K[Tab::SF][N], ynew[N], xerr[N];
#pragma unroll
            for (int i = 0; i < N; ++i) K[0][i] = k0[i];
            R::attempt(tc, q, y, K, h, ynew, xerr);
            bool accept = true, fail = false;
            if constexpr (Adaptive) {
                const double err = R::error_norm(sp.atol, sp.rtol, h, y, k0, xerr);
                accept = control_step<Tab>(h, err, dt, pc);
                fail = ++tries > sp.max_attempts;
            }
            if (accept) {
                ++count;
                const double tn = Adaptive ? t + h : sp.t0 + (double)count * sp.dt0;
                store_row(stored_step(tn, t));
                row += F;
                t = tn;
#pragma unroll
                for (int i = 0; i < N; ++i) {
                    y[i] = ynew[i];
                    if constexpr (Tab::FSAL) k0[i] = K[Tab::SF - 1][i];
                }
                finish = !begin_step();
            } else {
                ++rej;
            }
            if (fail) {
                st = LANE_MAX_FAIL;
                finish = true;
            }
        }
        if (finish) {
            if (st == LANE_OK) {
                store_row(0.0);
                if (!all_finite<N>(y)) st = LANE_NONFINITE;
            }
#pragma unroll
            for (int i = 0; i < N; ++i) a.y[(int64_t)i * B + b] = y[i];
            a.n_acc[b] = count;
            a.n_rej[b] = rej;
            a.status[b] = st;
            atomicMax(a.max_steps_seen, count);
            need = true;
        }
    }
}

// ---------------------------------------------------------------------------
// Reverse step (detail/backpropagation.hpp:83-158) on one stored row pair.
// ---------------------------------------------------------------------------
// NS seeds of one instance share the recomputed stages.
template <class Sys, class Tab, bool Opaque, int NS>
__device__ __forceinline__ void back_prop_step(const TabRegs<Tab, Opaque> &tc,
                                               const typename Sys::Params &q, double h,
                                               const double *yn, double (&lam)[NS][Sys::N],
                                               double (&pbar)[NS][Sys::P])
{
    // h = t_{n+1} - t_n as stored by the forward (the reference's GetDt).
    constexpr int N = Sys::N, S = Tab::S;
    using R = RK<Sys, Tab, Opaque>;
    double K[Tab::SF][N], X[S][N], Kb[NS][S][N];
#pragma unroll
    for (int m = 0; m < S; ++m) {
        R::stage_input(tc, m, h, yn, K, X[m]);
        Sys::rhs(q, X[m], K[m]);
    }
#pragma unroll
    for (int m = 0; m < S; ++m) {
        const double bh = tc.b[m] * h;
#pragma unroll
        for (int s = 0; s < NS; ++s)
#pragma unroll
            for (int i = 0; i < N; ++i) Kb[s][m][i] = bh * lam[s][i];
    }
#pragma unroll
    for (int m = S - 1; m >= 0; --m)
#pragma unroll
        for (int s = 0; s < NS; ++s) {
            double xi[N];
            Sys::vjp(q, X[m], Kb[s][m], xi, pbar[s]);
#pragma unroll
            for (int i = 0; i < N; ++i) lam[s][i] = lam[s][i] + xi[i];
#pragma unroll
            for (int j = 0; j < S; ++j) {
                if (j < m && Tab::A[m][j] != 0.0) {
#pragma unroll
                    for (int i = 0; i < N; ++i)
                        Kb[s][j][i] = Kb[s][j][i] + (xi[i] * tc.a[m][j]) * h;
                }
            }
        }
}

template <class Sys, class Tab, bool Opaque>
__device__ __forceinline__ void back_prop_step(const TabRegs<Tab, Opaque> &tc,
                                               const typename Sys::Params &q, double h,
                                               const double *yn, double (&lam)[Sys::N],
                                               double (&pbar)[Sys::P])
{
    back_prop_step<Sys, Tab, Opaque, 1>(tc, q, h, yn,
                                        reinterpret_cast<double (&)[1][Sys::N]>(lam),
                                        reinterpret_cast<double (&)[1][Sys::P]>(pbar));
}

template <int N>
__device__ __forceinline__ double terminal_cost(int cost, const double *w, const double *y,
                                                double *lam)
{
    double J = 0.0;
#pragma unroll
    for (int i = 0; i < N; ++i) {
        if (cost == COST_SUM) {
            J = J + y[i];
            lam[i] = 1.0;
        } else if (cost == COST_SQUARED_NORM) {
            J = fma(y[i], y[i], J);
            lam[i] = 2.0 * y[i];
        } else {
            J = fma(w[i], y[i], J);
            lam[i] = w[i];
        }
    }
    return J;
}

// ---------------------------------------------------------------------------
// Persistent reverse.  A work item is an instance with its seeds, or with a group
// of them (RevArgs::seeds_per_item): with few instances every seed has a lane of
// its own, with many a lane takes NS seeds through one sweep, which recomputes the
// stages once for all of them (RK4 oscillator, B=40000, two seeds, reverse alone
// 1.16 ms one after the other).
// ---------------------------------------------------------------------------
template <class Sys, class Tab, bool Lone, int NS>
__global__ void __launch_bounds__(256) k_rev(RevArgs a)
{
    const TabRegs<Tab, Lone> tc;
    constexpr int N = Sys::N, P = Sys::P, F = N + 2;
    const SolveParams sp = a.sp;
    const int64_t B = sp.B;
    const double qnan = __builtin_nan("");
    const RevItems items = rev_items(a);

    typename Sys::Params q;
    double lam[NS][N] = {}, pbar[NS][P] = {};
    int64_t b = 0;
    int32_t o = 0, o_end = 0, n = -1;  // seeds o .. o + NS - 1, of those below o_end
    bool need = true;
    const double *rows = nullptr;
    // rows n and n - 1 of the sweep, each loaded two steps before its own, so that
    // no step waits for memory (a step of a small system takes about 0.5 us, less
    // than a read from HBM)
    double h0 = 0.0, h1 = 0.0, y0[N] = {}, y1[N] = {};
    auto load_row = [&](int32_t k, double &h, double (&y)[N]) {
        const double *r = rows + (size_t)(k > 0 ? k : 0) * F;
        h = r[1];
#pragma unroll
        for (int i = 0; i < N; ++i) y[i] = r[2 + i];
    };
    // the seeds from o on, from the instance's last step
    auto start_sweep = [&]() {
        if (!a.cost) {
#pragma unroll
            for (int s = 0; s < NS; ++s)
#pragma unroll
                for (int i = 0; i < N; ++i) {
                    if (a.identity) lam[s][i] = o + s == i ? 1.0 : 0.0;
                    else if (o + s < o_end) lam[s][i] = a.lambda[((int64_t)(o + s) * N + i) * B + b];
                }
        }
#pragma unroll
        for (int s = 0; s < NS; ++s)
#pragma unroll
            for (int k = 0; k < P; ++k) pbar[s][k] = 0.0;
        n = a.n_acc[b] - 1;
        load_row(n, h0, y0);
        load_row(n - 1, h1, y1);
        wait_vmem();
    };

    for (;;) {
        if (need) {
            const int32_t k = atomicAdd(a.counter, 1);
            if (k >= B * items.parts) break;
            b = k;
            o = 0;
            if (items.parts > 1) {
                b = k / items.parts;
                o = (k - (int32_t)b * items.parts) * items.per;
            }
            o_end = o + items.per < items.seeds ? o + items.per : items.seeds;
            if (a.order) b = a.order[b];
            if (a.status[b] != LANE_OK) {
                for (; o < o_end; ++o) {
                    if (!a.identity)
                        for (int i = 0; i < N; ++i) a.lambda[((int64_t)o * N + i) * B + b] = qnan;
                    for (int j = 0; j < P; ++j) a.mu[((int64_t)o * P + j) * B + b] = qnan;
                }
                if (a.cost) a.J[b] = qnan;
                continue;
            }
            Sys::load(q, a.p, B, b, sp.kconst);
            rows = a.traj + (size_t)b * (size_t)(sp.cap + 1) * F;
            if (a.cost) {
                double yT[N];
#pragma unroll
                for (int i = 0; i < N; ++i) yT[i] = a.yT[(int64_t)i * B + b];
                a.J[b] = terminal_cost<N>(a.cost, a.cost_w, yT, lam[0]);
            }
            start_sweep();
            need = false;
        }
        if (n >= 0) {
            const double h = h0;
            double y[N];
            h0 = h1;
#pragma unroll
            for (int i = 0; i < N; ++i) {
                y[i] = y0[i];
                y0[i] = y1[i];
            }
            load_row(n - 2, h1, y1);
            // (the scheduler would move these loads to the end of the step)
            __builtin_amdgcn_sched_barrier(0);
            back_prop_step<Sys, Tab, Lone, NS>(tc, q, h, y, lam, pbar);
            --n;
        }
        if (n < 0) {
#pragma unroll
            for (int s = 0; s < NS; ++s) {
                if (o + s >= o_end) break;
                if (!a.identity) {
#pragma unroll
                    for (int i = 0; i < N; ++i)
                        a.lambda[((int64_t)(o + s) * N + i) * B + b] = lam[s][i];
                }
#pragma unroll
                for (int k = 0; k < P; ++k) {
                    double *m = a.mu + ((int64_t)(o + s) * P + k) * B + b;
                    *m = a.cost || a.identity ? 0.0 + pbar[s][k] : *m + pbar[s][k];
                }
            }
            o += NS;
            need = o >= o_end;
            if (!need) start_sweep();
        }
    }
}

// ---------------------------------------------------------------------------
// Plain GPU form
// ---------------------------------------------------------------------------
template <class Sys, class Tab, bool Adaptive>
__global__ void __launch_bounds__(256) k_plain_fwd(PlainFwdArgs a)
{
    if constexpr (Adaptive) load_ctrl_tables();
    constexpr int N = Sys::N;
    constexpr int F = 2 + N;  // fields (t_n, h_n, y_n)
    using R = RK<Sys, Tab>;
    const TabRegs<Tab, false> tc;
    const SolveParams sp = a.sp;
    const int64_t B = sp.B;
    const int64_t b = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (b >= B || a.st.done[b]) return;
    const int32_t step = a.step;

    typename Sys::Params q;
    Sys::load(q, a.p, B, b, sp.kconst);
    double y[N], K[Tab::SF][N], ynew[N], xerr[N];
#pragma unroll
    for (int i = 0; i < N; ++i) y[i] = a.y[(int64_t)i * B + b];
    double t = step == 0 ? sp.t0 : a.st.t[b];
    double dt = step == 0 ? sp.dt0 : a.st.dt[b];
    int32_t rej = step == 0 ? 0 : a.n_rej[b];
    double *row = a.traj + (size_t)step * F * B + b;

    const bool more = Adaptive ? less_with_sign(t, sp.t1, dt)
                               : less_eq_with_sign(t + sp.dt0, sp.t1, sp.dt0);
    int32_t st = LANE_OK;
    if (!more || step >= sp.cap) {
        if (more) {
            st = LANE_MAX_STEPS;
        } else {
            row[0] = t;
            row[(size_t)B] = 0.0;
#pragma unroll
            for (int i = 0; i < N; ++i) row[(size_t)(2 + i) * B] = y[i];
            if (!all_finite<N>(y)) st = LANE_NONFINITE;
        }
        a.status[b] = st;
        a.n_acc[b] = step;
        a.n_rej[b] = rej;
        a.st.done[b] = 1;
        atomicSub(a.st.active, 1);
        atomicMax(a.st.max_steps_seen, step);
        return;
    }
    row[0] = t;
#pragma unroll
    for (int i = 0; i < N; ++i) row[(size_t)(2 + i) * B] = y[i];
    if (Adaptive && less_with_sign(sp.t1, t + dt, dt)) dt = sp.t1 - t;
    if (Tab::FSAL && step > 0) {
#pragma unroll
        for (int i = 0; i < N; ++i) K[0][i] = a.st.k0[(int64_t)i * B + b];
    } else {
        Sys::rhs(q, y, K[0]);
    }
    if constexpr (Adaptive) {
        int32_t tries = 0;
        for (;;) {
            R::attempt(tc, q, y, K, dt, ynew, xerr);
            const double err = R::error_norm(sp.atol, sp.rtol, dt, y, K[0], xerr);
            double dt_next;
            const bool ok = control_step<Tab>(dt, err, dt_next);
            if (!ok) {
                ++rej;
            } else {
                const double tn = t + dt;
                row[(size_t)B] = stored_step(tn, t);
                t = tn;
            }
            dt = dt_next;
            ++tries;
            if (tries > sp.max_attempts) {
                if (ok) {
#pragma unroll
                    for (int i = 0; i < N; ++i) a.y[(int64_t)i * B + b] = ynew[i];
                }
                a.status[b] = LANE_MAX_FAIL;
                a.n_acc[b] = step + (ok ? 1 : 0);
                a.n_rej[b] = rej;
                a.st.done[b] = 1;
                atomicSub(a.st.active, 1);
                return;
            }
            if (ok) break;
        }
    } else {
        R::attempt(tc, q, y, K, sp.dt0, ynew, xerr);
        const double tn = sp.t0 + (double)(step + 1) * sp.dt0;
        row[(size_t)B] = stored_step(tn, t);
        t = tn;
    }
#pragma unroll
    for (int i = 0; i < N; ++i) a.y[(int64_t)i * B + b] = ynew[i];
    if constexpr (Tab::FSAL) {
#pragma unroll
        for (int i = 0; i < N; ++i) a.st.k0[(int64_t)i * B + b] = K[Tab::SF - 1][i];
    }
    a.st.t[b] = t;
    a.st.dt[b] = dt;
    a.n_rej[b] = rej;
    a.n_acc[b] = step + 1;
    a.status[b] = LANE_OK;
}

template <class Sys, class Tab>
__global__ void __launch_bounds__(256) k_plain_rev(PlainRevArgs a)
{
    constexpr int N = Sys::N, P = Sys::P;
    constexpr int F = 2 + N;
    const SolveParams sp = a.sp;
    const int64_t B = sp.B;
    const int64_t b = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (b >= B || a.status[b] != LANE_OK) return;
    const int32_t n = a.n_acc[b] - 1 - a.k;
    if (n < 0) return;

    typename Sys::Params q;
    Sys::load(q, a.p, B, b, sp.kconst);
    const double *row = a.traj + (size_t)n * F * B + b;
    const double h = row[(size_t)B];
    double yn[N], lam[N], pbar[P];
#pragma unroll
    for (int i = 0; i < N; ++i) yn[i] = row[(size_t)(2 + i) * B];
#pragma unroll
    for (int i = 0; i < N; ++i) lam[i] = a.lambda[(int64_t)i * B + b];
#pragma unroll
    for (int k = 0; k < P; ++k) pbar[k] = a.st.pbar[(int64_t)k * B + b];
    back_prop_step<Sys>(TabRegs<Tab, false>(), q, h, yn, lam, pbar);
#pragma unroll
    for (int i = 0; i < N; ++i) a.lambda[(int64_t)i * B + b] = lam[i];
#pragma unroll
    for (int k = 0; k < P; ++k) a.st.pbar[(int64_t)k * B + b] = pbar[k];
}

// ---------------------------------------------------------------------------
// Launchers and the dispatch table
// ---------------------------------------------------------------------------
// A launch whose waves have a SIMD each (at most one wave per SIMD of the 256
// CUs): its time is the waves' own instruction count, and it takes the kernels
// with the constants in vector registers.  Only small systems have them: the
// state of a larger one needs the registers.
constexpr int VA_LONE_THREADS = 256 * 4 * 64;

template <class Sys>
inline bool lone_waves(int grid, int block)
{
    return Sys::N <= 4 && (int64_t)grid * block <= VA_LONE_THREADS;
}

template <class Sys, class Tab, bool Ad>
struct Launch {
    static hipError_t fwd(const FwdArgs &a, int grid, int block, hipStream_t s)
    {
        if constexpr (Sys::N <= 4) {
            if (lone_waves<Sys>(grid, block)) {
                hipLaunchKernelGGL((k_fwd<Sys, Tab, Ad, true>), dim3(grid), dim3(block), 0, s, a);
                return hipGetLastError();
            }
        }
        hipLaunchKernelGGL((k_fwd<Sys, Tab, Ad, false>), dim3(grid), dim3(block), 0, s, a);
        return hipGetLastError();
    }
    // two seeds through one sweep where the state leaves room for both
    static constexpr bool kSeedPairs = Sys::N <= 4 && Sys::P <= 8;
    template <bool Lone>
    static hipError_t rev_as(const RevArgs &a, int grid, int block, hipStream_t s)
    {
        if constexpr (kSeedPairs) {
            if (rev_items(a).per > 1) {
                hipLaunchKernelGGL((k_rev<Sys, Tab, Lone, 2>), dim3(grid), dim3(block), 0, s, a);
                return hipGetLastError();
            }
        }
        hipLaunchKernelGGL((k_rev<Sys, Tab, Lone, 1>), dim3(grid), dim3(block), 0, s, a);
        return hipGetLastError();
    }
    static hipError_t rev(const RevArgs &a, int grid, int block, hipStream_t s)
    {
        if constexpr (Sys::N <= 4)
            if (lone_waves<Sys>(grid, block)) return rev_as<true>(a, grid, block, s);
        return rev_as<false>(a, grid, block, s);
    }
    static hipError_t pfwd(const PlainFwdArgs &a, int grid, int block, hipStream_t s)
    {
        hipLaunchKernelGGL((k_plain_fwd<Sys, Tab, Ad>), dim3(grid), dim3(block), 0, s, a);
        return hipGetLastError();
    }
    static hipError_t prev(const PlainRevArgs &a, int grid, int block, hipStream_t s)
    {
        hipLaunchKernelGGL((k_plain_rev<Sys, Tab>), dim3(grid), dim3(block), 0, s, a);
        return hipGetLastError();
    }
    static int occ_fwd(int block)
    {
        int nb = 0;
        if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, k_fwd<Sys, Tab, Ad, false>, block, 0) !=
            hipSuccess)
            return 1;
        return nb;
    }
    static int occ_rev(int block)
    {
        int nb = 0;
        if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, k_rev<Sys, Tab, false, 1>, block, 0) !=
            hipSuccess)
            return 1;
        return nb;
    }
    static int slots(int block) { return block; }
    static KernelSet make()
    {
        KernelSet k{};
        k.n = Sys::N;
        k.np = Sys::P;
        k.s_rev = Tab::S;
        k.s_fwd = Tab::SF;
        k.flop_rhs = Sys::FLOP_RHS;
        k.flop_vjp = Sys::FLOP_VJP;
        k.fwd = &fwd;
        k.rev = &rev;
        k.plain_fwd = &pfwd;
        k.plain_rev = &prev;
        k.occ_fwd = &occ_fwd;
        k.occ_rev = &occ_rev;
        k.slots = &slots;
        k.layout = 0;
        return k;
    }
};


enum { TAB_EULER = 1, TAB_RK4 = 2, TAB_CK54 = 3, TAB_DOPRI5 = 4, TAB_F78 = 5 };


template <class Sys>
inline bool pick_tableau(int tableau, int adaptive, KernelSet *out)
{
    if (adaptive) {
        switch (tableau) {
        case TAB_CK54: *out = Launch<Sys, CashKarp54, true>::make(); return true;
        case TAB_DOPRI5: *out = Launch<Sys, Dopri5, true>::make(); return true;
        case TAB_F78: *out = Launch<Sys, Fehlberg78, true>::make(); return true;
        default: return false;
        }
    }
    switch (tableau) {
    case TAB_EULER: *out = Launch<Sys, Euler, false>::make(); return true;
    case TAB_RK4: *out = Launch<Sys, RK4, false>::make(); return true;
    case TAB_CK54: *out = Launch<Sys, CashKarp54, false>::make(); return true;
    case TAB_DOPRI5: *out = Launch<Sys, Dopri5, false>::make(); return true;
    case TAB_F78: *out = Launch<Sys, Fehlberg78, false>::make(); return true;
    default: return false;
    }
}

}  // namespace va
