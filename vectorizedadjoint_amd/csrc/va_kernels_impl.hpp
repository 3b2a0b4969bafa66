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

// Slot s's rows, and row r among them (see RowLayout).
__device__ __forceinline__ int64_t slot_rows(const RowLayout &l, int64_t s)
{
    return (int64_t)((uint64_t)s / VA_ROW_TILE) * l.tile + (int64_t)(s & (VA_ROW_TILE - 1)) * l.lane;
}
template <int F>
__device__ __forceinline__ int64_t row_offset(const RowLayout &l, int32_t r)
{
    const uint32_t u = (uint32_t)r;
    return (int64_t)(u / VA_ROW_BLOCK) * l.blk + (u % VA_ROW_BLOCK) * F;
}

// A reverse's rows: (h, y) of row r of one slot, row 0 below it.  Five vector
// instructions of address per row, for a lone wave pays for each of them.
template <int F>
struct RowsBack {
    const double *p;   // the slot's row 0; always a slot of the store, also without an item
    uint32_t blk = 0;  // bytes between blocks of rows
    template <int N>
    __device__ __forceinline__ void load(int32_t r, double &h, double (&y)[N]) const
    {
        const uint32_t u = r > 0 ? (uint32_t)r : 0u;
        const char *at = (const char *)p + (uint64_t)(u / VA_ROW_BLOCK) * blk;
        const double *q = (const double *)(at + (uint64_t)(u % VA_ROW_BLOCK * (F * 8)));
        h = q[1];
#pragma unroll
        for (int i = 0; i < N; ++i) y[i] = q[2 + i];
    }
};

template <int N>
__device__ __forceinline__ bool all_finite(const double *y)
{
    bool ok = true;
#pragma unroll
    for (int i = 0; i < N; ++i) ok = ok && (fabs(y[i]) <= 1.7976931348623157e308);
    return ok;
}

// A wave's lines of four rows (N = 2, 128 bytes) on their way to or from the
// tiled store, each lane's in LDS.  The stride of 144 bytes leaves the lanes'
// 16-byte accesses, and the wave's accesses to eight lines at a time, without
// bank conflicts.  Every lane of the wave calls store() and load().
typedef double d2 __attribute__((ext_vector_type(2)));

struct WaveLines {
    d2 line[64][9];
    d2 *addr[64];
    int src[64];

    // Write the lines of the lanes with full set to to[] of each.
    __device__ __forceinline__ void store(bool full, int lane, double *to)
    {
        const uint64_t m = __builtin_amdgcn_ballot_w64(full);
        if (m == 0) return;
        const int n = __builtin_popcountll(m);
        const int rank = __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32),
                                                   __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0));
        if (full) {
            addr[rank] = reinterpret_cast<d2 *>(to);
            src[rank] = lane;
        }
        __builtin_amdgcn_wave_barrier();
        for (int j = lane >> 3; j < n; j += 8) addr[j][lane & 7] = line[src[j]][lane & 7];
        __builtin_amdgcn_wave_barrier();
    }

    // Chunk lane % 8 of the lines of lanes lane / 8 + 8 j, at from[] of each.
    __device__ __forceinline__ void load(int lane, const double *from, d2 (&v)[8])
    {
        addr[lane] = const_cast<d2 *>(reinterpret_cast<const d2 *>(from));
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int j = 0; j < 8; ++j) v[j] = addr[(lane >> 3) + 8 * j][lane & 7];
        __builtin_amdgcn_wave_barrier();
    }
    __device__ __forceinline__ void keep(int lane, const d2 (&v)[8])
    {
#pragma unroll
        for (int j = 0; j < 8; ++j) line[(lane >> 3) + 8 * j][lane & 7] = v[j];
        __builtin_amdgcn_wave_barrier();
    }
};

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
// registers 1.83 and 33.8; with rows three ahead in k_rev's Lone loop 1.73.)
//
// Lines (N = 2, tiled rows): a row's two 16-byte stores touch a line per lane
// each, and at 128 requests per row of a wave the path to L2 was the bound of a
// full chip (oscillator, B=2^20: forward 14.4 ms, 6.4 of them vector
// instructions).  A lane there gathers its line, four rows, in LDS; lanes whose
// lines are full hand them to the whole wave, which stores eight lines per
// instruction: forward 11.2 ms.
template <class Sys, class Tab, bool Adaptive, bool Lone, bool Lines = false>
__global__ void __launch_bounds__(256) k_fwd(FwdArgs a)
{
    static_assert(!Lines || Sys::N == 2, "lines of four rows are 128 bytes for N = 2");
    __shared__ WaveLines lines[Lines ? 4 : 1];
    const int lane = threadIdx.x & 63;
    WaveLines &wl = lines[Lines ? threadIdx.x >> 6 : 0];
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
    bool need = true, over = false;  // over (Lines): no instance left for this lane
    double *row = nullptr;  // row `count` of the instance (Lines: the first of its block)
    const int64_t row_wrap = a.rows.blk - (VA_ROW_BLOCK - 1) * F;  // to the next block of rows

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
    auto put_row = [&](double *to, double h) {
        to[0] = t;
        to[1] = h;
#pragma unroll
        for (int i = 0; i < N; ++i) to[2 + i] = y[i];
    };
    auto store_row = [&](double h) {
        if constexpr (Lines)
            put_row(reinterpret_cast<double *>(wl.line[lane] + 2 * (count % VA_ROW_BLOCK)), h);
        else
            put_row(row, h);
    };

    // one attempt, and after an accepted one the head of the next step
    auto attempt = [&](bool &finish, bool &full) {
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
            const double tn = Adaptive ? t + h : sp.t0 + (double)(count + 1) * sp.dt0;
            store_row(stored_step(tn, t));
            ++count;
            full = count % VA_ROW_BLOCK == 0;
            if constexpr (!Lines) row += full ? row_wrap : F;
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
    };

    for (;;) {
        bool finish = false, full = false;
        if (need && !over) {
            const int64_t k = atomicAdd(a.counter, 1);
            if constexpr (Lines) {
                over = k >= B;
            } else {
                if (k >= B) break;
            }
            if (!over) {
                b = a.order ? a.order[k] : k;
                if (a.slot) a.slot[b] = (int32_t)k;
                Sys::load(q, a.p, B, b, sp.kconst);
#pragma unroll
                for (int i = 0; i < N; ++i) y[i] = a.y[(int64_t)i * B + b];
                t = sp.t0;
                dt = sp.dt0;
                count = rej = 0;
                st = LANE_OK;
                need = false;
                row = a.traj + slot_rows(a.rows, a.slot ? k : b);
                wait_vmem();
                if constexpr (Tab::FSAL) Sys::rhs(q, y, k0);
                finish = !begin_step();
            }
        }
        if constexpr (Lines)
            if (__builtin_amdgcn_ballot_w64(!over) == 0) break;  // the wave, all at once
        if constexpr (Lone) {
            // (no refill until all of the wave's lanes are done: see VA_LONE_THREADS)
            while (!finish) attempt(finish, full);
        } else if (!finish && !over) {
            attempt(finish, full);
        }
        if constexpr (Lines) {
            wl.store(full, lane, row);
            if (full) row += a.rows.blk;
        }
        if (finish) {
            if constexpr (Lines) {  // the rows of a line that is not full
                const d2 *l = wl.line[lane];
                for (int r = 0; r < 2 * (count % VA_ROW_BLOCK); ++r)
                    reinterpret_cast<d2 *>(row)[r] = l[r];
                row += count % VA_ROW_BLOCK * F;
            }
            if (st == LANE_OK) {
                put_row(row, 0.0);
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
// Rows are loaded two steps ahead; for waves that run alone three steps share a
// trip, so that no row is copied between registers and the wait for it lies where
// it is used (Van der Pol, B=1024, reverse 0.78 ms with a copy and a wait per step,
// 0.69 so).
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
    // the rows of the next steps, each loaded two steps before its own, so that no
    // step waits for memory (a step of a small system takes about 0.6 us, less than
    // a read from HBM)
    double hr[3] = {}, yr[3][N] = {};
    RowsBack<F> rows{a.traj, (uint32_t)a.rows.blk * 8u};
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
#pragma unroll
        for (int s = 0; s < 3; ++s) rows.load(n - s, hr[s], yr[s]);
        wait_vmem();
    };

    // reverse step n, whose row is in slot s, and load row n - 3 there (a lane that
    // is done loads row 0: no branch around the load, so that the compiler's wait
    // for it comes where it is used)
    auto step = [&](int s) {
        if (n >= 0) back_prop_step<Sys, Tab, Lone, NS>(tc, q, hr[s], yr[s], lam, pbar);
        __builtin_amdgcn_sched_barrier(0);  // (the row's registers are free from here)
        rows.load(n - 3, hr[s], yr[s]);
        --n;
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
            rows.p = a.traj + slot_rows(a.rows, a.slot ? a.slot[b] : b);
            if (a.cost) {
                double yT[N];
#pragma unroll
                for (int i = 0; i < N; ++i) yT[i] = a.yT[(int64_t)i * B + b];
                a.J[b] = terminal_cost<N>(a.cost, a.cost_w, yT, lam[0]);
            }
            start_sweep();
            need = false;
        }
        if constexpr (Lone) {
            // three steps per trip, so that each slot keeps its registers; no refill
            // until all of the wave's lanes are done (see VA_LONE_THREADS)
            do {
                step(0);
                step(1);
                step(2);
            } while (__builtin_amdgcn_ballot_w64(n >= 0) != 0);
        } else if (n >= 0) {
            step(0);
            const double h = hr[0];
            hr[0] = hr[1];
            hr[1] = hr[2];
            hr[2] = h;
#pragma unroll
            for (int i = 0; i < N; ++i) {
                const double y = yr[0][i];
                yr[0][i] = yr[1][i];
                yr[1][i] = yr[2][i];
                yr[2][i] = y;
            }
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

// The same for one seed, N = 2 and a tiled store on a full chip, by lines of four
// rows: every fourth trip the wave keeps the lines its lanes need next in LDS and
// loads those after them, eight lines per instruction (a lane's own loads touch a
// line each: oscillator, B=2^20, reverse 11.6 ms, 6.0 of them vector
// instructions).  Row r is reversed in a trip with 3 - r = trip (mod 4), so all
// lanes need new lines at the same trip; an instance waits at most three trips for
// its first.  Reverse 8.0 ms.
template <class Sys, class Tab>
__global__ void __launch_bounds__(256) k_rev_lines(RevArgs a)
{
    constexpr int N = Sys::N, P = Sys::P, F = N + 2;
    static_assert(N == 2, "lines of four rows are 128 bytes for N = 2");
    __shared__ WaveLines lines[4];
    const int lane = threadIdx.x & 63;
    WaveLines &wl = lines[threadIdx.x >> 6];
    const TabRegs<Tab, false> tc;
    const int64_t B = a.sp.B;
    const double qnan = __builtin_nan("");

    typename Sys::Params q;
    double lam[N] = {}, pbar[P] = {};
    int64_t b = 0;
    int32_t n = -1;  // the next step to reverse
    bool need = true, over = false;
    const double *line = a.traj;  // the line with row n
    d2 v[8];                      // lines before those in LDS, as load() gives them

    for (;;) {
        // every lane finds an instance with steps left, or none
        bool fresh = false;
        while (need && !over) {
            const int64_t k = atomicAdd(a.counter, 1);
            over = k >= B;
            if (over) break;
            b = a.order ? a.order[k] : k;
            if (a.status[b] != LANE_OK) {
#pragma unroll
                for (int i = 0; i < N; ++i) a.lambda[(int64_t)i * B + b] = qnan;
                for (int j = 0; j < P; ++j) a.mu[(int64_t)j * B + b] = qnan;
                if (a.cost) a.J[b] = qnan;
                continue;
            }
            Sys::load(q, a.p, B, b, a.sp.kconst);
            if (a.cost) {
                double yT[N];
#pragma unroll
                for (int i = 0; i < N; ++i) yT[i] = a.yT[(int64_t)i * B + b];
                a.J[b] = terminal_cost<N>(a.cost, a.cost_w, yT, lam);
            } else {
#pragma unroll
                for (int i = 0; i < N; ++i) lam[i] = a.lambda[(int64_t)i * B + b];
            }
#pragma unroll
            for (int j = 0; j < P; ++j) pbar[j] = 0.0;
            n = a.n_acc[b] - 1;
            const int32_t last = n > 0 ? n : 0;
            line = a.traj + slot_rows(a.rows, a.slot ? a.slot[b] : b) +
                   (int64_t)(last / VA_ROW_BLOCK) * a.rows.blk;
            need = false;
            fresh = true;
            wait_vmem();
        }
        if (__builtin_amdgcn_ballot_w64(!over) == 0) break;  // the wave, all at once
        // a lane's first line was not loaded ahead
        if (__builtin_amdgcn_ballot_w64(fresh) != 0) wl.load(lane, line, v);
        wl.keep(lane, v);
        if (n >= VA_ROW_BLOCK) line -= a.rows.blk;
        wl.load(lane, line, v);
        __builtin_amdgcn_sched_barrier(0);  // the loads stay ahead of the steps
#pragma unroll 1
        for (int r = VA_ROW_BLOCK - 1; r >= 0; --r) {
            if (n >= 0 && !over && n % VA_ROW_BLOCK == r) {
                const double h = wl.line[lane][2 * r].y;
                const d2 yr = wl.line[lane][2 * r + 1];
                const double y[N] = {yr.x, yr.y};
                back_prop_step<Sys>(tc, q, h, y, lam, pbar);
                --n;
            }
        }
        if (n < 0 && !need && !over) {
#pragma unroll
            for (int i = 0; i < N; ++i) a.lambda[(int64_t)i * B + b] = lam[i];
#pragma unroll
            for (int j = 0; j < P; ++j) {
                double *m = a.mu + (int64_t)j * B + b;
                *m = a.cost || a.identity ? 0.0 + pbar[j] : *m + pbar[j];
            }
            need = true;
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
// with the constants in vector registers (Lone).  With more instances than lanes
// as well, where a wave takes new ones only when all of its own have ended: Van
// der Pol, B=131072 on 4096 lanes, forward 10.2 ms against 16.1 of the refilling
// kernel, in index order 16.5 / 17.6; Lotka-Volterra N=4, one lane each, on
// 16384 lanes 0.49 / 0.97 and 0.61 / 1.41.
constexpr int VA_LONE_THREADS = 256 * 4 * 64;
inline bool lone_waves(int grid, int block) { return (int64_t)grid * block <= VA_LONE_THREADS; }

// Only sweeps whose values fit beside the constants have such kernels: a lane has
// 512 registers, 256 doubles, and the compiler needs some third of them for
// intermediates.  Reverses with one seed, B=65536, Lone against not, by the doubles
// counted here: Lotka-Volterra N=4, Cash-Karp (107) 332 / 430 us; N=2, Fehlberg
// 7(8) (126) 129 / 131; N=3, Fehlberg (164) 185 / 241; N=4, Fehlberg (206, which
// puts 592 bytes per lane in scratch memory) 810 / 641 us.
constexpr int VA_LONE_DOUBLES = 168;

constexpr int count_nonzero(const double *v, int n)
{
    int c = 0;
    for (int k = 0; k < n; ++k) c += v[k] != 0.0;
    return c;
}
// the stage weights of the first `stages` stages, and the solution's
template <class Tab>
constexpr int stage_constants(int stages)
{
    int c = count_nonzero(Tab::B, Tab::S);
    for (int m = 1; m < stages; ++m) c += count_nonzero(Tab::A[m], m);
    return c;
}
// the embedded error's weights and the controller's pow (PowRegs)
template <class Tab>
constexpr int control_constants()
{
    if constexpr (Tab::HAS_ERR) return count_nonzero(Tab::DB, Tab::SF) + 17;
    else return 0;
}
template <class Sys, class Tab>
constexpr bool lone_forward(bool adaptive)
{
    return Sys::N <= 4 && Sys::N * Tab::SF + Sys::P + stage_constants<Tab>(Tab::SF) +
                                  (adaptive ? control_constants<Tab>() : 0) <=
                              VA_LONE_DOUBLES;
}
// replay: an observed reverse, which runs the forward's steps again
template <class Sys, class Tab, int NS>
constexpr bool lone_reverse(bool replay = false)
{
    return Sys::N <= 4 && (1 + NS) * (Sys::N * Tab::S + Sys::P) + stage_constants<Tab>(Tab::S) +
                                  (replay ? control_constants<Tab>() : 0) <=
                              VA_LONE_DOUBLES;
}

template <class Sys, class Tab, bool Ad>
struct Launch {
    static hipError_t fwd(const FwdArgs &a, int grid, int block, hipStream_t s)
    {
        if constexpr (lone_forward<Sys, Tab>(Ad)) {
            if (lone_waves(grid, block)) {
                hipLaunchKernelGGL((k_fwd<Sys, Tab, Ad, true>), dim3(grid), dim3(block), 0, s, a);
                return hipGetLastError();
            }
        }
        if constexpr (Sys::N == 2) {
            if (a.slot) {
                hipLaunchKernelGGL((k_fwd<Sys, Tab, Ad, false, true>), dim3(grid), dim3(block), 0,
                                   s, a);
                return hipGetLastError();
            }
        }
        hipLaunchKernelGGL((k_fwd<Sys, Tab, Ad, false>), dim3(grid), dim3(block), 0, s, a);
        return hipGetLastError();
    }
    // two seeds through one sweep where the state leaves room for both
    static constexpr bool kSeedPairs = Sys::N <= 4 && Sys::P <= 8;
    template <int NS>
    static hipError_t rev_as(const RevArgs &a, int grid, int block, hipStream_t s)
    {
        if constexpr (lone_reverse<Sys, Tab, NS>()) {
            if (lone_waves(grid, block)) {
                hipLaunchKernelGGL((k_rev<Sys, Tab, true, NS>), dim3(grid), dim3(block), 0, s, a);
                return hipGetLastError();
            }
        }
        if constexpr (Sys::N == 2 && NS == 1) {
            if (a.slot && rev_items(a).seeds == 1 && !a.identity) {
                hipLaunchKernelGGL((k_rev_lines<Sys, Tab>), dim3(grid), dim3(block), 0, s, a);
                return hipGetLastError();
            }
        }
        hipLaunchKernelGGL((k_rev<Sys, Tab, false, NS>), dim3(grid), dim3(block), 0, s, a);
        return hipGetLastError();
    }
    static hipError_t rev(const RevArgs &a, int grid, int block, hipStream_t s)
    {
        if constexpr (kSeedPairs)
            if (rev_items(a).per > 1) return rev_as<2>(a, grid, block, s);
        return rev_as<1>(a, grid, block, s);
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
