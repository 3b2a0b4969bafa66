// va_observed.hpp -- observation-cost forward and reverse sweeps (one lane per
// instance), with the trajectory stored in full or kept as checkpoints.
//
// No reference counterpart: the reference's cost is terminal only
// (examples/VanDerPol/main.cpp:98-117).  The forward is the controlled loop of
// lib/include/detail/runge_kutta.hpp:74-118 run segment by segment: a step that
// would pass the next observation time is shortened to land on it, as at t1
// (:98-101); after such a shortened step is accepted, the next step size is the
// larger of the controller's proposal and the size before shortening (what
// Boost.odeint 1.74 integrate_times does for controlled steppers).  At each
// observation time the running cost J += |y - y_obs_k|^2 is accumulated and the
// stored-point index recorded.  The reverse is the discrete adjoint of
// detail/backpropagation.hpp:83-158 with lambda += 2 (y_n - y_obs_k) at every
// observation point.
//
// Checkpoints.  With a trajectory budget too small for every row, an instance
// keeps `slots` checkpoints (t, dt to try, observations taken, y) at every
// `stride`-th accepted step; when the slots fill up, every other checkpoint is
// dropped and the stride doubles, so any step count up to slots * stride_max
// fits.  The reverse rebuilds each segment's rows from its checkpoint by
// replaying the controlled loop (the same decisions, so bit-identical rows, and
// f(y) from the checkpoint equals the FSAL value carried by the forward), then
// sweeps the segment backwards.  Memory: slots rows per instance plus
// stride_max rows per lane; work: one extra forward pass.
#pragma once

#include "va_kernels_impl.hpp"

namespace va {

// The time the controlled loop heads for after observation kobs - 1: observation
// kobs's time, or t1 once every observation is taken.  It waits for its load at
// once (s_waitcnt vmcnt(0)): it runs only where an observation is passed, and
// with the load retired there the steps in between test the target without
// waiting for the wave's earlier row stores (gfx9 counts loads and stores in
// one in-order counter).
__device__ __forceinline__ double obs_time(const double *obs_t, int K, int kobs, double t1)
{
    const double v = kobs < K ? obs_t[kobs] : t1;
    __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt 0; expcnt and lgkmcnt left at their maxima
    return v;
}

// The stored-point index of observation kobs, or -1 (no point) once kobs < 0.
__device__ __forceinline__ int32_t obs_point(const int32_t *orow, int kobs)
{
    return kobs >= 0 ? orow[kobs] : -1;
}

// Observation jumps at stored point `point` (state yn), newest observation first.
// `next` holds obs_point(orow, kobs) and is reloaded only when kobs moves, so
// the steps between observations test a register instead of waiting on a load.
template <int N>
__device__ __forceinline__ int obs_jumps(const int32_t *orow, const double *obs_y, int kobs,
                                         int32_t &next, int32_t point, const double *yn,
                                         double *lam)
{
    while (kobs >= 0 && next == point) {
#pragma unroll
        for (int i = 0; i < N; ++i) lam[i] = fma(2.0, yn[i] - obs_y[kobs * N + i], lam[i]);
        --kobs;
        next = obs_point(orow, kobs);
    }
    return kobs;
}

// ---------------------------------------------------------------------------
// Forward
// ---------------------------------------------------------------------------
// Structured and bounded like k_fwd: one branch per attempt besides the accept,
// no wait for memory in the loop but where an observation is passed, rows stored
// whole at the accept, the constants in vector registers for waves that run
// alone (Lone).  With the full store's rows loaded ahead in the reverse: solve of
// B=6000, mu to 10, full store, 4.71 -> 3.40 ms; B=262144, 4 GB, 27.2 -> 24.9 ms.
template <class Sys, class Tab, bool Ckpt, bool Lone>
__global__ void __launch_bounds__(256) k_obs_fwd(ObsFwdArgs a)
{
    load_ctrl_tables();
    constexpr int N = Sys::N;
    constexpr int F = N + 2, FC = N + 3;
    using R = RK<Sys, Tab, Lone>;
    const TabRegs<Tab, Lone> tc;
    const PowConsts<Lone> pc;
    const SolveParams sp = a.sp;
    const int64_t B = sp.B;
    const int32_t cap = (int32_t)sp.cap;
    const int K = a.K;

    typename Sys::Params q;
    double y[N], k0[N] = {};  // k0 = f(y)
    // tnext: the next target, obs_time(a.obs_t, K, kobs, sp.t1), reloaded only
    // when kobs moves, so a step's clipping test waits on no load
    double t = 0.0, dt = 0.0, dt_keep = 0.0, Jacc = 0.0, tnext = 0.0;
    int64_t b = 0;
    int32_t count = 0, rej = 0, tries = 0, st = LANE_OK, kobs = 0, stride = 1, nck = 0;
    bool need = true, clipped = false;
    double *row = nullptr, *ck = nullptr;  // row: row `count` of the full store
    const int64_t row_wrap = a.st.rows.blk - (VA_ROW_BLOCK - 1) * F;
    int32_t *orow = nullptr;

    // The head of the controlled loop at the point (t, y): the observations
    // reached here, then false when the instance is done (or has no room for
    // another step), else dt clipped to end at the next target.
    auto begin_step = [&]() {
        bool more = less_with_sign(t, tnext, dt);
        while (!more && kobs < K) {
            orow[kobs] = count;
#pragma unroll
            for (int i = 0; i < N; ++i) {
                const double d = y[i] - a.obs_y[kobs * N + i];
                Jacc = fma(d, d, Jacc);
            }
            ++kobs;
            tnext = obs_time(a.obs_t, K, kobs, sp.t1);
            more = less_with_sign(t, tnext, dt);
        }
        if (more && count >= cap) st = LANE_MAX_STEPS;
        more = more && count < cap;
        if constexpr (Ckpt) {
            // stride is a power of two (it starts at 1 and is only doubled), so
            // this is count % stride == 0 without the integer division's two
            // dozen instructions on every step
            if (more && (count & (stride - 1)) == 0) {
                if (nck >= a.st.slots) {
                    // drop every other checkpoint, double the spacing
                    for (int m = 1; m < a.st.slots / 2; ++m)
#pragma unroll
                        for (int f = 0; f < FC; ++f)
                            ck[(size_t)m * FC + f] = ck[(size_t)(2 * m) * FC + f];
                    stride *= 2;
                    nck = a.st.slots / 2;
                }
                double *c = ck + (size_t)nck * FC;
                c[0] = t;
                c[1] = dt;
                c[2] = (double)kobs;
#pragma unroll
                for (int i = 0; i < N; ++i) c[3 + i] = y[i];
                ++nck;
            }
        }
        dt_keep = dt;
        clipped = less_with_sign(tnext, t + dt, dt);
        dt = clipped ? tnext - t : dt;
        clipped = clipped && kobs < K;
        if constexpr (!Tab::FSAL) Sys::rhs(q, y, k0);
        tries = 0;
        return more;
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
            const int64_t k = atomicAdd(a.counter, 1);
            if (k >= B) break;
            b = a.order ? a.order[k] : k;
            Sys::load(q, a.p, B, b, sp.kconst);
#pragma unroll
            for (int i = 0; i < N; ++i) y[i] = a.y[(int64_t)i * B + b];
            t = sp.t0;
            dt = sp.dt0;
            Jacc = 0.0;
            stride = 1;
            if constexpr (Ckpt) {
                // Start from the spacing the previous solve of this instance reached
                // (its step count is still in n_acc until this one finishes): the
                // smallest with room for that many steps, so that a solve taking
                // the same steps again never fills the slots.  Each doubling moves
                // half the checkpoints, one lane at a time, and with one lane per
                // instance the whole wave waits for any lane that moves them (half
                // that spacing, which filled the slots once per solve, cost 10% of
                // the observed Van der Pol solve).  Any spacing gives the same
                // results: the reverse replays the forward from each checkpoint.
                if (a.order) stride = obs_first_stride(a.n_acc[b], a.st.slots, a.st.stride_max);
            }
            count = rej = kobs = nck = 0;
            st = LANE_OK;
            need = false;
            if constexpr (Ckpt) {
                ck = a.st.ck + (size_t)b * (size_t)a.st.slots * FC;
            } else {
                if (a.st.slot) a.st.slot[b] = (int32_t)k;
                row = a.st.traj + slot_rows(a.st.rows, a.st.slot ? k : b);
            }
            orow = a.st.obs_row + (size_t)b * (size_t)K;
            tnext = obs_time(a.obs_t, K, 0, sp.t1);  // waits for the loads above as well
            if constexpr (Tab::FSAL) Sys::rhs(q, y, k0);
            finish = !begin_step();
        }
        if (!finish) {
            const double h = dt;
            double Kst[Tab::SF][N], ynew[N], xerr[N];
#pragma unroll
            for (int i = 0; i < N; ++i) Kst[0][i] = k0[i];
            R::attempt(tc, q, y, Kst, h, ynew, xerr);
            const double err = R::error_norm(sp.atol, sp.rtol, h, y, k0, xerr);
            const bool accept = control_step<Tab>(h, err, dt, pc);
            const bool fail = ++tries > sp.max_attempts;
            if (accept) {
                const double tn = t + h;
                if constexpr (!Ckpt) {
                    store_row(stored_step(tn, t));
                    row += (count + 1) % VA_ROW_BLOCK ? F : row_wrap;
                }
                t = tn;
#pragma unroll
                for (int i = 0; i < N; ++i) {
                    y[i] = ynew[i];
                    if constexpr (Tab::FSAL) k0[i] = Kst[Tab::SF - 1][i];
                }
                if (clipped && fabs(dt_keep) > fabs(dt)) dt = dt_keep;
                ++count;
                finish = !begin_step();
            } else {
                ++rej;
                clipped = false;
            }
            if (fail) {
                st = LANE_MAX_FAIL;
                finish = true;
            }
        }
        if (finish) {
            if (st == LANE_OK) {
                if constexpr (!Ckpt) store_row(0.0);
                if (!all_finite<N>(y)) st = LANE_NONFINITE;
            }
#pragma unroll
            for (int i = 0; i < N; ++i) a.y[(int64_t)i * B + b] = y[i];
            a.J[b] = st == LANE_OK ? Jacc : __builtin_nan("");
            a.n_acc[b] = count;
            a.n_rej[b] = rej;
            a.status[b] = st;
            if constexpr (Ckpt) a.st.stride[b] = stride;
            atomicMax(a.max_steps_seen, count);
            need = true;
        }
    }
}

// ---------------------------------------------------------------------------
// Reverse
// ---------------------------------------------------------------------------

// Replay `len` accepted steps from the checkpoint c (t, dt to try, observations
// taken, y), running the forward's controlled loop with the same observation
// stops, and either (Rows) rebuild their rows (h_n, y_n) into seg, h_n =
// t_{n+1} - t_n, or (!Rows) store a checkpoint of the same form as c at the start
// of every `sub`-th step into seg (the level-2 checkpoints of a long segment).
// Field f of row / checkpoint k is seg[(k W + f) ss] with W = N+1 / N+3: the
// lanes' buffers are interleaved (ss = the grid's thread count), so a wave's
// stores and loads of one field coalesce.  One trip of the loop is one attempt,
// whether the lane starts a step or retries one, so the lanes of a wave do not
// wait for each other's rejected attempts step by step (with 64 lanes some lane
// rejects in most steps); the values formed are those of the forward.
template <class Sys, class Tab, bool Lone, bool Rows = true>
__device__ void recompute_segment(const TabRegs<Tab, Lone> &tc, const PowConsts<Lone> &pc,
                                  const typename Sys::Params &q, const SolveParams &sp,
                                  const double *obs_t, int K, const double *c, int32_t len,
                                  double *seg, int64_t ss, int32_t sub = 1)
{
    constexpr int N = Sys::N, FS = N + 1, FC = N + 3;
    using R = RK<Sys, Tab, Lone>;
    double y[N], k0[N];
    double t = c[0], dt = c[1], dt_keep = 0.0;
    int kobs = (int)c[2];
#pragma unroll
    for (int i = 0; i < N; ++i) y[i] = c[3 + i];
    double tnext = obs_time(obs_t, K, kobs, sp.t1);  // as in the forward
    // f(y) here equals the FSAL value the forward carried into this step: the
    // last stage input of DOPRI5 is y_{n+1} computed with the same operations.
    Sys::rhs(q, y, k0);
    int32_t k = 0, tries = 0;
    bool clipped = false;
    double *r = seg;  // field 0 of row k
    auto begin_step = [&]() {
        bool more = less_with_sign(t, tnext, dt);
        while (!more && kobs < K) {
            ++kobs;
            tnext = obs_time(obs_t, K, kobs, sp.t1);
            more = less_with_sign(t, tnext, dt);
        }
        if constexpr (!Rows) {
            if (k < len && k % sub == 0) {
                double *c2 = seg + (size_t)(k / sub) * FC * ss;
                c2[0] = t;
                c2[ss] = dt;
                c2[2 * ss] = (double)kobs;
#pragma unroll
                for (int i = 0; i < N; ++i) c2[(size_t)(3 + i) * ss] = y[i];
            }
        }
        dt_keep = dt;
        clipped = less_with_sign(tnext, t + dt, dt);
        dt = clipped ? tnext - t : dt;
        clipped = clipped && kobs < K;
        tries = 0;
    };
    begin_step();
    while (k < len) {
        const double h = dt;
        double Kst[Tab::SF][N], ynew[N], xerr[N];
#pragma unroll
        for (int i = 0; i < N; ++i) Kst[0][i] = k0[i];
        R::attempt(tc, q, y, Kst, h, ynew, xerr);
        const double err = R::error_norm(sp.atol, sp.rtol, h, y, k0, xerr);
        const bool ok = control_step<Tab>(h, err, dt, pc);
        // (an instance whose forward ended OK never exhausts its tries here; the
        // bound only keeps the loop finite)
        const bool stuck = ++tries > sp.max_attempts;
        if (ok) {
            const double tn = t + h;
            if constexpr (Rows) {
                r[0] = stored_step(tn, t);
#pragma unroll
                for (int i = 0; i < N; ++i) r[(size_t)(1 + i) * ss] = y[i];
                r += FS * ss;
            }
            t = tn;
#pragma unroll
            for (int i = 0; i < N; ++i) {
                y[i] = ynew[i];
                if constexpr (Tab::FSAL) k0[i] = Kst[Tab::SF - 1][i];
            }
            if constexpr (!Tab::FSAL) Sys::rhs(q, y, k0);
            if (clipped && fabs(dt_keep) > fabs(dt)) dt = dt_keep;
            ++k;
            begin_step();
        } else {
            clipped = false;
            if (stuck) {
                ++k;
                tries = 0;
            }
        }
    }
}

// ---------------------------------------------------------------------------
// Checkpointed reverse in pairs of waves (one level of checkpoints, segments
// of at most VA_OBS_PAIR_MAX_ROWS rows)
// ---------------------------------------------------------------------------
// A lane's reverse is two dependent chains one after the other, segment by
// segment: the replay of the controlled loop from the segment's checkpoint and
// the backward sweep over the replayed rows.  Here wave 2p of a block replays
// while wave 2p+1 sweeps backwards, for the same 64 instances (one per lane):
// in iteration i each replay lane rebuilds one segment into the row buffer of
// parity i & 1 and records which (instance, segment) it was; the backward lane
// of the same index reverses iteration i's segment while the replay lane
// rebuilds iteration i+1's into the other buffer.  The two buffers are the row
// buffers the one-wave reverse gives the two waves' threads, so the memory is
// the same.  The waves meet through two counters in LDS (iterations replayed,
// iterations reversed), written and polled by whole waves, so no lane waits
// on another lane of its own wave; every wait gives up after VA_OBS_SPIN_LIMIT
// polls, and then each wave writes NaN outputs for the instances it holds and
// stops.  The replay runs at most two iterations ahead.  Results are those of
// the one-wave reverse: the same rows, reversed in the same order.
// A wait lasts one iteration of the other wave: one segment replayed or
// reversed, at most VA_OBS_PAIR_MAX_ROWS steps (longer segments take the
// one-wave reverse), tens of milliseconds; a wait gives up only after some
// seconds of polls.
constexpr int VA_OBS_SPIN_LIMIT = 1 << 26;
constexpr int VA_OBS_PAIR_MAX_ROWS = 8192;

struct ObsPipe {
    int item_b[2][64];  // instance of each lane in the iterations of each parity (-1: idle)
    int item_j[2][64];  // its segment (-1: none; the instance's outputs only)
    int rep;            // iterations replayed
    int con;            // iterations reversed: a buffer is free again
    int abort_;         // a wait gave up
};

__device__ __forceinline__ int pipe_load(int *p)
{
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
__device__ __forceinline__ void pipe_store(int *p, int v)
{
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

// Wait until *ctr > k (the same word for every lane, so the whole wave leaves
// the loop together).  Returns false when the other wave gave up or, after
// VA_OBS_SPIN_LIMIT polls, gives up itself.
__device__ __forceinline__ bool pipe_wait(ObsPipe &P, int *ctr, int k)
{
    for (int spins = 0; spins < VA_OBS_SPIN_LIMIT; ++spins) {
        if (pipe_load(ctr) > k) {
            // the other wave's buffer and item writes before its count come first
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
            return true;
        }
        if (pipe_load(&P.abort_)) return false;
        __builtin_amdgcn_s_sleep(1);
    }
    pipe_store(&P.abort_, 1);
    return false;
}

template <int N, int P>
__device__ __forceinline__ void obs_nan_outputs(const ObsRevArgs &a, int64_t b)
{
    const int64_t B = a.sp.B;
    const double qnan = __builtin_nan("");
#pragma unroll
    for (int i = 0; i < N; ++i) a.dJdy0[(int64_t)i * B + b] = qnan;
    for (int k = 0; k < P; ++k) a.dJdp[(int64_t)k * B + b] = qnan;
}

// Replay wave: takes the instances (longest first) and rebuilds their segments,
// last first.
template <class Sys, class Tab, bool Lone>
__device__ void obs_rev_replay(const ObsRevArgs &a, ObsPipe &Pp, int pair, int lane)
{
    const TabRegs<Tab, Lone> tc;
    const PowConsts<Lone> pc;
    constexpr int N = Sys::N, P = Sys::P, FC = N + 3;
    const SolveParams sp = a.sp;
    const int64_t B = sp.B;
    const int K = a.K;
    const int64_t ss = (int64_t)gridDim.x * blockDim.x;
    const int64_t tbase = (int64_t)blockIdx.x * blockDim.x + pair * 128 + lane;
    typename Sys::Params q;
    int64_t b = -1;
    int32_t cnt = 0, stride = 1, j = -1;
    bool done = false, have = false;
    for (int it = 0;; ++it) {
        // this lane's item: the next segment of its instance, or a new instance
        bool seg_item = false;
        int64_t ib = -1;
        if (!done && !have) {
            const int64_t pos = atomicAdd(a.counter, 1);
            if (pos >= B) {
                done = true;
            } else {
                b = a.order ? a.order[pos] : pos;
                if (a.status[b] == LANE_OK) {
                    Sys::load(q, a.p, B, b, sp.kconst);
                    cnt = a.n_acc[b];
                    stride = a.st.stride[b];
                    j = (cnt + stride - 1) / stride - 1;
                    have = j >= 0;
                }
                ib = b;  // an instance without segments: its outputs only
            }
        }
        if (have) {
            ib = b;
            seg_item = true;
        }
        if (__builtin_amdgcn_ballot_w64(!done) == 0) {
            // the final iteration, all lanes idle: the backward wave stops at it
            if (!pipe_wait(Pp, &Pp.con, it - 2)) return;
            Pp.item_b[it & 1][lane] = -1;
            Pp.item_j[it & 1][lane] = -1;
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
            pipe_store(&Pp.rep, it + 1);
            return;
        }
        // the buffer of this parity was read by the backward wave's iteration it - 2
        if (!pipe_wait(Pp, &Pp.con, it - 2)) {
            // NaN outputs for every instance this lane handed over or holds
            for (int d = 1; d <= 2; ++d)
                if (it - d >= 0 && Pp.item_b[(it - d) & 1][lane] >= 0)
                    obs_nan_outputs<N, P>(a, Pp.item_b[(it - d) & 1][lane]);
            if (ib >= 0) obs_nan_outputs<N, P>(a, ib);
            return;
        }
        Pp.item_b[it & 1][lane] = (int)ib;
        Pp.item_j[it & 1][lane] = seg_item ? j : -1;
        if (seg_item) {
            const double *c = a.st.ck + ((size_t)b * (size_t)a.st.slots + (size_t)j) * FC;
            const int32_t n0 = j * stride;
            const int32_t len = (cnt - n0 < stride) ? cnt - n0 : stride;
            recompute_segment<Sys, Tab, Lone>(tc, pc, q, sp, a.obs_t, K, c, len,
                                              a.st.seg + tbase + (it & 1) * 64, ss);
            if (--j < 0) have = false;
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
        pipe_store(&Pp.rep, it + 1);
    }
}

// Backward wave: reverses each replayed segment and writes the outputs.
template <class Sys, class Tab, bool Lone>
__device__ void obs_rev_backward(const ObsRevArgs &a, ObsPipe &Pp, int pair, int lane)
{
    const TabRegs<Tab, Lone> tc;
    constexpr int N = Sys::N, P = Sys::P, FS = N + 1;
    const SolveParams sp = a.sp;
    const int64_t B = sp.B;
    const int K = a.K;
    const int64_t ss = (int64_t)gridDim.x * blockDim.x;
    const int64_t tbase = (int64_t)blockIdx.x * blockDim.x + pair * 128 + lane;
    typename Sys::Params q;
    double lam[N], pbar[P];
    int64_t cur = -1;  // the instance in progress
    int32_t stride = 1, cnt = 0, onext = -1;
    int kobs = -1;
    const int32_t *orow = nullptr;
    // state for instance b, reversed from its end
    auto start = [&](int64_t b) {
        Sys::load(q, a.p, B, b, sp.kconst);
        double yT[N];
#pragma unroll
        for (int i = 0; i < N; ++i) {
            lam[i] = 0.0;
            yT[i] = a.yT[(int64_t)i * B + b];
        }
        if (a.cost) a.J[b] = terminal_cost<N>(a.cost, a.cost_w, yT, lam);
#pragma unroll
        for (int k = 0; k < P; ++k) pbar[k] = 0.0;
        cnt = a.n_acc[b];
        stride = a.st.stride[b];
        orow = a.st.obs_row + (size_t)b * (size_t)K;
        onext = obs_point(orow, K - 1);
        kobs = obs_jumps<N>(orow, a.obs_y, K - 1, onext, cnt, yT, lam);
        cur = b;
    };
    auto finish = [&](int64_t b) {
#pragma unroll
        for (int i = 0; i < N; ++i) a.dJdy0[(int64_t)i * B + b] = lam[i];
        for (int k = 0; k < P; ++k) a.dJdp[(int64_t)k * B + b] = 0.0 + pbar[k];
        cur = -1;
    };
    for (int it = 0;; ++it) {
        if (!pipe_wait(Pp, &Pp.rep, it)) {
            if (cur >= 0) obs_nan_outputs<N, P>(a, cur);
            return;
        }
        const int ib = Pp.item_b[it & 1][lane];
        const int ij = Pp.item_j[it & 1][lane];
        if (__builtin_amdgcn_ballot_w64(ib >= 0) == 0) return;  // the replay wave is done
        if (ib >= 0) {
            if (ij < 0) {
                // no segments: a failed instance, or one with no accepted step
                if (a.status[ib] != LANE_OK) {
                    obs_nan_outputs<N, P>(a, ib);
                } else {
                    start(ib);
                    finish(ib);
                }
            } else {
                if (ib != cur) start(ib);
                const int32_t n0 = ij * stride;
                const int32_t len = (cnt - n0 < stride) ? cnt - n0 : stride;
                const double *seg = a.st.seg + tbase + (it & 1) * 64;
                // row k-1 is loaded while step k is reversed
                double hn = 0.0, yn[N] = {};
                auto load_row = [&](int32_t k) {
                    const double *r = seg + (size_t)k * FS * ss;
                    hn = r[0];
#pragma unroll
                    for (int i = 0; i < N; ++i) yn[i] = r[(size_t)(1 + i) * ss];
                };
                if (len > 0) load_row(len - 1);
                for (int32_t k = len - 1; k >= 0; --k) {
                    const double hk = hn;
                    double yk[N];
#pragma unroll
                    for (int i = 0; i < N; ++i) yk[i] = yn[i];
                    if (k > 0) load_row(k - 1);
                    back_prop_step<Sys>(tc, q, hk, yk, lam, pbar);
                    kobs = obs_jumps<N>(orow, a.obs_y, kobs, onext, n0 + k, yk, lam);
                }
                if (ij == 0) finish(ib);
            }
        }
        // this iteration's buffer may be rebuilt
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
        pipe_store(&Pp.con, it + 1);
    }
}

template <class Sys, class Tab, bool Ckpt, bool Lone>
__global__ void __launch_bounds__(256) k_obs_rev(ObsRevArgs a)
{
    if constexpr (Ckpt) {
        load_ctrl_tables();
        if (a.st.levels == 1 && a.st.seg_rows <= VA_OBS_PAIR_MAX_ROWS &&
            (blockDim.x & 127) == 0) {
            // pairs of waves (the condition is the same for the whole grid)
            __shared__ ObsPipe pipes[2];
            const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
            if (lane == 0 && (w & 1) == 0) {
                pipes[w >> 1].rep = 0;
                pipes[w >> 1].con = 0;
                pipes[w >> 1].abort_ = 0;
            }
            __syncthreads();
            if (w & 1) obs_rev_backward<Sys, Tab, Lone>(a, pipes[w >> 1], w >> 1, lane);
            else obs_rev_replay<Sys, Tab, Lone>(a, pipes[w >> 1], w >> 1, lane);
            return;
        }
    }
    const TabRegs<Tab, Lone> tc;
    const PowConsts<Lone && Ckpt> pc;
    constexpr int N = Sys::N, P = Sys::P;
    constexpr int F = N + 2, FC = N + 3, FS = N + 1;
    const SolveParams sp = a.sp;
    const int64_t B = sp.B;
    const int K = a.K;
    const double qnan = __builtin_nan("");
    const int64_t gtid = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    double *seg = nullptr;
    // lanes' segment buffers interleaved: field f of row k at seg[(k FS + f) ss]
    const int64_t ss = (int64_t)gridDim.x * blockDim.x;
    if constexpr (Ckpt) seg = a.st.seg + gtid;

    for (;;) {
        int64_t b = atomicAdd(a.counter, 1);
        if (b >= B) break;
        if (a.order) b = a.order[b];
        if (a.status[b] != LANE_OK) {
#pragma unroll
            for (int i = 0; i < N; ++i) a.dJdy0[(int64_t)i * B + b] = qnan;
            for (int k = 0; k < P; ++k) a.dJdp[(int64_t)k * B + b] = qnan;
            continue;
        }
        typename Sys::Params q;
        Sys::load(q, a.p, B, b, sp.kconst);
        double lam[N], pbar[P], yT[N];
#pragma unroll
        for (int i = 0; i < N; ++i) {
            lam[i] = 0.0;
            yT[i] = a.yT[(int64_t)i * B + b];
        }
        if (a.cost) a.J[b] = terminal_cost<N>(a.cost, a.cost_w, yT, lam);
#pragma unroll
        for (int k = 0; k < P; ++k) pbar[k] = 0.0;
        const int32_t cnt = a.n_acc[b];
        const int32_t *orow = a.st.obs_row + (size_t)b * (size_t)K;
        int32_t onext = obs_point(orow, K - 1);
        int kobs = obs_jumps<N>(orow, a.obs_y, K - 1, onext, cnt, yT, lam);
        if constexpr (!Ckpt) {
            const RowsBack<F> rows{
                a.st.traj + slot_rows(a.st.rows, a.st.slot ? a.st.slot[b] : b),
                (uint32_t)a.st.rows.blk * 8u};
            // rows loaded two steps before their own, three steps per trip (as in k_rev)
            double hr[3], yr[3][N];
            int32_t n = cnt - 1;
#pragma unroll
            for (int s = 0; s < 3; ++s) rows.load(n - s, hr[s], yr[s]);
            wait_vmem();
            auto step = [&](int s) {
                if (n >= 0) {
                    back_prop_step<Sys>(tc, q, hr[s], yr[s], lam, pbar);
                    kobs = obs_jumps<N>(orow, a.obs_y, kobs, onext, n, yr[s], lam);
                }
                __builtin_amdgcn_sched_barrier(0);
                rows.load(n - 3, hr[s], yr[s]);
                --n;
            };
            do {
                step(0);
                step(1);
                step(2);
            } while (__builtin_amdgcn_ballot_w64(n >= 0) != 0);
        } else {
            const int32_t stride = a.st.stride[b];
            const double *ck = a.st.ck + (size_t)b * (size_t)a.st.slots * FC;
            const int32_t nseg = (cnt + stride - 1) / stride;
            // reverse `len` rows from checkpoint c; the first is point n0
            auto reverse_rows = [&](const double *c, int32_t n0, int32_t len) {
                recompute_segment<Sys, Tab, Lone>(tc, pc, q, sp, a.obs_t, K, c, len, seg, ss);
                // row k-1 is loaded while step k is reversed, so no step waits
                // on its own row's loads
                double hn = 0.0, yn[N] = {};
                auto load_row = [&](int32_t k) {
                    const double *r = seg + (size_t)k * FS * ss;
                    hn = r[0];
#pragma unroll
                    for (int i = 0; i < N; ++i) yn[i] = r[(size_t)(1 + i) * ss];
                };
                if (len > 0) load_row(len - 1);
                for (int32_t k = len - 1; k >= 0; --k) {
                    const double hk = hn;
                    double yk[N];
#pragma unroll
                    for (int i = 0; i < N; ++i) yk[i] = yn[i];
                    if (k > 0) load_row(k - 1);
                    back_prop_step<Sys>(tc, q, hk, yk, lam, pbar);
                    kobs = obs_jumps<N>(orow, a.obs_y, kobs, onext, n0 + k, yk, lam);
                }
            };
            for (int32_t j = nseg - 1; j >= 0; --j) {
                const int32_t n0 = j * stride;
                const int32_t len = (cnt - n0 < stride) ? cnt - n0 : stride;
                if (len <= a.st.seg_rows) {
                    reverse_rows(ck + (size_t)j * FC, n0, len);
                    continue;
                }
                // two levels: level-2 checkpoints every `sub` steps of the segment,
                // then each sub-segment, last first (sub <= seg_rows and
                // ceil(len / sub) <= slots2 by the sizing in va_create)
                const int32_t sub = (len + a.st.slots2 - 1) / a.st.slots2;
                double *ck2 = a.st.ck2 + gtid;
                recompute_segment<Sys, Tab, Lone, false>(tc, pc, q, sp, a.obs_t, K,
                                                         ck + (size_t)j * FC, len, ck2, ss, sub);
                for (int32_t i = (len - 1) / sub; i >= 0; --i) {
                    double c2[FC];
#pragma unroll
                    for (int f = 0; f < FC; ++f) c2[f] = ck2[(size_t)(i * FC + f) * ss];
                    const int32_t m0 = i * sub;
                    const int32_t leni = (len - m0 < sub) ? len - m0 : sub;
                    reverse_rows(c2, n0 + m0, leni);
                }
            }
        }
#pragma unroll
        for (int i = 0; i < N; ++i) a.dJdy0[(int64_t)i * B + b] = lam[i];
        for (int k = 0; k < P; ++k) a.dJdp[(int64_t)k * B + b] = 0.0 + pbar[k];
    }
}

template <class Sys, class Tab>
struct LaunchObs {
    template <bool Lone>
    static hipError_t fwd_as(const ObsFwdArgs &a, int grid, int block, hipStream_t s)
    {
        if (a.st.ckpt)
            hipLaunchKernelGGL((k_obs_fwd<Sys, Tab, true, Lone>), dim3(grid), dim3(block), 0, s,
                               a);
        else
            hipLaunchKernelGGL((k_obs_fwd<Sys, Tab, false, Lone>), dim3(grid), dim3(block), 0, s,
                               a);
        return hipGetLastError();
    }
    template <bool Lone>
    static hipError_t rev_as(const ObsRevArgs &a, int grid, int block, hipStream_t s)
    {
        if (a.st.ckpt)
            hipLaunchKernelGGL((k_obs_rev<Sys, Tab, true, Lone>), dim3(grid), dim3(block), 0, s,
                               a);
        else
            hipLaunchKernelGGL((k_obs_rev<Sys, Tab, false, Lone>), dim3(grid), dim3(block), 0, s,
                               a);
        return hipGetLastError();
    }
    static hipError_t fwd(const ObsFwdArgs &a, int grid, int block, hipStream_t s)
    {
        if constexpr (lone_forward<Sys, Tab>(true))
            if (lone_waves(grid, block)) return fwd_as<true>(a, grid, block, s);
        return fwd_as<false>(a, grid, block, s);
    }
    static hipError_t rev(const ObsRevArgs &a, int grid, int block, hipStream_t s)
    {
        if constexpr (lone_reverse<Sys, Tab, 1>(true))
            if (lone_waves(grid, block)) return rev_as<true>(a, grid, block, s);
        return rev_as<false>(a, grid, block, s);
    }
    // the smaller occupancy of the two storage variants, so one sizing serves both
    static int occ_fwd(int block)
    {
        int n0 = 0, n1 = 0;
        if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&n0, k_obs_fwd<Sys, Tab, false, false>, block,
                                                         0) != hipSuccess ||
            hipOccupancyMaxActiveBlocksPerMultiprocessor(&n1, k_obs_fwd<Sys, Tab, true, false>, block,
                                                         0) != hipSuccess)
            return 1;
        return n0 < n1 ? n0 : n1;
    }
    static int occ_rev(int block)
    {
        int n0 = 0, n1 = 0;
        if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&n0, k_obs_rev<Sys, Tab, false, false>, block,
                                                         0) != hipSuccess ||
            hipOccupancyMaxActiveBlocksPerMultiprocessor(&n1, k_obs_rev<Sys, Tab, true, false>, block,
                                                         0) != hipSuccess)
            return 1;
        return n0 < n1 ? n0 : n1;
    }
    static void apply(KernelSet *k)
    {
        k->obs_fwd = &fwd;
        k->obs_rev = &rev;
        k->occ_obs_fwd = &occ_fwd;
        k->occ_obs_rev = &occ_rev;
    }
};

// Adds the observation kernels for the adaptive error steppers.
template <class Sys>
inline void pick_observed(int tableau, int adaptive, KernelSet *out)
{
    if (!adaptive) return;
    switch (tableau) {
    case TAB_CK54: LaunchObs<Sys, CashKarp54>::apply(out); break;
    case TAB_DOPRI5: LaunchObs<Sys, Dopri5>::apply(out); break;
    case TAB_F78: LaunchObs<Sys, Fehlberg78>::apply(out); break;
    default: break;
    }
}

}  // namespace va
