// va_kernels.hpp -- host-side launch interface of the HIP kernels (internal).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace va {

struct SolveParams {
    int64_t B;
    int64_t cap;          // accepted-step capacity per instance
    double t0, t1, dt0, atol, rtol, kconst;
    int32_t max_attempts;
    int32_t adaptive;
};

// Where the one-lane kernels keep an instance's rows (t, h, y), F = N + 2 doubles
// each: row r of storage slot s at traj[(s / 64) tile + (s % 64) lane +
// (r / 4) blk + (r % 4) F].  A handle's store is tiled: four rows of a slot lie
// together (128 bytes for N = 2, a cache line), beside those of the 63 other
// slots of its tile, and a forward stores the k-th instance it takes in slot k
// (slot[b] = k), so the lanes of a wave write one 8 KB block after another.
// With rows instance-major each lane was at an address of its own in a store of
// tens of GB, and address translation bound both sweeps (solve of the oscillator,
// B=2^20: 26.4 ms; tiled, and by the lines of k_fwd and k_rev_lines, 19.2 ms).
// slot == null: slot b is instance b's.
struct RowLayout {
    int64_t tile = 0, lane = 0, blk = 0;
};
constexpr int VA_ROW_TILE = 64, VA_ROW_BLOCK = 4;

// Rows instance-major, [B][cap + 1][F].
inline RowLayout rows_instance_major(int64_t cap, int F)
{
    return RowLayout{VA_ROW_TILE * (cap + 1) * F, (cap + 1) * F, VA_ROW_BLOCK * F};
}
inline int64_t row_blocks(int64_t cap) { return (cap + VA_ROW_BLOCK) / VA_ROW_BLOCK; }
inline RowLayout rows_tiled(int64_t cap, int F)
{
    const int64_t blk = (int64_t)VA_ROW_TILE * VA_ROW_BLOCK * F;
    return RowLayout{blk * row_blocks(cap), VA_ROW_BLOCK * F, blk};
}

// Persistent forward: each lane takes instances from *counter until B is reached.
struct FwdArgs {
    SolveParams sp;
    double *y;             // [N][B] in y0, out y(T)
    const double *p;       // [P][B]; Lotka-Volterra persistent kernels: [B][P]
    double *traj;          // rows (t, h, y), instance-major [B][cap+1][N+2] or as `rows` says
    int32_t *n_acc, *n_rej, *status;
    int32_t *counter;
    int32_t *max_steps_seen;
    const int32_t *order = nullptr;  // [B] or null: the k-th instance taken is order[k]
    const int32_t *split = nullptr;  // null: queue positions [0, B); else part 0 takes
    int32_t part = 0;                // [0, *split), part 1 takes [*split, B)
    RowLayout rows;                  // one-lane kernels
    int32_t *slot = nullptr;         // [B] or null, written
};

// Persistent reverse over the stored trajectory.
//   cost > 0: lambda computed from y(T) (read from yT) and written to dJdy0,
//             dJdp = sum p_bar, J written.
//   cost == 0: lambda [nout][N][B] in/out, mu [nout][P][B] += (reference semantics).
// The Lotka-Volterra persistent kernels take p as [B][P], store the dJ/dp sums
// [nout][B][P] in mu as they are, for either cost (the caller applies them),
// and set pbar_set[b] for each instance they wrote (when pbar_set is given);
// the long-instance kernels take p and mu as above.
struct RevArgs {
    SolveParams sp;
    const double *p;
    const double *traj;
    const int32_t *n_acc, *status;
    int32_t cost;
    const double *cost_w;  // [N] for the linear cost
    const double *yT;      // [N][B]
    double *J;
    double *lambda;        // [nout][N][B]
    double *mu;            // [nout][P][B]
    int32_t nout;
    int32_t *counter;
    const int32_t *order;  // [B] or null: the k-th instance taken is order[k]
    const int32_t *split = nullptr;  // as in FwdArgs; part 2 (rows_rev_head): the first blocks
    int32_t part = 0;                // take [0, *split) of the order, the queue holds the rest
    int32_t *pbar_set = nullptr;     // [B] or null
    // (cost == 0) seeds that one work item takes: 0 all of them, else items are
    // (instance, group of so many seeds) pairs.  See seeds_per_item() in va_capi.cpp.
    int32_t seeds_per_item = 0;
    // (cost == 0) the seeds are the unit vectors (nout = N): lambda is neither read
    // nor written, and mu = 0.0 + sum
    int32_t identity = 0;
    RowLayout rows;                  // one-lane kernels
    const int32_t *slot = nullptr;   // [B] or null
    // (Lotka-Volterra row kernels, several seeds) null, or a count of long instances:
    // where it is 0 an item is an instance with all of its seeds after all
    const int32_t *in_turn = nullptr;
};

// The work items of a reverse: groups of seeds per instance.
struct RevItems {
    int32_t seeds, per, parts;
};
__host__ __device__ inline RevItems rev_items(const RevArgs &a)
{
    RevItems r;
    r.seeds = a.cost ? 1 : a.nout;
    r.per = a.seeds_per_item > 0 ? a.seeds_per_item : r.seeds;
    r.parts = (r.seeds + r.per - 1) / r.per;
    return r;
}

// Whether the adaptive Lotka-Volterra row kernels of N species take part 2 in their
// reverse (the long instances' waves exchange by row broadcasts: N <= 16).
constexpr bool rows_rev_head(int n) { return n <= 16; }

// Plain form: one launch per accepted step, state in HBM, no refill, full
// trajectory store [step][field][B] with fields (t, y[N], K[S][N]).
struct PlainState {
    double *t, *dt;        // [B]
    double *k0;            // [N][B] f(y_n) carried for FSAL tableaus
    int32_t *done;         // [B]
    int32_t *active;       // 1 counter
    int32_t *max_steps_seen;
    double *pbar;          // [P][B] reverse accumulator
};

struct PlainFwdArgs {
    SolveParams sp;
    double *y;
    const double *p;
    double *traj;
    int32_t *n_acc, *n_rej, *status;
    PlainState st;
    int32_t step;
};

struct PlainRevArgs {
    SolveParams sp;
    const double *p;
    const double *traj;
    const int32_t *n_acc, *status;
    double *lambda;        // [N][B] seed in/out
    PlainState st;
    int32_t k;             // reverse launch index
};

// Observation cost (forced stops at obs_t, running cost, lambda jumps) with the
// trajectory either stored in full or kept as checkpoints.
struct ObsStore {
    int32_t ckpt;          // 0: full rows (t, h, y) in traj; 1: checkpoints in ck
    double *traj;          // rows (t, h, y), placed by `rows`
    double *ck;            // [B][slots][N+3] (t, dt to try, observations taken, y)
    int32_t slots;         // checkpoints per instance (even)
    int32_t stride_max;    // largest checkpoint spacing; slots * stride_max >= cap
    int32_t *stride;       // [B] spacing each instance ended with
    double *seg;           // [lanes][seg_rows][N+1] (h, y) rows recomputed by the reverse
    int32_t *obs_row;      // [B][K] stored-point index of each observation
    // two levels: a segment longer than seg_rows is replayed once to store level-2
    // checkpoints every `sub` steps (sub <= seg_rows) in ck2, then recomputed
    // sub-segment by sub-segment into seg
    int32_t levels = 1;
    int32_t seg_rows = 0;  // rows of the per-lane row buffer (stride_max with one level)
    int32_t slots2 = 0;    // level-2 checkpoints per lane
    double *ck2 = nullptr; // [lanes][slots2][N+3], lanes interleaved like seg
    RowLayout rows;        // of traj
    int32_t *slot = nullptr;
};

// The largest checkpoint spacing a solve of at most cap steps can need with `slots`
// checkpoints: the row buffers of the reverse are sized for it.  Spacings are
// powers of two; doubled only where a checkpoint is due and no slot is free, which
// with this one does not happen (slots * it >= cap, checkpoints lie below cap).
__host__ __device__ inline int32_t obs_stride_max(int64_t cap, int32_t slots)
{
    int32_t s = 1;
    while ((int64_t)s * slots < cap) s *= 2;
    return s;
}

// The spacing a solve starts from after one of `prev` accepted steps: the smallest
// with room for that many and never above stride_max, which the row buffers of
// the reverse are sized for (prev may be the cap itself, after an instance that
// ran out of steps).
__host__ __device__ inline int32_t obs_first_stride(int32_t prev, int32_t slots,
                                                    int32_t stride_max)
{
    int32_t s = 1;
    while (s < stride_max && (int64_t)s * slots <= prev) s *= 2;
    return s;
}

struct ObsFwdArgs {
    SolveParams sp;
    double *y;             // [N][B] in y0, out y(T)
    const double *p;
    int32_t *n_acc, *n_rej, *status;
    int32_t *counter;
    int32_t *max_steps_seen;
    const int32_t *order = nullptr;  // [B] or null: the k-th instance taken is order[k]
    const double *obs_t;   // [K]
    const double *obs_y;   // [K][N]
    int32_t K;
    double *J;             // [B]
    ObsStore st;
};

struct ObsRevArgs {
    SolveParams sp;
    const double *p;
    const double *yT;      // [N][B]
    const int32_t *n_acc, *status;
    const double *obs_y;   // [K][N]
    const double *obs_t;
    int32_t K;
    double *dJdy0;         // [N][B]
    double *dJdp;          // [P][B]
    int32_t *counter;
    const int32_t *order;
    int32_t cost;          // > 0: terminal cost added to the seed, J written
    const double *cost_w;
    double *J;
    ObsStore st;
};

// Lotka-Volterra with A shared by the batch (tiles of instances on MFMA).
struct SharedFwdArgs {
    SolveParams sp;
    double *y;             // [N][B] in y0, out y(T)
    const double *r;       // [N][B]
    const double *A;       // [N][N] row-major, shared
    double *traj;          // [B][cap+1][N+2]
    int32_t *n_acc, *n_rej, *status;
    int32_t *max_steps_seen;
};

struct SharedRevArgs {
    SolveParams sp;
    const double *r;
    const double *A;
    const double *traj;
    const int32_t *n_acc, *status;
    const int32_t *order;  // [B] longest first
    const double *lambda;  // [N][B] dJ/dy(T) (may alias dJdy0)
    double *dJdy0;         // [N][B]
    double *dJdr;          // [N][B]
    double *abar_part;     // [grid][N][N] per-workgroup partial dJ/dA
    double *gscr;          // [grid][waves][2][S][64][4] growth products and stage inputs of the step being reversed
};

// Layout version of KernelSet: kernel tables made in a caller's translation unit
// (VA_DEVICE_SYSTEM) are accepted with the library's size and a version it knows.
// Version 2 kernels read RevArgs::seeds_per_item, identity and the rows and slot
// members; version 1 kernels (the same table and argument layout up to those
// members) sweep all seeds of an instance one after the other, keep their rows
// instance-major, and are never given any of them.
constexpr int32_t VA_KERNEL_TABLE_VERSION = 2;
constexpr int32_t VA_KERNEL_TABLE_OLDEST = 1;

struct KernelSet {
    int32_t table_size = (int32_t)sizeof(KernelSet);
    int32_t table_version = VA_KERNEL_TABLE_VERSION;
    int n, np, s_rev, s_fwd;
    int flop_rhs, flop_vjp;
    hipError_t (*fwd)(const FwdArgs &, int grid, int block, hipStream_t);
    hipError_t (*rev)(const RevArgs &, int grid, int block, hipStream_t);
    // forward then reverse of each long-running instance, one block of three waves per
    // instance: grid = instances, block = 192 (null where absent)
    hipError_t (*long_fused)(const FwdArgs &, const RevArgs &, int grid, int block, hipStream_t);
    // the same instances' forward alone (one wave per instance) and reverse
    // alone (block 192: three waves per instance, one seed; block 256: one wave
    // per instance, any seeds) (null where absent)
    hipError_t (*long_fwd)(const FwdArgs &, int grid, int block, hipStream_t);
    hipError_t (*long_rev)(const RevArgs &, int grid, int block, hipStream_t);
    hipError_t (*plain_fwd)(const PlainFwdArgs &, int grid, int block, hipStream_t);
    hipError_t (*plain_rev)(const PlainRevArgs &, int grid, int block, hipStream_t);
    int (*occ_fwd)(int block);   // resident blocks per CU of the persistent kernels
    int (*occ_rev)(int block);
    int (*slots)(int block);     // instances one block holds at a time
    int layout;                  // 0: one lane per instance, 1: one group of N lanes per instance
    // observation-cost kernels (null where the system/tableau has none)
    hipError_t (*obs_fwd)(const ObsFwdArgs &, int grid, int block, hipStream_t);
    hipError_t (*obs_rev)(const ObsRevArgs &, int grid, int block, hipStream_t);
    int (*occ_obs_fwd)(int block);
    int (*occ_obs_rev)(int block);
    // shared-parameter kernels (layout 2), one workgroup per CU
    hipError_t (*shared_fwd)(const SharedFwdArgs &, int grid, hipStream_t);
    hipError_t (*shared_rev)(const SharedRevArgs &, int grid, hipStream_t);
    int shared_tile;
    int shared_waves;            // waves per workgroup of the shared-parameter kernels
};

// The kernels that order instances longest first (va_capi.cpp).
struct OrderArgs {
    const int32_t *n_acc, *n_rej, *status;
    int64_t B;
    int modes;       // bit 0: the reverse order, bit 1: the forward order
    int items;       // instances per thread, at most VA_ORDER_ITEMS (va_capi.cpp)
    const int32_t *from;  // the scatter takes instances in this order (null: index order)
    int32_t *work;   // per mode a histogram and cursors, cleared before
    int32_t *order[2], *n_long[2];
    int long_bucket[2];
};

hipError_t launch_glvs_reduce(const double *part, int nparts, double *out, hipStream_t s);

// Returns false when (system, n, tableau, adaptive) has no compiled kernels.
// instances_per_wave: 64 selects one lane per instance; 64/N (or 0 = default)
// selects the row-per-lane layout where the system has one.
bool get_kernels(int system, int n, int tableau, int adaptive, int instances_per_wave,
                 KernelSet *out);

hipError_t launch_plain_finish(double *lambda_out, const double *lambda_in, double *mu,
                               const double *pbar, const int32_t *status, int64_t B, int n, int np,
                               int grid, int block, hipStream_t s);
hipError_t launch_plain_cost(int cost, const double *cost_w, const double *yT, double *J,
                             double *lambda, const int32_t *status, int64_t B, int n, int grid,
                             int block, hipStream_t s);

}  // namespace va
