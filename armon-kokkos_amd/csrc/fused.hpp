// Fused Lagrange + remap sweeps: device state and launch interface.
#pragma once

#include "armon/armon.h"

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>

namespace armon {

// The CFL minimum of the current state is the least of kDtSlots accumulators (bit patterns of
// non-negative doubles), each on a cache line of its own: the waves of a sweep spread over them.
// Atomics on one word are served one after the other, some 4 ns each: with a single accumulator the
// 5632 waves of a 512^2 sweep took 24 us to end what they compute in 8.
constexpr int kDtSlots = 32;
struct alignas(128) DtSlot {
    unsigned long long bits;
};
constexpr unsigned long long kNoBound = 0x7FEFFFFFFFFFFFFFull;   // DBL_MAX

struct TimeStepConfig {
    double cfl, Dt, max_time;
    int max_cycles, cst_dt, dt_on_even_cycles;
};

// Time-stepping state kept on the device between cycles (armon_2D.cpp:229-252, 347-361).
struct StepState {
    double current_dt;
    double next_dt;
    double time;
    double error_dt;
    int cycle;
    int active;                      // 1 while the current cycle runs
    int error;                       // 1 after an invalid time step
    int error_cycle;

    bool running() const { return active && !error; }
    // How many cycles are left: 0 when the run has ended, else by the count of cycles, or by the time at
    // this state's time step and one or two more. A time step that does not lead to the end (a
    // constant one may be negative) leaves all of the count.
    int64_t left(const TimeStepConfig& c) const
    {
        if (!running() || !(time < c.max_time) || cycle >= c.max_cycles) return 0;
        const int64_t count = (int64_t) c.max_cycles - cycle;
        const double steps = (c.max_time - time) / current_dt;
        return steps >= 0 && steps < (double) count ? std::min(count, (int64_t) steps + 2) : count;
    }
};

struct DeviceState : StepState {
    DtSlot dt_min[kDtSlots];
};

inline TimeStepConfig step_config(const ArmonParams& p)
{
    return {p.cfl, p.Dt, p.max_time, p.max_cycles, p.cst_dt, p.dt_on_even_cycles};
}

// A cycle's time step is made from one state into another, in turn between two of them: by a kernel of
// its own, or by the cycle's first sweep (`prev` set), each of whose waves computes it for itself
// while one wave writes it down for the sweeps that follow. That saves a launch a cycle for some 30
// instructions a wave (7% of a sweep's) and a longer wait before its first stage, so it is done for
// sweeps of up to folded_cells() cells (0.9 M, 2.1 M). Cycle without -> with it, us: FP64 256^2
// 12.4 -> 11.0, 512^2 18.8 -> 17.9, 1024x768 37.0 -> 36.8, 1024^2 46.2 -> 46.5, 2048x1280 93.0 -> 95.5;
// FP32-mixed 512^2 13.2 -> 11.9, 1024^2 25.3 -> 24.4, 2048x1024 39.0 -> 39.1, 2048x1536 52.6 -> 53.4.
constexpr int64_t folded_cells(size_t element) { return element == 8 ? 7 << 17 : 1 << 21; }

enum { REDUCE_NO, REDUCE, REDUCE_UNSEEN };   // not, after a look at the accumulator, without one

// Everything a sweep kernel needs. Arrays use the reference layout: row-major with
// nb_ghosts ghost layers on every side, index(i, j) = index_start + j*row_length + i.
template <class T>
struct SweepArgs {
    const T* in_rho; const T* in_u; const T* in_v; const T* in_E;
    T* out_rho; T* out_u; T* out_v; T* out_E;
    const T* stale_p; const T* stale_c;   // pmat/cmat, read only for ghost layers beyond the stencil width
    DeviceState* st;                      // the cycle's state
    const DeviceState* prev;              // the state before the cycle's time step, where this sweep makes it
    TimeStepConfig step;
    int nx, ny, row_length, index_start, stencil_width;
    int seg_len;                          // Y sweep: rows per marching run (set by the launcher)
    int x_slots;                          // X sweep: slots per row, nx + 2 x the ghost layers read
    float x_inv_slots;                    // 1 / x_slots
    int dx_mode;                          // DX_POW2 (inv_dx = 1 / dx) or DX_RECIP (inv_dx = RN(1 / dx))
    int reduce;                           // whether and how the sweep adds to the CFL accumulators: REDUCE_*
    double gamma, dx, inv_dx, dt_factor;
    double lo_u, lo_v, hi_u, hi_v;        // BC factors: Left/Bottom (lo), Right/Top (hi)
    double cfl_dx, cfl_dy;
};

// Compile-time sweep variant: flux = 0 Godunov, 1..3 GAD with limiter None/Minmod/Superbee;
// proj = 1 (Euler) or 2 (Euler 2nd order); eos = 0 perfect gas, 1 Bizarrium.
struct SweepVariant {
    int flux, proj, eos;
};

// Ghost layers read by a sweep on each side: faces from -e to n+e (e = 1 + [Euler 2nd]),
// a GAD face reading one more cell each side (ranges.cpp:14-30, acoustic.cpp:51-63).
inline int read_extent(int flux, int proj) { return 2 + (flux > 0 ? 1 : 0) + (proj == 2 ? 1 : 0); }

template <class T>
void launch_sweep(int axis, const SweepVariant& v, const SweepArgs<T>& a, hipStream_t s);

// Output cells per X-sweep tile of `tile` threads (the single-domain sweep's: 256).
int x_tile_outputs(const SweepVariant& v, int tile = 256);

// The time step from `prev` into `st`.
void launch_time_step(const DeviceState* prev, DeviceState* st, const TimeStepConfig& c, hipStream_t s);

// ---- batched ensemble --------------------------------------------------------------------

// One domain of a batch: its slice of the packed arrays and its per-axis constants.
struct BatchDomain {
    long long offset;              // first element of the domain in the packed arrays
    int nx, ny, row_length, index_start;
    double dx[2], inv_dx[2];       // per axis; inv_dx = RN(1 / dx), for the batch's DX_RECIP division
    double cfl_dx, cfl_dy;
    double bc[4][2];               // per side (Left, Right, Top, Bottom): u, v factors
    int x_slots;                   // X sweep: slots per row (nx + 2 x the ghost layers read)
    float x_inv_slots;             // 1 / x_slots
};

// Domains start on multiples of a wave's 64 elements, so a wave's elements belong to one domain: the
// last whose offset is not past them.
template <class Domain>
__device__ __forceinline__ int domain_of(const Domain* domains, int n, int64_t element)
{
    int lo = 0, hi = n;
    while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        if (domains[mid].offset <= element) lo = mid;
        else hi = mid;
    }
    return lo;
}

// What the initial state of one domain of a batch is made of (init_test_states).
struct BatchInit {
    long long offset, cells;       // first element of the domain in the packed arrays, and how many
    int row_length, nb_ghosts, nx, ny, test;
    double size[2], origin[2], option;
    ArmonTestState states;
};

// The initial state of every domain in one launch, over the whole arrays (ARMON_FIELD_*).
void launch_batch_init(const BatchInit* domains, int n, int64_t elements, double* const arrays[ARMON_FIELD_COUNT],
                       hipStream_t s);

// Work items: an X tile (domain; row and slot within that row of the tile's first thread,
// see sweep_x_tile) or a Y run of one wave (domain, first column, output rows [y0, y1)).
struct BatchItemX { int domain, row, slot, pad; };
struct BatchItemY { int domain, x0, y0, y1; };

template <class T>
struct BatchArgs {
    const T* in_rho; const T* in_u; const T* in_v; const T* in_E;
    T* out_rho; T* out_u; T* out_v; T* out_E;
    const T* stale_p; const T* stale_c;
    const BatchDomain* domains;
    DeviceState* states;
    const DeviceState* prev;      // as SweepArgs::prev, with the domains' configurations
    const TimeStepConfig* steps;
    int stencil_width, reduce;
    double gamma, dt_factor;
};

// One launch sweeps every domain of the batch along `axis`: `grid` persistent blocks walk
// the work items (BatchItemX for X, BatchItemY for Y; with `b.prev` one block each, whatever `grid`); X tiles are `tile` cells wide (128,
// 256 or 512, the width the X items were cut for), `cpt` cells per thread (1, or 2 for tiles of
// 256 or 512 cells, one block per tile whatever `grid`). Y items are marching runs (`tile` 0) or LDS
// tiles (`tile` 1: y_tile_cols() x y_tile_outputs() cells, one block per tile).
template <class T>
void launch_batch_sweep(int axis, const SweepVariant& v, const BatchArgs<T>& b, const void* items, int nitems,
                        int grid, int tile, int cpt, hipStream_t s);

// Blocks of the batched sweep kernel of this variant (X tiles of `tile` threads) that fit on the
// device at once.
template <class T>
int batch_resident_blocks(int axis, const SweepVariant& v, int tile);

// Columns and output rows of a Y tile, and the number of cells up to which a sweep along y takes tiles.
constexpr int y_tile_cols() { return 16; }
constexpr int y_tile_rows() { return 32; }
inline int y_tile_outputs(const SweepVariant& v) { return y_tile_rows() - 2 * read_extent(v.flux, v.proj); }
constexpr int64_t y_tile_max_cells(size_t element) { return element == 8 ? 5 << 19 : 7 << 19; }   // 2.6 M, 3.7 M

// What a Y sweep computes either way, in lanes' cells, summed over its domains: as tiles all of their
// slots, as marches (runs of `run` rows; blocks of `cols` columns, one wave per 64) the rows with their
// warm-up.
struct YSweepWork {
    int64_t cells = 0, slots = 0, marched = 0, waves = 0;
    void add(const SweepVariant& v, int nx, int ny, int run, int cols)
    {
        const int64_t W = y_tile_outputs(v), runs = (ny + run - 1) / run;
        cells += (int64_t) nx * ny;
        slots += (int64_t) ((nx + y_tile_cols() - 1) / y_tile_cols()) * ((ny + W - 1) / W) * y_tile_cols() * y_tile_rows();
        marched += (int64_t) ((nx + cols - 1) / cols) * cols * (ny + 2 * read_extent(v.flux, v.proj) * runs);
        waves += (nx + 63) / 64 * runs;
    }
};

// Whether it takes tiles.
//  * Up to y_tile_max_cells() cells, where the tiles' rows are filled: a flat domain leaves most of a tile's
//    24 to 28 output rows empty, where a march has no row too many, so the slots must stay below 0.85 of
//    what the march costs, its rate growing with the waves w as w / (w + SIMDs) (y_run_rows). Y sweep with
//    GAD and second order, us (in brackets slots / cost), march / tile: FP64 100 000 x 8 (1.21) 36.8 / 55.1,
//    325 000 x 8 (1.66) 73 / 158, 56 000 x 25 (0.98) 53.5 / 68.1, 28 000 x 50 (0.74) 54 / 52; FP32
//    100 000 x 8 21.9 / 26.2, 66 666 x 12 (0.81) 24.2 / 22.2. Squares: 0.67 at most.
//  * Of any size, where a march's blocks have many columns past the domain, whose waves hold registers and
//    LDS to the end: slots below 0.7 (FP64) or 0.35 (FP32) of the march's lanes; a full width has 1.2. 20 M
//    cells, march / tile, FP64: Godunov and first order 4 columns 7785 / 1090, 64 (0.25) 551 / 320, 130
//    (0.57) 409 / 317; GAD and second order 100 (0.52) 653 / 486, 130 (0.67) 602 / 499, 180 (0.84) 449 / 473.
//    FP32: 64 (0.30) 317 / 225; Godunov and first order 100 (0.44) 185 / 194, 130 (0.57) 172 / 211.
bool y_takes_tiles(const YSweepWork& w, size_t element);
bool y_takes_tiles(const SweepVariant& v, size_t element, int nx, int ny);   // one domain's, against its best march

// The time step of every domain (one wave each), per-domain configuration.
void launch_batch_time_step(const DeviceState* prev, DeviceState* states, const TimeStepConfig* cfgs, int n,
                            hipStream_t s);

// ---- before and after the cycles -----------------------------------------------------------

// The arrays of one domain, or of every domain of a batch packed one after the other: the FP64 fields
// and, where the cycles run in them, the FP32 buffers.
struct FieldArrays {
    double *rho, *u, *v, *E, *p, *c, *g;
    double* other[4];     // FP64: the second state buffer (rho, u, v, E)
    float* f32[10];       // FP32-mixed: both state buffers, then p and c of stale ghost layers; or null
};

// What the first cycle finds: the EOS of the real cells into p, c and g, the CFL minimum of each
// domain's real cells into its state's accumulators (which must be clear), and a copy of every cell
// (ghosts included) in the cycles' buffers. With a null g, the fields p, c and g stay as they are. One pass over memory and one launch for all domains;
// `n` domains from `domains`, or the one of `one` when n is 1. `elements`: length of the arrays.
void launch_begin(const FieldArrays& f, const BatchDomain* domains, int n, const BatchDomain& one, int64_t elements,
                  DeviceState* states, int eos, double gamma, hipStream_t s);

// What the last cycle leaves, per domain after the cycles its state counts: the final state in rho, u, v
// and E, and in p, c and g the EOS of the last sweep's input over the real cells. Domains that ran no
// cycle are left alone.
void launch_finish(const FieldArrays& f, const BatchDomain* domains, int n, const BatchDomain& one, int64_t elements,
                   const DeviceState* states, int sweeps_per_cycle, int eos, double gamma, hipStream_t s);

// The states before the first cycle, for launch_begin.
void launch_clear(DeviceState* states, int n, hipStream_t s);

// ---- the host's view of a run ---------------------------------------------------------------

// Copies the time-stepping part of n states to `out`, which the device can write.
void launch_report(const DeviceState* states, int n, StepState* out, hipStream_t s);

// Reports of n states in pinned memory that the device writes: two, so that the host reads one while
// the other is on its way. Made with the first report; used from one stream.
class StateReports {
public:
    StateReports() = default;
    StateReports(const StateReports&) = delete;
    StateReports& operator=(const StateReports&) = delete;
    ~StateReports();
    void resize(int n) { n_ = n; }   // before the first report
    int size() const { return n_; }
    // Enqueues report k (the one in the place of report k - 2).
    void post(const DeviceState* states, int k, hipStream_t s);
    // Report k, once it has arrived.
    const StepState* wait(int k);

private:
    StepState* host_ = nullptr;
    hipEvent_t arrived_[2] = {};
    int n_ = 0;
};

// Runs chunks of up to `chunk` cycles until no state is running. `enqueue(n)` enqueues n cycles and returns
// the states after them; `config(d)` is the configuration of state d.
//
// The host learns of a chunk's end a report's round trip later, 20-30 us in which the device would idle
// (a quarter of a chunk of a 100^2 domain's cycles). So while one chunk runs, the next is enqueued
// behind it, unless the report before it says that no cycle will be left. Where that guess is wrong,
// as the time step changes, the run takes a little longer.
//
// Cycles after the end change no state, but their blocks take their time to come and go, 1.3 ns each: such an
// X sweep takes 352 us at 8192^2 in FP64 (270 900 blocks) and 177 in FP32 (133 300, two cells a thread), 95 and
// 41 at 4096^2, 24 and 14 at 2048^2. From kWholeChunks `cells` on, no more cycles are enqueued than the
// report leaves, the rest of a chunk launch by launch: 100 cycles of 8192^2 in chunks of 16, of which 12 are
// past the end, 190 -> 187 ms in FP64 and 94 -> 90 in FP32, 33 cycles of 4096^2 18.6 -> 17.0 and 9.6 -> 9.0.
// Smaller domains enqueue whole chunks, though the rest one by one would be the faster there too (100 cycles
// of 128^2 1.13 -> 1.10 ms, of 1024^2 4.83 -> 4.70, of 2048^2 14.9 -> 14.6): a run's graph launches, which
// the table of stage times counts, are then whole ones (20 cycles in chunks of 8 are 3).
constexpr int64_t kWholeChunks = 1 << 22;

template <class Enqueue, class Config>
void run_chunks(StateReports& reports, int chunk, int64_t cells, hipStream_t s, Enqueue&& enqueue, Config&& config)
{
    const int64_t least = cells < kWholeChunks ? chunk : 1;
    auto left = [&](const StepState* states) {
        int64_t most = 0;
        for (int d = 0; d < reports.size(); d++) most = std::max(most, states[d].left(config(d)));
        return most;
    };
    int64_t cycles = least;   // of the chunk that runs
    for (int d = 0; d < reports.size(); d++) cycles = std::max<int64_t>(cycles, config(d).max_cycles);
    cycles = std::min<int64_t>(cycles, chunk);
    const StepState* known = nullptr;   // the report before the chunk that runs
    reports.post(enqueue(cycles), 0, s);
    for (int k = 0;; k ^= 1) {
        int64_t next = known ? left(known) - cycles : 0;
        const bool ahead = next > 0;
        next = std::clamp<int64_t>(next, least, chunk);
        if (ahead) reports.post(enqueue(next), k ^ 1, s);
        known = reports.wait(k);
        const int64_t more = left(known);
        if (more == 0) return;
        if (!ahead) {
            next = std::clamp<int64_t>(more, least, chunk);
            reports.post(enqueue(next), k ^ 1, s);
        }
        cycles = next;
    }
}

// Element-wise conversion of an FP32 working buffer to a reference FP64 array.
void launch_convert_f2d(const float* in, double* out, int64_t n, hipStream_t s);

}  // namespace armon
