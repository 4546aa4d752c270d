// Fused Lagrange + remap sweep kernels (templates), instantiated by fused.hip for FP64 and
// by fused_fp32.hip for the FP32-mixed form, each with its own floating-point flags.
//
// One kernel per axis sweep performs, for every real cell, the whole per-axis chain of the
// reference (armon_2D.cpp:309-320): EOS -> boundary ghost synthesis -> Godunov / GAD face
// fluxes -> Lagrangian cell update -> first/second-order advection fluxes -> Euler
// projection, reading the state once and writing it once (out of place, ping-pong buffers).
//
//  * X sweep (k_sweep_x): one 256-thread block per tile of a stream of padded rows. Each
//    thread owns one cell of the tile (FP32: two; outputs plus an R-cell halo on each side, R =
//    ghost layers read); the stage results are exchanged through LDS between barriers. Loads and
//    stores are contiguous.
//  * Y sweep of large domains (k_sweep_y): one thread per column, marching down a run of rows.
//    Every stage's stencil neighbours along y live in the thread's own registers and LDS (a sliding
//    window); consecutive lanes touch consecutive columns.
//  * Y sweep of the others (k_sweep_y_tile): the X tile's stages on tiles of 16 columns.
//  * Both number their blocks XCD by XCD (xcd_block) so that each XCD's L2 serves a
//    contiguous part of the arrays.
//  * The batched ensemble (k_batch_x, k_batch_x1, k_batch_y, k_batch_y1) runs the same tile and
//    run bodies over a work list that spans many domains.
//
// Ghost cells are synthesised in registers: layers within the stencil width mirror the real
// cells with the side's velocity factors (halo_exchange.cpp:9-36); deeper layers keep their
// never-refilled values from the arrays, as in the reference.
//
// The CFL reduction of the next cycle (reductions.cpp:8-24) is folded into the epilogue of
// the last sweep of a cycle: it needs the new velocities and the sound speed of that sweep's
// input state, which is exactly what the reference's dt_CFL reads at the start of the next
// cycle (cmat is last written by the EOS of the last sweep).
#pragma once

#include "fused.hpp"
#include "device_math.hpp"
#include "xcd.hpp"

#include <algorithm>
#include <cfloat>
#include <stdexcept>
#include <string>
#include <type_traits>

namespace armon {
namespace sweep {

constexpr int kTile = 256;    // X sweep: cells per tile (FP64 single-domain sweep, batched default)
constexpr int kYBlock = 256;  // Y sweep: columns per block

// Y march: rows per unrolled loop body (FP64: 4 rows spill, 1 row moves its windows, 982 -> 992 us at
// 8192^2) and the minimum waves per SIMD the register allocation must allow.
#ifndef ARMON_Y_UNROLL_FP64
#define ARMON_Y_UNROLL_FP64 2
#endif
#ifndef ARMON_Y_UNROLL_FP32
#define ARMON_Y_UNROLL_FP32 2
#endif
constexpr int kYUnrollFp64 = ARMON_Y_UNROLL_FP64, kYUnrollFp32 = ARMON_Y_UNROLL_FP32;
constexpr int kYWaves = 3, kYWavesFirstOrder = 4;   // 168 and 128 VGPRs

template <class T>
struct Cell {
    T rho, un, ut, E, p, c;   // un: velocity along the sweep axis, ut: across it
    T y;                      // shared_recip(rho)
};

__device__ __forceinline__ double bits_to_double(unsigned long long b) { return __longlong_as_double((long long) b); }
__device__ __forceinline__ unsigned long long double_to_bits(double d) { return (unsigned long long) __double_as_longlong(d); }

__device__ __forceinline__ bool finite_d(double x)
{
    return (double_to_bits(x) & 0x7FF0000000000000ull) != 0x7FF0000000000000ull;
}

// Element at `byte` bytes past a base that is the same for the whole wave: the base stays in scalar
// registers and the lanes' offsets in one 32-bit register for all arrays.
template <class T>
__device__ __forceinline__ T load_at(const T* base, unsigned byte)
{
    return *reinterpret_cast<const T*>(reinterpret_cast<const char*>(base) + byte);
}
template <class T>
__device__ __forceinline__ void store_at(T* base, unsigned byte, T v)
{
    *reinterpret_cast<T*>(reinterpret_cast<char*>(base) + byte) = v;
}

// EOS of one cell (fluid_eos.cpp:9-62) with y = shared_recip(rho). The perfect gas is evaluated in
// the working precision T; the Bizarrium EOS always in FP64, because its `e - eps_k0` and
// `p - pk0` terms cancel to a few digits near the reference density (p and c rounded to T).
template <class T, int EOS>
__device__ __forceinline__ void cell_eos(double gamma, T rho, T u, T v, T E, T y, T& p, T& c)
{
    if constexpr (EOS == 0) {
        perfect_gas_pc<T>((T) gamma, rho, E, u, v, y, p, c);
    } else {
        double pd, cd;
        const double yd = sizeof(T) == 8 ? (double) y : shared_recip<double>((double) rho);
        bizarrium_pc((double) rho, (double) E, (double) u, (double) v, yd, pd, cd);
        p = (T) pd;
        c = (T) cd;
    }
}

// A tile's cell in two parts: its loads (fetch_cell), which depend on nothing but the launch, and the
// cell from them (make_cell). The tiles' kernels issue the loads before they wait for the cycle's
// time step, so that the two latencies overlap: a block of a small sweep spends as long on them as
// on its arithmetic.
template <class T>
struct LoadedCell {
    T rho, u, v, E;
    unsigned offset;   // bytes past the base
    int mirror;        // 0 real, 1 low side, 2 high side
    bool stale;
};

// Cell `k` (along the sweep axis, `n` real cells) of the pencil whose cell 0 lies `first` elements
// past `base` (the same for the whole wave) and whose cells lie `stride` apart. Real cells are
// loaded; ghost layers 1..stencil_width mirror real cells; deeper ghost layers are read as they are.
// The byte offsets fit 32 bits: a row has fewer than 2^23 real cells (the fused engine takes no longer
// ones) and at most 8.4 M with its ghosts, as a domain's index allows 2^31 - 1 cells in all; an X tile
// stays within one such row or some short ones, a Y tile within 31 rows of its base, 2.1 GB in FP64.
template <class T>
__device__ __forceinline__ LoadedCell<T> fetch_cell(const SweepArgs<T>& a, int64_t base, int first, int k, int stride,
                                                    int n)
{
    LoadedCell<T> l;
    int kk = k;
    l.mirror = 0;
    l.stale = false;
    if (__builtin_expect((unsigned) k >= (unsigned) n, 0)) {
        if (k < 0) {
            if (-k <= a.stencil_width) { kk = -k - 1; l.mirror = 1; }
            else l.stale = true;
        } else {
            if (k - n + 1 <= a.stencil_width) { kk = 2 * n - 1 - k; l.mirror = 2; }
            else l.stale = true;
        }
    }
    l.offset = (unsigned) (first + kk * stride) * (unsigned) sizeof(T);
    l.rho = load_at(a.in_rho + base, l.offset);
    l.u = load_at(a.in_u + base, l.offset);
    l.v = load_at(a.in_v + base, l.offset);
    l.E = load_at(a.in_E + base, l.offset);
    return l;
}

// A mirror ghost has the real cell's rho and E, its p and c too (halo_exchange.cpp:23-30: the EOS of the
// unscaled state) and its velocities times the side's factors; a stale one p and c from
// stale_p/stale_c.
template <class T, int AXIS, int EOS>
__device__ __forceinline__ Cell<T> make_cell(const SweepArgs<T>& a, int64_t base, const LoadedCell<T>& l)
{
    Cell<T> cell;
    T u = l.u, v = l.v;
    cell.y = shared_recip<T>(l.rho);
    cell_eos<T, EOS>(a.gamma, l.rho, u, v, l.E, cell.y, cell.p, cell.c);
    if (__builtin_expect(l.stale | (l.mirror != 0), 0)) {
        if (l.stale) {
            cell.p = load_at(a.stale_p + base, l.offset);
            cell.c = load_at(a.stale_c + base, l.offset);
        } else {
            u = u * (T) (l.mirror == 1 ? a.lo_u : a.hi_u);
            v = v * (T) (l.mirror == 1 ? a.lo_v : a.hi_v);
        }
    }
    cell.rho = l.rho;
    cell.E = l.E;
    cell.un = AXIS == 0 ? u : v;
    cell.ut = AXIS == 0 ? v : u;
    return cell;
}

// The Y march loads a row's state one row before it makes the cell: where row `k` comes from (the same
// for the whole wave: the row it is read at, the mirror side or staleness), then the cell from the loaded
// state.
struct RowSource {
    int row;
    int mirror;
    bool stale;
};

// STALE = false: the caller guarantees that the stencil width covers every ghost layer read
// (|k| beyond the domain is at most the read extent), so no layer is stale.
template <class T, bool STALE = true>
__device__ __forceinline__ RowSource row_source(const SweepArgs<T>& a, int k)
{
    RowSource s{k, 0, false};
    if (k < 0) {
        if (!STALE || -k <= a.stencil_width) { s.row = -k - 1; s.mirror = 1; }
        else s.stale = true;
    } else if (k >= a.ny) {
        if (!STALE || k - a.ny + 1 <= a.stencil_width) { s.row = 2 * a.ny - 1 - k; s.mirror = 2; }
        else s.stale = true;
    }
    return s;
}

// The first cell of row `row` within an array (64-bit, in scalar registers).
template <class T>
__device__ __forceinline__ int64_t row_start(const SweepArgs<T>& a, int row)
{
    return (int64_t) a.index_start + (int64_t) row * a.row_length;
}

template <class T, int EOS, bool STALE = true>
__device__ __forceinline__ Cell<T> make_row_cell(const SweepArgs<T>& a, const RowSource& s, unsigned column, T rho, T u,
                                                 T v, T E)
{
    Cell<T> cell;
    cell.y = shared_recip<T>(rho);
    if (STALE && s.stale) {
        cell.p = load_at(a.stale_p + row_start(a, s.row), column);
        cell.c = load_at(a.stale_c + row_start(a, s.row), column);
    } else {
        cell_eos<T, EOS>(a.gamma, rho, u, v, E, cell.y, cell.p, cell.c);   // unscaled, as make_cell
    }
    if (s.mirror == 1) {
        u = u * (T) a.lo_u;
        v = v * (T) a.lo_v;
    } else if (s.mirror == 2) {
        u = u * (T) a.hi_u;
        v = v * (T) a.hi_v;
    }
    cell.rho = rho;
    cell.E = E;
    cell.un = v;
    cell.ut = u;
    return cell;
}

template <class T>
__device__ __forceinline__ Cell<T> benign_cell()
{
    Cell<T> c;
    c.rho = T(1); c.un = T(0); c.ut = T(0); c.E = T(1); c.p = T(1); c.c = T(1); c.y = T(1);
    return c;
}

// `v` of the lane that a DPP control names, this lane's where that reaches no lane.
template <int CTRL>
__device__ __forceinline__ double dpp(double v)
{
    const uint64_t b = double_to_bits(v);
    const int lo = (int) (uint32_t) b, hi = (int) (b >> 32);
    const uint32_t l = (uint32_t) __builtin_amdgcn_update_dpp(lo, lo, CTRL, 0xF, 0xF, false);
    const uint32_t h = (uint32_t) __builtin_amdgcn_update_dpp(hi, hi, CTRL, 0xF, 0xF, false);
    return bits_to_double((unsigned long long) h << 32 | l);
}

// Minimum over the wave, in lane 63 (no NaN among the operands): neighbours, pairs and halves of each
// row of 16 lanes, then row 0 into 1 and 2 into 3, then rows 0-1 into 2-3.
__device__ __forceinline__ double wave_min_last(double v)
{
    v = __builtin_fmin(v, dpp<0xB1>(v));    // quad_perm [1,0,3,2]
    v = __builtin_fmin(v, dpp<0x4E>(v));    // quad_perm [2,3,0,1]
    v = __builtin_fmin(v, dpp<0x141>(v));   // row_half_mirror
    v = __builtin_fmin(v, dpp<0x140>(v));   // row_mirror
    v = __builtin_fmin(v, dpp<0x142>(v));   // row_bcast:15
    return __builtin_fmin(v, dpp<0x143>(v));   // row_bcast:31
}

// Merges a per-lane CFL bound into one of the state's accumulators, which the blocks share out among
// themselves. An accumulator only falls, so a wave whose bound is not below what it reads there (some
// earlier value at most) has nothing to add, and most waves of a large sweep need no atomic. The waves
// of a small one end together and would read the cleared value, 0.3-0.5 us later: they add unseen.
__device__ __forceinline__ void reduce_cfl(DeviceState* st, int mode, double local)
{
    unsigned long long* slot = &st->dt_min[(blockIdx.x + (threadIdx.x >> 6)) % kDtSlots].bits;
    unsigned long long seen = ~0ull;
    if (mode == REDUCE) seen = __hip_atomic_load(slot, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const unsigned long long bits = double_to_bits(wave_min_last(local));
    if ((threadIdx.x & 63) == 63 && bits < seen) atomicMin(slot, bits);
}

// The least of a state's accumulators, for every lane of the calling wave.
__device__ __forceinline__ double least_bound(const DeviceState* st)
{
    const int lane = threadIdx.x & 63;
    const double v = lane < kDtSlots ? bits_to_double(st->dt_min[lane].bits) : DBL_MAX;
    const uint64_t b = double_to_bits(wave_min_last(v));
    const uint32_t lo = (uint32_t) __builtin_amdgcn_readlane((int) (uint32_t) b, 63);
    const uint32_t hi = (uint32_t) __builtin_amdgcn_readlane((int) (b >> 32), 63);
    return bits_to_double((unsigned long long) hi << 32 | lo);
}

// ---------------------------------------------------------------------------------------
// Time step (armon_2D.cpp:212-252 and the loop condition of :347)
// ---------------------------------------------------------------------------------------

struct NextStep {
    double current_dt, next_dt, time, error_dt;
    int cycle, active, error, error_cycle;
};

// The next cycle's step from the state `st` and the CFL minimum of its current fields; called by a
// whole wave, whose lanes all compute it.
__device__ __forceinline__ NextStep next_step(const DeviceState* st, const TimeStepConfig& c)
{
    NextStep s{st->current_dt, st->next_dt, st->time, st->error_dt, st->cycle, 0, st->error, st->error_cycle};
    // before the checks, so that the bounds are on their way together with the state (0.4 us a small sweep)
    const double dt = least_bound(st);
    if (s.error || !(s.time < c.max_time && s.cycle < c.max_cycles)) return s;
    double current = s.next_dt;
    double next;
    if (c.cst_dt) {
        next = c.Dt;
    } else if (!c.dt_on_even_cycles || (s.cycle % 2 == 0) || current == 0) {
        double local;
        if (!finite_d(dt) || dt <= 0) local = dt;
        else if (current == 0) local = c.cfl * dt;
        else local = kmin(c.cfl * dt, 1.05 * current);
        if (!finite_d(local) || local <= 0) {
            s.error = 1;
            s.error_cycle = s.cycle;
            s.error_dt = local;
            return s;
        }
        next = local;
    } else {
        next = current;
    }
    if (s.cycle == 0) current = next;
    s.current_dt = current;
    s.next_dt = next;
    s.time += current;
    s.cycle += 1;
    s.active = 1;
    return s;
}

// Writes it down, by one whole wave, with the bounds of the fields to come cleared.
__device__ __forceinline__ void write_step(DeviceState* st, const NextStep& s)
{
    if ((threadIdx.x & 63) < kDtSlots) st->dt_min[threadIdx.x & 63].bits = kNoBound;
    if ((threadIdx.x & 63) != 0) return;
    st->current_dt = s.current_dt;
    st->next_dt = s.next_dt;
    st->time = s.time;
    st->error_dt = s.error_dt;
    st->cycle = s.cycle;
    st->active = s.active;
    st->error = s.error;
    st->error_cycle = s.error_cycle;
}

// Whether the cycle runs, and its dt: as its time step left them or, with FOLD, made here and written
// down by the first wave of the block that is told to (`writer`: one block of the launch). A compile
// time choice: the other way's code alone, behind a branch that is never taken, made the X sweep 2%
// (FP64) and 6% (FP32) slower at 8192^2.
template <bool FOLD, class T>
__device__ __forceinline__ bool begin_sweep(const SweepArgs<T>& a, bool writer, double& dt)
{
    if constexpr (!FOLD) {
        dt = a.st->current_dt;
        return a.st->active != 0;
    } else {
        const NextStep s = next_step(a.prev, a.step);
        if (writer && threadIdx.x < 64) write_step(a.st, s);
        dt = s.current_dt;
        return s.active != 0;
    }
}

// The CFL bound of the cells that a thread has seen (cfl_cell), kept as the largest wave speeds: a
// correctly rounded dx / a never grows with a, so the smallest bound is the one of the largest speed,
// and the divisions are made once. max(|u + c|, |u - c|) is |u| + |c| with the same rounding. A cell
// whose x bound is NaN has no bound, one whose y bound is NaN only that of x, as comparisons that a
// NaN loses leave it: a NaN speed counts as none (its high half cleared).
struct CflSpeeds {
    double x = 0, y = 0;
    __device__ __forceinline__ void add(double u, double v, double c)
    {
        const bool nan_x = !(u + c == u + c), nan_y = !(v + c == v + c);
        x = __builtin_fmax(x, speed(u, c, nan_x));
        y = __builtin_fmax(y, speed(v, c, (bool) ((int) nan_x | (int) nan_y)));
    }
    __device__ __forceinline__ double bound(double dx, double dy) const
    {
        return __builtin_fmin(DBL_MAX, __builtin_fmin(dx / x, dy / y));
    }
    static __device__ __forceinline__ double speed(double u, double c, bool none)
    {
        const uint64_t b = double_to_bits(__builtin_fabs(u) + __builtin_fabs(c));
        const uint32_t hi = none ? 0u : (uint32_t) (b >> 32);
        return bits_to_double((unsigned long long) hi << 32 | (uint32_t) b);
    }
};

// ---------------------------------------------------------------------------------------
// X sweep: LDS-staged row tiles
// ---------------------------------------------------------------------------------------

// LDS of one tile of CELLS slots whose neighbours along the axis lie S slots apart. The values that
// neighbours read together are stored together, 16 bytes (or 8) an access, and each slot's
// neighbours are reached by constant offsets from its own address: 2S slots of padding before the
// tile and S after it stand for the neighbours that the tile's end slots do not have (what is read
// there is never written by anyone and reaches no output, as outputs lie R slots inside).
//   stages 0-2: a0 = rho dx, un | a1 = p, rho c     b, f = Godunov's A, B     w = the face's u*, p*
//   stages 3-4: a0 = rho, rho un | a1 = rho ut, rho E   b = L, 1/L | c = 1/S (see tile_sweep)
//   stages 4-5: the advection fluxes, in FP64 in w and f, in FP32 in a0 and a1 after one more barrier
// FP64: 88 bytes a slot, 22.8 KB for a tile of 256: 7 blocks fit in a CU's 160 KB. FP32: 40 bytes, 20.6
// KB for a tile of 512, 7 blocks too. X sweep at 8192^2: FP64 846 us (96 bytes, 6 blocks: 892; the
// tile of before, which divided everywhere and exchanged single words: 914), FP32 408 us (48 bytes
// and no barrier more: 433; before: 416).
template <class T>
struct alignas(2 * sizeof(T)) Pair {
    T x, y;
};
template <class T>
struct alignas(16) Quad {
    T x, y, z, w;
};

// GAD, E2: whether the scheme has those stages (without either, b and c are not there: 64 bytes, 8 blocks).
template <class T, int CELLS, int S, bool GAD, bool E2>
struct TileLds;

template <int CELLS, int S, bool GAD, bool E2>
struct TileLds<double, CELLS, S, GAD, E2> {
    static constexpr int N = CELLS + 3 * S;
    static constexpr bool kFluxBarrier = false;
    using P = Pair<double>;
    P a0_[N], a1_[N], b_[GAD || E2 ? N : 1], w_[N], f_[N];
    double c_[E2 ? N : 1];
    __device__ __forceinline__ P& a0(int t) { return a0_[t + 2 * S]; }
    __device__ __forceinline__ P& a1(int t) { return a1_[t + 2 * S]; }
    __device__ __forceinline__ P& w(int t) { return w_[t + 2 * S]; }
    __device__ __forceinline__ void put_differences(int t, P A, P B)
    {
        b_[t + 2 * S] = A;
        f_[t + 2 * S] = B;
    }
    __device__ __forceinline__ P get_A(int t) { return b_[t + 2 * S]; }
    __device__ __forceinline__ P get_B(int t) { return f_[t + 2 * S]; }
    __device__ __forceinline__ void put_state(int t, double dm, double un, double p, double rc)
    {
        a0(t) = {dm, un};
        a1(t) = {p, rc};
    }
    __device__ __forceinline__ void get_state(int t, double& dm, double& un, double& p, double& rc)
    {
        const P l = a0(t), h = a1(t);
        dm = l.x; un = l.y; p = h.x; rc = h.y;
    }
    // what the slopes read: rho and the products rho u, rho v, rho E
    __device__ __forceinline__ void put_carried(int t, double rho, double un, double ut, double E)
    {
        a0(t) = {rho, rho * un};
        a1(t) = {rho * ut, rho * E};
    }
    __device__ __forceinline__ void get_carried(int t, double (&q)[4])
    {
        const P l = a0(t), h = a1(t);
        q[0] = l.x; q[1] = l.y; q[2] = h.x; q[3] = h.y;
    }
    __device__ __forceinline__ void put_lengths(int t, double L, double yL, double yS)
    {
        b_[t + 2 * S] = {L, yL};
        c_[t + 2 * S] = yS;
    }
    // around the donor cell t: its length and 1/L, the sums of its length and its neighbours'
    // lengths and their reciprocals
    __device__ __forceinline__ void get_lengths(int t, double& L, double& yL, double& lo, double& y_lo, double& hi,
                                                double& y_hi)
    {
        const P l = b_[t + 2 * S];
        L = l.x;
        yL = l.y;
        lo = L + b_[t + S].x;
        hi = b_[t + 3 * S].x + L;
        y_lo = c_[t + 2 * S];
        y_hi = c_[t + 3 * S];
    }
    __device__ __forceinline__ void put_flux(int t, const double (&f)[4])
    {
        w(t) = {f[0], f[1]};
        f_[t + 2 * S] = {f[2], f[3]};
    }
    __device__ __forceinline__ void get_flux(int t, double (&f)[4])
    {
        const P l = w(t), h = f_[t + 2 * S];
        f[0] = l.x; f[1] = l.y; f[2] = h.x; f[3] = h.y;
    }
};

template <int CELLS, int S, bool GAD, bool E2>
struct TileLds<float, CELLS, S, GAD, E2> {
    static constexpr int N = CELLS + 3 * S;
    using P = Pair<float>;
    using Q = Quad<float>;
    static constexpr bool kFluxBarrier = true;
    Q a_[N], b_[GAD || E2 ? N : 1];   // a: the state, what the slopes read, then the fluxes; b: Godunov's A and B, then the lengths
    P w_[N];
    __device__ __forceinline__ void put_differences(int t, P A, P B) { b_[t + 2 * S] = {A.x, A.y, B.x, B.y}; }
    __device__ __forceinline__ P get_A(int t)
    {
        const Q v = b_[t + 2 * S];
        return {v.x, v.y};
    }
    __device__ __forceinline__ P get_B(int t)
    {
        const Q v = b_[t + 2 * S];
        return {v.z, v.w};
    }
    __device__ __forceinline__ P& w(int t) { return w_[t + 2 * S]; }
    __device__ __forceinline__ void put_state(int t, float dm, float un, float p, float rc)
    {
        a_[t + 2 * S] = {dm, un, p, rc};
    }
    __device__ __forceinline__ void get_state(int t, float& dm, float& un, float& p, float& rc)
    {
        const Q v = a_[t + 2 * S];
        dm = v.x; un = v.y; p = v.z; rc = v.w;
    }
    // the state itself: its products are taken by the reader, as a flux fuses one of them
    __device__ __forceinline__ void put_carried(int t, float rho, float un, float ut, float E)
    {
        a_[t + 2 * S] = {rho, un, ut, E};
    }
    __device__ __forceinline__ void get_carried(int t, float (&q)[4])
    {
        const Q v = a_[t + 2 * S];
        q[0] = v.x; q[1] = v.y; q[2] = v.z; q[3] = v.w;
    }
    __device__ __forceinline__ void put_lengths(int t, float L, float yL, float yS)
    {
        b_[t + 2 * S] = {L, yL, yS, 0.0f};
    }
    __device__ __forceinline__ void get_lengths(int t, float& L, float& yL, float& lo, float& y_lo, float& hi,
                                                float& y_hi)
    {
        const Q l = b_[t + 2 * S], h = b_[t + 3 * S];
        L = l.x;
        yL = l.y;
        y_lo = l.z;
        y_hi = h.z;
        lo = hi = 0.0f;   // a quotient is the numerator times the reciprocal
    }
    __device__ __forceinline__ void put_flux(int t, const float (&f)[4]) { a_[t + 2 * S] = {f[0], f[1], f[2], f[3]}; }
    __device__ __forceinline__ void get_flux(int t, float (&f)[4])
    {
        const Q v = a_[t + 2 * S];
        f[0] = v.x; f[1] = v.y; f[2] = v.z; f[3] = v.w;
    }
};

template <class T, int FLUX, int PROJ, int CELLS, int S>
using SchemeLds = TileLds<T, CELLS, S, (FLUX > 0), PROJ == 2>;

// The whole per-axis chain of one tile, from the loaded cells (EOS done) to the projected ones:
// thread t computes the slots slot[0..CPT), and cell[] holds their new rho, un, ut, E afterwards
// (c stays the input state's). Every thread of the block calls it; outputs are right for the slots
// whose R neighbours on both sides are in the tile.
//
// What neighbours need is computed once and handed over through LDS: besides the states and fluxes
// these are each cell's Lagrangian length L = dx + dt (u*_right - u*_left), the sum S of its length
// and the lower neighbour's, and the refined reciprocals of both, over which the update, the slopes
// and the length factor of the advection divide (2 reciprocals where there were 4 divisions, and no
// length computed more than twice). The arithmetic of each result is the reference's, so FP64 keeps
// the bits of dividing everywhere; operands outside shared_recip's ranges take the divisions.
template <class T, int FLUX, int PROJ, int DXM, int CELLS, int S, int CPT>
__device__ __forceinline__ void tile_sweep(T dx, T inv_dx, T dt, SchemeLds<T, FLUX, PROJ, CELLS, S>& sm, const int (&slot)[CPT],
                                           Cell<T> (&cell)[CPT])
{
    constexpr bool GAD = FLUX > 0;
    constexpr bool E2 = PROJ == 2;
    // Stage 0: what the faces read.
    T dm[CPT], rc[CPT], dtdm[CPT];
    int bad[CPT];
#pragma unroll
    for (int k = 0; k < CPT; k++) {
        dm[k] = cell[k].rho * dx;
        rc[k] = cell[k].rho * cell[k].c;
        sm.put_state(slot[k], dm[k], cell[k].un, cell[k].p, rc[k]);
        dtdm[k] = mass_quotient<DXM>(dt, dm[k], cell[k].y, inv_dx);
        bad[k] = unusable(dtdm[k]);
        if (__builtin_expect(bad[k], 0)) dtdm[k] = dv<T>(dt, dm[k]);
    }
    __syncthreads();

    // Stages 1-2: the flux at face t, between the cells t-S and t.
    T us[CPT], ps[CPT];
    {
        T dm_m[CPT], un_m[CPT], p_m[CPT], rc_m[CPT];
#pragma unroll
        for (int k = 0; k < CPT; k++) {
            sm.get_state(slot[k] - S, dm_m[k], un_m[k], p_m[k], rc_m[k]);
            face_godunov<T>(rc_m[k], rc[k], un_m[k], cell[k].un, p_m[k], cell[k].p, us[k], ps[k]);
        }
        if constexpr (GAD) {
            Pair<T> A[CPT], B[CPT];
#pragma unroll
            for (int k = 0; k < CPT; k++) {
                A[k] = {us[k] - un_m[k], ps[k] - p_m[k]};
                B[k] = {cell[k].un - us[k], cell[k].p - ps[k]};
                sm.put_differences(slot[k], A[k], B[k]);
            }
            __syncthreads();
#pragma unroll
            for (int k = 0; k < CPT; k++) {
                const Pair<T> above = sm.get_A(slot[k] + S), below = sm.get_B(slot[k] - S);
                const T theta = gad_theta<T>(dt, dm_m[k], dm[k], rc_m[k], rc[k]);
                us[k] = gad_star<FLUX - 1, T>(theta, us[k], A[k].x, above.x, B[k].x, below.x);
                ps[k] = gad_star<FLUX - 1, T>(theta, ps[k], A[k].y, above.y, B[k].y, below.y);
            }
        }
    }
#pragma unroll
    for (int k = 0; k < CPT; k++) sm.w(slot[k]) = {us[k], ps[k]};
    __syncthreads();

    // Stage 3: Lagrangian update of cell t from the faces t and t+S.
    T us_m[CPT], us_p[CPT], L[CPT];
#pragma unroll
    for (int k = 0; k < CPT; k++) {
        const Pair<T> wp = sm.w(slot[k] + S);
        us_p[k] = wp.x;
        L[k] = dx + dt * (us_p[k] - us[k]);
        const T yL = shared_recip<T>(L[k]);
        cell[k].un += dtdm[k] * (ps[k] - wp.y);
        cell[k].E += dtdm[k] * (ps[k] * us[k] - wp.y * us_p[k]);
        cell[k].rho = quot<T>(dm[k], L[k], yL);
        if (__builtin_expect(bad[k] | unusable(yL), 0)) cell[k].rho = dv<T>(dm[k], L[k]);
        if constexpr (E2) {
            us_m[k] = sm.w(slot[k] - S).x;
            const T L_m = dx + dt * (us[k] - us_m[k]);
            const T sum = L[k] + L_m;
            sm.put_lengths(slot[k], L[k], yL, shared_recip<T>(sum));
        }
        sm.put_carried(slot[k], cell[k].rho, cell[k].un, cell[k].ut, cell[k].E);
    }
    __syncthreads();

    // Stage 4: the advection flux at face t, from the donor cell t or t-S.
    T f[CPT][4];
#pragma unroll
    for (int k = 0; k < CPT; k++) {
        const T disp = dt * us[k];
        const int d = disp > 0 ? slot[k] - S : slot[k];
        T q[4];
        sm.get_carried(d, q);
        if constexpr (E2) {
            T qm[4], qp[4];
            sm.get_carried(d - S, qm);
            sm.get_carried(d + S, qp);
            T Ld, yLd, lo, y_lo, hi, y_hi;
            sm.get_lengths(d, Ld, yLd, lo, y_lo, hi, y_hi);
            const T lf = length_factor<T>(donor_length<T>(dx, dt, disp, us_m[k], us_p[k]), Ld, yLd);
            T r_m, r_p, slope[4];
            slope_ratios<T>(Ld, lo, y_lo, hi, y_hi, r_m, r_p);
#pragma unroll
            for (int i = 0; i < 4; i++) {
                // FP64 tiles hold the products
                const T c = sizeof(T) == 8 ? q[i] : carried(q, i), m = sizeof(T) == 8 ? qm[i] : carried(qm, i),
                        p = sizeof(T) == 8 ? qp[i] : carried(qp, i);
                slope[i] = slope_minmod_t<T>(r_p * (p - c), r_m * (c - m));
            }
            donor_flux_2<T>(disp, lf, q, slope, f[k]);
        } else {
            donor_flux_1<T>(disp, q, f[k]);
        }
    }
    if constexpr (SchemeLds<T, FLUX, PROJ, CELLS, S>::kFluxBarrier) __syncthreads();
#pragma unroll
    for (int k = 0; k < CPT; k++) sm.put_flux(slot[k], f[k]);
    __syncthreads();

    // Stage 5: projection of cell t.
#pragma unroll
    for (int k = 0; k < CPT; k++) {
        T fp[4];
        sm.get_flux(slot[k] + S, fp);
        project<DXM, T>(dx, inv_dx, L[k], f[k], fp, cell[k].rho, cell[k].un, cell[k].ut, cell[k].E);
    }
}

// One X tile of the domain described by `a`; `begin(dt)` gives the cycle's dt, or false where the cycle
// does not run (the same for the whole block). Called by all TILE / CPT threads of a block; each thread
// computes CPT cells of the tile, at slots t, t + TILE / CPT, ... (consecutive lanes on consecutive slots
// for every load and store).
//
// The rows of the domain are laid end to end as a stream of slots, each row taking
// x_slots = nx + 2R slots (its R ghost cells on each side, then the next row). A tile covers
// TILE consecutive slots, starting at slot `k0` of row `j0`; consecutive tiles overlap by 2R
// slots, and the slots [R, TILE - R) of a tile that hold real cells are its outputs. A cell's
// result depends only on the cells within R of it in its own row, so a tile may span the end
// of one row and the start of the next; no thread is spent on a tile's share of a row end.
template <class T, int FLUX, int PROJ, int EOS, int DXM, int TILE = kTile, int CPT = 1, class Begin>
__device__ __forceinline__ void sweep_x_tile(const SweepArgs<T>& a, Begin&& begin, int j0, int k0,
                                             SchemeLds<T, FLUX, PROJ, TILE, 1>& sm)
{
    constexpr int R = 2 + (FLUX > 0 ? 1 : 0) + (PROJ == 2 ? 1 : 0);
    constexpr int NT = TILE / CPT;
    static_assert(TILE % CPT == 0, "a tile is a whole number of cells per thread");

    int slot[CPT], jc[CPT], kc[CPT];
    bool in_range[CPT];
    LoadedCell<T> loaded[CPT];
    Cell<T> cell[CPT];
    // Row jc and cell kc (-R <= kc < nx + R) of each slot: n = k0 + t < x_slots + TILE. Rows of
    // at least TILE slots: n < 2 x_slots. Shorter rows: the float quotient is within one of the
    // exact one and a single correction makes it exact. (The test on the row length is the
    // block's, taken once, so that only one of the two ways is executed.)
    if (a.x_slots >= TILE) {
#pragma unroll
        for (int c = 0; c < CPT; c++) {
            const int n = k0 + (int) threadIdx.x + c * NT;
            const int dj = n >= a.x_slots ? 1 : 0;
            jc[c] = dj;
            kc[c] = n - (dj ? a.x_slots : 0) - R;
        }
    } else {
#pragma unroll
        for (int c = 0; c < CPT; c++) {
            const int n = k0 + (int) threadIdx.x + c * NT;
            int dj = (int) ((float) n * a.x_inv_slots);
            int r = n - dj * a.x_slots;
            if (r < 0) { dj--; r += a.x_slots; }
            else if (r >= a.x_slots) { dj++; r -= a.x_slots; }
            jc[c] = dj;
            kc[c] = r - R;
        }
    }
    // Offsets within the arrays count from the tile's first row less its R ghost cells, so that they
    // are small, unsigned and shared by all arrays, and the bases stay in scalar registers.
    const int64_t base = (int64_t) a.index_start + (int64_t) j0 * a.row_length - R;
    const int rows_left = a.ny - j0;
#pragma unroll
    for (int c = 0; c < CPT; c++) {
        slot[c] = threadIdx.x + c * NT;
        in_range[c] = jc[c] < rows_left;       // false for slots past the last row
        if (in_range[c]) loaded[c] = fetch_cell<T>(a, base, jc[c] * a.row_length + R, kc[c], 1, a.nx);
    }
    double cycle_dt;
    if (!begin(cycle_dt)) return;
    const T dt = (T) (cycle_dt * a.dt_factor);
#pragma unroll
    for (int c = 0; c < CPT; c++)
        cell[c] = in_range[c] ? make_cell<T, 0, EOS>(a, base, loaded[c]) : benign_cell<T>();
    tile_sweep<T, FLUX, PROJ, DXM, TILE, 1, CPT>((T) a.dx, (T) a.inv_dx, dt, sm, slot, cell);

    CflSpeeds speeds;
#pragma unroll
    for (int c = 0; c < CPT; c++) {
        const int t = slot[c];
        if (t >= R && t < TILE - R && in_range[c] && (unsigned) kc[c] < (unsigned) a.nx) {
            const unsigned o = (unsigned) (jc[c] * a.row_length + R + kc[c]) * (unsigned) sizeof(T);
            store_at(a.out_rho + base, o, cell[c].rho);
            store_at(a.out_u + base, o, cell[c].un);
            store_at(a.out_v + base, o, cell[c].ut);
            store_at(a.out_E + base, o, cell[c].E);
            if (a.reduce) speeds.add((double) cell[c].un, (double) cell[c].ut, (double) cell[c].c);
        }
    }
    if (a.reduce) reduce_cfl(a.st, a.reduce, speeds.bound(a.cfl_dx, a.cfl_dy));
}

// Tile of the single-domain X sweep per element type: FP64 tiles of 256 cells at one cell per
// thread; FP32 tiles of 512 cells at two cells per thread (256 threads), which measured faster for
// the FP32-mixed sweep (408 us at 8192^2, one cell per thread 468) and slower for the FP64 one. The
// LDS leaves room for 7 waves per SIMD (8 without GAD and second order), so the kernels are held to the
// 72 (64) VGPRs that so many have.
template <class T>
struct XTile {
    static constexpr int cells = 256, cpt = 1;
};
template <>
struct XTile<float> {
    static constexpr int cells = 512, cpt = 2;
};

template <class T, int FLUX, int PROJ, int EOS, int DXM, bool FOLD>
__global__ void __launch_bounds__(XTile<T>::cells / XTile<T>::cpt) __attribute__((amdgpu_waves_per_eu(FLUX > 0 || PROJ == 2 ? 7 : 8)))
        k_sweep_x(SweepArgs<T> a)
{
    constexpr int TILE = XTile<T>::cells;
    constexpr int W = TILE - 2 * (2 + (FLUX > 0 ? 1 : 0) + (PROJ == 2 ? 1 : 0));
    __shared__ SchemeLds<T, FLUX, PROJ, TILE, 1> sm;
    const int s0 = xcd_block(blockIdx.x, gridDim.x) * W;   // first slot of the tile
    const int j0 = s0 / a.x_slots;
    sweep_x_tile<T, FLUX, PROJ, EOS, DXM, TILE, XTile<T>::cpt>(
            a, [&](double& dt) { return begin_sweep<FOLD>(a, blockIdx.x == 0, dt); }, j0, s0 - j0 * a.x_slots, sm);
}

// ---------------------------------------------------------------------------------------
// Y sweep: register march down columns
// ---------------------------------------------------------------------------------------

template <class T, int N>
__device__ __forceinline__ void push(T (&w)[N], T v)
{
#pragma unroll
    for (int i = 0; i < N - 1; i++) w[i] = w[i + 1];
    w[N - 1] = v;
}

// What a thread of the march keeps in LDS until a later row, off the arithmetic's dependency chains
// (a slot is read before the row that wraps round to it writes it): the parts of a cell that the
// faces do not read and, for the CFL bound, its sound speed.
// The update takes them two rows later with GAD, else one; the bound R rows later, with GAD 3 or 4.
template <class T, int FLUX, int PROJ>
struct MarchLds {
    static constexpr int kRows = FLUX > 0 ? 2 : 1, kBounds = FLUX > 0 ? 4 : PROJ == 2 ? 3 : 2;
    Pair<T> ut_E[kRows][kYBlock];
    T dtdm[kRows][kYBlock], c[kBounds][kYBlock];
};

// What else waits for the next row or two: the reciprocal of an updated cell's length, its slopes and
// its state once the next cell is there, and a face's advection fluxes. In FP64 in LDS too (32 VGPRs
// fewer: with register windows the unrolled march does not fit the 168 of 3 waves per SIMD; 48 KB
// with the rest, 3 blocks a CU); in FP32 in registers, where the march has them (100 VGPRs) and is
// 4% faster so (494 -> 472 us at 8192^2).
//
// E2: whether the projection is of second order; in first order only the fluxes wait.
template <class T, bool E2>
struct MarchWindows;

template <bool E2>
struct MarchWindows<double, E2> {
    struct SecondOrder {
        double yL[2][kYBlock];
        Pair<double> cell[2][kYBlock], slope[2][kYBlock];
    };
    struct FirstOrder {};
    struct Lds : std::conditional_t<E2, SecondOrder, FirstOrder> {
        Pair<double> flux[2][kYBlock];
    };
    Lds* lds;
    static __device__ __forceinline__ void swap(Pair<double> (&at)[2][kYBlock], const double (&put)[4], double (&got)[4])
    {
        get(at, got);
        at[0][threadIdx.x] = {put[0], put[1]};
        at[1][threadIdx.x] = {put[2], put[3]};
    }
    static __device__ __forceinline__ void get(const Pair<double> (&at)[2][kYBlock], double (&v)[4])
    {
        const Pair<double> l = at[0][threadIdx.x], h = at[1][threadIdx.x];
        v[0] = l.x; v[1] = l.y; v[2] = h.x; v[3] = h.y;
    }
    __device__ __forceinline__ void init(Lds* at) { lds = at; }
    __device__ __forceinline__ void cell(const double (&put)[4], double (&got)[4]) { swap(lds->cell, put, got); }
    __device__ __forceinline__ void flux(const double (&put)[4], double (&got)[4]) { swap(lds->flux, put, got); }
    __device__ __forceinline__ void slope_below(double (&v)[4]) const { get(lds->slope, v); }
    __device__ __forceinline__ double yL_below(int U) const { return lds->yL[U & 1][threadIdx.x]; }
    __device__ __forceinline__ double yL_own(int U) const { return lds->yL[(U - 1) & 1][threadIdx.x]; }
    __device__ __forceinline__ void put(int U, const double (&slope)[4], double yL)
    {
        double old[4];
        swap(lds->slope, slope, old);
        lds->yL[U & 1][threadIdx.x] = yL;
    }
};

template <bool E2>
struct MarchWindows<float, E2> {
    struct Lds {};
    float cell_[4], flux_[4], slope_[4], yL_[2];
    static __device__ __forceinline__ void swap(float (&at)[4], const float (&put)[4], float (&got)[4])
    {
#pragma unroll
        for (int k = 0; k < 4; k++) {
            got[k] = at[k];
            at[k] = put[k];
        }
    }
    __device__ __forceinline__ void init(Lds*)
    {
#pragma unroll
        for (int k = 0; k < 4; k++) cell_[k] = flux_[k] = slope_[k] = 1.0f;
        yL_[0] = yL_[1] = 1.0f;
    }
    __device__ __forceinline__ void cell(const float (&put)[4], float (&got)[4]) { swap(cell_, put, got); }
    __device__ __forceinline__ void flux(const float (&put)[4], float (&got)[4]) { swap(flux_, put, got); }
    __device__ __forceinline__ void slope_below(float (&v)[4]) const
    {
#pragma unroll
        for (int k = 0; k < 4; k++) v[k] = slope_[k];
    }
    __device__ __forceinline__ float yL_below(int) const { return yL_[0]; }
    __device__ __forceinline__ float yL_own(int) const { return yL_[1]; }
    __device__ __forceinline__ void put(int, const float (&slope)[4], float yL)
    {
#pragma unroll
        for (int k = 0; k < 4; k++) slope_[k] = slope[k];
        yL_[0] = yL_[1];
        yL_[1] = yL;
    }
};

template <size_t BYTES>
struct Unused {
    char bytes[BYTES];
};
template <>
struct Unused<0> {};

// A block's LDS: one in a kernel, also where that holds two copies of the march. In FP64 GAD and second order
// take 48 KB, for 3 blocks a CU, as their registers allow; the others 40 KB, for 4, with what they need
// (18 to 40 KB) and some unused. With 3 blocks they took 8% longer on the mean of 50 sizes of 6 M to 60 M
// cells (GAD and first order 60 M in 7745 columns 792 us and 745 with 4; Godunov and second order in 520
// columns 1023 and 898). With 5 Godunov and first order, bound by memory, took up to 20% longer in 60 M
// cells (4000 columns 720 us with 3 or 4 and 870).
template <class T, int FLUX, int PROJ>
struct MarchParts {
    MarchLds<T, FLUX, PROJ> keep;
    typename MarchWindows<T, PROJ == 2>::Lds windows;
};
template <class T, int FLUX, int PROJ>
struct MarchBlockLds : MarchParts<T, FLUX, PROJ>,
                       Unused<sizeof(T) == 8 && sizeof(MarchParts<T, FLUX, PROJ>) < 40960
                                      ? 40960 - sizeof(MarchParts<T, FLUX, PROJ>) : 0> {};

// The march state of one column of a Y run: sliding windows of the stage results along y. Each row's
// state is loaded one row before it is used (with STALE = false, when the stencil width covers the
// read extent so that no ghost layer is stale, the march then loads nothing else).
//
// Per row it makes the cell n, Godunov's face n, the final face F, the update of the cell U below it,
// the slopes of the cell below that, the advection flux at a face A and the projection of the cell P
// below A. What several rows or stages need is made once: the differences A and B of a face, theta,
// the Lagrangian lengths, their sums and the reciprocals of both, the differences and slopes of the
// carried quantities (per cell, whichever face takes them).
template <class T, int FLUX, int PROJ, int EOS, int DXM, bool STALE>
struct YColumn {
    static constexpr int GAD = FLUX > 0 ? 1 : 0;
    static constexpr int E2 = PROJ == 2 ? 1 : 0;
    static constexpr int R = 2 + GAD + E2;

    // Windows, oldest first.
    T dm[3], un[3];                       // cells n-2, n-1, n
    T rc, p;                              // cell n
    T theta[2], g_u[2], g_p[2];           // faces n-1, n
    Pair<T> A[2], B[3];                   // faces n-1, n; n-2, n-1, n
    T us[4], ps[2];                       // final faces F-3..F; F-1, F (F = n - GAD)
    T L[3], S[2], yS[2];                  // cells U-2, U-1, U; U-1, U (U = F - 1)
    T q[2][4];                            // updated cells U-1, U: rho, un, ut, E
    T dq[2][4];                           // carried quantities: U-1 over U-2, U over U-1
    T nx_rho, nx_u, nx_v, nx_E;           // the next row's state
    unsigned column;                      // byte offset of the column within a row
    bool lane_ok;                         // false for lanes past the domain
    CflSpeeds speeds;                     // of the column's outputs
    MarchWindows<T, PROJ == 2> windows;

    __device__ __forceinline__ void init(int x, bool ok, typename MarchWindows<T, PROJ == 2>::Lds* lds)
    {
        windows.init(lds);
        column = (unsigned) x * (unsigned) sizeof(T);
        lane_ok = ok;
#pragma unroll
        for (int i = 0; i < 3; i++) {
            dm[i] = L[i] = T(1);
            un[i] = T(0);
            B[i] = {T(0), T(0)};
        }
        rc = p = T(1);
#pragma unroll
        for (int i = 0; i < 2; i++) {
            theta[i] = g_u[i] = g_p[i] = ps[i] = T(0);
            A[i] = {T(0), T(0)};
            S[i] = yS[i] = T(1);
            q[i][0] = q[i][3] = T(1);
            q[i][1] = q[i][2] = T(0);
#pragma unroll
            for (int k = 0; k < 4; k++) dq[i][k] = T(0);
        }
#pragma unroll
        for (int i = 0; i < 4; i++) us[i] = T(0);
        nx_rho = T(1); nx_u = T(0); nx_v = T(0); nx_E = T(1);
    }

    __device__ __forceinline__ void fetch(const SweepArgs<T>& a, int k)
    {
        if (lane_ok) {
            const int64_t row = row_start(a, row_source<T, STALE>(a, k).row);
            nx_rho = load_at(a.in_rho + row, column);
            nx_u = load_at(a.in_u + row, column);
            nx_v = load_at(a.in_v + row, column);
            nx_E = load_at(a.in_E + row, column);
        }
    }

    // Row n of a run that outputs rows [y0, y1).
    __device__ __forceinline__ void step(const SweepArgs<T>& a, T dt, T dx, T inv_dx, int n, int y0, int y1,
                                         MarchLds<T, FLUX, PROJ>& keep)
    {
        const int t = threadIdx.x;
        // Keeps the column's offset out of the loop-invariant addresses that the compiler would make
        // of it and the arrays' bases (16 VGPRs, and a 64-bit sum per access): base and row stay scalar.
        asm("" : "+v"(column));
        // the next load is issued after this row's cell is made: a stale layer's p, c loads are
        // waited for there
        const Cell<T> cn = lane_ok ? make_row_cell<T, EOS, STALE>(a, row_source<T, STALE>(a, n), column, nx_rho, nx_u,
                                                                  nx_v, nx_E)
                                   : benign_cell<T>();
        if (n + 1 < y1 + R) fetch(a, n + 1);
        const T rc_m = rc, p_m = p;
        push(dm, cn.rho * dx);
        push(un, cn.un);
        rc = cn.rho * cn.c;
        p = cn.p;
        T dtdm = mass_quotient<DXM>(dt, dm[2], cn.y, inv_dx);
        if (__builtin_expect(unusable(dtdm), 0)) dtdm = dv<T>(dt, dm[2]);
        // what is left of cell U (the one before n, or two before it) and the sound speed of cell n-R
        constexpr int W = GAD ? 0 : 1;    // window index of cell U among n-2, n-1, n
        constexpr unsigned kBounds = MarchLds<T, FLUX, PROJ>::kBounds;
        const int row = GAD ? n & 1 : 0;
        const unsigned bound = (unsigned) (n + 4) % kBounds, bound_P = (unsigned) (n + 4 + (int) kBounds - R) % kBounds;
        const Pair<T> rest = keep.ut_E[row][t];
        const T dtdm_U = keep.dtdm[row][t];
        const T c_P = keep.c[bound_P][t];
        keep.ut_E[row][t] = {cn.ut, cn.E};
        keep.dtdm[row][t] = dtdm;
        keep.c[bound][t] = cn.c;

        // Godunov at face n (cells n-1 | n).
        T gu, gp;
        face_godunov<T>(rc_m, rc, un[1], un[2], p_m, p, gu, gp);
        // Final flux at face F: GAD at F = n-1 (cells n-2 | n-1, Godunov n-2, n-1, n), else F = n.
        if constexpr (GAD) {
            push(g_u, gu);
            push(g_p, gp);
            push(A, Pair<T>{gu - un[1], gp - p_m});
            push(B, Pair<T>{un[2] - gu, p - gp});
            push(us, gad_star<FLUX - 1, T>(theta[1], g_u[0], A[0].x, A[1].x, B[1].x, B[0].x));
            push(ps, gad_star<FLUX - 1, T>(theta[1], g_p[0], A[0].y, A[1].y, B[1].y, B[0].y));
            push(theta, gad_theta<T>(dt, dm[1], dm[2], rc_m, rc));
        } else {
            push(us, gu);
            push(ps, gp);
        }

        // Lagrangian update of cell U = F-1 from the faces U and F.
        const int U = n - 2 + W;
        const T len = dx + dt * (us[3] - us[2]);
        push(L, len);
        const T yL = shared_recip<T>(len);
        T rho = quot<T>(dm[W], len, yL);
        // a mass out of quot()'s range came with a density out of shared_recip's
        if (__builtin_expect(unusable(rho) | too_small(dm[W]), 0)) rho = dv<T>(dm[W], len);
        T u = un[W], E = rest.y;
        u += dtdm_U * (ps[0] - ps[1]);
        E += dtdm_U * (ps[0] * us[2] - ps[1] * us[3]);
        T older[4];                       // cell U-2
        if constexpr (E2) windows.cell(q[1], older);
#pragma unroll
        for (int k = 0; k < 4; k++) q[0][k] = q[1][k];
        q[1][0] = rho; q[1][1] = u; q[1][2] = rest.x; q[1][3] = E;

        // Advection flux at face A.
        const T disp = dt * us[E2 ? 1 : 2];
        T f[4];
        if constexpr (E2) {
            push(S, L[2] + L[1]);
            push(yS, shared_recip<T>(S[1]));
            // the slopes of cell U-1
            T r_m, r_p, slope[4];
            slope_ratios<T>(L[1], S[0], yS[0], S[1], yS[1], r_m, r_p);
#pragma unroll
            for (int k = 0; k < 4; k++) {
                dq[0][k] = dq[1][k];
                dq[1][k] = carried(q[1], k) - carried(q[0], k);
                slope[k] = slope_minmod_t<T>(r_p * dq[1][k], r_m * dq[0][k]);
            }
            // A = U-1: the cells A-1 = U-2 and A = U-1
            const T Dx = donor_length<T>(dx, dt, disp, us[0], us[2]);
            T from[4];
            if (disp > 0) {
                windows.slope_below(from);
                flux_from(disp, length_factor<T>(Dx, L[0], windows.yL_below(U)), older, from, f);
            } else {
                flux_from(disp, length_factor<T>(Dx, L[1], windows.yL_own(U)), q[0], slope, f);
            }
            windows.put(U, slope, yL);
        } else {
            // A = U: the cells A-1 = U-1 and A = U
            const T none[4] = {T(0), T(0), T(0), T(0)};
            if (disp > 0) flux_from(disp, T(0), q[0], none, f);
            else flux_from(disp, T(0), q[1], none, f);
        }
        T below[4];                       // the fluxes of face P
        windows.flux(f, below);

        // Projection of cell P = A-1 = n-R from the faces P and A.
        const int P = n - R;
        if (P >= y0 && P < y1 && lane_ok) {
            const T(&c)[4] = E2 ? older : q[0];
            T r = c[0], un_P = c[1], ut_P = c[2], e = c[3];
            project<DXM, T>(dx, inv_dx, L[E2 ? 0 : 1], below, f, r, un_P, ut_P, e);
            const int64_t row = row_start(a, P);
            store_at(a.out_rho + row, column, r);
            store_at(a.out_u + row, column, ut_P);   // ut is the x velocity in a Y sweep
            store_at(a.out_v + row, column, un_P);
            store_at(a.out_E + row, column, e);
            if (a.reduce) speeds.add((double) ut_P, (double) un_P, (double) c_P);
        }
    }

    // The flux from the donor cell `c`.
    static __device__ __forceinline__ void flux_from(T disp, T lf, const T (&c)[4], const T (&slope)[4], T (&f)[4])
    {
        T d[4] = {c[0], c[1], c[2], c[3]};
        if constexpr (sizeof(T) == 8) {
#pragma unroll
            for (int k = 1; k < 4; k++) d[k] = c[0] * c[k];
        }
        if constexpr (E2) donor_flux_2<T>(disp, lf, d, slope, f);
        else donor_flux_1<T>(disp, d, f);
    }
};

// One Y run: column x (a lane at or past nx marches benign cells and writes nothing), output
// rows [y0, y1), with the cycle's dt. The whole wave must call it with the same y0, y1.
//
// SYNC: every wave of the block marches the same rows (of adjacent columns) and meets a block
// barrier after every 4 rows, so that the block's loads and stores of a row stay within 4 rows
// of each other. Waves that march independently drift apart by many rows, and the pieces that
// each wave reads and writes per array and row (512 bytes in FP64) then fall in different DRAM
// pages: a copy with the FP64 march's access pattern and no arithmetic (ymarch_copy.hip) moves
// 4.2 TB/s that way and 4.6 TB/s with a barrier every 1-8 rows. With the barrier the FP32-mixed
// march is 9% faster and the FP64 march 3.6% (and with stale layers, Godunov and first-order
// projection, us per sweep at 8192^2 without -> with: FP64 968 -> 909, FP32 568 -> 489).
// `idle` waves (past the last column) take part in the barriers only. SYNC needs the same number
// of rows for the whole block: the loop-free batched kernel takes it for a block whose 4 waves
// hold live runs of equal length (most blocks, as the runs are listed longest first) and the
// independent march otherwise.
template <class T, int FLUX, int PROJ, int EOS, int DXM, bool STALE, bool SYNC = false>
__device__ __forceinline__ void sweep_y_run(const SweepArgs<T>& a, T dt, int x, int y0, int y1,
                                            MarchBlockLds<T, FLUX, PROJ>& lds, bool idle = false)
{
    using Col = YColumn<T, FLUX, PROJ, EOS, DXM, STALE>;
    constexpr int R = Col::R;
    // a row counter from 0 keeps the loop and the row index in scalar registers (counting
    // from y0 - R, the compiler carried the row index in a vector register)
    const int rows = y1 - y0 + 2 * R;
    // SYNC marches whole groups of 4 rows: up to 3 steps past the run, which load nothing (the
    // row-ahead load stops at the run's last row; without stale layers a cell is made from the
    // loaded state alone) and store nothing (outputs are rows [y0, y1) only). With stale layers,
    // whose p and c a step loads, those steps are left out.
    const int groups = (rows + 3) / 4;
    if constexpr (SYNC) {
        if (idle) {
            for (int g = 0; g < groups; ++g) __syncthreads();
            return;
        }
    }
    Col col;
    auto& keep = lds.keep;
    col.init(x, x < a.nx, &lds.windows);
    col.fetch(a, y0 - R);
    if constexpr (SYNC) {
        for (int g = 0; g < groups; ++g) {
#pragma unroll(sizeof(T) == 8 ? kYUnrollFp64 : kYUnrollFp32)
            for (int k = 0; k < 4; ++k)
                if (!STALE || 4 * g + k < rows)
                    col.step(a, dt, (T) a.dx, (T) a.inv_dx, y0 - R + 4 * g + k, y0, y1, keep);
            __syncthreads();
        }
    } else {
        // not unrolled: step()'s empty asm keeps the compiler from it, and two rows a turn by hand (with the
        // rest of the rows after it) measured no faster
        for (int i = 0; i < rows; ++i) col.step(a, dt, (T) a.dx, (T) a.inv_dx, y0 - R + i, y0, y1, keep);
    }
    if (a.reduce) reduce_cfl(a.st, a.reduce, col.speeds.bound(a.cfl_dx, a.cfl_dy));
}

template <class T, int FLUX, int PROJ, int EOS, int DXM, bool STALE>
__global__ void __launch_bounds__(kYBlock) __attribute__((amdgpu_waves_per_eu(PROJ == 2 ? kYWaves : kYWavesFirstOrder)))
        k_sweep_y(SweepArgs<T> a, int ncolblk)
{
    if (!a.st->active) return;
    const T dt = (T) (a.st->current_dt * a.dt_factor);
    const int bid = xcd_block(blockIdx.x, gridDim.x);   // runs in segment-major order
    const int seg = bid / ncolblk;
    const int x = (bid - seg * ncolblk) * kYBlock + threadIdx.x;
    const bool idle = x - (int) (threadIdx.x & 63) >= a.nx;   // a wave past the last column
    const int y0 = seg * a.seg_len;
    __shared__ MarchBlockLds<T, FLUX, PROJ> lds;
    sweep_y_run<T, FLUX, PROJ, EOS, DXM, STALE, true>(a, dt, x, y0, min(y0 + a.seg_len, a.ny), lds, idle);
}

// ---------------------------------------------------------------------------------------
// Y sweep of domains too small to fill the chip with marches: LDS tiles
// ---------------------------------------------------------------------------------------

// One Y tile: the columns [x0, x0 + COLS) and the output rows [y0, y0 + ROWS - 2R) of the domain
// described by `a` (`begin` as for sweep_x_tile), through the stages of tile_sweep with neighbours a tile
// row apart. Called by NT threads, each with COLS ROWS / NT cells of one column.
template <class T, int FLUX, int PROJ, int EOS, int DXM, int COLS, int ROWS, int NT, class Begin>
__device__ __forceinline__ void sweep_y_tile(const SweepArgs<T>& a, Begin&& begin, int x0, int y0,
                                             SchemeLds<T, FLUX, PROJ, COLS * ROWS, COLS>& sm)
{
    constexpr int R = 2 + (FLUX > 0 ? 1 : 0) + (PROJ == 2 ? 1 : 0);
    constexpr int CPT = COLS * ROWS / NT;
    static_assert(NT % COLS == 0 && COLS * ROWS % NT == 0, "a thread's cells are in one column");
    const int col = threadIdx.x % COLS, x = x0 + col;
    // offsets count from the tile's first row (a mirror's real cell never lies above it)
    const int64_t base = (int64_t) a.index_start + (int64_t) (y0 - R) * a.row_length + x0;
    int slot[CPT], row[CPT];
    bool in_range[CPT];
    LoadedCell<T> loaded[CPT];
    Cell<T> cell[CPT];
#pragma unroll
    for (int c = 0; c < CPT; c++) {
        slot[c] = threadIdx.x + c * NT;
        row[c] = threadIdx.x / COLS + c * (NT / COLS);
        const int k = y0 - R + row[c];
        in_range[c] = x < a.nx && k < a.ny + R;
        if (in_range[c])
            loaded[c] = fetch_cell<T>(a, base, col + (R - y0) * a.row_length, k, a.row_length, a.ny);
    }
    double cycle_dt;
    if (!begin(cycle_dt)) return;
    const T dt = (T) (cycle_dt * a.dt_factor);
#pragma unroll
    for (int c = 0; c < CPT; c++)
        cell[c] = in_range[c] ? make_cell<T, 1, EOS>(a, base, loaded[c]) : benign_cell<T>();
    tile_sweep<T, FLUX, PROJ, DXM, COLS * ROWS, COLS, CPT>((T) a.dx, (T) a.inv_dx, dt, sm, slot, cell);
    CflSpeeds speeds;
#pragma unroll
    for (int c = 0; c < CPT; c++) {
        if (row[c] >= R && row[c] < ROWS - R && x < a.nx && y0 - R + row[c] < a.ny) {
            const unsigned o = (unsigned) (col + row[c] * a.row_length) * (unsigned) sizeof(T);
            store_at(a.out_rho + base, o, cell[c].rho);
            store_at(a.out_u + base, o, cell[c].ut);   // ut is the x velocity in a Y sweep
            store_at(a.out_v + base, o, cell[c].un);
            store_at(a.out_E + base, o, cell[c].E);
            if (a.reduce) speeds.add((double) cell[c].ut, (double) cell[c].un, (double) cell[c].c);
        }
    }
    if (a.reduce) reduce_cfl(a.st, a.reduce, speeds.bound(a.cfl_dx, a.cfl_dy));
}

// Tiles of 16 columns x 32 rows: 128 bytes of a row in FP64, and 24 of the 32 rows are outputs. FP64:
// one cell a thread, 49 KB of LDS, 3 blocks a CU; FP32: two cells a thread. Of the shapes measured
// (4 to 32 columns, 24 to 96 rows, 1 to 4 cells a thread; Y sweep at 512^2 / 1024^2, us): FP64 16x32
// 12.1 / 27.8, 8x64 12.9 / 27.1, 16x64 19 / 37, 32x32 18 / 39; FP32 16x32 10.5 / 16.9, 16x64 at two cells
// 10.4 / 17.2, at one cell 11.5 / 20.4.
//
// A march has a wave per 64 columns and run, which works through its rows one after the other, some
// 1.5 us each; a tile has a thread per cell or two. The march is the cheaper per cell (its runs are
// longer than 24 rows, and nothing passes through LDS) once its waves fill the chip: us per Y sweep,
// march / tile, FP64 512^2 24.7 / 12.1, 1024^2 35.9 / 27.8, 2048^2 86 / 92; FP32 512^2 16.9 / 10.5,
// 1024^2 23 / 16.9, 2048^2 40 / 41. y_takes_tiles() has the rule.
template <class T>
struct YTile {
    static constexpr int cols = y_tile_cols(), rows = y_tile_rows(), threads = sizeof(T) == 8 ? 512 : 256;
};

template <class T, int FLUX, int PROJ, int EOS, int DXM, bool FOLD>
__global__ void __launch_bounds__(YTile<T>::threads) k_sweep_y_tile(SweepArgs<T> a, int ncolblk)
{
    using Y = YTile<T>;
    constexpr int W = Y::rows - 2 * (2 + (FLUX > 0 ? 1 : 0) + (PROJ == 2 ? 1 : 0));
    __shared__ SchemeLds<T, FLUX, PROJ, Y::cols * Y::rows, Y::cols> sm;
    const int bid = xcd_block(blockIdx.x, gridDim.x);
    const int band = bid / ncolblk;
    sweep_y_tile<T, FLUX, PROJ, EOS, DXM, Y::cols, Y::rows, Y::threads>(
            a, [&](double& dt) { return begin_sweep<FOLD>(a, blockIdx.x == 0, dt); }, (bid - band * ncolblk) * Y::cols,
            band * W, sm);
}

// ---------------------------------------------------------------------------------------
// Batched ensemble: persistent blocks over the work items of every domain
// ---------------------------------------------------------------------------------------

// How the batched sweeps divide by the cell sizes, the same for every domain: the
// reciprocal-corrected quotient in FP64 (exact for powers of two too), the FP32-mixed division
// (a native reciprocal) in FP32.
template <class T>
constexpr int kBatchDxMode = sizeof(T) == 8 ? DX_RECIP : DX_DIVIDE;

template <bool FOLD = false, class T>
__device__ __forceinline__ SweepArgs<T> batch_domain_args(const BatchArgs<T>& b, int d, int axis)
{
    const BatchDomain& D = b.domains[d];
    SweepArgs<T> a;
    a.in_rho = b.in_rho + D.offset;
    a.in_u = b.in_u + D.offset;
    a.in_v = b.in_v + D.offset;
    a.in_E = b.in_E + D.offset;
    a.out_rho = b.out_rho + D.offset;
    a.out_u = b.out_u + D.offset;
    a.out_v = b.out_v + D.offset;
    a.out_E = b.out_E + D.offset;
    a.stale_p = b.stale_p + D.offset;
    a.stale_c = b.stale_c + D.offset;
    a.st = b.states + d;
    if constexpr (FOLD) {
        a.prev = b.prev + d;
        a.step = b.steps[d];
    }
    a.nx = D.nx;
    a.ny = D.ny;
    a.row_length = D.row_length;
    a.index_start = D.index_start;
    a.stencil_width = b.stencil_width;
    a.seg_len = 0;
    a.reduce = b.reduce;
    a.gamma = b.gamma;
    a.dx = D.dx[axis];
    a.inv_dx = D.inv_dx[axis];
    a.dt_factor = b.dt_factor;
    const int lo = axis == 0 ? 0 : 3, hi = axis == 0 ? 1 : 2;   // Left/Right or Bottom/Top
    a.lo_u = D.bc[lo][0];
    a.lo_v = D.bc[lo][1];
    a.hi_u = D.bc[hi][0];
    a.hi_v = D.bc[hi][1];
    a.cfl_dx = D.cfl_dx;
    a.cfl_dy = D.cfl_dy;
    a.x_slots = D.x_slots;
    a.x_inv_slots = D.x_inv_slots;
    return a;
}

template <class T, int FLUX, int PROJ, int EOS, int TILE>
__global__ void __launch_bounds__(TILE) k_batch_x(BatchArgs<T> b, const BatchItemX* __restrict__ items, int nitems)
{
    __shared__ SchemeLds<T, FLUX, PROJ, TILE, 1> sm;
    for (int it = blockIdx.x; it < nitems; it += gridDim.x) {
        const BatchItemX item = items[it];
        const DeviceState* st = b.states + item.domain;
        if (!st->active) continue;   // the same for the whole block
        const SweepArgs<T> a = batch_domain_args(b, item.domain, 0);
        sweep_x_tile<T, FLUX, PROJ, EOS, kBatchDxMode<T>, TILE>(
                a, [&](double& dt) { dt = st->current_dt; return true; }, item.row, item.slot, sm);
        __syncthreads();             // the next item reuses the LDS
    }
}

// One block per X item (the launch configuration the autotuner usually picks): no item loop,
// so the tile body keeps the single-domain kernel's register budget. TILE cells per tile,
// CPT cells per thread.
template <class T, int FLUX, int PROJ, int EOS, bool FOLD, int TILE, int CPT = 1>
__global__ void __launch_bounds__(TILE / CPT) k_batch_x1(BatchArgs<T> b, const BatchItemX* __restrict__ items)
{
    __shared__ SchemeLds<T, FLUX, PROJ, TILE, 1> sm;
    const BatchItemX item = items[xcd_block(blockIdx.x, gridDim.x)];
    const SweepArgs<T> a = batch_domain_args<FOLD>(b, item.domain, 0);
    // a domain's first tile writes its step
    sweep_x_tile<T, FLUX, PROJ, EOS, kBatchDxMode<T>, TILE, CPT>(
            a, [&](double& dt) { return begin_sweep<FOLD>(a, item.row == 0 && item.slot == 0, dt); }, item.row,
            item.slot, sm);
}

// One block per Y tile.
template <class T, int FLUX, int PROJ, int EOS, bool FOLD>
__global__ void __launch_bounds__(YTile<T>::threads) k_batch_y_tile(BatchArgs<T> b, const BatchItemY* __restrict__ items)
{
    using Y = YTile<T>;
    __shared__ SchemeLds<T, FLUX, PROJ, Y::cols * Y::rows, Y::cols> sm;
    const BatchItemY item = items[xcd_block(blockIdx.x, gridDim.x)];
    const SweepArgs<T> a = batch_domain_args<FOLD>(b, item.domain, 1);
    sweep_y_tile<T, FLUX, PROJ, EOS, kBatchDxMode<T>, Y::cols, Y::rows, Y::threads>(
            a, [&](double& dt) { return begin_sweep<FOLD>(a, item.x0 == 0 && item.y0 == 0, dt); }, item.x0, item.y0, sm);
}

template <class T, int FLUX, int PROJ, int EOS, bool STALE>
__global__ void __launch_bounds__(kYBlock) __attribute__((amdgpu_waves_per_eu(3)))
        k_batch_y(BatchArgs<T> b, const BatchItemY* __restrict__ items, int nitems)
{
    __shared__ MarchBlockLds<T, FLUX, PROJ> lds;
    const int lane = threadIdx.x & 63;
    const int nwaves = (gridDim.x * blockDim.x) >> 6;
    // the item index is uniform across the wave: keep it (and what is loaded through it) scalar
    const int first = __builtin_amdgcn_readfirstlane((int) ((blockIdx.x * blockDim.x + threadIdx.x) >> 6));
    for (int it = first; it < nitems; it += nwaves) {
        const BatchItemY item = items[it];
        const DeviceState* st = b.states + item.domain;
        if (!st->active) continue;   // the same for the whole wave
        const SweepArgs<T> a = batch_domain_args(b, item.domain, 1);
        const int x = item.x0 + lane;
        sweep_y_run<T, FLUX, PROJ, EOS, kBatchDxMode<T>, STALE>(a, (T) (st->current_dt * b.dt_factor), x,
                                                                item.y0, item.y1, lds);
    }
}

// One wave per Y item (the launch configuration the autotuner usually picks): no item loop, so
// the run body keeps the single-domain kernel's register budget. The work list is sorted by run
// length and otherwise keeps each domain's runs in column order, so a block's 4 waves are mostly
// adjacent columns of one run: when all 4 waves have active items of the same row count, the
// block marches them with the block barrier of sweep_y_run (same trip count for every wave),
// which keeps their accesses of a row together in DRAM.
template <class T, int FLUX, int PROJ, int EOS, bool STALE>
__global__ void __launch_bounds__(kYBlock) __attribute__((amdgpu_waves_per_eu(PROJ == 2 ? kYWaves : kYWavesFirstOrder)))
        k_batch_y1(BatchArgs<T> b, const BatchItemY* __restrict__ items, int nitems)
{
    __shared__ MarchBlockLds<T, FLUX, PROJ> lds;
    const int lane = threadIdx.x & 63;
    const int it = __builtin_amdgcn_readfirstlane((int) ((blockIdx.x * blockDim.x + threadIdx.x) >> 6));
    BatchItemY item{0, 0, 0, 0};
    bool live = it < nitems;
    if (live) {
        item = items[it];
        live = b.states[item.domain].active != 0;
    }
    // in the march's LDS: 16 bytes more would leave room for a block less
    int* rows_of_wave = reinterpret_cast<int*>(&lds);
    if (lane == 0) rows_of_wave[threadIdx.x >> 6] = live ? item.y1 - item.y0 : -1;
    __syncthreads();
    bool sync = true;
#pragma unroll
    for (int w = 0; w < kYBlock / 64; w++) sync = sync && rows_of_wave[w] == rows_of_wave[0] && rows_of_wave[w] >= 0;
    __syncthreads();
    if (!live) return;   // the whole wave; never in a synchronised block
    const DeviceState* st = b.states + item.domain;
    const SweepArgs<T> a = batch_domain_args(b, item.domain, 1);
    const int x = item.x0 + lane;
    const T dt = (T) (st->current_dt * b.dt_factor);
    if (sync) {
        sweep_y_run<T, FLUX, PROJ, EOS, kBatchDxMode<T>, STALE, true>(a, dt, x, item.y0, item.y1, lds);
        return;
    }
    sweep_y_run<T, FLUX, PROJ, EOS, kBatchDxMode<T>, STALE>(a, dt, x, item.y0, item.y1, lds);
}

// X tiles covering a stream of `slots` slots (tiles of W outputs overlapping by 2R): the last
// real cell sits R slots before the end.
inline int64_t x_tiles(int64_t slots, int R, int W) { return (slots - 2 * R + W - 1) / W; }

inline unsigned grid_for(int64_t n, int block, int64_t max_blocks)
{
    int64_t g = (n + block - 1) / block;
    if (g > max_blocks) g = max_blocks;
    if (g < 1) g = 1;
    return (unsigned) g;
}

// How the tiles of a single domain add to its CFL accumulators (see reduce_cfl): up to 4096 waves without
// a look. Cycle with -> without it, us: 128^2 FP64 10.2 -> 9.9, 512^2 FP32 (2816 waves) 13.1 -> 12.0,
// 512^2 FP64 (5632) 17.8 -> 18.1, 1024^2 FP64 (22 016) 45.6 -> 50.5.
inline int reduce_mode(int reduce, int64_t blocks, int threads)
{
    return reduce && blocks * (threads / 64) <= 4096 ? REDUCE_UNSEEN : reduce;
}

// Blocks of `block` threads of `kernel` resident on the whole device at once.
inline int resident_blocks(const void* kernel, int block)
{
    int dev = 0, per_cu = 0, cus = 0;
    if (hipGetDevice(&dev) != hipSuccess) return 0;
    if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess) return 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kernel, block, 0) != hipSuccess) return 0;
    return per_cu * cus;
}

// SIMDs of the current device (4 per CU), looked up once per device.
inline int device_simds()
{
    static int cached[64] = {};
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 1024;
    if (cached[dev] == 0) {
        int cus = 0;
        if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus <= 0)
            return 1024;
        cached[dev] = 4 * cus;
    }
    return cached[dev];
}

// Rows per marching run of the Y sweep, for a domain of nx x ny cells whose stencil reads
// `halo` cells each side. A run of L output rows marches L + 2 halo rows (the warm-up), and a
// wave of 64 columns marches one run, so shorter runs give more waves for more redundant work.
// The rate of the march grows with the waves in flight as w / (w + SIMDs) (measured on MI355X
// from 512^2 to 8192^2: the best L is 8 rows at 512^2, 16 at 1024^2, 32 at 2048^2, 32-64 at
// 4096^2 and 64-128 at 8192^2), so L minimises (1 + 2 halo / L) (1 + SIMDs / waves) over the
// powers of two from 8 to 128, the larger L on a tie. The number of runs per column is a
// multiple of the XCD count when the column has at least that many, so that each XCD's
// contiguous share of the blocks (xcd_block) is a set of whole row bands.
inline int y_run_rows(int nx, int ny, int halo)
{
    if (ny <= 8) return ny > 0 ? ny : 1;
    const double simds = (double) device_simds();
    const double groups = (double) ((nx + 63) / 64);
    int best = ny;
    double best_cost = 0;
    for (int L = 8; L <= 128; L *= 2) {
        int nseg = (ny + L - 1) / L;
        if (nseg >= kXcds) nseg = (nseg + kXcds - 1) / kXcds * kXcds;
        const int len = (ny + nseg - 1) / nseg;
        nseg = (ny + len - 1) / len;
        const double cost = (1.0 + 2.0 * halo / len) * (1.0 + simds / (groups * nseg));
        if (L == 8 || cost <= best_cost * (1.0 + 1e-3)) {
            best = len;
            best_cost = cost;
        }
    }
    return best;
}

inline void check_launch(const char* what)
{
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) throw std::runtime_error(std::string(what) + ": " + hipGetErrorString(e));
}

template <class T, int F, int P, int E, int DXM>
void launch_variant(int axis, const SweepArgs<T>& a, hipStream_t s)
{
    constexpr int R = 2 + (F > 0 ? 1 : 0) + (P == 2 ? 1 : 0);
    if (axis == 0) {
        constexpr int W = XTile<T>::cells - 2 * R;
        SweepArgs<T> b = a;
        b.x_slots = a.nx + 2 * R;
        b.x_inv_slots = 1.0f / (float) b.x_slots;
        const int64_t tiles = x_tiles((int64_t) a.ny * b.x_slots, R, W);
        const dim3 grid((unsigned) tiles), block(XTile<T>::cells / XTile<T>::cpt);
        b.reduce = reduce_mode(a.reduce, tiles, XTile<T>::cells / XTile<T>::cpt);
        if (a.prev) k_sweep_x<T, F, P, E, DXM, true><<<grid, block, 0, s>>>(b);
        else k_sweep_x<T, F, P, E, DXM, false><<<grid, block, 0, s>>>(b);
        check_launch("sweep_x");
    } else {
        using Y = YTile<T>;
        // a run length that the caller gives is a march's
        if (a.seg_len <= 0 && y_takes_tiles(SweepVariant{F, P, E}, sizeof(T), a.nx, a.ny)) {
            constexpr int W = Y::rows - 2 * R;
            const int nc = (a.nx + Y::cols - 1) / Y::cols, nb = (a.ny + W - 1) / W;
            const dim3 grid((unsigned) (nc * nb)), block(Y::threads);
            SweepArgs<T> b = a;
            b.reduce = reduce_mode(a.reduce, (int64_t) nc * nb, Y::threads);
            if (a.prev) k_sweep_y_tile<T, F, P, E, DXM, true><<<grid, block, 0, s>>>(b, nc);
            else k_sweep_y_tile<T, F, P, E, DXM, false><<<grid, block, 0, s>>>(b, nc);
            check_launch("sweep_y_tile");
            return;
        }
        if (a.prev) throw std::logic_error("the march makes no time step");
        // Each block marches down a run of rows of its 256 columns (the warm-up is paid once
        // per run); blocks are numbered row band by row band (segment-major).
        const int ncolblk = (a.nx + kYBlock - 1) / kYBlock;
        SweepArgs<T> b = a;
        b.seg_len = a.seg_len > 0 ? std::min(a.seg_len, a.ny) : y_run_rows(a.nx, a.ny, R);
        const int nseg = (a.ny + b.seg_len - 1) / b.seg_len;
        const dim3 grid((unsigned) (ncolblk * nseg));
        if (a.stencil_width >= R)
            k_sweep_y<T, F, P, E, DXM, false><<<grid, dim3(kYBlock), 0, s>>>(b, ncolblk);
        else
            k_sweep_y<T, F, P, E, DXM, true><<<grid, dim3(kYBlock), 0, s>>>(b, ncolblk);
        check_launch("sweep_y");
    }
}

// The division by dx of the single-domain sweeps: a multiply for a power of two, else the
// reciprocal-corrected quotient in FP64 and the FP32-mixed division in FP32.
template <class T, int F, int P, int E>
void launch_dx_dispatch(int axis, const SweepArgs<T>& a, hipStream_t s)
{
    constexpr int other = sizeof(T) == 8 ? DX_RECIP : DX_DIVIDE;
    if (a.dx_mode == DX_POW2) launch_variant<T, F, P, E, DX_POW2>(axis, a, s);
    else launch_variant<T, F, P, E, other>(axis, a, s);
}

template <class T, int F, int P>
void launch_eos_dispatch(int axis, int eos, const SweepArgs<T>& a, hipStream_t s)
{
    if (eos == 0) launch_dx_dispatch<T, F, P, 0>(axis, a, s);
    else launch_dx_dispatch<T, F, P, 1>(axis, a, s);
}

template <class T, int F>
void launch_proj_dispatch(int axis, const SweepVariant& v, const SweepArgs<T>& a, hipStream_t s)
{
    if (v.proj == 2) launch_eos_dispatch<T, F, 2>(axis, v.eos, a, s);
    else launch_eos_dispatch<T, F, 1>(axis, v.eos, a, s);
}

template <class T, int F, int P, int E, int TILE>
void launch_batch_x(const BatchArgs<T>& b, const BatchItemX* items, int nitems, int grid, hipStream_t s)
{
    if (b.prev)
        k_batch_x1<T, F, P, E, true, TILE><<<dim3((unsigned) nitems), dim3(TILE), 0, s>>>(b, items);
    else if (grid >= nitems)
        k_batch_x1<T, F, P, E, false, TILE><<<dim3((unsigned) nitems), dim3(TILE), 0, s>>>(b, items);
    else
        k_batch_x<T, F, P, E, TILE><<<dim3((unsigned) grid), dim3(TILE), 0, s>>>(b, items, nitems);
}

// Two cells per thread: one block per tile of TILE cells (TILE / 2 threads).
template <class T, int F, int P, int E, int TILE>
void launch_batch_x2(const BatchArgs<T>& b, const BatchItemX* items, int nitems, hipStream_t s)
{
    if (b.prev) k_batch_x1<T, F, P, E, true, TILE, 2><<<dim3((unsigned) nitems), dim3(TILE / 2), 0, s>>>(b, items);
    else k_batch_x1<T, F, P, E, false, TILE, 2><<<dim3((unsigned) nitems), dim3(TILE / 2), 0, s>>>(b, items);
}

// X: `tile` cells per tile (128, 256 or 512), `cpt` cells per thread (1; or 2 for tiles of 256
// or 512 cells, one block per tile); `grid` blocks, or one per tile when grid >= nitems. Y: marching
// runs, or LDS tiles (`tile` 1).
template <class T, int F, int P, int E>
void launch_batch_variant(int axis, const BatchArgs<T>& b, const void* items, int nitems, int grid, int tile, int cpt,
                          hipStream_t s)
{
    if (nitems <= 0) return;
    if (axis == 0) {
        const auto* x_items = static_cast<const BatchItemX*>(items);
        if (cpt == 2) {
            if (tile == 512) launch_batch_x2<T, F, P, E, 512>(b, x_items, nitems, s);
            else if (tile == 256) launch_batch_x2<T, F, P, E, 256>(b, x_items, nitems, s);
            else throw std::invalid_argument("2 cells per thread needs X tiles of 256 or 512 cells");
        } else {
            switch (tile) {
            case 128: launch_batch_x<T, F, P, E, 128>(b, x_items, nitems, grid, s); break;
            case 512: launch_batch_x<T, F, P, E, 512>(b, x_items, nitems, grid, s); break;
            default: launch_batch_x<T, F, P, E, 256>(b, x_items, nitems, grid, s); break;
            }
        }
    } else {
        constexpr int R = 2 + (F > 0 ? 1 : 0) + (P == 2 ? 1 : 0);
        const auto* y_items = static_cast<const BatchItemY*>(items);
        const int waves_per_block = kYBlock / 64;
        if (tile == 1) {
            const dim3 grid((unsigned) nitems), block(YTile<T>::threads);
            if (b.prev) k_batch_y_tile<T, F, P, E, true><<<grid, block, 0, s>>>(b, y_items);
            else k_batch_y_tile<T, F, P, E, false><<<grid, block, 0, s>>>(b, y_items);
            check_launch("batch_y_tile");
            return;
        }
        if ((int64_t) grid * waves_per_block >= nitems) {
            const unsigned g1 = (unsigned) ((nitems + waves_per_block - 1) / waves_per_block);
            if (b.stencil_width >= R)
                k_batch_y1<T, F, P, E, false><<<dim3(g1), dim3(kYBlock), 0, s>>>(b, y_items, nitems);
            else
                k_batch_y1<T, F, P, E, true><<<dim3(g1), dim3(kYBlock), 0, s>>>(b, y_items, nitems);
        } else if (b.stencil_width >= R) {
            k_batch_y<T, F, P, E, false><<<dim3((unsigned) grid), dim3(kYBlock), 0, s>>>(b, y_items, nitems);
        } else {
            k_batch_y<T, F, P, E, true><<<dim3((unsigned) grid), dim3(kYBlock), 0, s>>>(b, y_items, nitems);
        }
    }
    check_launch(axis == 0 ? "batch_x" : "batch_y");
}

template <class T, int F, int P, int E>
int batch_variant_resident(int axis, int tile)
{
    if (axis != 0) return resident_blocks((const void*) k_batch_y<T, F, P, E, false>, kYBlock);
    switch (tile) {
    case 128: return resident_blocks((const void*) k_batch_x<T, F, P, E, 128>, 128);
    case 512: return resident_blocks((const void*) k_batch_x<T, F, P, E, 512>, 512);
    default: return resident_blocks((const void*) k_batch_x<T, F, P, E, 256>, 256);
    }
}

// Calls fn.template operator()<F, P, E>() for the variant's compile-time parameters.
template <class Fn>
auto with_variant(const SweepVariant& v, Fn&& fn)
{
    auto by_eos = [&](auto f, auto p) {
        return v.eos == 0 ? fn.template operator()<decltype(f)::value, decltype(p)::value, 0>()
                          : fn.template operator()<decltype(f)::value, decltype(p)::value, 1>();
    };
    auto by_proj = [&](auto f) {
        return v.proj == 2 ? by_eos(f, std::integral_constant<int, 2>{}) : by_eos(f, std::integral_constant<int, 1>{});
    };
    switch (v.flux) {
    case 0: return by_proj(std::integral_constant<int, 0>{});
    case 1: return by_proj(std::integral_constant<int, 1>{});
    case 2: return by_proj(std::integral_constant<int, 2>{});
    default: return by_proj(std::integral_constant<int, 3>{});
    }
}

}  // namespace sweep

template <class T>
void launch_sweep(int axis, const SweepVariant& v, const SweepArgs<T>& a, hipStream_t s)
{
    switch (v.flux) {
    case 0: sweep::launch_proj_dispatch<T, 0>(axis, v, a, s); break;
    case 1: sweep::launch_proj_dispatch<T, 1>(axis, v, a, s); break;
    case 2: sweep::launch_proj_dispatch<T, 2>(axis, v, a, s); break;
    default: sweep::launch_proj_dispatch<T, 3>(axis, v, a, s); break;
    }
}

template <class T>
void launch_batch_sweep(int axis, const SweepVariant& v, const BatchArgs<T>& b, const void* items, int nitems, int grid,
                        int tile, int cpt, hipStream_t s)
{
    sweep::with_variant(v, [&]<int F, int P, int E>() {
        sweep::launch_batch_variant<T, F, P, E>(axis, b, items, nitems, grid, tile, cpt, s);
        return 0;
    });
}

template <class T>
int batch_resident_blocks(int axis, const SweepVariant& v, int tile)
{
    return sweep::with_variant(v,
                               [&]<int F, int P, int E>() { return sweep::batch_variant_resident<T, F, P, E>(axis, tile); });
}

}  // namespace armon
