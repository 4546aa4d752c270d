// Fused engine, FP64 instantiation of the sweep kernels (sweep_kernels.hpp), plus the kernels of
// the time step and of what comes before the first cycle and after the last one.
#include "internal.hpp"
#include "sweep_kernels.hpp"

#include <cfloat>
#include <stdexcept>
#include <string>

namespace armon {

using namespace sweep;

namespace {

__global__ void k_time_step(const DeviceState* prev, DeviceState* st, TimeStepConfig c)
{
    write_step(st, next_step(prev, c));
}

// One wave per domain.
__global__ void __launch_bounds__(256) k_batch_time_step(const DeviceState* prev, DeviceState* states,
                                                         const TimeStepConfig* cfgs, int n)
{
    const int d = (blockIdx.x * blockDim.x + threadIdx.x) >> 6;
    if (d < n) write_step(states + d, next_step(prev + d, cfgs[d]));
}

__global__ void k_f2d(const float* in, double* out, int64_t n)
{
    for (int64_t k = (int64_t) blockIdx.x * blockDim.x + threadIdx.x; k < n; k += (int64_t) gridDim.x * blockDim.x)
        out[k] = (double) in[k];
}

__global__ void __launch_bounds__(64) k_clear(DeviceState* states)
{
    DeviceState& st = states[blockIdx.x];
    if (threadIdx.x < kDtSlots) st.dt_min[threadIdx.x].bits = kNoBound;
    if (threadIdx.x == 63) static_cast<StepState&>(st) = StepState{};
}

__global__ void __launch_bounds__(64) k_report(const DeviceState* states, int n, StepState* out)
{
    const int d = blockIdx.x * blockDim.x + threadIdx.x;
    if (d < n) out[d] = states[d];
}

// Whether element `i` of a domain is one of its real cells.
__device__ __forceinline__ bool real_cell(const BatchDomain& d, int64_t i)
{
    const int g = d.index_start % d.row_length;   // ghost layers: index_start = (row_length + 1) g
    const unsigned row = (unsigned) i / (unsigned) d.row_length, col = (unsigned) i - row * (unsigned) d.row_length;
    return row - (unsigned) g < (unsigned) d.ny && col - (unsigned) g < (unsigned) d.nx;
}

__device__ __forceinline__ void full_eos(int eos, double gamma, double rho, double u, double v, double E, double& p,
                                         double& c, double& g)
{
    if (eos == 0) perfect_gas<double>(gamma, rho, E, u, v, p, c, g);
    else bizarrium(rho, E, u, v, p, c, g);
}

// Both kernels: one element a thread. They are bound by memory (FP64: 12 words an element in begin).
__global__ void __launch_bounds__(256) k_begin(FieldArrays f, const BatchDomain* domains, int n, BatchDomain one,
                                               int64_t elements, DeviceState* states, int eos, double gamma)
{
    const int64_t e = (int64_t) blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t wave = (int64_t) blockIdx.x * blockDim.x + __builtin_amdgcn_readfirstlane((int) threadIdx.x);
    if (wave >= elements) return;
    const int which = n == 1 ? 0 : domain_of(domains, n, wave);
    const BatchDomain d = n == 1 ? one : domains[which];
    CflSpeeds speeds;
    if (e < elements) {
        const double rho = f.rho[e], u = f.u[e], v = f.v[e], E = f.E[e];
        double p, c, g;
        if (real_cell(d, e - d.offset)) {
            full_eos(eos, gamma, rho, u, v, E, p, c, g);
            if (f.g) {
                f.p[e] = p;
                f.c[e] = c;
                f.g[e] = g;
            }
            speeds.add(u, v, c);
        } else if (f.f32[0]) {
            p = f.p[e];
            c = f.c[e];
        }
        if (f.f32[0]) {
            f.f32[0][e] = f.f32[4][e] = (float) rho;
            f.f32[1][e] = f.f32[5][e] = (float) u;
            f.f32[2][e] = f.f32[6][e] = (float) v;
            f.f32[3][e] = f.f32[7][e] = (float) E;
            f.f32[8][e] = (float) p;
            f.f32[9][e] = (float) c;
        } else {
            f.other[0][e] = rho;
            f.other[1][e] = u;
            f.other[2][e] = v;
            f.other[3][e] = E;
        }
    }
    reduce_cfl(states + which, REDUCE, speeds.bound(d.cfl_dx, d.cfl_dy));
}

__global__ void __launch_bounds__(256) k_finish(FieldArrays f, const BatchDomain* domains, int n, BatchDomain one,
                                                int64_t elements, const DeviceState* states, int sweeps_per_cycle,
                                                int eos, double gamma)
{
    const int64_t e = (int64_t) blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t wave = (int64_t) blockIdx.x * blockDim.x + __builtin_amdgcn_readfirstlane((int) threadIdx.x);
    if (wave >= elements) return;
    const int which = n == 1 ? 0 : domain_of(domains, n, wave);
    const BatchDomain d = n == 1 ? one : domains[which];
    const int64_t sweeps = (int64_t) states[which].cycle * sweeps_per_cycle;
    if (sweeps == 0 || e >= elements) return;
    const bool second = sweeps & 1;   // the final state is in the second buffer, the last input in the first
    const bool real = real_cell(d, e - d.offset);
    double rho, u, v, E;              // the last sweep's input
    if (f.f32[0]) {
        float* const* in = second ? f.f32 : f.f32 + 4;
        float* const* out = second ? f.f32 + 4 : f.f32;
        if (real) {
            rho = (double) in[0][e];
            u = (double) in[1][e];
            v = (double) in[2][e];
            E = (double) in[3][e];
        }
        f.rho[e] = (double) out[0][e];
        f.u[e] = (double) out[1][e];
        f.v[e] = (double) out[2][e];
        f.E[e] = (double) out[3][e];
    } else if (second) {
        if (real) {
            rho = f.rho[e];
            u = f.u[e];
            v = f.v[e];
            E = f.E[e];
        }
        f.rho[e] = f.other[0][e];
        f.u[e] = f.other[1][e];
        f.v[e] = f.other[2][e];
        f.E[e] = f.other[3][e];
    } else if (real) {
        rho = f.other[0][e];
        u = f.other[1][e];
        v = f.other[2][e];
        E = f.other[3][e];
    }
    if (real) {
        double p, c, g;
        full_eos(eos, gamma, rho, u, v, E, p, c, g);
        f.p[e] = p;
        f.c[e] = c;
        f.g[e] = g;
    }
}

}  // namespace

template void launch_sweep<double>(int, const SweepVariant&, const SweepArgs<double>&, hipStream_t);
template void launch_batch_sweep<double>(int, const SweepVariant&, const BatchArgs<double>&, const void*, int, int, int,
                                       int, hipStream_t);
template int batch_resident_blocks<double>(int, const SweepVariant&, int);

int x_tile_outputs(const SweepVariant& v, int tile) { return tile - 2 * read_extent(v.flux, v.proj); }

bool y_takes_tiles(const YSweepWork& w, size_t element)
{
    const double slots = (double) w.slots, marched = (double) w.marched;
    if (slots <= (element == 8 ? 0.7 : 0.35) * marched) return true;
    return w.cells <= y_tile_max_cells(element) &&
           slots <= 0.85 * marched * (1.0 + (double) device_simds() / (double) w.waves);
}

bool y_takes_tiles(const SweepVariant& v, size_t element, int nx, int ny)
{
    YSweepWork w;
    w.add(v, nx, ny, y_run_rows(nx, ny, read_extent(v.flux, v.proj)), kYBlock);
    return y_takes_tiles(w, element);
}

void launch_time_step(const DeviceState* prev, DeviceState* st, const TimeStepConfig& c, hipStream_t s)
{
    k_time_step<<<1, 64, 0, s>>>(prev, st, c);
    check_launch("time_step");
}

void launch_batch_time_step(const DeviceState* prev, DeviceState* states, const TimeStepConfig* cfgs, int n,
                            hipStream_t s)
{
    k_batch_time_step<<<(unsigned) ((n + 3) / 4), 256, 0, s>>>(prev, states, cfgs, n);
    check_launch("batch_time_step");
}

static unsigned element_blocks(int64_t elements)
{
    const int64_t g = (elements + 255) / 256;
    if (g > INT32_MAX) throw std::runtime_error("too many elements for one launch");
    return (unsigned) g;
}

void launch_begin(const FieldArrays& f, const BatchDomain* domains, int n, const BatchDomain& one, int64_t elements,
                  DeviceState* states, int eos, double gamma, hipStream_t s)
{
    k_begin<<<element_blocks(elements), 256, 0, s>>>(f, domains, n, one, elements, states, eos, gamma);
    check_launch("begin");
}

void launch_finish(const FieldArrays& f, const BatchDomain* domains, int n, const BatchDomain& one, int64_t elements,
                   const DeviceState* states, int sweeps_per_cycle, int eos, double gamma, hipStream_t s)
{
    k_finish<<<element_blocks(elements), 256, 0, s>>>(f, domains, n, one, elements, states, sweeps_per_cycle, eos,
                                                      gamma);
    check_launch("finish");
}

void launch_clear(DeviceState* states, int n, hipStream_t s)
{
    k_clear<<<(unsigned) n, 64, 0, s>>>(states);
    check_launch("clear");
}

void launch_report(const DeviceState* states, int n, StepState* out, hipStream_t s)
{
    k_report<<<(unsigned) ((n + 63) / 64), 64, 0, s>>>(states, n, out);
    check_launch("report");
}

StateReports::~StateReports()
{
    for (hipEvent_t e : arrived_)
        if (e) (void) hipEventDestroy(e);
    if (host_) (void) hipHostFree(host_);
}

void StateReports::post(const DeviceState* states, int k, hipStream_t s)
{
    if (!host_) {
        for (hipEvent_t& e : arrived_)
            if (!e) hip_check(hipEventCreateWithFlags(&e, hipEventDisableTiming), "hipEventCreate");
        void* p = nullptr;
        hip_check(hipHostMalloc(&p, 2 * sizeof(StepState) * (size_t) n_, hipHostMallocDefault), "hipHostMalloc(reports)");
        host_ = static_cast<StepState*>(p);
    }
    launch_report(states, n_, host_ + (k & 1) * (size_t) n_, s);
    hip_check(hipEventRecord(arrived_[k & 1], s), "hipEventRecord");
}

const StepState* StateReports::wait(int k)
{
    hip_check(hipEventSynchronize(arrived_[k & 1]), "hipEventSynchronize");
    return host_ + (k & 1) * (size_t) n_;
}

void launch_convert_f2d(const float* in, double* out, int64_t n, hipStream_t s)
{
    k_f2d<<<grid_for(n, 256, 8192), 256, 0, s>>>(in, out, n);
    check_launch("convert_f2d");
}

}  // namespace armon
