// Fused engine, FP64 instantiation of the sweep kernels (sweep_kernels.hpp), plus the
// device time step, the CFL reduction of a whole state, the EOS of a whole state and the
// FP32 <-> FP64 conversions used by the FP32-mixed form.
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

__global__ void k_reset_min(DeviceState* st) { st->dt_min[threadIdx.x].bits = kNoBound; }

template <class T>
__global__ void __launch_bounds__(256) k_cfl_real(DeviceState* st, const T* u, const T* v, const T* c, int nx, int ny,
                                                  int row_length, int index_start, double cfl_dx, double cfl_dy)
{
    double local = DBL_MAX;
    const int64_t total = (int64_t) nx * ny;
    for (int64_t k = (int64_t) blockIdx.x * blockDim.x + threadIdx.x; k < total; k += (int64_t) gridDim.x * blockDim.x) {
        const int j = (int) (k / nx), i = (int) (k - (int64_t) j * nx);
        const int idx = index_start + j * row_length + i;
        local = kmin(local, cfl_cell<double>(cfl_dx, cfl_dy, (double) u[idx], (double) v[idx], (double) c[idx], 1.0));
    }
    reduce_cfl(st, local);
}

__global__ void k_d2f(const double* in, float* out, int64_t n)
{
    for (int64_t k = (int64_t) blockIdx.x * blockDim.x + threadIdx.x; k < n; k += (int64_t) gridDim.x * blockDim.x)
        out[k] = (float) in[k];
}

__global__ void k_f2d(const float* in, double* out, int64_t n)
{
    for (int64_t k = (int64_t) blockIdx.x * blockDim.x + threadIdx.x; k < n; k += (int64_t) gridDim.x * blockDim.x)
        out[k] = (double) in[k];
}

template <class T>
__global__ void __launch_bounds__(256) k_eos_real(const T* rho, const T* u, const T* v, const T* E, double* p,
                                                  double* c, double* g, int eos, double gamma, int nx, int ny,
                                                  int row_length, int index_start)
{
    const int64_t total = (int64_t) nx * ny;
    for (int64_t k = (int64_t) blockIdx.x * blockDim.x + threadIdx.x; k < total; k += (int64_t) gridDim.x * blockDim.x) {
        const int j = (int) (k / nx), i = (int) (k - (int64_t) j * nx);
        const int idx = index_start + j * row_length + i;
        double pd, cd, gd;
        if (eos == 0) perfect_gas<double>(gamma, (double) rho[idx], (double) E[idx], (double) u[idx], (double) v[idx], pd, cd, gd);
        else bizarrium((double) rho[idx], (double) E[idx], (double) u[idx], (double) v[idx], pd, cd, gd);
        p[idx] = pd;
        c[idx] = cd;
        g[idx] = gd;
    }
}

}  // namespace

template void launch_sweep<double>(int, const SweepVariant&, const SweepArgs<double>&, hipStream_t);
template void launch_batch_sweep<double>(int, const SweepVariant&, const BatchArgs<double>&, const void*, int, int, int,
                                       int, hipStream_t);
template int batch_resident_blocks<double>(int, const SweepVariant&, int);

int x_tile_outputs(const SweepVariant& v, int tile) { return tile - 2 * read_extent(v.flux, v.proj); }

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

template <class T>
void launch_cfl_real(DeviceState* st, const T* u, const T* v, const T* c, int nx, int ny, int row_length,
                     int index_start, double cfl_dx, double cfl_dy, hipStream_t s)
{
    k_reset_min<<<1, kDtSlots, 0, s>>>(st);
    check_launch("cfl_reset");
    k_cfl_real<T><<<grid_for((int64_t) nx * ny, 256, 2048), 256, 0, s>>>(st, u, v, c, nx, ny, row_length, index_start,
                                                                         cfl_dx, cfl_dy);
    check_launch("cfl_real");
}

template void launch_cfl_real<double>(DeviceState*, const double*, const double*, const double*, int, int, int, int,
                                      double, double, hipStream_t);
template void launch_cfl_real<float>(DeviceState*, const float*, const float*, const float*, int, int, int, int,
                                     double, double, hipStream_t);

void launch_convert_d2f(const double* in, float* out, int64_t n, hipStream_t s)
{
    k_d2f<<<grid_for(n, 256, 8192), 256, 0, s>>>(in, out, n);
    check_launch("convert_d2f");
}

void launch_convert_f2d(const float* in, double* out, int64_t n, hipStream_t s)
{
    k_f2d<<<grid_for(n, 256, 8192), 256, 0, s>>>(in, out, n);
    check_launch("convert_f2d");
}

template <class T>
void launch_eos_real(const T* rho, const T* u, const T* v, const T* E, double* p, double* c, double* g, int eos,
                     double gamma, int nx, int ny, int row_length, int index_start, hipStream_t s)
{
    k_eos_real<T><<<grid_for((int64_t) nx * ny, 256, 8192), 256, 0, s>>>(rho, u, v, E, p, c, g, eos, gamma, nx, ny,
                                                                          row_length, index_start);
    check_launch("eos_real");
}

template void launch_eos_real<double>(const double*, const double*, const double*, const double*, double*, double*,
                                      double*, int, double, int, int, int, int, hipStream_t);
template void launch_eos_real<float>(const float*, const float*, const float*, const float*, double*, double*,
                                     double*, int, double, int, int, int, int, hipStream_t);

}  // namespace armon
