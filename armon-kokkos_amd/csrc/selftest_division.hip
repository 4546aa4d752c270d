// Self-tests of the shortened FP64 sequences of device_math.hpp, on the device: the
// shared-divisor quotients (with_divisor: three quotients over one divisor against the
// compiler's IEEE a / b) and the square root (sqrt_t<double> against the compiler's
// __builtin_sqrt), bit for bit, for operands drawn over the whole FP64 range (subnormals, zeros
// of both signs, infinities, NaNs), around the bounds of the ranges where the short sequences
// are taken, and in the range of physical states. Built as its own library,
// libarmon_selftest.so; the solver library does not contain it.
#include <hip/hip_runtime.h>

#include <cstdint>

#include "device_math.hpp"

namespace {

__device__ uint64_t splitmix64(uint64_t& s)
{
    uint64_t z = (s += 0x9E3779B97F4A7C15ull);
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    return z ^ (z >> 31);
}

__device__ double from_bits(uint64_t b) { return __builtin_bit_cast(double, b); }
__device__ uint64_t to_bits(double d) { return __builtin_bit_cast(uint64_t, d); }

// A double with unbiased exponent e (normal range) or biased exponent 0 (subnormal) when e is
// below -1022, a random mantissa (or zero, one time in eight) and the given sign.
__device__ double with_exponent(uint64_t& s, int e, bool negative)
{
    const uint64_t r = splitmix64(s);
    const uint64_t mant = (r & 7) == 0 ? 0 : (r >> 12);
    const uint64_t biased = e < -1022 ? 0 : (uint64_t) (e + 1023);
    return from_bits(((uint64_t) negative << 63) | (biased << 52) | (mant & 0xFFFFFFFFFFFFFull));
}

__device__ double special(uint64_t r)
{
    switch (r % 8) {
    case 0: return 0.0;
    case 1: return -0.0;
    case 2: return __builtin_huge_val();
    case 3: return -__builtin_huge_val();
    case 4: return __builtin_nan("");
    case 5: return from_bits(1);                       // smallest subnormal
    case 6: return from_bits(0x000FFFFFFFFFFFFFull);   // largest subnormal
    default: return from_bits(0x7FEFFFFFFFFFFFFFull);  // largest finite
    }
}

__device__ double draw_divisor(uint64_t& s)
{
    const uint64_t r = splitmix64(s);
    const bool neg = (r >> 8) & 1;
    const int span = (int) ((r >> 16) & 0xFFFF);
    switch (r & 7) {
    case 0: return with_exponent(s, -1075 + span % 2099, neg);   // every exponent, both signs
    case 1: return with_exponent(s, -210 + span % 421, false);   // around the divisor range
    case 2: {                                                     // at its bounds
        const int e[6] = {-201, -200, -199, 199, 200, 201};
        return with_exponent(s, e[span % 6], false);
    }
    case 3: return special(r >> 20);
    default: return with_exponent(s, -20 + span % 41, false);   // physical states
    }
}

__device__ double draw_numerator(uint64_t& s)
{
    const uint64_t r = splitmix64(s);
    const bool neg = (r >> 8) & 1;
    const int span = (int) ((r >> 16) & 0xFFFF);
    switch (r & 7) {
    case 0: return with_exponent(s, -1075 + span % 2099, neg);
    case 1: return with_exponent(s, -610 + span % 921, neg);     // around the numerator range
    case 2: {
        const int e[6] = {-601, -600, -599, 299, 300, 301};
        return with_exponent(s, e[span % 6], neg);
    }
    case 3: return neg ? -0.0 : 0.0;
    case 4: return special(r >> 20);
    default: return with_exponent(s, -30 + span % 61, neg);
    }
}

// counts[0]: quotients whose bits differ from a / b; counts[1]: triples that took the shared
// sequence (every operand inside its range); first[0..3]: b, a0, a1, a2 of a differing triple.
__global__ void __launch_bounds__(256) k_check_shared_divisor(uint64_t seed, int64_t n, unsigned long long* counts,
                                                               double* first, int* first_taken)
{
    unsigned long long bad = 0, fast = 0;
    for (int64_t i = (int64_t) blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t) gridDim.x * blockDim.x) {
        uint64_t s = seed ^ ((uint64_t) i * 0xD1B54A32D192ED03ull);
        const double b = draw_divisor(s);
        const double a0 = draw_numerator(s), a1 = draw_numerator(s), a2 = draw_numerator(s);
        double q0, q1, q2;
        armon::with_divisor(b, [&](auto div) {
            q0 = div(a0);
            q1 = div(a1);
            q2 = div(a2);
        });
        const int miss = (int) (to_bits(q0) != to_bits(a0 / b)) + (int) (to_bits(q1) != to_bits(a1 / b))
                + (int) (to_bits(q2) != to_bits(a2 / b));
        bad += (unsigned long long) miss;
        fast += (unsigned long long) (armon::shared_divisor_ok(b) & armon::shared_numerator_ok(a0)
                                      & armon::shared_numerator_ok(a1) & armon::shared_numerator_ok(a2));
        if (miss && atomicCAS(first_taken, 0, 1) == 0) {
            first[0] = b;
            first[1] = a0;
            first[2] = a1;
            first[3] = a2;
        }
    }
    if (bad) atomicAdd(&counts[0], bad);
    if (fast) atomicAdd(&counts[1], fast);
}

__device__ double draw_radicand(uint64_t& s)
{
    const uint64_t r = splitmix64(s);
    const bool neg = ((r >> 8) & 15) == 0;
    const int span = (int) ((r >> 16) & 0xFFFF);
    switch (r & 7) {
    case 0: return with_exponent(s, -1075 + span % 2099, neg);   // every exponent
    case 1: return with_exponent(s, -777 + span % 21, false);    // around 2^-767
    case 2: return special(r >> 20);
    case 3: return with_exponent(s, 1013 + span % 11, false);    // near the largest finite
    default: return with_exponent(s, -30 + span % 61, false);    // physical states
    }
}

// counts[0]: roots whose bits differ from __builtin_sqrt; counts[1]: operands that took the
// short sequence; first[0]: the operand of a differing root.
__global__ void __launch_bounds__(256) k_check_sqrt(uint64_t seed, int64_t n, unsigned long long* counts,
                                                     double* first, int* first_taken)
{
    unsigned long long bad = 0, fast = 0;
    for (int64_t i = (int64_t) blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t) gridDim.x * blockDim.x) {
        uint64_t s = seed ^ ((uint64_t) i * 0xD1B54A32D192ED03ull);
        const double x = draw_radicand(s);
        const int miss = (int) (to_bits(armon::sqrt_t<double>(x)) != to_bits(__builtin_sqrt(x)));
        bad += (unsigned long long) miss;
        fast += (unsigned long long) armon::sqrt_core_ok(x);
        if (miss && atomicCAS(first_taken, 0, 1) == 0) first[0] = x;
    }
    if (bad) atomicAdd(&counts[0], bad);
    if (fast) atomicAdd(&counts[1], fast);
}

// Values as the sweeps' stages meet them and as they should not: mostly physical states, one in
// eight a difference that vanishes or nearly does, one in sixteen anything at all.
__device__ double draw_value(uint64_t& s, bool positive)
{
    const uint64_t r = splitmix64(s);
    const bool neg = !positive && ((r >> 8) & 1);
    const int span = (int) ((r >> 16) & 0xFFFF);
    switch (r & 15) {
    case 0: return (r >> 40) & 1 ? special(r >> 20) : with_exponent(s, -1075 + span % 2099, (r >> 41) & 1);
    case 1: return neg ? -0.0 : 0.0;
    case 2: return with_exponent(s, -1075 + span % 1000, neg);
    default: return with_exponent(s, -12 + span % 25, neg);
    }
}

__device__ bool same(double a, double b) { return to_bits(a) == to_bits(b) || (!(a == a) && !(b == b)); }

// The fused sweeps' form of each stage against the plain one (godunov, gad_correct with every
// limiter, the two divisions of cell_update, advection_flux_2 for both donors, projection in both
// ways of dividing by dx, both equations of state). counts[0]: results that differ; counts[1]: samples whose
// shared reciprocals all served; first[0]: the index of a differing sample, first[1]: the stages.
__global__ void __launch_bounds__(256) k_check_stages(uint64_t seed, int64_t n, unsigned long long* counts,
                                                       double* first, int* first_taken)
{
    using namespace armon;
    unsigned long long bad = 0, fast = 0;
    for (int64_t i = (int64_t) blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t) gridDim.x * blockDim.x) {
        uint64_t s = seed ^ ((uint64_t) i * 0xD1B54A32D192ED03ull);
        const bool pow2 = splitmix64(s) & 1;
        const double dx = pow2 ? with_exponent(s, -12, false) : 1.0 / (double) (3 + splitmix64(s) % 10000);
        const double dx2 = pow2 ? 0x1p-12 : dx, inv_dx = 1.0 / dx2;
        const double dt = (splitmix64(s) & 63) == 0 ? draw_value(s, true) : dx2 * 0x1p-3 * with_exponent(s, 0, false);
        double rho[4], c[4], u[4], v[4], E[4], us[4];
        for (int k = 0; k < 4; k++) {
            rho[k] = draw_value(s, true);
            c[k] = draw_value(s, true);
            u[k] = draw_value(s, false);
            v[k] = draw_value(s, false);
            E[k] = draw_value(s, true);
            us[k] = k && (splitmix64(s) & 7) == 0 ? us[k - 1] : draw_value(s, false);
        }
        int wrong = 0;
        bool shared = true;
        {   // faces: p stands in E's place
            double a, b, x, y;
            godunov<double, false>(rho[1], rho[0], c[1], c[0], u[1], u[0], E[1], E[0], a, b);
            face_godunov<double>(rho[0] * c[0], rho[1] * c[1], u[0], u[1], E[0], E[1], x, y);
            wrong |= (same(a, x) && same(b, y) ? 0 : 1);
            auto gad = [&]<int L>() {
                gad_correct<L, double>(dt, dx2, rho[0], rho[1], c[0], c[1], u[0], u[1], E[0], E[1], us[0], v[0], us[1],
                                       v[1], us[2], v[2], a, b);
                const double th = gad_theta<double>(dt, rho[0] * dx2, rho[1] * dx2, rho[0] * c[0], rho[1] * c[1]);
                x = gad_star<L, double>(th, us[1], us[1] - u[0], us[2] - u[1], u[1] - us[1], u[0] - us[0]);
                y = gad_star<L, double>(th, v[1], v[1] - E[0], v[2] - E[1], E[1] - v[1], E[0] - v[0]);
                wrong |= (same(a, x) && same(b, y) ? 0 : 2);
            };
            gad.template operator()<0>();
            gad.template operator()<1>();
            gad.template operator()<2>();
        }
        {   // update: rho and dt / dm
            const double y = shared_recip<double>(rho[0]), dm = rho[0] * dx2;
            double q = pow2 ? mass_quotient<DX_POW2>(dt, dm, y, inv_dx) : mass_quotient<DX_RECIP>(dt, dm, y, inv_dx);
            const int no = unusable(q);
            if (no) q = dt / dm;
            wrong |= (same(q, dt / dm) ? 0 : 4);
            const double L = dx2 + dt * (us[1] - us[0]), yL = shared_recip<double>(L);
            double r = quot<double>(dm, L, yL);
            if (no | unusable(yL)) r = dm / L;
            shared &= !(no | unusable(yL));
            wrong |= (same(r, dm / L) ? 0 : 8);
            // the march's way out of the shared reciprocal, which knows the mass and not its density
            double m = quot<double>(dm, L, yL);
            if (unusable(m) | too_small(dm)) m = dm / L;
            wrong |= (same(m, dm / L) ? 0 : 8);
            double p0, c0, g0, p1, c1;
            perfect_gas<double>(1.4, rho[0], E[0], u[0], v[0], p0, c0, g0);
            perfect_gas_pc<double>(1.4, rho[0], E[0], u[0], v[0], y, p1, c1);
            wrong |= (same(p0, p1) && same(c0, c1) ? 0 : 16);
            // Bizarrium's densities lie about 1e4
            const double heavy = (splitmix64(s) & 7) ? 1e4 * with_exponent(s, 0, false) : rho[1];
            const double eh = (splitmix64(s) & 3) ? 1e6 * with_exponent(s, 0, false) : E[1];
            bizarrium(heavy, eh, u[1], v[1], p0, c0, g0);
            bizarrium_pc(heavy, eh, u[1], v[1], shared_recip<double>(heavy), p1, c1);
            wrong |= (same(p0, p1) && same(c0, c1) ? 0 : 128);
        }
        {   // advection from the donor 1 with neighbours 0 and 2; its faces carry us[1] and us[2]
            double L[3], yS[4], q[3][4];
            for (int k = 0; k < 3; k++) {
                L[k] = dx2 + dt * (us[k + 1] - us[k]);
                q[k][0] = rho[k];
                q[k][1] = rho[k] * u[k];
                q[k][2] = rho[k] * v[k];
                q[k][3] = rho[k] * E[k];
            }
            for (int k = 1; k < 3; k++) yS[k] = shared_recip<double>(L[k] + L[k - 1]);
            for (int up = 0; up < 2; up++) {
                // up: the face above the donor (u* > 0 there), else the face below it
                const double disp = dt * us[up ? 2 : 1];
                if (up ? !(disp > 0) : disp > 0) continue;
                const double plain = up ? -(dx2 - dt * us[1]) : dx2 + dt * us[2];
                const double Dx = donor_length<double>(dx2, dt, disp, us[1], us[2]);
                double a[4], f[4];
                advection_flux_2<double>(dx2, dt, disp, plain, us[0], us[1], us[2], us[3], rho[0], rho[1], rho[2],
                                         u[0], u[1], u[2], v[0], v[1], v[2], E[0], E[1], E[2], a[0], a[1], a[2], a[3]);
                double r_m, r_p, slope[4];
                slope_ratios<double>(L[1], L[1] + L[0], yS[1], L[2] + L[1], yS[2], r_m, r_p);
                for (int k = 0; k < 4; k++)
                    slope[k] = slope_minmod_t<double>(r_p * (q[2][k] - q[1][k]), r_m * (q[1][k] - q[0][k]));
                donor_flux_2<double>(disp, length_factor<double>(Dx, L[1], shared_recip<double>(L[1])), q[1], slope,
                                     f);
                for (int k = 0; k < 4; k++) wrong |= (same(a[k], f[k]) ? 0 : 32);
            }
        }
        {   // projection, from fluxes of any kind
            const double f[4] = {draw_value(s, false), draw_value(s, false), draw_value(s, false), draw_value(s, false)};
            const double fp[4] = {draw_value(s, false), (splitmix64(s) & 3) ? f[1] : draw_value(s, false),
                                  draw_value(s, false), draw_value(s, false)};
            double a[4] = {rho[0], u[0], v[0], E[0]}, b[4] = {rho[0], u[0], v[0], E[0]};
            const double L = dx2 + dt * (us[1] - us[0]);
            if (pow2) {
                projection<DX_POW2, double, false>(dx2, inv_dx, dt, us[0], us[1], f[0], fp[0], f[1], fp[1], f[2], fp[2],
                                                   f[3], fp[3], a[0], a[1], a[2], a[3]);
                project<DX_POW2, double>(dx2, inv_dx, L, f, fp, b[0], b[1], b[2], b[3]);
            } else {
                projection<DX_RECIP, double, false>(dx2, inv_dx, dt, us[0], us[1], f[0], fp[0], f[1], fp[1], f[2],
                                                    fp[2], f[3], fp[3], a[0], a[1], a[2], a[3]);
                project<DX_RECIP, double>(dx2, inv_dx, L, f, fp, b[0], b[1], b[2], b[3]);
            }
            for (int k = 0; k < 4; k++) wrong |= (same(a[k], b[k]) ? 0 : 64);
        }
        bad += (unsigned long long) (wrong != 0);
        fast += (unsigned long long) shared;
        if (wrong && atomicCAS(first_taken, 0, 1) == 0) {
            first[0] = (double) i;
            first[1] = (double) wrong;
        }
    }
    if (bad) atomicAdd(&counts[0], bad);
    if (fast) atomicAdd(&counts[1], fast);
}

using CheckKernel = void (*)(uint64_t, int64_t, unsigned long long*, double*, int*);

// Runs one check kernel over n samples and copies its two counts and, when a sample failed,
// its nfirst operands back. Returns 0, or the HIP error code.
int run_check(CheckKernel kernel, uint64_t seed, int64_t n, uint64_t* mismatches, uint64_t* taken_short,
              double* first_bad, int nfirst)
{
    unsigned long long* counts = nullptr;
    double* first = nullptr;
    int* taken = nullptr;
    hipError_t e = hipMalloc((void**) &counts, 2 * sizeof(unsigned long long));
    if (e == hipSuccess) e = hipMalloc((void**) &first, 4 * sizeof(double));
    if (e == hipSuccess) e = hipMalloc((void**) &taken, sizeof(int));
    if (e == hipSuccess) e = hipMemset(counts, 0, 2 * sizeof(unsigned long long));
    if (e == hipSuccess) e = hipMemset(taken, 0, sizeof(int));
    if (e == hipSuccess) {
        hipLaunchKernelGGL(kernel, dim3(2048), dim3(256), 0, 0, seed, n, counts, first, taken);
        e = hipGetLastError();
    }
    if (e == hipSuccess) e = hipDeviceSynchronize();
    unsigned long long h[2] = {0, 0};
    int t = 0;
    if (e == hipSuccess) e = hipMemcpy(h, counts, sizeof(h), hipMemcpyDeviceToHost);
    if (e == hipSuccess) e = hipMemcpy(&t, taken, sizeof(int), hipMemcpyDeviceToHost);
    if (e == hipSuccess && t) e = hipMemcpy(first_bad, first, nfirst * sizeof(double), hipMemcpyDeviceToHost);
    if (e == hipSuccess) {
        *mismatches = h[0];
        *taken_short = h[1];
    }
    (void) hipFree(counts);
    (void) hipFree(first);
    (void) hipFree(taken);
    return (int) e;
}

}  // namespace

// Checks n triples drawn from seed. mismatches: quotients that differ from a / b; shared:
// triples that took the shared sequence; first_bad: b, a0, a1, a2 of one differing triple
// (untouched when none differs). Returns 0, or the HIP error code.
extern "C" __attribute__((visibility("default"))) int armon_selftest_shared_divisor(
        uint64_t seed, int64_t n, uint64_t* mismatches, uint64_t* shared, double* first_bad)
{
    return run_check(k_check_shared_divisor, seed, n, mismatches, shared, first_bad, 4);
}

// Checks n square roots drawn from seed. mismatches: roots that differ from __builtin_sqrt;
// fast: operands that took the short sequence; first_bad: the operand of one differing root
// (untouched when none differs). Returns 0, or the HIP error code.
extern "C" __attribute__((visibility("default"))) int armon_selftest_sqrt(uint64_t seed, int64_t n,
                                                                          uint64_t* mismatches, uint64_t* fast,
                                                                          double* first_bad)
{
    return run_check(k_check_sqrt, seed, n, mismatches, fast, first_bad, 1);
}

// Checks n samples of the sweeps' stages drawn from seed. mismatches: samples with a result whose
// bits differ from the plain form's; shared: samples whose shared reciprocals served; first_bad: the
// index of one differing sample and the stages that differ (1 Godunov, 2 GAD, 4 dt / dm, 8 dm / L,
// 16 EOS, 32 advection, 64 projection, 128 Bizarrium's EOS). Returns 0, or the HIP error code.
extern "C" __attribute__((visibility("default"))) int armon_selftest_stages(uint64_t seed, int64_t n,
                                                                            uint64_t* mismatches, uint64_t* shared,
                                                                            double* first_bad)
{
    return run_check(k_check_stages, seed, n, mismatches, shared, first_bad, 2);
}
