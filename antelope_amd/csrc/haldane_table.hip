// haldane_table.hip - set-up of a 2-band context on the device: the laser rows of
// every step and stage, the adaptive stepper's field table, and the k points.
//
// A context's own cost matters next to a short solve: the host took 0.12 us per
// table row (16 sines and cosines) and 10 ns per k point and then copied them
// over; 300 x 300 k, 86,168 rows: create 10.9 ms that way, 0.30 ms here.
#include <cstring>

#include "haldane_setup.hpp"

namespace sbe {
namespace {

using namespace dev;

__global__ __launch_bounds__(256) void haldane_table_kernel(const TableArgs a, double *__restrict__ tab,
                                                            float *__restrict__ tab32)
{
    table_row(a, static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x, tab, tab32);
}

// the initial state (blocks below nstate) and the laser rows (the others) of an FP64 solve in one
// launch: neither needs the other, and at 5 and 6 us each they would wait in turn (40 x 40 k points,
// 64 steps without allocation: 55.7 -> 52.2 us the call)
__global__ __launch_bounds__(256) void haldane_begin_kernel(const HaldaneArgs h, int fermi, double ef, int nstate,
                                                            const TableArgs a, double *__restrict__ tab)
{
    const int b = static_cast<int>(blockIdx.x);
    if (b < nstate) {
        const int64_t k = static_cast<int64_t>(b) * 256 + threadIdx.x;
        if (k < h.nk_stride) init_point<double>(h, k, h.nval, fermi, ef);
        return;
    }
    table_row(a, static_cast<int64_t>(b - nstate) * 256 + threadIdx.x, tab, nullptr);
}

// A - A(t_min) and the consistent dA/dt = -E at t_n, summed in pulse order
__global__ __launch_bounds__(256) void field_table_kernel(const TableArgs a, int64_t rows, double *__restrict__ at)
{
    const int64_t n = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (n >= rows) return;
    const double tn = a.atmin + a.dt * static_cast<double>(n);
    double s[2] = {0.0, 0.0}, g[2] = {0.0, 0.0};
    for (int p = 0; p < a.npulses; ++p) {
        double pa[3], pe[3];
        pulse_field(a.pulses[p], tn, true, pa, pe);
        for (int c = 0; c < 2; ++c) {
            s[c] += pa[c];
            g[c] -= pe[c];
        }
    }
    at[4 * n] = s[0] - a.A_at_min[0];
    at[4 * n + 1] = s[1] - a.A_at_min[1];
    at[4 * n + 2] = g[0];
    at[4 * n + 3] = g[1];
}

__global__ __launch_bounds__(256) void kgrid_kernel(const GridArgs g, int64_t k_begin, int64_t nk, int64_t nk_stride,
                                                    double *__restrict__ kpts)
{
    const int64_t o = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (o >= nk_stride) return;
    double k[3] = {0.0, 0.0, 0.0}, w = 0.0;
    if (o < nk) w = grid_point(g, k_begin + o, k);
    for (int c = 0; c < 3; ++c) kpts[c * nk_stride + o] = k[c];
    kpts[3 * nk_stride + o] = w;
}

unsigned blocks(int64_t n) { return static_cast<unsigned>((n + 255) / 256); }

}  // namespace

TableArgs table_args(const Laser &L, const Tableau &t, int nstage, double t1, const double va[3][2], const double vb[3][2])
{
    TableArgs a{};
    a.npulses = static_cast<int32_t>(L.pulses.size());
    for (size_t p = 0; p < L.pulses.size() && p < static_cast<size_t>(kMaxDevicePulses); ++p) a.pulses[p] = L.pulses[p];
    a.consistent = L.consistent ? 1 : 0;
    a.nstage = nstage;
    for (int j = 0; j < 3; ++j) a.A_at_min[j] = L.A_at_min[j];
    a.atmin = L.atmin;
    a.dt = L.dt;
    a.t1 = t1;
    for (int i = 0; i < 7; ++i) a.c[i] = t.c[i];
    std::memcpy(a.va, va, sizeof a.va);
    std::memcpy(a.vb, vb, sizeof a.vb);
    a.nsteps = L.nt;
    return a;
}

hipError_t launch_haldane_table(const TableArgs &a, double *tab, float *tab32, hipStream_t s)
{
    if (a.npulses > kMaxDevicePulses || a.nstage < 1 || a.nstage > 7) return hipErrorInvalidValue;
    if (a.nsteps <= 0) return hipSuccess;
    haldane_table_kernel<<<blocks(a.nsteps * a.nstage), 256, 0, s>>>(a, tab, tab32);
    return hipGetLastError();
}

hipError_t launch_haldane_begin(const HaldaneArgs &h, int init_type, double ef, const TableArgs &a, double *tab,
                                hipStream_t s)
{
    if (h.precision != SBE_PREC_FP64 || a.plain || a.npulses > kMaxDevicePulses || a.nstage < 1 || a.nstage > 7 ||
        a.nsteps < 1)
        return hipErrorInvalidValue;
    const unsigned nstate = blocks(h.nk_stride);
    haldane_begin_kernel<<<nstate + blocks(a.nsteps * a.nstage), 256, 0, s>>>(
        h, init_type == SBE_INIT_FERMI_DIRAC, ef, static_cast<int>(nstate), a, tab);
    return hipGetLastError();
}

hipError_t launch_field_table(const TableArgs &a, int64_t rows, double *at, hipStream_t s)
{
    if (a.npulses > kMaxDevicePulses) return hipErrorInvalidValue;
    field_table_kernel<<<blocks(rows), 256, 0, s>>>(a, rows, at);
    return hipGetLastError();
}

hipError_t launch_kgrid(const GridArgs &g, int64_t k_begin, int64_t nk, int64_t nk_stride, double *kpts, hipStream_t s)
{
    kgrid_kernel<<<blocks(nk_stride), 256, 0, s>>>(g, k_begin, nk, nk_stride, kpts);
    return hipGetLastError();
}

}  // namespace sbe
