// haldane_setup.hpp - set-up of a 2-band solve on the device, per point: the initial state of a k
// point and the laser row of a step and stage (haldane.hip, haldane_table.hip).
#pragma once

#include "haldane_dev.hpp"

namespace sbe {
namespace dev {

// Initial state (SBEs.h:284-364): rho_H = diag(occupations) at k, rho = U rho_H U^dag
// -> n = f0 + f1, s = (f1 - f0) dh(k). Padding points get a zero state.
template <typename R>
__device__ __forceinline__ void init_point(const HaldaneArgs &a, int64_t k, int nval, int fermi, double ef)
{
    const int64_t ks = a.nk_stride;
    R *st = static_cast<R *>(a.state);
    double n = 0, sx = 0, sy = 0, sz = 0;
    if (k < a.nk) {
        const double kx = a.kpts[k], ky = a.kpts[ks + k];
        double er[6], ei[6];
        for (int j = 0; j < 3; ++j) {
            sincos(kx * a.va[j][0] + ky * a.va[j][1], &ei[j], &er[j]);
            sincos(kx * a.vb[j][0] + ky * a.vb[j][1], &ei[j + 3], &er[j + 3]);
        }
        const Vec3<double> d = dvec<double>(er, ei, a.t1, a.c3, a.M0);
        const double d0 = a.c0 * (er[3] + er[4] + er[5]);
        const double dn = sqrt(d.x * d.x + d.y * d.y + d.z * d.z);
        double hx = 0, hy = 0, hz = -1;  // degenerate point: eigenbasis = orbital basis
        if (dn > 0) { hx = d.x / dn; hy = d.y / dn; hz = d.z / dn; }
        double f0, f1;
        if (fermi) {
            const double kT = 300.0 / 3.15775024804e5;
            f0 = 1.0 / (exp((d0 - dn - ef) / kT) + 1.0);
            f1 = 1.0 / (exp((d0 + dn - ef) / kT) + 1.0);
            const double sum = f0 + f1;
            f0 /= sum;
            f1 /= sum;
        } else {
            f0 = nval > 0 ? 1.0 : 0.0;
            f1 = nval > 1 ? 1.0 : 0.0;
        }
        n = f0 + f1;
        sx = (f1 - f0) * hx;
        sy = (f1 - f0) * hy;
        sz = (f1 - f0) * hz;
    }
    st[k] = static_cast<R>(n);
    st[ks + k] = static_cast<R>(sx);
    st[2 * ks + k] = static_cast<R>(sy);
    st[3 * ks + k] = static_cast<R>(sz);
    if (StateT<R>::kComp) {
        // compensation = -(low part) so that value = hi - c is exact in FP64
        st[4 * ks + k] = static_cast<R>(static_cast<double>(static_cast<R>(n)) - n);
        st[5 * ks + k] = static_cast<R>(static_cast<double>(static_cast<R>(sx)) - sx);
        st[6 * ks + k] = static_cast<R>(static_cast<double>(static_cast<R>(sy)) - sy);
        st[7 * ks + k] = static_cast<R>(static_cast<double>(static_cast<R>(sz)) - sz);
    }
}

// A(t) less its value at atmin, the sum of the pulses in order
__device__ __forceinline__ void field_at(const TableArgs &a, double t, double A[3])
{
    A[0] = A[1] = A[2] = 0.0;
    for (int p = 0; p < a.npulses; ++p) {
        double pa[3], pe[3];
        pulse_field(a.pulses[p], t, a.consistent != 0, pa, pe);
        for (int j = 0; j < 3; ++j) A[j] += pa[j];
    }
    for (int j = 0; j < 3; ++j) A[j] -= a.A_at_min[j];
}

// row i = (step - step0) nstage + stage of the laser table
__device__ __forceinline__ void table_row(const TableArgs &a, int64_t i, double *__restrict__ tab,
                                          float *__restrict__ tab32)
{
    if (i >= a.nsteps * a.nstage) return;
    const int64_t n = a.step0 + i / a.nstage;
    const int s = static_cast<int>(i % a.nstage);
    const double tn = a.atmin + a.dt * static_cast<double>(n);
    const double tn1 = a.atmin + a.dt * static_cast<double>(n + 1);
    // the stage at c = 1 is taken at t_{n+1} itself, so its row is the next step's first row bit
    // for bit (the step kernels carry it across steps)
    double A[3];
    field_at(a, a.c[s] == 1.0 ? tn1 : tn + a.c[s] * a.dt, A);
    if (a.plain) {
        tab[2 * i] = A[0];
        tab[2 * i + 1] = A[1];
        if (tab32) {
            tab32[2 * i] = static_cast<float>(A[0]);
            tab32[2 * i + 1] = static_cast<float>(A[1]);
        }
        return;
    }
    double *row = tab + i * 12;
    for (int j = 0; j < 3; ++j) {
        const double pa = A[0] * a.va[j][0] + A[1] * a.va[j][1];
        const double pb = A[0] * a.vb[j][0] + A[1] * a.vb[j][1];
        double sa, ca, sb, cb;
        sincos(pa, &sa, &ca);
        sincos(pb, &sb, &cb);
        row[2 * j] = a.t1 * ca;  // NN part carries t1
        row[2 * j + 1] = a.t1 * sa;
        row[6 + 2 * j] = cb;
        row[7 + 2 * j] = sb;
        if (tab32) {
            float *r32 = tab32 + i * 12;
            r32[2 * j] = static_cast<float>(a.t1 * ca);
            r32[2 * j + 1] = static_cast<float>(a.t1 * sa);
            r32[6 + 2 * j] = static_cast<float>(cb);
            r32[7 + 2 * j] = static_cast<float>(sb);
        }
    }
}

}  // namespace dev
}  // namespace sbe
