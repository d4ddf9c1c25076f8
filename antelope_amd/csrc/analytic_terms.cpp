// analytic_terms.cpp - the trigonometric sums of the analytic classes, read
// off by a discrete Fourier transform of the class's own H(k): every class
// but MultiWSM is a trigonometric polynomial on a lattice of bond components.
#include <algorithm>
#include <cmath>
#include <complex>

#include "analytic.hpp"
#include "analytic_terms.hpp"

namespace sbe {
namespace {

using cplx = std::complex<double>;
constexpr double kTwoPi = 6.28318530717958647692;

// products and sizes without std::complex's care for infinities and overflow (ten times the time,
// at every footprint query); a NaN stays one
cplx mul(const cplx &a, const cplx &b)
{
    return cplx(a.real() * b.real() - a.imag() * b.imag(), a.real() * b.imag() + a.imag() * b.real());
}
double size(const cplx &a) { return std::fabs(a.real()) + std::fabs(a.imag()); }

// Per class: the spacings u of its bond components (k.v_t = sum_i n_i u_i k_i
// with integers n_i, |n_i| <= reach), the sign of J against dH/dk, and which
// component of v each current slot differentiates (-1: the slot is zero).
struct Layout {
    double u[3] = {0, 0, 0};
    int reach = 4;
    double sign = -1.0, gscale = 1.0;
    int slot[3] = {0, 1, 2};
};

bool layout(int kind, const double *p, Layout &L)
{
    const double r3 = std::sqrt(3.0);
    auto set = [&](double x, double y) { L.u[0] = x, L.u[1] = y; };
    switch (kind) {
    case SBE_MODEL_WILSON_MASS: set(p[3], p[4]); return true;
    case SBE_MODEL_SQUARE_SBAND: set(p[2], p[2]); L.sign = -0.5; return true;  // only J(0,1): half of -dH/dk
    case SBE_MODEL_KANE_MELE: set(0.5 * r3 * p[5], 0.5 * p[5]); return true;
    case SBE_MODEL_XYH_LATTICE: set(0.5 * p[3], 0.5 * p[3] / r3); L.sign = 1.0; return true;
    case SBE_MODEL_TMDC: set(0.5 * p[0], 0.5 * r3 * p[0]); L.sign = 1.0; return true;
    case SBE_MODEL_HALDANE_2L: set(0.5 * r3 * p[8], 0.5 * p[8]); return true;
    case SBE_MODEL_BI2SE3_SURF: {
        double c[10];
        am::bi2se3_consts(c);
        set(0.5 * c[9], 0.5 * c[9] / r3);
        return true;
    }
    case SBE_MODEL_WDSM_TAAS:  // x and y slots: d/dkx and d/dkz without the factor a0 (WDSM_TaAs.h:170-185)
        L.u[0] = L.u[1] = L.u[2] = p[4];
        L.reach = 1;
        L.gscale = 1.0 / p[4];
        L.slot[1] = 2;
        L.slot[2] = -1;
        return true;
    default: return false;
    }
}

void eval(int kind, int N, const double *params, const double *k, std::vector<cplx> &H, std::vector<cplx> *J)
{
    const size_t nn = static_cast<size_t>(N) * N;
    std::vector<double2> h(nn, make_double2(0.0, 0.0)), j(3 * nn, make_double2(0.0, 0.0));
    am::analytic_eval(kind, N, params, k, h.data(), J ? j.data() : nullptr, J ? j.data() + nn : nullptr,
                      J ? j.data() + 2 * nn : nullptr);
    H.resize(nn);
    for (size_t e = 0; e < nn; ++e) H[e] = cplx(h[e].x, h[e].y);
    if (!J) return;
    J->resize(3 * nn);
    for (size_t e = 0; e < 3 * nn; ++e) (*J)[e] = cplx(j[e].x, j[e].y);
}

}  // namespace

bool analytic_terms(int kind, int N, const double *params, AnalyticTerms &out)
{
    Layout lay;
    out = AnalyticTerms{};
    if (!am::is_analytic(kind) || N < 1 || N > 8 || !layout(kind, params, lay)) return false;
    const int nn = N * N, L = 2 * lay.reach + 1;
    const int Ld[3] = {L, L, lay.u[2] != 0.0 ? L : 1};
    // samples on the L_x x L_y x L_z points of one period and their transform
    std::vector<std::vector<cplx>> smp;
    double hmax = 0.0;
    for (int x = 0; x < Ld[0]; ++x)
        for (int y = 0; y < Ld[1]; ++y)
            for (int z = 0; z < Ld[2]; ++z) {
                const double k[3] = {kTwoPi * x / Ld[0] / lay.u[0], kTwoPi * y / Ld[1] / lay.u[1],
                                     Ld[2] > 1 ? kTwoPi * z / Ld[2] / lay.u[2] : 0.0};
                std::vector<cplx> H;
                eval(kind, N, params, k, H, nullptr);
                for (const cplx &v : H) hmax = std::max(hmax, size(v));
                smp.push_back(std::move(H));
            }
    if (!std::isfinite(hmax)) return false;
    // e^{-2 pi i m / L} by index modulo L
    std::vector<cplx> root[3];
    for (int d = 0; d < 3; ++d)
        for (int m = 0; m < Ld[d]; ++m)
            root[d].push_back(std::polar(1.0, -kTwoPi * m / Ld[d]));
    // the transform of every element, one axis at a time (elements that are zero throughout stay so)
    const size_t stride[3] = {static_cast<size_t>(Ld[1]) * Ld[2], static_cast<size_t>(Ld[2]), 1};
    std::vector<std::vector<cplx>> tr(nn);
    for (int e = 0; e < nn; ++e) {
        std::vector<cplx> &f = tr[e];
        f.reserve(smp.size());
        bool any = false;
        for (const std::vector<cplx> &H : smp) {
            f.push_back(H[e]);
            any = any || H[e] != cplx(0.0);
        }
        for (int d = 0; d < 3 && any; ++d) {
            if (Ld[d] == 1) continue;
            cplx line[2][9];
            for (size_t q = 0; q < f.size(); ++q) {
                if ((q / stride[d]) % Ld[d] != 0) continue;  // the first point of each line
                for (int x = 0; x < Ld[d]; ++x) line[0][x] = f[q + x * stride[d]];
                for (int n = 0; n < Ld[d]; ++n) {
                    line[1][n] = 0.0;
                    for (int x = 0; x < Ld[d]; ++x) line[1][n] += mul(line[0][x], root[d][(n * x) % Ld[d]]);
                }
                for (int n = 0; n < Ld[d]; ++n) f[q + n * stride[d]] = line[1][n];
            }
        }
        for (cplx &v : f) v /= static_cast<double>(smp.size());
    }
    auto coef = [&](int nx, int ny, int nz, int e) {
        auto wrap = [&](int d, int n) { return static_cast<size_t>((n % Ld[d] + Ld[d]) % Ld[d]); };
        return tr[e][wrap(0, nx) * stride[0] + wrap(1, ny) * stride[1] + wrap(2, nz)];
    };
    auto clean = [&](cplx v) {  // rounding residue of the transform
        return cplx(std::fabs(v.real()) < 1e-15 * hmax ? 0.0 : v.real(), std::fabs(v.imag()) < 1e-15 * hmax ? 0.0 : v.imag());
    };
    auto hermitian = [&](const std::vector<cplx> &M, std::vector<double> &dst) {
        for (int i = 0; i < N; ++i)
            for (int j = 0; j < N; ++j) {
                const cplx v = 0.5 * (M[i * N + j] + std::conj(M[j * N + i]));
                dst.push_back(v.real());
                dst.push_back(v.imag());
            }
    };
    std::vector<cplx> M(nn), P(nn), Q(nn);
    for (int e = 0; e < nn; ++e) M[e] = clean(coef(0, 0, 0, e));
    hermitian(M, out.m0);
    const int rz = Ld[2] > 1 ? lay.reach : 0;
    for (int nx = 0; nx <= lay.reach; ++nx)
        for (int ny = -lay.reach; ny <= lay.reach; ++ny)
            for (int nz = -rz; nz <= rz; ++nz) {
                if (nx == 0 && (ny < 0 || (ny == 0 && nz <= 0))) continue;  // one of each +-v pair
                double big = 0.0;
                for (int e = 0; e < nn; ++e) {
                    const cplx a = coef(nx, ny, nz, e), b = coef(-nx, -ny, -nz, e);
                    P[e] = clean(a + b);
                    Q[e] = clean(cplx(b.imag() - a.imag(), a.real() - b.real()));  // i (a - b)
                    big = std::max({big, size(P[e]), size(Q[e])});
                }
                if (big < 1e-13 * hmax) continue;
                if (out.T == kMaxTerms) return false;
                const double v[3] = {nx * lay.u[0], ny * lay.u[1], nz * lay.u[2]};
                for (int c = 0; c < 3; ++c) {
                    out.vec[out.T][c] = v[c];
                    out.grad[out.T][c] = lay.slot[c] >= 0 ? v[lay.slot[c]] * lay.gscale : 0.0;
                }
                hermitian(P, out.p);
                hermitian(Q, out.q);
                ++out.T;
            }
    for (int e = 0; e < nn; ++e) {
        out.scale.push_back(lay.sign);
        out.scale.push_back(0.0);
    }
    if (kind == SBE_MODEL_KANE_MELE) {
        // Rashba elements (KaneMele.h:138-176): (0,3), (1,2), (2,1) are +dH/dk, (3,0) is too but
        // for its missing factor i tR, so the Hermitian part at (0,3) is (1 + i / tR) / 2 dH/dk
        const double x = 0.5 / params[2];
        const int e[4] = {3, 6, 9, 12};
        const cplx f[4] = {cplx(0.5, x), 1.0, 1.0, cplx(0.5, -x)};
        for (int i = 0; i < 4; ++i) {
            out.scale[2 * e[i]] = f[i].real();
            out.scale[2 * e[i] + 1] = f[i].imag();
        }
    }
    // the form against the class at points off the sampling grid
    for (int s = 1; s <= 6; ++s) {
        const double k[3] = {(0.37 * s - 1.1) / lay.u[0], (0.53 * s - 1.7) / lay.u[1],
                             lay.u[2] != 0.0 ? (0.29 * s - 0.6) / lay.u[2] : 0.0};
        std::vector<cplx> H, J;
        eval(kind, N, params, k, H, &J);
        double jmax = 0.0;
        for (const cplx &v : J) jmax = std::max(jmax, size(v));
        double cs[kMaxTerms], sn[kMaxTerms];
        for (int t = 0; t < out.T; ++t) {
            const double th = k[0] * out.vec[t][0] + k[1] * out.vec[t][1] + k[2] * out.vec[t][2];
            cs[t] = std::cos(th);
            sn[t] = std::sin(th);
        }
        for (int e = 0; e < nn; ++e) {
            const cplx scale(out.scale[2 * e], out.scale[2 * e + 1]);
            cplx h(out.m0[2 * e], out.m0[2 * e + 1]), g[3] = {0.0, 0.0, 0.0};
            for (int t = 0; t < out.T; ++t) {
                const size_t o = 2 * (static_cast<size_t>(t) * nn + e);
                const cplx p(out.p[o], out.p[o + 1]), q(out.q[o], out.q[o + 1]);
                h += p * cs[t] + q * sn[t];
                const cplx dh = mul(scale, q * cs[t] - p * sn[t]);
                for (int c = 0; c < 3; ++c) g[c] += out.grad[t][c] * dh;
            }
            if (!(size(h - H[e]) <= 1e-12 * hmax)) return false;
            const int tr = (e % N) * N + e / N;
            for (int c = 0; c < 3; ++c) {
                const cplx jh = 0.5 * (J[static_cast<size_t>(c) * nn + e] + std::conj(J[static_cast<size_t>(c) * nn + tr]));
                if (!(size(g[c] - jh) <= 1e-12 * std::max(jmax, hmax))) return false;
            }
        }
    }
    return true;
}

}  // namespace sbe
