// tile_eig.hpp - the per-k operations of the N-band RK stage and sample on
// register tiles (tile16.hpp, tile_small.hpp): warm-started eigenvectors, the
// band-diagonal part of a matrix, the stage derivative. T is the tile type;
// buf is the wave's LDS transpose buffer (16x16 tiles; unused by small ones).
#pragma once

#include "nband.hpp"
#include "tile_small.hpp"

namespace sbe {
namespace tile {

// U <- U (3I - U^dag U) / 2 (Newton-Schulz: unitarity error e -> ~e^2); returns
// e = max |U^dag U - I| before the step (over the wave). Columns longer than 1.3
// are first scaled below 1: the step diverges from sqrt(3) on.
template <class T>
__device__ __forceinline__ double orthonormalize(T &U, T &Ut, int N, cd *buf)
{
    const int c = Shape<T>::col();
    const T G = cmm(U, true, U);
    double e = 0.0, g = 0.0;
#pragma unroll
    for (int r = 0; r < Shape<T>::E; ++r) {
        const bool dg = Shape<T>::row(r) == c;
        const double dr = G.re[r] - (dg ? 1.0 : 0.0);
        e = fmax(e, fmax(fabs(dr), fabs(G.im[r])));
        g = fmax(g, fabs(G.re[r]));
    }
    e = wave_max_dpp(e);
    double s1 = 1.5, s2 = -0.5;
    if (e > 0.7) {
        g = wave_max_dpp(g);
        if (g > 1.7) {
            s1 = 1.0 / sqrt(N * g);
            s2 = 0.0;
        }
    }
    T S;
#pragma unroll
    for (int r = 0; r < Shape<T>::E; ++r) {
        S.re[r] = (Shape<T>::row(r) == c ? s1 : 0.0) + s2 * G.re[r];
        S.im[r] = s2 * G.im[r];
    }
    U = cmm(Ut, false, S);
    Ut = transpose(U, buf);
    return e;
}

// 1 / (D/2 + s sqrt(D^2/4 + w2)), s = the sign of D, from the hardware estimates with one
// cubic step each (their errors cubed: rounding is what is left)
__device__ __forceinline__ double inv_angle(double D, double w2, double s)
{
    const double x = fma(0.25 * D, D, w2);
    const double q0 = __builtin_amdgcn_rsq(x);
    const double e = fma(-(x * q0), q0, 1.0);
    const double q = fma(q0 * e, fma(0.375, e, 0.5), q0);
    const double y = fma(s * x, q, 0.5 * D);
    const double v = __builtin_amdgcn_rcp(y);
    const double h = fma(-y, v, 1.0);
    return fma(v, fma(h, h, h), v);
}

constexpr double kRefineFar = 0.09, kRefineLast2 = 1e-12, kRefineLast1 = 1e-16;  // squares of 0.3, 1e-6, 1e-8

// K_ij = W_ij / (D/2 + s sqrt(D^2/4 + |W_ij|^2)), D = W_jj - W_ii: the 2x2 Jacobi angles
// of a nearly diagonal W; 0 on the diagonal and outside N x N, and with SIFT for registers r
// with bit r of off and where |W_ij|^2 > most D^2 (an angle above about sqrt(most)). Returns
// the larger of max |K|^2 and more, over the wave.
template <bool SIFT, class T>
__device__ __forceinline__ double angles(const T &W, T &K, int N, unsigned off, double most, double more, double &lam_c)
{
    constexpr int E = Shape<T>::E;
    const int c = Shape<T>::col();
    double lam_r[E], k2 = more;
    diag_bcast(W, lam_r, lam_c);
#pragma unroll
    for (int r = 0; r < E; ++r) {
        const int i = Shape<T>::row(r);
        const double w2 = W.re[r] * W.re[r] + W.im[r] * W.im[r];
        const double D = lam_c - lam_r[r];
        const double s = (D > 0.0 || (D == 0.0 && i < c)) ? 1.0 : -1.0;
        // (1e-280: below it the root's estimate would leave its range)
        bool on = i != c && i < N && c < N && w2 > 1e-280;
        if (SIFT) on = on && !(off >> r & 1) && !(w2 > most * D * D);
        const double inv = on ? inv_angle(D, on ? w2 : 1.0, s) : 0.0;
        K.re[r] = W.re[r] * inv;
        K.im[r] = W.im[r] * inv;
        k2 = fmax(k2, K.re[r] * K.re[r] + K.im[r] * K.im[r]);
    }
    k2 = wave_max_dpp(k2);
    // the same in every lane: a scalar, so that the branches on it are
    return __hiloint2double(__builtin_amdgcn_readfirstlane(__double2hiint(k2)),
                            __builtin_amdgcn_readfirstlane(__double2loint(k2)));
}

// (X + f X^dag) / 2, f = 1 or -1
template <class T>
__device__ __forceinline__ T half_sum(const T &X, double f, cd *buf)
{
    const T Xt = transpose(X, buf);
    T F;
#pragma unroll
    for (int r = 0; r < Shape<T>::E; ++r) {
        F.re[r] = 0.5 * (X.re[r] + f * Xt.re[r]);
        F.im[r] = 0.5 * (X.im[r] - f * Xt.im[r]);
    }
    return F;
}

// Warm-started eigenvectors of the Hermitian part of H (as zheevr, which
// reads one triangle; H from FP16-split sums is Hermitian only to their
// error): U (and its transpose Ut) in, refined U, Ut out.
//
// W = U^dag H U is nearly diagonal, W = L + E. One round takes the angles to second
// order: with K the angles of W, the angles X of the Hermitian part F of W + E K (what K
// leaves of W at second order), U <- U (I + X + X^2/2). F is Hermitian bit for bit, so X is
// exactly anti-Hermitian and the rotation unitary to X^4/8 however small a gap it divides by.
// What is left off the diagonal is of third order, times the ratio of the largest gap to the
// smallest: a round that starts at max|K| < 1e-6 is the last, one that starts below 1e-8 needs
// K's anti-Hermitian part alone. Three products a round against four of a first-order round, and
// no second round where a first-order scheme would need one. Later rounds take W from H again
// with G = U^dag U = I + e: W - e (W_ii + W_jj) / 2 is W in orthonormal columns to order e^2, and
// - e / 2 in the rotation makes the columns so (error ~e^2, so no round is the last while e is
// above 1e-8); ortho asks for that in the last round also when it is the first. Between RK
// stages of the 16-band workload (max|K| ~ 2e-2) 9 products against 14 of first-order rounds,
// of weak fields 5 against 9.
//
// Where bands meet, elements of W at its rounding (4 x 2^-52 max|W_ii|) have angles that are
// noise; from the third round on (others have ended) those above 1e-6 are left out: as rotations
// they would never end. 60 random 16-band matrices of eight exactly degenerate pairs in
// FP64: at most 26 rounds to a unitary U (6e-16) with nothing above 5e-16 off the diagonal; without
// that and the limit on e 30 rounds left U non-unitary by 0.2.
// Far starts (max|K| > 0.3 or columns off by 3e-3) take damped first-order rotations with
// Newton-Schulz steps until they are near. The columns keep the order of the warm start.
// herm: Hin is Hermitian to rounding already (FP64 sums), no symmetrization; lam_out:
// this lane's column of the diagonal before the last rotation (the band energies, for
// ranking: off by the squares of the last angles).
template <class T>
__device__ __forceinline__ void eig_refine(const T &Hin, T &U, T &Ut, int N, cd *buf, bool ortho = true, bool herm = false,
                                           double *lam_out = nullptr)
{
    constexpr int E = Shape<T>::E;
    const int c = Shape<T>::col();
    const T H = herm ? Hin : half_sum(Hin, 1.0, buf);
    T W = cmm(U, true, cmm(H, true, U));  // U^dag (H U)
    double lam_last = 0.0;
    T G;  // e = U^dag U - I, where formed
    bool have_e = false, done = false;
    unsigned off = 0;  // registers of elements left out
    double e2 = 0.0;  // 1e4 max |e|^2 of this lane: e below 1e-8 where below kRefineLast2
    auto form_e = [&]() {
        G = cmm(U, true, U);
#pragma unroll
        for (int r = 0; r < E; ++r) G.re[r] -= Shape<T>::row(r) == c ? 1.0 : 0.0;
        have_e = true;
    };
    for (int it = 0; it < 30 && !done; ++it) {
        T K, V;
        const double m2 = angles<false>(W, K, N, 0, 0.0, e2, lam_last);
        if (!(m2 > kRefineFar)) {  // (a NaN ends here, in the state it makes non-finite)
            done = !(m2 >= kRefineLast2);
            if (m2 >= kRefineLast1) {
                T F;  // W + E K, then its Hermitian part
                {
                    T Eo;
#pragma unroll
                    for (int r = 0; r < E; ++r) {
                        const bool dg = Shape<T>::row(r) == c;
                        Eo.re[r] = dg ? 0.0 : W.re[r];
                        Eo.im[r] = dg ? 0.0 : W.im[r];
                    }
                    F = cmm(Eo, true, K);
                }
#pragma unroll
                for (int r = 0; r < E; ++r) {
                    F.re[r] += W.re[r];
                    F.im[r] += W.im[r];
                }
                F = half_sum(F, 1.0, buf);
                // (in the last round an angle above 2e-6 is one of bands that nearly meet, coupled
                // at second order alone: left to the next refinement)
                (void)angles<true>(F, K, N, off, done ? 4.0 * kRefineLast2 : HUGE_VAL, 0.0, lam_last);
                T Kn;  // X^T's tile is -conj(X)
#pragma unroll
                for (int r = 0; r < E; ++r) {
                    Kn.re[r] = -K.re[r];
                    Kn.im[r] = -K.im[r];
                }
                const T K2 = cmm(Kn, true, K);
#pragma unroll
                for (int r = 0; r < E; ++r) {
                    V.re[r] = fma(0.5, K2.re[r], K.re[r]);
                    V.im[r] = fma(0.5, K2.im[r], K.im[r]);
                }
            } else {
                V = half_sum(K, -1.0, buf);
            }
            if (done && ortho && !have_e) form_e();
#pragma unroll
            for (int r = 0; r < E; ++r) {
                V.re[r] += Shape<T>::row(r) == c ? 1.0 : 0.0;
                if (have_e) {
                    V.re[r] = fma(-0.5, G.re[r], V.re[r]);
                    V.im[r] = fma(-0.5, G.im[r], V.im[r]);
                }
            }
            U = cmm(Ut, false, V);  // U V
            Ut = transpose(U, buf);
            if (done) break;
        } else {
            // far from converged (a cold-like start): rotations of norm 1 at most
            K = half_sum(K, -1.0, buf);
            double fr = 0.0;
#pragma unroll
            for (int r = 0; r < E; ++r) fr += K.re[r] * K.re[r] + K.im[r] * K.im[r];
            fr = wave_sum(fr);
            const double f = fr > 1.0 ? 1.0 / sqrt(fr) : 1.0;
            T Kn;
#pragma unroll
            for (int r = 0; r < E; ++r) {
                K.re[r] *= f;
                K.im[r] *= f;
                Kn.re[r] = -K.re[r];
                Kn.im[r] = -K.im[r];
            }
            const T K2 = cmm(Kn, true, K);
#pragma unroll
            for (int r = 0; r < E; ++r) {
                V.re[r] = K.re[r] + 0.5 * K2.re[r] + (Shape<T>::row(r) == c ? 1.0 : 0.0);
                V.im[r] = K.im[r] + 0.5 * K2.im[r];
            }
            U = cmm(Ut, false, V);
            Ut = transpose(U, buf);
            for (int q = 0; q < 16; ++q)
                if (orthonormalize(U, Ut, N, buf) < 1e-8) break;
        }
        W = cmm(U, true, cmm(H, true, U));
        form_e();
        double lr[E], lc;
        diag_bcast(W, lr, lc);
        e2 = 0.0;
#pragma unroll
        for (int r = 0; r < E; ++r) {
            const double h = -0.5 * (lr[r] + lc);
            W.re[r] = fma(h, G.re[r], W.re[r]);
            W.im[r] = fma(h, G.im[r], W.im[r]);
            e2 = fmax(e2, 1e4 * (G.re[r] * G.re[r] + G.im[r] * G.im[r]));
        }
        if (it >= 2) {
            W = half_sum(W, 1.0, buf);  // so that W_ij and W_ji go together
            const double fl = 0x1p-50 * wave_max_dpp(fabs(lc));
            off = 0;
#pragma unroll
            for (int r = 0; r < E; ++r) {
                const double w2 = W.re[r] * W.re[r] + W.im[r] * W.im[r], D = lc - lr[r];
                if (Shape<T>::row(r) != c && w2 <= fl * fl && w2 > kRefineLast2 * D * D) {
                    off |= 1u << r;
                    W.re[r] = W.im[r] = 0.0;
                }
            }
        }
    }
    if (!done)
        for (int q = 0; q < 16; ++q)
            if (orthonormalize(U, Ut, N, buf) < 1e-8) break;
    if (lam_out) *lam_out = lam_last;
}

// The band-diagonal part of y, U diag(U^dag y U) U^dag, and this lane's column
// of its diagonal d = (U^dag y U)_cc (two products)
template <class T>
__device__ __forceinline__ T band_diag(const T &Y, const T &U, const T &Ut, double &d)
{
    const T G = cmm(Y, true, U);  // y U
    d = col_dot(U, G);            // (U^dag y U)_cc
    double dr[Shape<T>::E];
    col_to_row(&U, d, dr);
    T Ud;  // (U diag(d))^T's tile: row i of U^T times d_i
#pragma unroll
    for (int r = 0; r < Shape<T>::E; ++r) {
        Ud.re[r] = Ut.re[r] * dr[r];
        Ud.im[r] = Ut.im[r] * dr[r];
    }
    return cmm(Ud, false, Ut, true);  // U diag(d) U^dag (B = U^dag: tile conj(U^T))
}

// The stage derivative at y given H~^T's tile (HERM: H~'s own tile, H~ Hermitian, so
// that H~^T's tile is its conjugate) and (dephasing on) y's band-diagonal part M:
// -i(H~ y - (H~ y)^dag) - g2 y - (g1 - g2) M.
template <bool HERM, class T>
__device__ __forceinline__ T stage_derivative_m(const NbArgs &a, const T &Y, const T &HtT, const T &M, cd *buf)
{
    const T P = cmm(HtT, HERM, Y);  // H~ y
    const T Pt = transpose(P, buf);
    T X;  // -i (P - P^dag)
#pragma unroll
    for (int r = 0; r < Shape<T>::E; ++r) {
        const double dr = P.re[r] - Pt.re[r], di = P.im[r] + Pt.im[r];
        X.re[r] = di;
        X.im[r] = -dr;
    }
    if (a.deph) {
        const double g2 = a.gam2, g12 = a.gam1 - a.gam2;
#pragma unroll
        for (int r = 0; r < Shape<T>::E; ++r) {
            X.re[r] -= g2 * Y.re[r] + g12 * M.re[r];
            X.im[r] -= g2 * Y.im[r] + g12 * M.im[r];
        }
    }
    return X;
}

// The same with U, U^T given (M formed here when dephasing)
template <class T>
__device__ __forceinline__ T stage_derivative(const NbArgs &a, const T &Y, const T &HtT, const T &U, const T &Ut, cd *buf)
{
    T M{};
    if (a.deph) {
        double d;
        M = band_diag(Y, U, Ut, d);
    }
    return stage_derivative_m<false>(a, Y, HtT, M, buf);
}

// Y = B + s X
template <class T>
__device__ __forceinline__ void axpy_tile(T &Y, const T &X, double s, const T &B)
{
#pragma unroll
    for (int r = 0; r < Shape<T>::E; ++r) {
        Y.re[r] = fma(s, X.re[r], B.re[r]);
        Y.im[r] = fma(s, X.im[r], B.im[r]);
    }
}

}  // namespace tile
}  // namespace sbe
